/* Host stand-in for the part of the HIP runtime that the box's bookkeeping calls
 * (memory, streams, events; kernels do not run), for CPU tests of what a box
 * holds and of failing calls.  Loaded before libmcac_gpu.so with global symbols. */
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#define MAX_BLOCKS 4096
#define MAX_DEVICES 4
static struct { void *p; size_t n; } blocks[MAX_BLOCKS];
static size_t live_bytes;
static int device, fail_streams, streams, events[MAX_DEVICES];

size_t fake_device_bytes(void) { return live_bytes; }
void fake_fail_streams(int on) { fail_streams = on; }
int fake_streams(void) { return streams; }
int fake_events(int dev) { return events[dev]; }

int hipSetDevice(int d) { device = d; return 0; }
int hipDeviceGetAttribute(int *v, int what, int d) { (void)what, (void)d; *v = 100000; return 0; }
int hipDeviceSynchronize(void) { return 0; }
int hipGetLastError(void) { return 0; }
const char *hipGetErrorString(int e) { (void)e; return "fake"; }
int hipMemGetInfo(size_t *f, size_t *t) { *t = (size_t)1 << 38; *f = *t - live_bytes; return 0; }
int hipMalloc(void **p, size_t n) {
    for (int i = 0; i < MAX_BLOCKS; ++i)
        if (!blocks[i].p) {
            blocks[i].p = *p = malloc(n ? n : 1);
            blocks[i].n = n;
            live_bytes += n;
            return 0;
        }
    return 2;
}
int hipFree(void *p) {
    for (int i = 0; p && i < MAX_BLOCKS; ++i)
        if (blocks[i].p == p) {
            live_bytes -= blocks[i].n;
            blocks[i].p = NULL;
            free(p);
            return 0;
        }
    return p ? 1 : 0;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = malloc(n ? n : 1); return 0; }
int hipHostFree(void *p) { free(p); return 0; }
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void)flags; *d = h; return 0; }
int hipMemcpy(void *d, const void *s, size_t n, int kind) { (void)kind; memcpy(d, s, n); return 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *st) { (void)kind, (void)st; memcpy(d, s, n); return 0; }
int hipMemset(void *d, int v, size_t n) { memset(d, v, n); return 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *st) { (void)st; memset(d, v, n); return 0; }
int hipStreamCreateWithFlags(void **st, unsigned flags) {
    (void)flags;
    if (fail_streams) return 2;
    *st = malloc(1);
    ++streams;
    return 0;
}
int hipStreamDestroy(void *st) { free(st); --streams; return 0; }
int hipStreamQuery(void *st) { (void)st; return 0; }
int hipStreamSynchronize(void *st) { (void)st; return 0; }
int hipEventCreateWithFlags(void **e, unsigned flags) { (void)flags; *e = malloc(1); ++events[device]; return 0; }
int hipEventCreate(void **e) { return hipEventCreateWithFlags(e, 0); }
int hipEventDestroy(void *e) { free(e); return 0; }
int hipEventRecord(void *e, void *st) { (void)e, (void)st; return 0; }
int hipEventSynchronize(void *e) { (void)e; return 0; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a, (void)b; *ms = 0; return 0; }
typedef struct { uint32_t x, y, z; } dims;
int __hipPushCallConfiguration(dims g, dims b, size_t lds, void *st) { (void)g, (void)b, (void)lds, (void)st; return 0; }
int __hipPopCallConfiguration(dims *g, dims *b, size_t *lds, void **st) {
    memset(g, 0, sizeof *g);
    memset(b, 0, sizeof *b);
    *lds = 0;
    *st = NULL;
    return 0;
}
int hipLaunchKernel(const void *f, dims g, dims b, void **args, size_t lds, void *st) {
    (void)f, (void)g, (void)b, (void)args, (void)lds, (void)st;
    return 0;
}
