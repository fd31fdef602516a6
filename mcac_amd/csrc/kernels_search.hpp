// Contact search of one MC step (a4 + a6 + a7 + a8 + a9 + a13).
//
// k_filter   gathers the aggregates of the reference's visited Verlet cells
//            (CSR cells, skipping dirty entries, plus the whole dirty list),
//            runs the bounding-sphere sweep (sphere_contact.cpp:47-125 on
//            (CoM, rmax), aggregat_list.cpp:510-532) and appends the survivors
//            with their multimap key (bounding distance, visit rank, label).
// k_solve    splits the spheres of all survivors into tiles over the
//            participating blocks (lexicographic (d, i, j) minimum per
//            candidate, aggregat_distance.cpp:24-44); the last participating block
//            reduces per candidate, orders the candidates like the multimap,
//            runs the reference early-exit scan (aggregat_list.cpp:459-482),
//            moves the aggregate (aggregat.cpp:148-161) when it is small, and
//            publishes the result to pinned host memory.
// k_step     both in one launch for small movers with few survivors; k_steps and
//            k_steps_group do so for several consecutive steps of one box or of
//            many, searched side by side and carried out in order by the block
//            that finishes last.  k_step_grid: both in one launch for the others.
// k_translate moves the spheres of a large mover.
#pragma once
#include "grid_form.hpp"
#include "kernels_common.hpp"
#include "kernels_merge.hpp"

namespace mcac_dev {

// Where a search's survivors go: the box's candidate buffer (the grid forms).
struct BoxSink {
    const DevBox &b;
    int cap;
    __device__ __forceinline__ void operator()(int id, int rank, double d, int2, int) const {
        const unsigned int slot = atomicAdd(&b.ss->nfilt, 1u);
        if (slot < static_cast<unsigned int>(cap)) {
            b.cand_db[slot] = d;
            b.cand_rank[slot] = rank;
            b.cand_id[slot] = id;
        } else {
            atomicOr(&b.ss->overflow, 1u);
        }
    }
};

// The moves of a step's predecessors in the same launch, assumed without
// contact (a step behind a contact is not carried out): the newest one of each
// mover, in LDS.  The search takes these aggregates from here instead of from
// the box, where the moves are carried out at the launch's end.  n = 0 and
// self = -1 for a step that has no predecessor.
struct Moved {
    int n;                                   // entries (id -1: superseded by a later one)
    int self;                                // the step's own mover's entry, -1: it has not moved
    int id[kMaxSteps], cell[kMaxSteps];
    double x[kMaxSteps], y[kMaxSteps], z[kMaxSteps], r[kMaxSteps];  // centre of mass and rmax
    double rx[kMaxSteps], ry[kMaxSteps], rz[kMaxSteps];             // centre - relative centre: its spheres' origin
    int2 info[kMaxSteps];                                           // as DevBox::cinfo
};

// Positions of spheres as a step sees them: an aggregate with entry m >= 0 of
// the moved set has its spheres at that move's origin + relative position, the
// values its move stores (aggregat.cpp:148-161).
template <bool kMoved> struct Places {
    const DevBox &b;
    const Moved *mv;
    __device__ __forceinline__ void operator()(int m, int sp, double &x, double &y, double &z) const {
        if (kMoved && m >= 0) {
            x = mv->rx[m] + b.srx[sp];
            y = mv->ry[m] + b.sry[sp];
            z = mv->rz[m] + b.srz[sp];
        } else {
            x = b.sx[sp];
            y = b.sy[sp];
            z = b.sz[sp];
        }
    }
    // the mover's sphere of this thread
    template <class Sphere>
    __device__ __forceinline__ void of(int m, const Sphere &s, double &x, double &y, double &z) const {
        const bool moved = kMoved && m >= 0;
        x = moved ? mv->rx[m] + s.rx : s.x;
        y = moved ? mv->ry[m] + s.ry : s.y;
        z = moved ? mv->rz[m] + s.rz : s.z;
    }
};

// FP32 broad phase: can the candidate's bounding sphere (centre c, radius rc)
// come within the mover's radius rs of the sweep segment p1 + t dir, t in
// [0, dist]?  Every swept-sphere contact within dist passes (the contact point
// lies on the segment); with dist + rs + rc < L/2 only the minimum image can
// be that close, and `margin` (far above FP32 rounding of box-sized
// coordinates) keeps the test conservative.
__device__ __forceinline__ bool capsule_pass32(float p1x, float p1y, float p1z, float rs, float4 c, float dx_,
                                               float dy_, float dz_, float dist, float L, float margin) {
    const float half = 0.5f * L;
    float d[3] = {c.x - p1x, c.y - p1y, c.z - p1z};
#pragma unroll
    for (int l = 0; l < 3; ++l) {
        if (d[l] < -half) d[l] += L;
        else if (d[l] >= half) d[l] -= L;
    }
    float t = d[0] * dx_ + d[1] * dy_ + d[2] * dz_;
    t = t < 0.f ? 0.f : (t > dist ? dist : t);
    const float ex = d[0] - t * dx_, ey = d[1] - t * dy_, ez = d[2] - t * dz_;
    const float R = rs + c.w + margin;
    return ex * ex + ey * ey + ez * ez <= R * R;
}

// Per-thread counts of the filter: appended candidates << 32 | aggregates in the window.
constexpr unsigned long long kAppendOne = 1ull << 32;
constexpr unsigned long long kTicketOne = 1ull << 56;

// A gated step enqueued behind a step that found a contact (or handed its
// solve over) does nothing; the host releases a gate value by passing it as
// `released` to the steps it enqueues afterwards.
__device__ __forceinline__ bool behind_gate(const DevBox &b, const SearchArgs &a) {
    if (!a.gated) return false;
    const unsigned long long g = b.ss->gate;
    return g != 0ull && g < a.seq && g > a.released;
}

// Bounds of the visited cells, loaded by lane v of wave 0 for cell v of a
// host-supplied window of at most 64 cells (valid = 0: filter_phase loads them).
struct CellBounds {
    int valid, c0, sz;
};

__device__ __forceinline__ CellBounds load_cell_bounds(const DevBox &b, const SearchArgs &a, const CellTable *ct) {
    CellBounds cb{0, 0, 0};
    const int lj = a.len[1], lk = a.len[2];
    const int V = a.len[0] * lj * lk;
    if (!a.known || V > 64) return cb;
    if (ct && ct->n == V) {  // the host's table (in LDS): lane v takes cell v's pair
        cb.valid = 1;
        const int v = static_cast<int>(threadIdx.x);
        if (v < V) {
            cb.c0 = ct->c0[v];
            cb.sz = ct->sz[v];
        }
        return cb;
    }
    cb.valid = 1;
    const int v = static_cast<int>(threadIdx.x), n = a.n_div;
    if (v < V) {
        const int oi = v / (lj * lk), rem = v - oi * (lj * lk), oj = rem / lk, ok = rem - oj * lk;
        const int c = (window_offset(a.b1[0] + oi, 0, n) * n + window_offset(a.b1[1] + oj, 0, n)) * n +
                      window_offset(a.b1[2] + ok, 0, n);
        cb.c0 = b.cstart[c];
        cb.sz = b.cstart[c + 1] - cb.c0;
    }
    return cb;
}

// Largest c of the n entries with pre[c] <= w (pre ascending from 0).
template <class T> __device__ __forceinline__ int last_not_above(const T *pre, int n, T w) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (pre[mid] <= w) lo = mid;
        else hi = mid;
    }
    return lo;
}

// Bounds of the visited cells in LDS.
struct FilterLds {
    int win[6], nvisit;
    double q[4];
    int pre[kMaxVisit + 1], cbeg[kMaxVisit];
};

// Filter work of block vb of the vg blocks on this step: the aggregates of the
// reference's visited Verlet cells and the dirty list, bounding sweep,
// survivors to `append` (id, visit rank, bounding distance, cinfo, moved-set
// entry; shared by every form of the search).  With skip the
// work is read-only (a step behind a closed gate appends nothing).  nd: entries
// of the dirty list.  kMoved: the aggregates of the moved set are taken from
// there, by the first block.
template <bool kMoved, class Sink>
__device__ __forceinline__ unsigned long long filter_phase(const DevBox &b, const SearchArgs &a, unsigned vb,
                                                           unsigned vg, const CellBounds &cb, bool skip, FilterLds &u,
                                                           int nd, const Moved *mv, const Sink &append) {
    int *const pre = u.pre, *const cbeg = u.cbeg;
    const int n = a.n_div;
    int b1i, b1j, b1k, li, lj, lk, V;
    double sx, sy, sz, sr;
    if (a.known) {
        // window and mover data from the host mirror (verlet.cpp:57-78)
        b1i = a.b1[0];
        b1j = a.b1[1];
        b1k = a.b1[2];
        li = a.len[0];
        lj = a.len[1];
        lk = a.len[2];
        sx = a.sx;
        sy = a.sy;
        sz = a.sz;
        sr = a.srmax;
        V = li * lj * lk;
    } else {
        if (threadIdx.x == 0) {
            double src[3] = {b.ax[a.src], b.ay[a.src], b.az[a.src]};
            double vec[3] = {a.lpm * a.dir[0], a.lpm * a.dir[1], a.lpm * a.dir[2]};
            double mindist = b.armax[a.src] + a.maxradius;  // aggregat_list.cpp:492
            int b1[3], len[3];
            verlet_window(src, vec, mindist, n, a.L, b1, len);
            for (int l = 0; l < 3; ++l) {
                u.win[l] = b1[l];
                u.win[3 + l] = len[l];
                u.q[l] = src[l];
            }
            u.q[3] = b.armax[a.src];
            u.nvisit = len[0] * len[1] * len[2];
        }
        __syncthreads();
        b1i = u.win[0];
        b1j = u.win[1];
        b1k = u.win[2];
        li = u.win[3];
        lj = u.win[4];
        lk = u.win[5];
        sx = u.q[0];
        sy = u.q[1];
        sz = u.q[2];
        sr = u.q[3];
        V = u.nvisit;
    }
    const int gtid = static_cast<int>(vb * blockDim.x + threadIdx.x);
    const int gstride = static_cast<int>(vg * blockDim.x);
    unsigned long long cnt = 0;
    int total;  // entries of the visited cells (or of the whole list for a very wide window)
    if (V <= 64) {
        // one wave: lane v loads cell v's start and size and the prefix runs in
        // registers (wave shuffles); one barrier publishes it
        if (threadIdx.x < 64) {
            const int v = threadIdx.x;
            int sz = 0, c0 = 0;
            if (v < V && cb.valid) {
                c0 = cb.c0;
                sz = cb.sz;
            } else if (v < V) {
                int oi = v / (lj * lk), rem = v - oi * (lj * lk), oj = rem / lk, ok = rem - oj * lk;
                int ci = window_offset(b1i + oi, 0, n), cj = window_offset(b1j + oj, 0, n),
                    ck = window_offset(b1k + ok, 0, n);
                int c = (ci * n + cj) * n + ck;
                c0 = b.cstart[c];
                sz = b.cstart[c + 1] - c0;
            }
            const int incl = wave_inclusive_scan(sz);
            if (v < V) {
                cbeg[v] = c0;
                pre[v] = incl - sz;
            }
            if (v == 63) pre[V] = incl;
        }
        lds_barrier();
        total = pre[V];
    } else if (V <= kMaxVisit) {
        // sizes and starts of the visited cells in visit order, then their prefix
        for (int v = threadIdx.x; v < V; v += blockDim.x) {
            int oi = v / (lj * lk), rem = v - oi * (lj * lk), oj = rem / lk, ok = rem - oj * lk;
            int ci = window_offset(b1i + oi, 0, n), cj = window_offset(b1j + oj, 0, n),
                ck = window_offset(b1k + ok, 0, n);
            int c = (ci * n + cj) * n + ck;
            const int c0 = b.cstart[c];
            cbeg[v] = c0;
            pre[v] = b.cstart[c + 1] - c0;
        }
        lds_barrier();
        block_exclusive_scan(pre, V);
        total = pre[V];
    } else {
        total = b.cstart[n * n * n];  // every entry of the build
        lds_barrier();
    }
    // one index space: cell entries, then the aggregates moved since the build
    // (at their current cell), so that both kinds run side by side
    int gone[kMaxSteps];  // the mover and the moved set: not taken from the box
    int own = a.src;
    if (kMoved)
        for (int m = 0; m < kMaxSteps; ++m) gone[m] = m < mv->n ? mv->id[m] : -1;
    auto elsewhere = [&](int id) {
        bool e = id == own;
        if (kMoved) {
#pragma unroll
            for (int m = 0; m < kMaxSteps; ++m) e = e || id == gone[m];
        }
        return e;
    };
    unsigned long long n32 = 0, kept32 = 0, miss32 = 0;
    const float fx = static_cast<float>(sx), fy = static_cast<float>(sy), fz = static_cast<float>(sz);
    const float fr = static_cast<float>(sr), fdx = static_cast<float>(a.dir[0]), fdy = static_cast<float>(a.dir[1]);
    const float fdz = static_cast<float>(a.dir[2]), flpm = static_cast<float>(a.lpm), fL = static_cast<float>(a.L);
    // the bounding sweep of one aggregate: the exact one only where the sound
    // pre-test cannot rule a contact out
    const SweepTest sw = sweep_test(a.dir, a.lpm, a.L);
    auto bounding = [&](double x, double y, double z, double r) {
        if (sw.usable && sr + r <= sw.limit &&
            !sweep_may_touch(sw, nearest_image(x - sx, sw.hx, sw), nearest_image(y - sy, sw.hy, sw),
                             nearest_image(z - sz, sw.hz, sw), sr + r))
            return kInf;
        return swept_sphere(sx, sy, sz, sr, x, y, z, r, a.dir[0], a.dir[1], a.dir[2], a.lpm, a.L);
    };
    if (kMoved && vb == 0u && static_cast<int>(threadIdx.x) < mv->n && mv->id[threadIdx.x] >= 0 &&
        mv->id[threadIdx.x] != own) {
        const int m = threadIdx.x, c = mv->cell[m];
        const int oi = window_offset(c / (n * n), b1i, n), oj = window_offset((c / n) % n, b1j, n),
                  ok = window_offset(c % n, b1k, n);
        if (oi < li && oj < lj && ok < lk) {
            cnt += 1;
            const double d = bounding(mv->x[m], mv->y[m], mv->z[m], mv->r[m]);
            if (d < a.lpm && !skip) {
                append(mv->id[m], (oi * lj + oj) * lk + ok, d, mv->info[m], m);
                cnt += kAppendOne;
            }
        }
    }
    if (a.prec == 0 && V <= kMaxVisit && total > gstride) {
        // FP64 sweep with several entries per thread (a block that takes a
        // window alone): kSweep entries per pass have their rank searches and
        // row loads in flight together instead of one load latency per entry
        constexpr int kSweep = 4;
        int top = 1;
        while (2 * top < V) top *= 2;
        for (int w0 = gtid; w0 < total; w0 += kSweep * gstride) {
            int rk[kSweep] = {}, idv[kSweep];
            double xv[kSweep], yv[kSweep], zv[kSweep], rv[kSweep];
            int pv[kSweep];
            for (int s = top; s > 0; s >>= 1) {  // largest v with pre[v] <= w, as above
#pragma unroll
                for (int u = 0; u < kSweep; ++u) {
                    const int m = rk[u] + s;
                    if (m < V && pre[m] <= w0 + u * gstride) rk[u] = m;
                }
            }
#pragma unroll
            for (int u = 0; u < kSweep; ++u) {
                const int w = w0 + u * gstride;
                idv[u] = a.src;
                xv[u] = yv[u] = zv[u] = 0.0;
                rv[u] = -1.0;
                pv[u] = 0;
                if (w < total) {
                    const int pos = cbeg[rk[u]] + (w - pre[rk[u]]);
                    pv[u] = pos;
                    idv[u] = b.citems[pos];
                    xv[u] = b.cpx[pos];
                    yv[u] = b.cpy[pos];
                    zv[u] = b.cpz[pos];
                    rv[u] = b.cpr[pos];
                }
            }
#pragma unroll
            for (int u = 0; u < kSweep; ++u) {
                if (rv[u] < 0.0 || elsewhere(idv[u])) continue;  // past the end, moved since the build, or the mover
                cnt += 1;
                const double d = bounding(xv[u], yv[u], zv[u], rv[u]);
                if (d < a.lpm && !skip) {
                    append(idv[u], rk[u], d, b.cinfo[pv[u]], -1);
                    cnt += kAppendOne;
                }
            }
        }
        for (int i = gtid; i < nd; i += gstride) {  // the dirty list, as below
            const int id = b.dirty_list[i];
            const int c = b.dpcell[i];
            if (c < 0 || elsewhere(id)) continue;
            int oi = window_offset(c / (n * n), b1i, n), oj = window_offset((c / n) % n, b1j, n),
                ok = window_offset(c % n, b1k, n);
            if (oi >= li || oj >= lj || ok >= lk) continue;
            cnt += 1;
            const double d = bounding(b.dpx[i], b.dpy[i], b.dpz[i], b.dpr[i]);
            if (d < a.lpm && !skip) {
                append(id, (oi * lj + oj) * lk + ok, d, b.dinfo[i], -1);
                cnt += kAppendOne;
            }
        }
        return cnt;
    }
    for (int w = gtid; w < total + nd; w += gstride) {
        int id, rank;
        double x, y, z, r;
        int2 info;
        if (w < total) {
            int pos;
            if (V <= kMaxVisit) {
                int lo = 0, hi = V;  // largest v with pre[v] <= w
                while (hi - lo > 1) {
                    int mid = (lo + hi) >> 1;
                    if (pre[mid] <= w) lo = mid;
                    else hi = mid;
                }
                rank = lo;
                pos = cbeg[lo] + (w - pre[lo]);
            } else {
                pos = w;
            }
            if (a.prec > 0) {
                // FP32 broad phase: 16 B per entry; only its survivors read the FP64 row
                const float4 f = b.cf[pos];
                if (f.w < 0.f || (kMoved && elsewhere(b.citems[pos]))) continue;  // moved since the build
                const bool pass = capsule_pass32(fx, fy, fz, fr, f, fdx, fdy, fdz, flpm, fL, a.margin32);
                n32 += 1;
                if (!pass) {
                    if (a.prec == 2) {  // would the FP64 filter have kept it?
                        const int id2 = b.citems[pos];
                        const double d2 = swept_sphere(sx, sy, sz, sr, b.cpx[pos], b.cpy[pos], b.cpz[pos],
                                                       b.cpr[pos], a.dir[0], a.dir[1], a.dir[2], a.lpm, a.L);
                        if (!elsewhere(id2) && d2 < a.lpm) miss32 += 1;
                    }
                    continue;
                }
                kept32 += 1;
            }
            id = b.citems[pos];
            x = b.cpx[pos];
            y = b.cpy[pos];
            z = b.cpz[pos];
            r = b.cpr[pos];
            info = b.cinfo[pos];
            if (r < 0.0 || elsewhere(id)) continue;  // moved since the build, or the mover
            if (V > kMaxVisit) {
                const int c = ref_cell(x, y, z, n, a.L);
                int oi = window_offset(c / (n * n), b1i, n), oj = window_offset((c / n) % n, b1j, n),
                    ok = window_offset(c % n, b1k, n);
                if (oi >= li || oj >= lj || ok >= lk) continue;
                rank = (oi * lj + oj) * lk + ok;
            }
        } else {
            const int i = w - total;
            id = b.dirty_list[i];
            const int c = b.dpcell[i];
            x = b.dpx[i];
            y = b.dpy[i];
            z = b.dpz[i];
            r = b.dpr[i];
            info = b.dinfo[i];
            if (c < 0 || elsewhere(id)) continue;
            int oi = window_offset(c / (n * n), b1i, n), oj = window_offset((c / n) % n, b1j, n),
                ok = window_offset(c % n, b1k, n);
            if (oi >= li || oj >= lj || ok >= lk) continue;
            rank = (oi * lj + oj) * lk + ok;
        }
        cnt += 1;
        const double d = bounding(x, y, z, r);
        if (d < a.lpm && !skip) {
            append(id, rank, d, info, -1);
            cnt += kAppendOne;
        }
    }
    if (a.prec == 2) {  // FP32 broad-phase accounting, one atomic per block and counter
        n32 = block_sum(n32);
        kept32 = block_sum(kept32);
        miss32 = block_sum(miss32);
        if (threadIdx.x == 0) {
            atomicAdd(&b.ss->fp32_tested, n32);
            atomicAdd(&b.ss->fp32_kept, kept32);
            if (miss32) atomicAdd(&b.ss->fp32_missed, miss32);
        }
    }
    return cnt;
}

__global__ __launch_bounds__(kBlock) void k_filter(DevBox b, SearchArgs a) {
    if (behind_gate(b, a)) return;
    __shared__ FilterLds u;
    const unsigned long long tot =
        block_sum(filter_phase<false>(b, a, blockIdx.x, gridDim.x, CellBounds{0, 0, 0}, false, u, a.dirty_n, nullptr,
                                      BoxSink{b, a.cap})) & 0xffffffffull;
    if (threadIdx.x == 0 && tot) atomicAdd(&b.ss->nquery, tot);
}

// A finished search: the contact and the search's counts (aggregat_list.cpp:459-482).
struct StepPick {
    double dist;                // distance of the contact, +inf: none
    long long ms, os, oagg;     // its spheres and other aggregate, -1: none
    long long tpairs;           // sphere pairs of the survivors
    unsigned long long nquery;  // aggregates of the visited cells tested
    unsigned int nfilt;         // candidates appended (may exceed the capacity)
    int overflow;
    int src_slot;               // packed cell entry of the mover (-1: none)
    int handover;               // survivors left to the grid form: no contact known
    int on, pad;                // size of the other aggregate
};

// Survivors of a one-launch step (at most kStepCands), kept in LDS by the
// finishing block: bounding distance, visit rank, label, size and member
// segment (or ~ its only sphere), moved-set entry, exact minimum, and the
// multimap order.
struct StepCands {
    double db[kStepCands], ex[kStepCands];
    int ms[kStepCands], os[kStepCands];  // spheres of the minimum
    int rank[kStepCands], id[kStepCands], nk[kStepCands], sk[kStepCands], mv[kStepCands], order[kStepCands];
    double mx[kThreadPairs], my[kThreadPairs], mz[kThreadPairs], mr[kThreadPairs];  // a small mover's spheres
    int msp[kThreadPairs];
    int pre[kStepCands + 1];  // spheres before each survivor's
    unsigned int n;           // survivors of a search by one block (may exceed kStepCands)
};

// Sphere of the mover a thread places when it applies a step, loaded early
// when the mover has at most one sphere per thread.
struct MoverSphere {
    int loaded;  // the block loaded the mover (uniform)
    int sp;      // this thread's sphere, -1: none
    double rx, ry, rz;     // relative position
    double x, y, z, r;     // position in the box, radius
};

__device__ __forceinline__ MoverSphere load_mover_sphere(const DevBox &b, const SearchArgs &a) {
    MoverSphere m{a.n_mov <= kBlock, -1, 0., 0., 0., 0., 0., 0., 0.};
    if (m.loaded && static_cast<int>(threadIdx.x) < a.n_mov) {
        m.sp = b.members[a.start + threadIdx.x];
        m.rx = b.srx[m.sp];
        m.ry = b.sry[m.sp];
        m.rz = b.srz[m.sp];
    }
    return m;
}

// What a step loads first that no other step changes while it is queued
// behind them without a contact: the mover's packed-entry slot (thread 0) and
// its spheres with their relative positions.  The persistent engine loads it
// while the previous step finishes.
struct StepPrefetch {
    int src_slot;
    MoverSphere mover;
};

__device__ __forceinline__ StepPrefetch prefetch_step(const DevBox &b, const SearchArgs &a) {
    StepPrefetch p;
    p.src_slot = (threadIdx.x == 0) ? b.cslot[a.src] : -1;
    p.mover = load_mover_sphere(b, a);
    return p;
}

// Pair solve of a step's survivors (aggregat_distance.cpp:24-44): per candidate
// the lexicographic (d, i, j) minimum of the swept-sphere distances between the
// mover's spheres i and the candidate's spheres j.  The candidates' spheres form
// one index space (sphere w of all candidates, cpre[c] the first of candidate c)
// worked on in tiles of kBlock spheres, so that a tile's loads are in flight
// together whatever the candidates' sizes.  Most pairs cannot touch on the way:
// a sphere of the tile is kept only if the sweep of the mover's bounding ball
// (taken from its spheres here, not from its stored rmax) may reach it, and of
// the pairs of kept spheres with the mover's only those whose own sweep may
// touch (sweep_may_touch, sound, so every finite distance is still computed)
// take the exact swept sphere with its divisions and square root, and of those
// only the ones whose earliest contact is not above the candidate's minimum so
// far.  The solve is bound by the FP64 of the pairs: with every pair exact a
// search of a 700-sphere mover among 125 such aggregates took 756 us, this way
// 109 us; searches of 100-sphere movers 21 us, this way 11 us.
constexpr int kMoverTile = 512;  // mover spheres in LDS at a time
struct SolveLds {
    double mx[kMoverTile], my[kMoverTile], mz[kMoverTile], mr[kMoverTile];
    // kept spheres of the tile: nearest image to the mover, stored position, radius
    double qx[kBlock], qy[kBlock], qz[kBlock], px[kBlock], py[kBlock], pz[kBlock], pr[kBlock];
    int cand[kBlock], idx[kBlock];                // their candidate (from the tile's first) and sphere number in it
    int sp[kBlock], msp[kMoverTile];              // sphere indices
    int bms[kBlock], bos[kBlock];                 // per candidate of the tile: spheres of pmin
    unsigned long long dmin[kBlock];              // per candidate of the tile: least distance (ordered bits)
    unsigned long long pmin[kBlock];              // and least pair index at it
    double rd[kBlock];                            // minimum of each kept sphere over the mover's
    long long rp[kBlock];
    double wmax[kBlock / 64];
    int wcnt[kBlock / 64];
    int found;
};

// A block filters, then solves, then merges: the three use the same LDS.
union StepLds {
    FilterLds filter;
    SolveLds solve;
    MergeLds merge;
};

// Orders the F candidates like the reference's std::multimap (bounding
// distance, visit rank, label) and runs its early-exit scan over the exact
// distances (from LDS when lc is given, else cand_exact / cand_pair): the
// contact, in pick, by thread 0.
__device__ __forceinline__ void scan_candidates(const DevBox &b, unsigned int F, int ssrc, const StepCands *lc,
                                                int *order, StepPick &pick) {
    if (lc) {
        for (unsigned int c = threadIdx.x; c < F; c += blockDim.x) {
            const double dc = lc->db[c];
            const int rc = lc->rank[c], ic = lc->id[c];
            unsigned int pos = 0;
            for (unsigned int e = 0; e < F; ++e) {
                const double de = lc->db[e];
                const int re = lc->rank[e];
                pos += (de < dc || (de == dc && (re < rc || (re == rc && lc->id[e] < ic)))) ? 1u : 0u;
            }
            order[pos] = static_cast<int>(c);
        }
        if (F > 0) lds_barrier();
    } else {
        for (unsigned int c = threadIdx.x; c < F; c += blockDim.x) {
            const double dc = b.cand_db[c];
            const int rc = b.cand_rank[c], ic = b.cand_id[c];
            unsigned int pos = 0;
            for (unsigned int e = 0; e < F; ++e) {
                double de = b.cand_db[e];
                int re = b.cand_rank[e];
                pos += (de < dc || (de == dc && (re < rc || (re == rc && b.cand_id[e] < ic)))) ? 1u : 0u;
            }
            order[pos] = static_cast<int>(c);
        }
        if (F > 0) __syncthreads();  // order and exact distances come from other threads
    }
    if (threadIdx.x == 0) {
        double closest = kInf;
        int best = -1;
        for (unsigned int pos = 0; pos < F; ++pos) {
            const int c = order[pos];
            if (closest <= 0.) break;
            if (closest < (lc ? lc->db[c] : b.cand_db[c])) break;
            const double ex = lc ? lc->ex[c] : b.cand_exact[c];
            if (ex < closest) {
                closest = ex;
                best = c;
            }
        }
        pick.dist = closest;
        pick.ms = pick.os = pick.oagg = -1;
        pick.on = 0;
        if (best >= 0) {
            if (lc) {
                pick.ms = lc->ms[best];
                pick.os = lc->os[best];
                pick.oagg = lc->id[best];
                pick.on = lc->nk[best];
            } else {
                const long long p = b.cand_pair[best];
                const int k = b.cand_id[best];
                const long long nk = b.acount[k];
                const int sk = b.astart[k];
                const long long i = p / nk, j = p - i * nk;
                pick.ms = b.members[ssrc + i];
                pick.os = b.members[sk + j];
                pick.oagg = k;
                pick.on = static_cast<int>(nk);
            }
        }
    }
}

// Carries out a finished search in the box: moves the aggregate, merges on a
// contact when asked to, writes the record (publishing it unless the caller
// publishes later) and resets the search counters.  pick is read by thread 0
// only.  Returns (in thread 0) whether the step closed the gate for the steps
// queued behind it.
template <bool kCaps>
__device__ __forceinline__ bool apply_step(const DevBox &b, const SearchArgs &a, const StepPick &pick,
                                           const MoverSphere &m, bool publish, MergeLds &u) {
    constexpr int kAutomerge = kCaps ? 2 : 1;  // the merges this kernel carries
    bool closed = false;
    const long long nsrc = a.n_mov;
    const int ssrc = a.start;
    __shared__ double s_ref[3];
    __shared__ StepRecord srec;  // assembled here, copied to host memory by one wave
    SearchState *s = b.ss;
    int other_n = 0, other_start = 0, keep_cap = 0;  // of a contact's merge (thread 0)
    if (threadIdx.x == 0) {
        // every load of this thread comes before its stores (no reloads through global memory)
        const double closest = pick.dist;
        if (pick.oagg >= 0 && closest <= a.lpm && a.automerge == kAutomerge) {
            const int o = static_cast<int>(pick.oagg);
            other_n = pick.on;
            other_start = b.astart[o];
            keep_cap = b.acap[a.src < o ? a.src : o];
        }
        // calcul.cpp:128-130 and aggregat.cpp:148-153
        const int contact = closest <= a.lpm;
        const double move = contact ? closest : a.lpm;
        double old[3], rc3[3], rmax_src;
        if (a.known) {
            old[0] = a.sx, old[1] = a.sy, old[2] = a.sz;
            rc3[0] = a.srx, rc3[1] = a.sry, rc3[2] = a.srz;
            rmax_src = a.srmax;
        } else {
            old[0] = b.ax[a.src], old[1] = b.ay[a.src], old[2] = b.az[a.src];
            rc3[0] = b.arx[a.src], rc3[1] = b.ary[a.src], rc3[2] = b.arz[a.src];
            rmax_src = b.armax[a.src];
        }
        double ncom[3], nref[3];
        int ncell;
        if (!contact && a.nc_ok) {  // the full move, computed by the host with the same operations
            for (int l = 0; l < 3; ++l) {
                ncom[l] = a.nc_com[l];
                nref[l] = a.nc_ref[l];
                s_ref[l] = nref[l];
            }
            ncell = a.nc_cell;
        } else {
            for (int l = 0; l < 3; ++l) {
                ncom[l] = periodic_position(old[l] + a.dir[l] * move, a.L);
                nref[l] = ncom[l] - rc3[l];
                s_ref[l] = nref[l];
            }
            ncell = ref_cell(ncom[0], ncom[1], ncom[2], a.n_div, a.L);
        }
        StepRecord *o = &srec;
        o->dist = closest;
        o->move = move;
        o->ms = pick.ms;
        o->os = pick.os;
        o->oagg = pick.oagg;
        o->contact = contact;
        o->status = pick.overflow ? MCAC_E_CAPACITY : 0;
        o->nquery = pick.nquery;
        o->nfilt = pick.nfilt;
        o->npairs = static_cast<unsigned long long>(pick.tpairs);
        o->skipped = 0;
        o->merged_inline = 0;
        o->m_new_start = 0;
        o->m_new_cap = 0;
        o->dirty_count = a.dirty_n + ((a.apply && a.dirty_slot >= 0) ? 1 : 0);
        for (int l = 0; l < 3; ++l) {
            s->newcom[l] = ncom[l];
            s->refpos[l] = nref[l];
        }
        s->newcell = ncell;
        if (a.apply) {
            b.ax[a.src] = ncom[0];
            b.ay[a.src] = ncom[1];
            b.az[a.src] = ncom[2];
            b.acell[a.src] = ncell;
            if (a.dirty_slot >= 0) {  // first move since the cell-list build
                b.dirty[a.src] = 1;
                b.dirty_list[a.dirty_slot] = a.src;
                b.dslot[a.src] = a.dirty_slot;
                s->dirty_count = static_cast<unsigned int>(a.dirty_slot + 1);
                if (pick.src_slot >= 0) {
                    b.cpr[pick.src_slot] = -1.0;
                    b.cf[pick.src_slot].w = -1.f;
                }
            }
            set_dirty_entry(b, a.dirty_pos, ncom[0], ncom[1], ncom[2], rmax_src, ncell);
            b.dinfo[a.dirty_pos] = make_int2(a.n_mov, a.n_mov == 1 && m.loaded ? ~m.sp : a.start);
        }
        if (a.gated && contact) s->gate = a.seq;  // the steps behind wait for the merge
        closed = a.gated && contact;
        s->nfilt = 0;
        s->nquery = 0;
        s->overflow = 0;
        s->done_solve = 0;
        s->grid_bar = 0;
    }
    lds_barrier();  // s_ref
    if (a.apply && a.translate_in_finish && m.loaded) {
        if (m.sp >= 0) {
            b.sx[m.sp] = s_ref[0] + m.rx;
            b.sy[m.sp] = s_ref[1] + m.ry;
            b.sz[m.sp] = s_ref[2] + m.rz;
        }
    } else if (a.apply && a.translate_in_finish) {
        const double r0 = s_ref[0], r1 = s_ref[1], r2 = s_ref[2];
        for (int t = threadIdx.x; t < nsrc; t += blockDim.x) {
            int sp = b.members[ssrc + t];
            b.sx[sp] = r0 + b.srx[sp];
            b.sy[sp] = r1 + b.sry[sp];
            b.sz[sp] = r2 + b.srz[sp];
        }
    }
    // merge in the same launch (AggregatList::merge, aggregat_list.cpp:367-410)
    // when the merged aggregate is small and its member segment fits
    if (a.automerge == kAutomerge && a.apply && a.translate_in_finish) {
        __shared__ MergeArgs s_ma;
        __shared__ int s_inline;
        if (threadIdx.x == 0) {
            s_inline = 0;
            if (srec.contact) {
                const int oagg = static_cast<int>(srec.oagg);
                const int keep = a.src < oagg ? a.src : oagg, rem = a.src < oagg ? oagg : a.src;
                const int nk = (keep == a.src) ? a.n_mov : other_n;
                const int nr = (rem == a.src) ? a.n_mov : other_n;
                const int start_k = (keep == a.src) ? a.start : other_start;
                const int start_r = (rem == a.src) ? a.start : other_start;
                const int n = nk + nr;
                int new_start = start_k, new_cap = keep_cap;
                bool fits = n <= kSmallMerge;
                if (fits && n > new_cap) {  // a fresh segment of twice the merged size
                    new_cap = (2 * n > 4) ? 2 * n : 4;
                    fits = a.pool_used + new_cap <= a.pool_cap;
                    new_start = static_cast<int>(a.pool_used);
                }
                if (fits) {
                    MergeArgs m{};
                    m.ms = srec.ms;
                    m.os = srec.os;
                    m.magg = a.src;
                    m.oagg = oagg;
                    m.keep = keep;
                    m.rem = rem;
                    m.n_k = nk;
                    m.n_r = nr;
                    m.new_start = new_start;
                    m.start_k = start_k;
                    m.start_r = start_r;
                    m.n_div = a.n_div;
                    m.cap_k = new_cap;
                    m.volsurf = kCaps ? 1 : 0;
                    m.L = a.L;
                    s_ma = m;
                    s_inline = 1;
                    srec.m_new_start = new_start;
                    srec.m_new_cap = new_cap;
                }
            }
        }
        lds_barrier();
        if (s_inline) {
            // the merge takes the mover's sphere positions from s_ref: its
            // loads do not wait for the placements above
            merge_small_block<kCaps>(b, s_ma, srec.merge, s_ref, u);
            if (threadIdx.x == 0) srec.merged_inline = 1;  // thread 0 also copies the record
        }
    }
    // the record body in one coalesced write, then the sequence number
    constexpr int kWords = static_cast<int>(offsetof(StepRecord, seq) / sizeof(unsigned long long));
    static_assert(offsetof(StepRecord, seq) % sizeof(unsigned long long) == 0, "record body in 8-byte words");
    if (threadIdx.x < 64) {
        if (static_cast<int>(threadIdx.x) < kWords)
            reinterpret_cast<unsigned long long *>(a.out)[threadIdx.x] =
                reinterpret_cast<const unsigned long long *>(&srec)[threadIdx.x];
        if (threadIdx.x == 0 && publish) {
            __threadfence_system();
            __hip_atomic_store(&a.out->seq, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
        }
    }
    return closed;
}

// Bits of a double whose unsigned order is the doubles' order.
__device__ __forceinline__ unsigned long long ordered_bits(double d) {
    const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(d));
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ __forceinline__ double from_ordered_bits(unsigned long long u) {
    return __longlong_as_double(static_cast<long long>((u >> 63) ? (u & 0x7fffffffffffffffull) : ~u));
}

// The mover's spheres [i0, i0 + nt) into LDS; returns the radius around centre
// that holds them (block-uniform).
template <class Where>
__device__ __forceinline__ double load_mover_tile(const DevBox &b, SolveLds &u, int ssrc, long long i0, int nt,
                                                  const double centre[3], int self, const Where &where,
                                                  const MoverSphere *own = nullptr) {
    double far = 0.0;
    for (int t = threadIdx.x; t < nt; t += blockDim.x) {
        double x, y, z, r;
        int sp;
        if (own) {  // the thread's sphere, loaded with the step's first loads
            sp = own->sp;
            r = own->r;
            where.of(self, *own, x, y, z);
        } else {
            sp = b.members[ssrc + i0 + t];
            r = b.sr[sp];
            where(self, sp, x, y, z);
        }
        u.mx[t] = x;
        u.my[t] = y;
        u.mz[t] = z;
        u.mr[t] = r;
        u.msp[t] = sp;
        const double d0 = x - centre[0], d1 = y - centre[1], d2 = z - centre[2];
        const double f = __builtin_sqrt(d0 * d0 + d1 * d1 + d2 * d2) + r;
        far = !(f <= far) ? f : far;  // a NaN stays: nothing is pruned then
    }
    for (int off = 32; off > 0; off >>= 1) {
        const double o = __shfl_xor(far, off, 64);
        far = !(o <= far) ? o : far;
    }
    if ((threadIdx.x & 63) == 0) u.wmax[threadIdx.x >> 6] = far;
    lds_barrier();
    far = u.wmax[0];
    for (int w = 1; w < kBlock / 64; ++w) far = !(u.wmax[w] <= far) ? u.wmax[w] : far;
    return far;
}

// One tile: thread t holds sphere number j of candidate cl (counted from the
// tile's first; cl < 0: no sphere), listed at member slot m (`member` itself
// where that is known, else -1), of an aggregate
// with moved-set entry `entry`, against the nt mover spheres in LDS (numbers i0 ...).  Returns whether some pair of the tile
// has a finite distance: then u.dmin / u.pmin hold the minima of its ncl (at
// most kBlock) candidates, candidate cl's for thread cl, where they are at most
// `best` (thread cl's: the candidate's minimum over earlier tiles; u.pmin stays
// ~0 where no pair of the tile is).  nk(cl): its size.
template <class Where, class Size>
__device__ __forceinline__ bool solve_tile(const DevBox &b, const SearchArgs &a, const SweepTest &sw, SolveLds &u,
                                           const double centre[3], double reach, long long i0, int nt, int cl,
                                           long long j, long long m, int member, int entry, const Where &where, int ncl,
                                           double best,
                                           Size &&nk) {
    double x = 0, y = 0, z = 0, r = 0, q0 = 0, q1 = 0, q2 = 0;
    bool keep = false;
    int sp = -1;
    if (cl >= 0) {
        sp = member >= 0 ? member : b.members[m];
        r = b.sr[sp];
        where(entry, sp, x, y, z);
        const double d0 = nearest_image(x - centre[0], sw.hx, sw), d1 = nearest_image(y - centre[1], sw.hy, sw),
                     d2 = nearest_image(z - centre[2], sw.hz, sw);
        q0 = centre[0] + d0;
        q1 = centre[1] + d1;
        q2 = centre[2] + d2;
        // where the image nearest to the centre need not be the nearest to every
        // mover sphere it is kept, and marked by a NaN
        const bool near = sw.usable && reach + r <= sw.limit;
        if (!near) q0 = __builtin_nan("");
        keep = !near || sweep_may_touch(sw, d0, d1, d2, reach + r);
    }
    const unsigned long long ball = __ballot(keep);
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    lds_barrier();  // the tile before has been read
    if (lane == 0) u.wcnt[wv] = __popcll(ball);
    if (threadIdx.x == 0) u.found = 0;
    if (static_cast<int>(threadIdx.x) < ncl) {
        u.dmin[threadIdx.x] = ordered_bits(best);
        u.pmin[threadIdx.x] = ~0ull;
    }
    lds_barrier();
    int base = 0, kept = 0;
    for (int w = 0; w < kBlock / 64; ++w) {
        if (w < wv) base += u.wcnt[w];
        kept += u.wcnt[w];
    }
    if (kept == 0) return false;  // uniform
    if (keep) {
        const int e = base + __popcll(ball & ((1ull << lane) - 1ull));
        u.qx[e] = q0;
        u.qy[e] = q1;
        u.qz[e] = q2;
        u.px[e] = x;
        u.py[e] = y;
        u.pz[e] = z;
        u.pr[e] = r;
        u.cand[e] = cl;
        u.idx[e] = static_cast<int>(j);
        u.sp[e] = sp;
    }
    lds_barrier();
    // a kept sphere by g lanes, each over every g-th mover sphere
    int g = 1;
    while (g < nt && g < 64) g *= 2;
    const int sub = lane & (g - 1), per = kBlock / g;
    for (int e0 = 0; e0 < kept; e0 += per) {
        const int e = e0 + static_cast<int>(threadIdx.x) / g;
        double d = kInf;
        long long p = 0x7fffffffffffffffLL;
        if (e < kept) {
            const double s0 = u.qx[e], s1 = u.qy[e], s2 = u.qz[e], sr = u.pr[e];
            const long long n = nk(u.cand[e]);
            for (int i = sub; i < nt; i += g) {
                const double m0 = u.mx[i], m1 = u.my[i], m2 = u.mz[i], mr = u.mr[i];
                double d0 = s0 - m0, d1 = s1 - m1, d2 = s2 - m2;
                bool tested = true;
                if (s0 != s0) {  // not near: the pair's own nearest image
                    tested = sw.usable && mr + sr <= sw.limit;
                    d0 = nearest_image(u.px[e] - m0, sw.hx, sw);
                    d1 = nearest_image(u.py[e] - m1, sw.hy, sw);
                    d2 = nearest_image(u.pz[e] - m2, sw.hz, sw);
                }
                if (tested) {
                    double earliest;
                    if (!sweep_may_touch(sw, d0, d1, d2, mr + sr, &earliest)) continue;
                    // a pair that cannot come below the candidate's minimum so far
                    if (earliest > from_ordered_bits(__hip_atomic_load(&u.dmin[u.cand[e]], __ATOMIC_RELAXED,
                                                                       __HIP_MEMORY_SCOPE_WORKGROUP)))
                        continue;
                }
                const double v = swept_sphere(m0, m1, m2, mr, u.px[e], u.py[e], u.pz[e], sr, a.dir[0], a.dir[1],
                                              a.dir[2], a.lpm, a.L);
                lexmin(d, p, v, (i0 + i) * n + u.idx[e]);
                if (v < kInf) atomicMin(&u.dmin[u.cand[e]], ordered_bits(v));
            }
        }
        if (__any(d < kInf)) {
            for (int off = g >> 1; off > 0; off >>= 1) {
                const double od = __shfl_xor(d, off, 64);
                const long long op = __shfl_xor(p, off, 64);
                lexmin(d, p, od, op);
            }
        }
        if (sub == 0 && e < kept) {
            u.rd[e] = d;
            u.rp[e] = p;
            if (d < kInf) u.found = 1;
        }
    }
    lds_barrier();
    if (!u.found) return false;
    // every thread passes the barriers
    const int e = threadIdx.x;
    const bool least = e < kept && u.rd[e] < kInf && ordered_bits(u.rd[e]) == u.dmin[u.cand[e]];
    if (least) atomicMin(&u.pmin[u.cand[e]], static_cast<unsigned long long>(u.rp[e]));
    lds_barrier();
    if (least && u.pmin[u.cand[e]] == static_cast<unsigned long long>(u.rp[e])) {
        u.bms[u.cand[e]] = u.msp[(u.rp[e] - u.idx[e]) / nk(u.cand[e]) - i0];
        u.bos[u.cand[e]] = u.sp[e];
    }
    lds_barrier();
    return true;
}

// The counters of a search's grid (grid_form.hpp).
constexpr unsigned long long kGridWaitTicks = 2000000;  // 20 ms of the 100 MHz constant clock
struct SearchGrid {
    SearchState *s;
    unsigned long long since = 0;
    __device__ __forceinline__ void publish() const { release_to_device(); }
    __device__ __forceinline__ void arrive() {
        atomicAdd(&s->grid_bar, 1u);
        since = wall_clock64();
    }
    __device__ __forceinline__ bool out_of_time() const { return wall_clock64() - since > kGridWaitTicks; }
    __device__ __forceinline__ unsigned arrived() const {
        return __hip_atomic_load(&s->grid_bar, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __device__ __forceinline__ void pause() const { __builtin_amdgcn_s_sleep(1); }
    __device__ __forceinline__ void give_up() const { atomicExch(&s->grid_fail, 1u); }
    __device__ __forceinline__ unsigned ticket() const { return atomicAdd(&s->done_solve, 1u); }
};

// Pair solve of the survivors filtered for step a: the tiles of the candidates'
// spheres over the blocks of the grid, and the last block to finish reduces the
// tiles' minima per candidate and finishes the step.
__device__ __forceinline__ void solve_phase(const DevBox &b, const SearchArgs &a, StepLds &lds) {
    __shared__ long long cpre[kMaxPlan + 1];
    SolveLds &u = lds.solve;
    __shared__ bool last;
    unsigned int F = b.ss->nfilt;
    if (F > static_cast<unsigned int>(a.cap)) F = static_cast<unsigned int>(a.cap);
    const long long nsrc = a.n_mov;
    const int ssrc = a.start;
    double centre[3] = {a.sx, a.sy, a.sz};
    if (!a.known) centre[0] = b.ax[a.src], centre[1] = b.ay[a.src], centre[2] = b.az[a.src];
    const SweepTest sw = sweep_test(a.dir, a.lpm, a.L);
    const Places<false> where{b, nullptr};
    const int n_movers = static_cast<int>((nsrc + kMoverTile - 1) / kMoverTile);
    double reach = 0.0;
    int nt = 0, in_lds = -1;
    auto mover_tile = [&](int q) {  // mover spheres q kMoverTile ... into LDS (uniform)
        if (q == in_lds) return;
        lds_barrier();
        nt = static_cast<int>(nsrc - static_cast<long long>(q) * kMoverTile < kMoverTile
                                  ? nsrc - static_cast<long long>(q) * kMoverTile : kMoverTile);
        reach = load_mover_tile(b, u, ssrc, static_cast<long long>(q) * kMoverTile, nt, centre, -1, where);
        in_lds = q;
    };
    // a few candidates' member segments are loaded once, into LDS
    constexpr unsigned int kStaged = 256;
    __shared__ int s_csk[kStaged];
    const bool staged = F <= kStaged;
    long long spheres = 0;
    const bool fits = F <= static_cast<unsigned int>(kMaxPlan);
    for (unsigned int c = threadIdx.x; c < F; c += blockDim.x) {
        const int k = b.cand_id[c];
        const int nk = b.acount[k];
        if (staged) s_csk[c] = b.astart[k];
        if (fits) cpre[c] = nk;
        spheres += nk;
    }
    spheres = block_sum(spheres);
    __shared__ long long s_spheres;
    if (threadIdx.x == 0) s_spheres = spheres;
    __syncthreads();
    // tiles of 64 to kBlock spheres: narrow ones spread a few large survivors
    // over more blocks
    const long long T = s_spheres;
    const long long want = (T + gridDim.x - 1) / gridDim.x;
    const long long W = want >= kBlock ? kBlock : (want <= 64 ? 64 : (want + 63) / 64 * 64);
    const long long tiles = (T + W - 1) / W;
    const bool planned = fits && tiles + F <= a.part_cap;
    if (planned) {
        block_exclusive_scan(cpre, static_cast<int>(F));
        for (long long g = blockIdx.x; g < tiles; g += gridDim.x) {
            const long long w0 = g * W, w = w0 + threadIdx.x, w1 = w0 + W < T ? w0 + W : T;
            const int c0 = last_not_above(cpre, static_cast<int>(F), w0);
            const int c1 = last_not_above(cpre, static_cast<int>(F), w1 - 1);
            int cl = -1;
            long long j = 0, m = 0;
            if (w < w1) {
                const int c = last_not_above(cpre, static_cast<int>(F), w);
                cl = c - c0;
                j = w - cpre[c];
                m = (staged ? s_csk[c] : b.astart[b.cand_id[c]]) + j;
            }
            // tile g of candidate c: its minimum at part[g + c] (g + c is its own)
            double bd = kInf;
            long long bp = 0x7fffffffffffffffLL;
            for (int q = 0; q < n_movers; ++q) {
                mover_tile(q);
                if (solve_tile(b, a, sw, u, centre, reach, static_cast<long long>(q) * kMoverTile, nt, cl, j, m,
                               -1, -1, where, c1 - c0 + 1, bd, [&](int e) { return cpre[c0 + e + 1] - cpre[c0 + e]; }) &&
                    static_cast<int>(threadIdx.x) <= c1 - c0 && u.pmin[threadIdx.x] != ~0ull)
                    lexmin(bd, bp, from_ordered_bits(u.dmin[threadIdx.x]), static_cast<long long>(u.pmin[threadIdx.x]));
            }
            if (static_cast<int>(threadIdx.x) <= c1 - c0) {
                b.part_d[g + c0 + threadIdx.x] = bd;
                b.part_p[g + c0 + threadIdx.x] = bp;
            }
        }
    } else {  // very many survivors (or partials): a candidate at a time by a block
        for (unsigned int c = blockIdx.x; c < F; c += gridDim.x) {
            const int k = b.cand_id[c];
            const long long nk = b.acount[k], sk = b.astart[k];
            double bd = kInf;
            long long bp = 0x7fffffffffffffffLL;
            for (int q = 0; q < n_movers; ++q) {
                mover_tile(q);
                for (long long w0 = 0; w0 < nk; w0 += kBlock) {
                    const long long j = w0 + threadIdx.x;
                    if (solve_tile(b, a, sw, u, centre, reach, static_cast<long long>(q) * kMoverTile, nt,
                                   j < nk ? 0 : -1, j, sk + j, -1, -1, where, 1, bd, [&](int) { return nk; }) &&
                        threadIdx.x == 0 && u.pmin[0] != ~0ull)
                        lexmin(bd, bp, from_ordered_bits(u.dmin[0]), static_cast<long long>(u.pmin[0]));
                }
            }
            if (threadIdx.x == 0) {
                b.cand_exact[c] = bd;
                b.cand_pair[c] = (bd < kInf) ? bp : -1;
            }
        }
    }
    __syncthreads();  // the block's partials are written
    if (threadIdx.x == 0) {
        SearchGrid grid{b.ss};
        last = grid_part(grid, gridDim.x, blockIdx.x < (planned ? tiles : static_cast<long long>(F)));
    }
    __syncthreads();
    if (!last) return;
    acquire_from_device();
    if (planned) {
        // per-candidate reduction of the tiles' minima: a candidate in a few
        // tiles by one thread, one in many by the whole block
        constexpr long long kThreadTiles = 8;
        for (unsigned int c = threadIdx.x; c < F; c += blockDim.x) {
            const long long g0 = cpre[c] / W, g1 = (cpre[c + 1] - 1) / W + 1;
            if (g1 - g0 > kThreadTiles) continue;
            double bd = kInf;
            long long bp = 0x7fffffffffffffffLL;
            for (long long g = g0; g < g1; ++g) lexmin(bd, bp, b.part_d[g + c], b.part_p[g + c]);
            b.cand_exact[c] = bd;
            b.cand_pair[c] = (bd < kInf) ? bp : -1;
        }
        for (unsigned int c = 0; c < F; ++c) {
            const long long g0 = cpre[c] / W, g1 = (cpre[c + 1] - 1) / W + 1;
            if (g1 - g0 <= kThreadTiles) continue;  // uniform over the block
            double bd = kInf;
            long long bp = 0x7fffffffffffffffLL;
            for (long long g = g0 + threadIdx.x; g < g1; g += blockDim.x) lexmin(bd, bp, b.part_d[g + c], b.part_p[g + c]);
            block_lexmin(bd, bp);
            if (threadIdx.x == 0) {
                b.cand_exact[c] = bd;
                b.cand_pair[c] = (bd < kInf) ? bp : -1;
            }
        }
    }
    __syncthreads();  // every candidate's minimum before the ordered scan reads them
    __shared__ StepPick pick;
    scan_candidates(b, F, ssrc, nullptr, b.order, pick);
    if (threadIdx.x == 0) {
        pick.nquery = b.ss->nquery;
        pick.nfilt = b.ss->nfilt;
        pick.overflow = b.ss->overflow != 0u;
        pick.src_slot = b.cslot[a.src];
        pick.tpairs = nsrc * T;
        pick.handover = 0;
    }
    apply_step<false>(b, a, pick, MoverSphere{0, -1, 0., 0., 0., 0., 0., 0., 0.}, true, lds.merge);
}

__global__ __launch_bounds__(kBlock) void k_solve(DevBox b, SearchArgs a) {
    if (behind_gate(b, a)) return;  // the host knows it is skipped: no record
    __shared__ StepLds lds;
    solve_phase(b, a, lds);
}

// One launch for a large mover: k_filter's work, a grid-wide barrier in place
// of the boundary between k_filter and k_solve, then k_solve's work by the same
// blocks; the same arithmetic in the same order, so the same step.  The grid
// is small enough to be resident at once (at most kFilterBlocks blocks, half
// the CUs; one box stream, launches in order); a block that waits past kGridWaitTicks at the
// barrier gives up and sets grid_fail, the step then publishes no record (the block
// takes no ticket, so none is the last) and the host reports a device error instead
// of waiting without end.
__global__ __launch_bounds__(kBlock) void k_step_grid(DevBox b, SearchArgs a) {
    if (behind_gate(b, a)) return;  // every block reads the same gate: the host knows it is skipped
    __shared__ StepLds lds;
    const unsigned long long tot =
        block_sum(filter_phase<false>(b, a, blockIdx.x, gridDim.x, CellBounds{0, 0, 0}, false, lds.filter, a.dirty_n,
                                      nullptr, BoxSink{b, a.cap})) & 0xffffffffull;
    __shared__ int s_ok;
    if (threadIdx.x == 0) {
        if (tot) atomicAdd(&b.ss->nquery, tot);
        SearchGrid grid{b.ss};
        s_ok = grid_meet(grid, gridDim.x) ? 1 : 0;
    }
    __syncthreads();
    if (!s_ok) return;
    acquire_from_device();  // every block's candidates are visible to this one
    solve_phase(b, a, lds);
}

// Survivors of a step: into LDS when one block takes the step, else into the
// step's share of the box's candidate buffer.
struct StepSink {
    const DevBox &b;
    StepCands &sc;
    int q, slots;  // the step's number and its share of the buffer (-1: LDS)
    __device__ __forceinline__ void operator()(int id, int rank, double d, int2 info, int entry) const {
        if (slots < 0) {
            const unsigned int c = atomicAdd(&sc.n, 1u);
            if (c >= static_cast<unsigned int>(kStepCands)) return;  // counted: left to the grid form
            sc.id[c] = id;
            sc.rank[c] = rank;
            sc.db[c] = d;
            sc.nk[c] = info.x;
            sc.sk[c] = info.y;
            sc.mv[c] = entry;
        } else {
            const unsigned int c = atomicAdd(&b.ss->step_nfilt[q], 1u);
            if (c >= static_cast<unsigned int>(slots)) return;
            b.cand_id[q * slots + c] = id;
            b.cand_rank[q * slots + c] = rank;
            b.cand_db[q * slots + c] = d;
            b.step_info[q * kStepCands + c] = make_int4(info.x, info.y, entry, 0);
        }
    }
};

// Search of one step, number q of its launch, by vg blocks (vb is this one):
// every block filters its share of the Verlet window; the last block to finish
// (ticket) solves the sphere pairs of the survivors, orders them and has the
// contact in pick (thread 0).  More survivors or pairs than one block should
// take are left to the grid form (pick.handover).  Nothing of the box changes.
// nd: dirty-list entries; mv: its predecessors' moves (kMoved); ct: bounds of
// the visited cells from the host (in LDS), or null.  gate_open: the caller
// knows the gate is open for this step; otherwise the gate is read with the
// first loads and a step behind it does no more than read-only filter work.
// Returns 0 for a step behind the gate, 1 where this block took part, 2 where it
// finished the search, 3 where it leaves it to the grid form (uniform over the
// block).
template <bool kMoved>
__device__ __forceinline__ int search_step(const DevBox &b, const SearchArgs &a, unsigned vb, unsigned vg, int q,
                                           int nd, const Moved *mv, bool gate_open, const CellTable *ct, StepLds &lds,
                                           StepCands &sc, StepPick &pick, MoverSphere &mover, const StepPrefetch *pre) {
    // independent loads first, so that their latencies overlap: the gate, the
    // mover's cell entry and sphere indices, the bounds of the visited cells
    const unsigned long long gate = (!gate_open && a.gated) ? b.ss->gate : 0ull;
    const bool mload = a.n_mov <= kBlock;
    int src_slot = -1, msp = -1;
    if (pre) {
        src_slot = pre->src_slot;
        msp = pre->mover.sp;
    } else {
        src_slot = (threadIdx.x == 0) ? b.cslot[a.src] : -1;
        msp = (mload && static_cast<int>(threadIdx.x) < a.n_mov) ? b.members[a.start + threadIdx.x] : -1;
    }
    const CellBounds cb = load_cell_bounds(b, a, ct);
    const bool skip = gate != 0ull && gate < a.seq && gate > a.released;
    mover = MoverSphere{mload, msp, 0., 0., 0., 0., 0., 0., 0.};
    if (pre) mover = pre->mover;
    if (msp >= 0) {
        if (!pre) {
            mover.rx = b.srx[msp];
            mover.ry = b.sry[msp];
            mover.rz = b.srz[msp];
        }
        mover.x = b.sx[msp];
        mover.y = b.sy[msp];
        mover.z = b.sz[msp];
        mover.r = b.sr[msp];
    }
    if (threadIdx.x == 0) sc.n = 0u;  // filter_phase appends behind a barrier
    const int share = a.cap / kMaxSteps < kStepCands ? a.cap / kMaxSteps : kStepCands;
    const StepSink sink{b, sc, q, vg > 1 ? share : -1};
    const unsigned long long cnt =
        block_sum(filter_phase<kMoved>(b, a, vb, vg, cb, skip, lds.filter, nd, mv, sink));
    if (skip) return 0;
    // one atomic per block: finished blocks, appended candidates, visited aggregates
    __shared__ bool last;
    __shared__ unsigned long long s_total;
    if (vg > 1) {
        if (threadIdx.x == 0) {
            const unsigned long long mine = kTicketOne + cnt;
            if (cnt >= kAppendOne) release_to_device();  // most blocks have written nothing
            const unsigned long long old = atomicAdd(&b.ss->step_tick[q], mine);
            last = (old >> 56) == vg - 1u;
            s_total = old + mine;
        }
        __syncthreads();
        if (!last) return 1;
        if (static_cast<unsigned int>((s_total >> 32) & 0xffffffull) > 0u) acquire_from_device();
        if (threadIdx.x == 0) {  // for the next launch
            b.ss->step_tick[q] = 0ull;
            b.ss->step_nfilt[q] = 0u;
        }
    } else {
        if (threadIdx.x == 0) s_total = cnt;
        lds_barrier();
    }
    const unsigned long long total = s_total;
    const unsigned int nfilt = static_cast<unsigned int>((total >> 32) & 0xffffffull);
    // past the box's candidate capacity the grid form reports it
    const unsigned int most = static_cast<unsigned int>(vg > 1 ? share : (a.cap < kStepCands ? a.cap : kStepCands));
    const unsigned int F = nfilt < most ? nfilt : most;
    const long long nsrc = a.n_mov;
    const int ssrc = a.start;
    const Places<kMoved> where{b, mv};
    const int self = kMoved ? mv->self : -1;
    if (threadIdx.x == 0) {
        pick.nquery = total & 0xffffffffull;
        pick.nfilt = nfilt;
        pick.overflow = 0;
        pick.src_slot = src_slot;
        pick.tpairs = 0;
        pick.handover = 0;
    }
    if (F > 0 || nfilt > F) {
        // survivors into LDS: label, size, member segment, bounding key, and
        // the prefix of the sizes
        long long tp = 0;
        for (unsigned int c = threadIdx.x; c < F; c += blockDim.x) {
            if (vg > 1) {
                sc.id[c] = b.cand_id[q * share + c];
                sc.db[c] = b.cand_db[q * share + c];
                sc.rank[c] = b.cand_rank[q * share + c];
                const int4 v = b.step_info[q * kStepCands + c];
                sc.nk[c] = v.x;
                sc.sk[c] = v.y;
                sc.mv[c] = v.z;
            }
            tp += nsrc * sc.nk[c];
        }
        if (mload && nsrc <= kThreadPairs && threadIdx.x < nsrc) {
            // a small mover's spheres, loaded with the step's first loads
            const int t = threadIdx.x;
            sc.msp[t] = mover.sp;
            sc.mr[t] = mover.r;
            where.of(self, mover, sc.mx[t], sc.my[t], sc.mz[t]);
        }
        const long long tpairs = block_sum(tp);
        __shared__ int s_over;
        __shared__ long long s_most;  // most pairs a survivor brings
        if (threadIdx.x == 0) {
            s_over = nfilt > most || tpairs > (a.lpm < 0.25 * a.L ? kStepPairs : kStepExactPairs);
            pick.tpairs = tpairs;
            pick.handover = s_over;
        }
        if (threadIdx.x < 64) {  // block_sum's barrier published the sizes
            const int nk = threadIdx.x < F ? sc.nk[threadIdx.x] : 0;
            const int incl = wave_inclusive_scan(nk);
            if (threadIdx.x < F) sc.pre[threadIdx.x + 1] = incl;
            int big = nk;
            for (int off = 32; off > 0; off >>= 1) {
                const int o = __shfl_xor(big, off, 64);
                big = o > big ? o : big;
            }
            if (threadIdx.x == 0) {
                sc.pre[0] = 0;
                s_most = nsrc * big;
            }
        }
        static_assert(kStepCands <= 64, "the prefix of the survivors' sizes is one wave's");
        lds_barrier();
        if (s_over) return 3;
        // exact sphere-pair distances, lexicographic (d, i, j) minimum per
        // candidate: when every candidate has at most kThreadPairs pairs
        // (monomers), one thread walks a candidate's in (i, j) order (strict <
        // keeps the first minimum); else all candidates' spheres in tiles
        if (s_most <= kThreadPairs && mload) {
            if (threadIdx.x < F) {
                const unsigned int c = threadIdx.x;
                const int nk = sc.nk[c];  // this thread's own entries
                const int sk = sc.sk[c];
                double bd = kInf;
                int bi = -1, bj = -1;
                for (int i = 0; i < nsrc; ++i)
                    for (int j = 0; j < nk; ++j) {
                        const int sj = sk < 0 ? ~sk : b.members[sk + j];
                        double x2, y2, z2;
                        where(sc.mv[c], sj, x2, y2, z2);
                        const double d = swept_sphere(sc.mx[i], sc.my[i], sc.mz[i], sc.mr[i], x2, y2, z2, b.sr[sj],
                                                      a.dir[0], a.dir[1], a.dir[2], a.lpm, a.L);
                        if (d < bd) {
                            bd = d;
                            bi = sc.msp[i];
                            bj = sj;
                        }
                    }
                sc.ex[c] = bd;
                sc.ms[c] = bi;
                sc.os[c] = bj;
            }
            lds_barrier();
        } else {
            SolveLds &u = lds.solve;
            const SweepTest sw = sweep_test(a.dir, a.lpm, a.L);
            double centre[3] = {a.sx, a.sy, a.sz};
            if (!a.known) centre[0] = b.ax[a.src], centre[1] = b.ay[a.src], centre[2] = b.az[a.src];
            const int T = sc.pre[F];
            double bd = kInf;  // thread c: candidate c's minimum
            long long bp = 0x7fffffffffffffffLL;
            int bi = -1, bj = -1;
            for (long long i0 = 0; i0 < nsrc; i0 += kMoverTile) {
                const int nt = static_cast<int>(nsrc - i0 < kMoverTile ? nsrc - i0 : kMoverTile);
                if (i0 > 0) lds_barrier();
                const double reach = load_mover_tile(b, u, ssrc, i0, nt, centre, self, where, mload ? &mover : nullptr);
                for (int w0 = 0; w0 < T; w0 += kBlock) {
                    const int w = w0 + static_cast<int>(threadIdx.x);
                    int c = -1, j = 0, m = 0, e = -1, one = -1;
                    if (w < T) {
                        c = last_not_above(sc.pre, static_cast<int>(F), w);
                        j = w - sc.pre[c];
                        m = sc.sk[c] + j;
                        e = sc.mv[c];
                        if (sc.sk[c] < 0) one = ~sc.sk[c];
                    }
                    if (solve_tile(b, a, sw, u, centre, reach, i0, nt, c, j, m, one, e, where, static_cast<int>(F), bd,
                                   [&](int k) { return static_cast<long long>(sc.nk[k]); }) &&
                        threadIdx.x < F && u.pmin[threadIdx.x] != ~0ull) {
                        const double d = from_ordered_bits(u.dmin[threadIdx.x]);
                        const long long p = static_cast<long long>(u.pmin[threadIdx.x]);
                        if (d < bd || (d == bd && p < bp)) {
                            bd = d;
                            bp = p;
                            bi = u.bms[threadIdx.x];
                            bj = u.bos[threadIdx.x];
                        }
                    }
                }
            }
            if (threadIdx.x < F) {
                sc.ex[threadIdx.x] = bd;
                sc.ms[threadIdx.x] = bi;
                sc.os[threadIdx.x] = bj;
            }
            lds_barrier();
        }
    }
    scan_candidates(b, F, ssrc, &sc, sc.order, pick);
    return 2;
}

// A step left to the grid form: its record says so, and the gate closes for the
// steps queued behind it (thread 0).
__device__ __forceinline__ void hand_over(const DevBox &b, const SearchArgs &a, bool publish) {
    if (a.gated) b.ss->gate = a.seq;
    StepRecord *o = a.out;
    o->status = kPendingSolve;
    o->contact = 0;
    o->skipped = 0;
    if (publish) {
        __threadfence_system();
        __hip_atomic_store(&o->seq, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// One MC step for a small mover, searched by vg blocks and carried out by the
// one that finishes the search.  publish: publish the record (else wave 0
// writes its body and the caller publishes the sequence number later, after a
// system-scope fence).  Returns (in thread 0) whether the step closed the gate.
// role (optional, LDS, set by thread 0): as search_step's result.
template <bool kCaps>
__device__ __forceinline__ bool step_body(const DevBox &b, const SearchArgs &a, unsigned vb, unsigned vg,
                                          bool gate_open, const CellTable *ct, bool publish, int *role = nullptr,
                                          const StepPrefetch *pre = nullptr) {
    __shared__ StepLds lds;
    __shared__ StepCands sc;
    __shared__ StepPick pick;
    MoverSphere mover;
    const int r = search_step<false>(b, a, vb, vg, 0, a.dirty_n, nullptr, gate_open, ct, lds, sc, pick, mover, pre);
    if (role && threadIdx.x == 0) *role = r < 2 ? r : 2;
    if (r < 2) return false;
    if (r == 3) {
        if (threadIdx.x == 0) hand_over(b, a, publish);
        return a.gated != 0;
    }
    return apply_step<kCaps>(b, a, pick, mover, publish, lds.merge);
}

// Kernel arguments read where the launch put them, in constant memory, when
// they are needed: taken by value, the box's 70 pointers are all loaded first
// and most of them spilled (219 spilled scalars against 35; a run of 2347
// monomers 189 ms against 175).
template <class T> __device__ __forceinline__ const T &kernel_arguments() {
    using Const = const T __attribute__((address_space(4)));
    return *(const T *)(Const *)__builtin_amdgcn_kernarg_segment_ptr();
}

struct StepOne {
    DevBox b;
    SearchArgs a;
};
template <bool kCaps> __global__ __launch_bounds__(kBlock) void k_step(StepOne) {
    const StepOne &k = kernel_arguments<StepOne>();
    step_body<kCaps>(k.b, k.a, blockIdx.x, gridDim.x, false, nullptr, true);
}

// Several consecutive queued steps of a box in one launch (at most kMaxSteps).
// A step is a chain of dependent loads of about 8 us in which one workgroup
// hardly uses its CU, and a step without a contact only moves its mover by a
// vector that the host knows beforehand.  So all steps of the launch search at
// the same time, each by its own blocks, against the box as it is before the
// launch with the moves of its predecessors put in (Moved); the last block to
// finish carries the steps out in order up to the first contact (or hand-over),
// behind which the others do nothing, as they would behind the gate.  Every
// step sees the very values it would see in launches of its own.
// A launch of up to eight takes 23.4 us on average (2347 monomers; a single step's
// 7.6): the searches, a ticket among a step's blocks and one among the steps, then
// the moves, their records and, on a contact, the merge, by one block.  Against
// eight launches of one that is less than half; how the 16 us beyond a step divide
// has not been measured.
struct StepsLds {
    StepLds lds;
    StepCands sc;
    StepPick pick;
    Moved mv;
    SearchArgs args[kMaxSteps];
    StepPick picks[kMaxSteps];
    StepRecord head[kMaxSteps];
    int over, last;
};

// Fills the moved set of step q from its predecessors' arguments.
template <class Args>
__device__ __forceinline__ void set_moved(Moved &mv, int q, int src, const Args &args) {
    if (static_cast<int>(threadIdx.x) < q) {
        const int p = threadIdx.x;
        const SearchArgs &e = args(p);
        int id = e.src;
        for (int r = p + 1; r < q; ++r)
            if (args(r).src == e.src) id = -1;  // moved again later
        mv.id[p] = id;
        mv.cell[p] = e.nc_cell;
        mv.x[p] = e.nc_com[0];
        mv.y[p] = e.nc_com[1];
        mv.z[p] = e.nc_com[2];
        mv.r[p] = e.srmax;
        mv.rx[p] = e.nc_ref[0];
        mv.ry[p] = e.nc_ref[1];
        mv.rz[p] = e.nc_ref[2];
        mv.info[p] = make_int2(e.n_mov, e.start);
    }
    if (threadIdx.x == 0) {
        int self = -1;
        for (int p = 0; p < q; ++p)
            if (args(p).src == src) self = p;
        mv.n = q;
        mv.self = self;
    }
}

// Carries out the nj searched steps in u.args / u.picks in order up to the first
// contact or hand-over and publishes their records (whole block).
template <bool kCaps> __device__ __forceinline__ void commit_steps(const DevBox &b, StepsLds &u, int nj) {
    SearchState *s = b.ss;
    // a step whose move the host does not know (the only one of its launch) is
    // carried out as one with a contact; a lane looks at a step
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool stops = lane < nj && (!u.args[lane].nc_ok || u.picks[lane].handover || u.picks[lane].dist <= u.args[lane].lpm);
    const unsigned long long stop = __ballot(stops);
    const int f = stop ? __ffsll(static_cast<long long>(stop)) - 1 : nj;
    constexpr int kHead = static_cast<int>(offsetof(StepRecord, merge) / sizeof(unsigned long long));
    static_assert(offsetof(StepRecord, merge) % sizeof(unsigned long long) == 0, "record head in 8-byte words");
    // moves without contact: a wave per step; a mover that moves again later in
    // the launch is placed by its last move
    for (int q = wave; q < f; q += kBlock / 64) {
        const SearchArgs &a = u.args[q];
        bool later = false;
        for (int p = q + 1; p < f; ++p) later = later || u.args[p].src == a.src;
        int first_sphere = 0;  // lane 0's
        if (!later)
            for (int t = lane; t < a.n_mov; t += 64) {
                const int sp = b.members[a.start + t];
                if (t == 0) first_sphere = sp;
                b.sx[sp] = a.nc_ref[0] + b.srx[sp];
                b.sy[sp] = a.nc_ref[1] + b.sry[sp];
                b.sz[sp] = a.nc_ref[2] + b.srz[sp];
            }
        if (lane == 0) {
            const StepPick &pk = u.picks[q];
            StepRecord &o = u.head[q];
            o.dist = pk.dist;
            o.move = a.lpm;
            o.ms = pk.ms;
            o.os = pk.os;
            o.oagg = pk.oagg;
            o.contact = 0;
            o.status = 0;
            o.nquery = pk.nquery;
            o.nfilt = pk.nfilt;
            o.npairs = static_cast<unsigned long long>(pk.tpairs);
            o.skipped = 0;
            o.dirty_count = a.dirty_n + (a.dirty_slot >= 0 ? 1 : 0);
            o.merged_inline = o.m_new_start = o.m_new_cap = o.pad = 0;
            if (a.dirty_slot >= 0) {  // first move since the cell-list build
                b.dirty[a.src] = 1;
                b.dirty_list[a.dirty_slot] = a.src;
                b.dslot[a.src] = a.dirty_slot;
                if (pk.src_slot >= 0) {
                    b.cpr[pk.src_slot] = -1.0;
                    b.cf[pk.src_slot].w = -1.f;
                }
            }
            if (!later) {
                b.ax[a.src] = a.nc_com[0];
                b.ay[a.src] = a.nc_com[1];
                b.az[a.src] = a.nc_com[2];
                b.acell[a.src] = a.nc_cell;
                set_dirty_entry(b, a.dirty_pos, a.nc_com[0], a.nc_com[1], a.nc_com[2], a.srmax, a.nc_cell);
                b.dinfo[a.dirty_pos] = make_int2(a.n_mov, a.n_mov == 1 ? ~first_sphere : a.start);
            }
        }
    }
    if (threadIdx.x == 0) {
        for (int q = f - 1; q >= 0; --q)
            if (u.args[q].dirty_slot >= 0) {  // slots are handed out in order
                s->dirty_count = static_cast<unsigned int>(u.args[q].dirty_slot + 1);
                break;
            }
        s->steps_done = 0u;
    }
    __syncthreads();  // the moves are in the box for the step that follows; the heads are in LDS
    if (wave == kBlock / 64 - 1 && f > 0) {
        // records of the moves, published while the contact below is carried out
        for (int i = lane; i < f * kHead; i += 64)
            reinterpret_cast<unsigned long long *>(u.args[i / kHead].out)[i % kHead] =
                reinterpret_cast<const unsigned long long *>(&u.head[i / kHead])[i % kHead];
        __threadfence_system();
        if (lane < f)
            __hip_atomic_store(&u.args[lane].out->seq, u.args[lane].seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (f >= nj) return;
    if (u.picks[f].handover) {
        if (threadIdx.x == 0) hand_over(b, u.args[f], true);
        return;
    }
    const MoverSphere mover = load_mover_sphere(b, u.args[f]);
    apply_step<kCaps>(b, u.args[f], u.picks[f], mover, true, u.lds.merge);
}

// The rest of a step's launch once its arguments are known: args(p) gives those
// of step p <= q, fetch(p) loads all of step p's into LDS (for p < nj, when
// every step has finished its search).
template <bool kCaps, class Args, class Fetch>
__device__ __forceinline__ void run_steps(const DevBox &b, StepsLds &u, const SearchArgs &a, int q, int nj,
                                          int nd, unsigned vb, unsigned vg, const Args &args, const Fetch &fetch) {
    set_moved(u.mv, q, a.src, args);
    lds_barrier();
    MoverSphere mover;
    const int r = search_step<true>(b, a, vb, vg, q, nd, &u.mv, false, nullptr, u.lds, u.sc, u.pick, mover, nullptr);
    if (r < 2) return;
    if (threadIdx.x == 0) {
        if (nj > 1) {
            b.picks[q] = u.pick;
            release_to_device();
            u.last = atomicAdd(&b.ss->steps_done, 1u) == static_cast<unsigned int>(nj) - 1u;
        } else {
            u.picks[0] = u.pick;
            u.last = 1;
        }
    }
    __syncthreads();
    if (!u.last) return;
    if (nj > 1) {
        acquire_from_device();
        constexpr int kPickWords = static_cast<int>(sizeof(StepPick) / sizeof(unsigned long long));
        for (int i = threadIdx.x; i < nj * kPickWords; i += blockDim.x)
            reinterpret_cast<unsigned long long *>(u.picks)[i] = reinterpret_cast<const unsigned long long *>(b.picks)[i];
    }
    fetch();
    __syncthreads();
    commit_steps<kCaps>(b, u, nj);
}

constexpr int kArgWords = static_cast<int>(sizeof(SearchArgs) / sizeof(unsigned long long));
static_assert(sizeof(SearchArgs) % sizeof(unsigned long long) == 0 && sizeof(StepPick) % sizeof(unsigned long long) == 0,
              "copied in 8-byte words");

struct StepSet {
    DevBox b;
    int nj, pad;
    SearchArgs a[kMaxSteps];
};

// Steps of one box, blockIdx.y the step and blockIdx.x its block.
template <bool kCaps> __global__ __launch_bounds__(kBlock) void k_steps(StepSet) {
    __shared__ StepsLds u;
    const StepSet &set = kernel_arguments<StepSet>();
    const int q = static_cast<int>(blockIdx.y);
    const SearchArgs &a = set.a[q];
    const unsigned vg = static_cast<unsigned>(a.vg);
    if (blockIdx.x >= vg) return;
    run_steps<kCaps>(set.b, u, a, q, set.nj, a.run_dirty, blockIdx.x, vg,
              [&](int p) -> const SearchArgs & { return set.a[p]; },
              [&] {
                  for (int i = threadIdx.x; i < set.nj * kArgWords; i += blockDim.x)
                      reinterpret_cast<unsigned long long *>(u.args)[i] =
                          reinterpret_cast<const unsigned long long *>(set.a)[i];
              });
}

// Steps of many boxes: blockIdx.y a box and blockIdx.x its step, one block each
// (windows of few aggregates).  The runs are in pinned host memory; a block
// reads its own step's arguments and of its predecessors what the moved set
// takes (the first kMoveWords words), and leaves its own in device memory for
// the block that carries the steps out.
struct BoxRun {
    const DevBox *box;  // device copy of the box's descriptor
    int nj, pad;
    SearchArgs a[kMaxSteps];
};
constexpr int kMoveWords = static_cast<int>(offsetof(SearchArgs, known) / sizeof(unsigned long long));
static_assert(offsetof(SearchArgs, known) % sizeof(unsigned long long) == 0, "move part in 8-byte words");

__global__ __launch_bounds__(kBlock) void k_steps_group(const BoxRun *runs) {
    __shared__ StepsLds u;
    __shared__ unsigned long long head[2];
    const BoxRun *run = runs + blockIdx.y;
    const int q = static_cast<int>(blockIdx.x);
    for (int i = threadIdx.x; i < 2 + kArgWords + q * kMoveWords; i += blockDim.x) {
        if (i < 2) {
            head[i] = reinterpret_cast<const unsigned long long *>(run)[i];
        } else if (i < 2 + kArgWords) {
            const int w = i - 2;
            reinterpret_cast<unsigned long long *>(&u.args[q])[w] =
                reinterpret_cast<const unsigned long long *>(&run->a[q])[w];
        } else {
            const int p = (i - 2 - kArgWords) / kMoveWords, w = (i - 2 - kArgWords) - p * kMoveWords;
            reinterpret_cast<unsigned long long *>(&u.args[p])[w] =
                reinterpret_cast<const unsigned long long *>(&run->a[p])[w];
        }
    }
    __syncthreads();
    const int nj = __builtin_amdgcn_readfirstlane(static_cast<int>(head[1] & 0xffffffffull));
    if (q >= nj) return;
    const unsigned lo = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(head[0] & 0xffffffffull));
    const unsigned hi = __builtin_amdgcn_readfirstlane(static_cast<unsigned>(head[0] >> 32));
    using Const = const DevBox __attribute__((address_space(4)));
    const DevBox &b = *(const DevBox *)(Const *)((static_cast<unsigned long long>(hi) << 32) | lo);
    if (nj > 1)
        for (int i = threadIdx.x; i < kArgWords; i += blockDim.x)
            reinterpret_cast<unsigned long long *>(&b.sargs[q])[i] =
                reinterpret_cast<const unsigned long long *>(&u.args[q])[i];
    const SearchArgs &a = u.args[q];
    run_steps<false>(b, u, a, q, nj, a.run_dirty, 0u, 1u, [&](int p) -> const SearchArgs & { return u.args[p]; },
              [&] {
                  if (nj > 1)
                      for (int i = threadIdx.x; i < nj * kArgWords; i += blockDim.x)
                          reinterpret_cast<unsigned long long *>(u.args)[i] =
                              reinterpret_cast<const unsigned long long *>(b.sargs)[i];
              });
}

// Persistent form of k_step for one box: a resident grid takes the queued
// steps from a ring in pinned host memory, in order, instead of one launch
// per step.  Block 0 alone polls the ring; it copies job k into device memory
// (the box's eng_jobs slot) and publishes its decision for k (run, exit, or
// quit after idle_ticks of clock without a job) in eng_decision; the other
// blocks wait for that decision, which usually comes while the previous step
// still runs.  Each block then loads what the step reads of the mover (no
// queued step changes it unless it closes the gate) and waits until the last
// step that ran is done: its finishing block writes eng_done = 2 k + (1 if it
// closed the gate) after the step's device writes and before it publishes the
// record to the host, so the next step starts one host round trip earlier.
// Every engine step is gated and its released floor never decreases, so a
// step is behind the gate exactly when the last step that ran closed it and
// was not released by it; the first step of a launch reads the gate itself.
// Blocks beyond a job's share of the grid (vg) follow the steps without work.
// Every wait is bounded (a wait that runs out ends the grid and reports reason
// -1), so the grid always ends.
constexpr unsigned long long kEngineWaitFactor = 8;  // a block's wait for the others: 8 idle periods

__device__ __forceinline__ void copy_words(unsigned long long *dst, const unsigned long long *src, int n) {
    for (int i = threadIdx.x; i < n; i += blockDim.x) dst[i] = src[i];
}

__global__ __launch_bounds__(kBlock) void k_step_engine(DevBox b, const EngineJob *ring, EngineCtl *ctl,
                                                        unsigned long long first, unsigned long long idle_ticks,
                                                        unsigned long long launch_no) {
    __shared__ EngineJob job;
    __shared__ int s_cmd, s_run;
    constexpr int kJobWords = static_cast<int>(offsetof(EngineJob, seq) / sizeof(unsigned long long));
    static_assert(offsetof(EngineJob, seq) % sizeof(unsigned long long) == 0, "job body in 8-byte words");
    SearchState *s = b.ss;
    unsigned long long last = 0;      // the last job that ran in this launch (0: none yet)
    unsigned long long last_seq = 0;  // its step's sequence number
    unsigned long long busy = 0, idle = 0, steps = 0;
    unsigned long long k = first;
    int reason = kEngineExit;
    for (;; ++k) {
        const int slot = static_cast<int>(k % kEngineRing);
        if (threadIdx.x == 0) {
            const unsigned long long t0 = wall_clock64();
            int cmd = -1;
            if (blockIdx.x == 0) {
                cmd = kEngineQuit;
                while (wall_clock64() - t0 <= idle_ticks) {
                    if (__hip_atomic_load(&ring[slot].seq, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM) == k) {
                        cmd = ring[slot].cmd == kEngineExit ? kEngineExit : kEngineRun;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                idle += wall_clock64() - t0;
            } else {
                const unsigned long long limit = kEngineWaitFactor * idle_ticks;
                while (wall_clock64() - t0 <= limit) {
                    const unsigned long long d =
                        __hip_atomic_load(&s->eng_decision, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
                    if ((d >> 2) > k) {  // block 0 has gone on: job k ran
                        cmd = kEngineRun;
                        break;
                    }
                    if ((d >> 2) == k && (d & 3ull) != 0ull) {
                        cmd = static_cast<int>(d & 3ull);
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
            }
            s_cmd = cmd;
        }
        __syncthreads();
        const int cmd = s_cmd;
        if (blockIdx.x == 0) {
            if (cmd == kEngineRun) {
                copy_words(reinterpret_cast<unsigned long long *>(&job),
                           reinterpret_cast<const unsigned long long *>(&ring[slot]), kJobWords);
                __syncthreads();
                copy_words(reinterpret_cast<unsigned long long *>(&b.eng_jobs[slot]),
                           reinterpret_cast<const unsigned long long *>(&job), kJobWords);
                __syncthreads();
            }
            if (threadIdx.x == 0) {
                __threadfence();  // the job copy before the decision
                __hip_atomic_store(&s->eng_decision, k * 4ull + static_cast<unsigned long long>(cmd),
                                   __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            }
        } else if (cmd == kEngineRun) {
            copy_words(reinterpret_cast<unsigned long long *>(&job),
                       reinterpret_cast<const unsigned long long *>(&b.eng_jobs[slot]), kJobWords);
            __syncthreads();
        }
        if (cmd != kEngineRun) {
            reason = cmd;
            break;
        }
        const unsigned vg = job.vg < 1 ? 1u : (job.vg > static_cast<int>(gridDim.x) ? gridDim.x : static_cast<unsigned>(job.vg));
        const bool works = blockIdx.x < vg;
        const SearchArgs a = job.a;  // in registers for the step, as a launch's kernel arguments are
        StepPrefetch pre{};
        if (works) pre = prefetch_step(b, a);  // in flight during the wait below
        unsigned long long t_start = 0;
        if (threadIdx.x == 0) {
            int run = 1;
            if (last == 0) {
                run = behind_gate(b, a) ? 0 : 1;
            } else {
                const unsigned long long t0 = wall_clock64(), limit = kEngineWaitFactor * idle_ticks;
                unsigned long long w = 0;
                run = -1;
                while (wall_clock64() - t0 <= limit) {
                    w = __hip_atomic_load(&s->eng_done, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
                    if ((w >> 1) >= last) {
                        run = 1;
                        break;
                    }
                    __builtin_amdgcn_s_sleep(1);
                }
                if (run == 1 && (w >> 1) > last) {
                    // later steps ran without this block: the word of `last` is in its slot
                    w = __hip_atomic_load(&b.eng_closed[last % kEngineRing], __ATOMIC_RELAXED,
                                          __HIP_MEMORY_SCOPE_AGENT);
                    if ((w >> 1) != last) run = -1;
                }
                if (run == 1) {
                    // behind_gate with the gate closed by `last` (or open)
                    const bool closed = (w & 1ull) != 0ull;
                    run = (a.gated && closed && last_seq > a.released) ? 0 : 1;
                }
            }
            t_start = wall_clock64();
            s_run = run;
        }
        __syncthreads();
        const int run = s_run;
        if (run < 0) {
            reason = -1;
            break;
        }
        if (!run) continue;  // behind the gate: no block works on it, no record
        last = k;
        last_seq = a.seq;
        if (!works) continue;
        const CellTable *ct = job.cells.n > 0 ? &job.cells : nullptr;
        int role = 0;
        __shared__ int s_role;
        const bool closed = step_body<false>(b, a, blockIdx.x, vg, true, ct, false, &s_role, &pre);
        __syncthreads();
        role = s_role;
        if (role == 2 && threadIdx.x == 0) {
            // the step's device writes, then eng_done for the other blocks,
            // then the record for the host
            const unsigned long long word = (k << 1) | (closed ? 1ull : 0ull);
            b.eng_closed[slot] = word;
            __threadfence();
            __hip_atomic_store(&s->eng_done, word, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
            __threadfence_system();
            __hip_atomic_store(&a.out->seq, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            busy += wall_clock64() - t_start;
            steps += 1;
        }
    }
    if (threadIdx.x == 0) {
        if (steps) {
            atomicAdd(&s->eng_steps, steps);
            atomicAdd(&s->eng_busy, busy);
        }
        if (blockIdx.x == 0) atomicAdd(&s->eng_idle, idle);
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        ctl->stopped_at = k;
        ctl->reason = reason;
        __threadfence_system();
        __hip_atomic_store(&ctl->launches_ended, launch_no, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    } else if (reason == -1 && threadIdx.x == 0) {
        ctl->reason = -1;
        __threadfence_system();
    }
}

// a13 for a large mover: sphere positions from the refpos of the last search.
__global__ __launch_bounds__(kBlock) void k_translate(DevBox b, int src, int gated, unsigned long long seq,
                                                      unsigned long long released) {
    const SearchState *s = b.ss;
    const unsigned long long g = s->gate;
    if (gated && g != 0ull && g < seq && g > released) return;  // the step was skipped
    const int n = b.acount[src];
    const int st = b.astart[src];
    const double r0 = s->refpos[0], r1 = s->refpos[1], r2 = s->refpos[2];
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) {
        int sp = b.members[st + t];
        b.sx[sp] = r0 + b.srx[sp];
        b.sy[sp] = r1 + b.sry[sp];
        b.sz[sp] = r2 + b.srz[sp];
    }
}

// Aggregate::translate by a given vector: new position, cell and refpos.
__global__ void k_set_move(DevBox b, int src, double v0, double v1, double v2, int n_div, double L) {
    SearchState *s = b.ss;
    const double v[3] = {v0, v1, v2};
    const double old[3] = {b.ax[src], b.ay[src], b.az[src]};
    const double rc3[3] = {b.arx[src], b.ary[src], b.arz[src]};
    for (int l = 0; l < 3; ++l) {
        s->newcom[l] = periodic_position(old[l] + v[l], L);
        s->refpos[l] = s->newcom[l] - rc3[l];
    }
    s->newcell = ref_cell(s->newcom[0], s->newcom[1], s->newcom[2], n_div, L);
    b.ax[src] = s->newcom[0];
    b.ay[src] = s->newcom[1];
    b.az[src] = s->newcom[2];
    b.acell[src] = s->newcell;
    mark_dirty(b, src);
    set_dirty_entry(b, b.dslot[src], s->newcom[0], s->newcom[1], s->newcom[2], b.armax[src], s->newcell);
    b.dinfo[b.dslot[src]] = entry_info(b, src);
}

__global__ void k_swept_batch(long long n, const double *p1, const double *r1, const double *p2, const double *r2,
                              const double *dir, const double *dist, double L, double *out) {
    for (long long i = blockIdx.x * static_cast<long long>(blockDim.x) + threadIdx.x; i < n;
         i += static_cast<long long>(gridDim.x) * blockDim.x)
        out[i] = swept_sphere(p1[3 * i], p1[3 * i + 1], p1[3 * i + 2], r1[i], p2[3 * i], p2[3 * i + 1], p2[3 * i + 2],
                              r2[i], dir[3 * i], dir[3 * i + 1], dir[3 * i + 2], dist[i], L);
}

}  // namespace mcac_dev
