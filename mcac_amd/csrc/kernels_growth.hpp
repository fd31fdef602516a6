// Surface growth of every sphere and the whole-box aggregate update that
// follows it (calcul.cpp:155-205 with individual_surf_reactions off and
// full_aggregate_update_frequency 1, volsurf_method none):
//   Sphere::croissance_surface   sphere.cpp:113-120 (r + u_sg dt, 4/3 pi r^3, 4 pi r^2)
//   Aggregate::update            aggregat.cpp:284-288: compute_volume_surface
//                                (:321-390, sphere sums), compute_mass_center
//                                (:431-452), compute_max_radius (:453-464),
//                                compute_giration_radius (:465-483)
// A wave, or eight lanes of one, walk an aggregate's member list in chunks of as
// many spheres; every lane adds the chunk's terms in list order (broadcast by
// shuffles), so each sum is the reference's sequential FP64 sum.  The merge
// caches (sums the next merge continues) are rewritten from the grown spheres.
#pragma once
#include "kernels_common.hpp"

namespace mcac_dev {

constexpr double kVolumeFactorD = 4 * kPi / 3;  // constants.hpp:114
constexpr double kSurfaceFactorD = 4 * kPi;     // constants.hpp:115

struct GrowOut {
    double *vol, *surf, *rsum, *rg, *rmax;  // by position in ids
    int *flag;
};
constexpr int kGrowSmall = 1, kGrowSplit = 2, kGrowLeft = 4;

// One aggregate by kLanes lanes (aligned, all active): id at position at, with n > 0
// spheres in the segment st.  The contact search's copies of CoM and rmax follow
// in place: a dirty aggregate's dirty-list entry, or the packed cell entry of one
// still in the cell it was built in; kGrowLeft tells that its growth took it out of
// its built cell (the entry is stale: the cell list must be rebuilt before the
// next search).  With grow = 0 the spheres keep their radii, volumes and surfaces
// (the update alone); kGrowSmall tells that a sphere of the aggregate is at or
// below rp_min after growing (oxidation removes it).
template <int kLanes>
__device__ __forceinline__ void grow_one(const DevBox &b, int at, int id, int n, int st, double dr, int grow,
                                         double rp_min, double L, int n_div, const GrowOut &o) {
    const int lane = static_cast<int>(threadIdx.x & (kLanes - 1));
    // grow, then volume, surface, sum of vol * relative position, radius sum
    // and sum of vol * r^2 in list order
    double V = 0.0, S = 0.0, vx = 0.0, vy = 0.0, vz = 0.0, rs = 0.0, brg = 0.0;
    double r = 0.0, vol = 0.0, rx = 0.0, ry = 0.0, rz = 0.0;
    int small = 0, s0 = 0;
    for (int c0 = 0; c0 < n; c0 += kLanes) {
        const int i = c0 + lane;
        double surf = 0.0;
        r = vol = rx = ry = rz = 0.0;
        if (i < n) {
            const int s = b.members[st + i];
            if (c0 == 0) s0 = s;
            r = b.sr[s];
            rx = b.srx[s];
            ry = b.sry[s];
            rz = b.srz[s];
            if (grow) {
                r = r + dr;  // PhysicalModel::grow: r + u_sg * dt, dr = u_sg * dt
                const double r2 = r * r;
                const double r3 = r2 * r;
                vol = kVolumeFactorD * r3;
                surf = kSurfaceFactorD * r2;
                b.sr[s] = r;
                b.svol[s] = vol;
                b.ssurf[s] = surf;
            } else {
                vol = b.svol[s];
                surf = b.ssurf[s];
            }
            small |= (r <= rp_min) ? 1 : 0;
        }
        const double tx = rx * vol, ty = ry * vol, tz = rz * vol, t2 = vol * (r * r);
        const int m = (n - c0 < kLanes) ? n - c0 : kLanes;
        for (int j = 0; j < m; ++j) {
            V = V + __shfl(vol, j, kLanes);
            S = S + __shfl(surf, j, kLanes);
            vx = vx + __shfl(tx, j, kLanes);
            vy = vy + __shfl(ty, j, kLanes);
            vz = vz + __shfl(tz, j, kLanes);
            rs = rs + __shfl(r, j, kLanes);
            brg = brg + __shfl(t2, j, kLanes);
        }
    }
    const double cx = vx / V, cy = vy / V, cz = vz / V;  // r /= agregat_volume
    // distances to the centre of mass, rmax and sum of vol * dc^2 in list order
    double rmax = 0.0, arg = 0.0;
    for (int c0 = 0; c0 < n; c0 += kLanes) {
        const int i = c0 + lane;
        if (n > kLanes) {  // else still in registers
            r = vol = rx = ry = rz = 0.0;
            if (i < n) {
                const int s = b.members[st + i];
                rx = b.srx[s];
                ry = b.sry[s];
                rz = b.srz[s];
                r = b.sr[s];  // written above by this lane
                vol = b.svol[s];
            }
        }
        const double dx = rx - cx, dy = ry - cy, dz = rz - cz;
        const double dc = __builtin_sqrt(dx * dx + dy * dy + dz * dz);
        const double far = r + dc, term = vol * (dc * dc);
        const int m = (n - c0 < kLanes) ? n - c0 : kLanes;
        for (int j = 0; j < m; ++j) {
            rmax = smax(rmax, __shfl(far, j, kLanes));
            arg = arg + __shfl(term, j, kLanes);
        }
    }
    const double rg = __builtin_sqrt(__builtin_fabs((arg + 3. / 5. * brg) / V));
    int flag = 0;
    {
        const int base = static_cast<int>(threadIdx.x & 63) & ~(kLanes - 1);
        const unsigned long long mine = kLanes == 64 ? ~0ull : ((1ull << (kLanes & 63)) - 1ull) << base;
        if (__ballot(small) & mine) flag = kGrowSmall;
    }
    if (lane != 0) return;
    // set_position(sphere 0 + r_cm) wraps into the box (aggregat.cpp:109-118)
    const double px = periodic_position(b.sx[s0] + cx, L);
    const double py = periodic_position(b.sy[s0] + cy, L);
    const double pz = periodic_position(b.sz[s0] + cz, L);
    b.avol[id] = V;
    b.asurf[id] = S;
    b.csvx[id] = vx;
    b.csvy[id] = vy;
    b.csvz[id] = vz;
    b.csr[id] = rs;
    b.csvr2[id] = brg;
    b.arx[id] = cx;
    b.ary[id] = cy;
    b.arz[id] = cz;
    b.ax[id] = px;
    b.ay[id] = py;
    b.az[id] = pz;
    const int cell = ref_cell(px, py, pz, n_div, L);
    const int built = b.acell[id];
    b.acell[id] = cell;
    b.armax[id] = rmax;
    if (b.dirty[id]) {
        set_dirty_entry(b, b.dslot[id], px, py, pz, rmax, cell);
    } else {
        const int cs = b.cslot[id];
        if (cs >= 0 && cell == built) {
            b.cpx[cs] = px;
            b.cpy[cs] = py;
            b.cpz[cs] = pz;
            b.cpr[cs] = rmax;
            b.cf[cs] = make_float4(static_cast<float>(px), static_cast<float>(py), static_cast<float>(pz),
                                   static_cast<float>(rmax));
        } else {
            flag |= kGrowLeft;
        }
    }
    b.arg[id] = rg;
    o.vol[at] = V;
    o.surf[at] = S;
    o.rsum[at] = rs;
    o.rg[at] = rg;
    o.rmax[at] = rmax;
    o.flag[at] = flag;
}

// ids[0..n_ids) may hold dead ids (count 0): their outputs are not written.
// kLanes lanes an aggregate.  What bounds it is the chain of loads from an id to its
// spheres, so the more aggregates are under way the better: a wave for each while
// the chip holds them all at once (kGrowPacked), eight lanes beyond that if the
// aggregates are small (kGrowPackedMean spheres on average); those of more than
// kGrowWide spheres are left to the whole wave afterwards (else one large
// aggregate would end long after the rest).  A call's time, a wave each -> eight
// lanes: 100000 aggregates of 8 spheres 436 -> 307 us (this kernel 44 us of it, the
// copy back 79), 30000 of 16 201 -> 130, 10000 of 16 84 -> 59, 25000 of 32 244 ->
// 263, 9000 of 32 109 -> 143.
constexpr int kGrowPacked = 8192;  // aggregates: 256 compute units with 32 waves each
constexpr int kGrowPackedMean = 16;
constexpr int kGrowWide = 32;
template <int kLanes>
__global__ __launch_bounds__(kBlock) void k_grow_update(DevBox b, const int *ids, int n_ids, double dr, int grow,
                                                       double rp_min, double L, int n_div, GrowOut o) {
    const int at = static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) / kLanes);
    int id = 0, n = 0, st = 0;
    if (at < n_ids) {
        id = ids[at];
        n = b.acount[id];
        st = b.astart[id];
    }
    if constexpr (kLanes == 64) {
        if (n > 0) grow_one<64>(b, at, id, n, st, dr, grow, rp_min, L, n_div, o);
    } else {
        if (n > 0 && n <= kGrowWide) grow_one<kLanes>(b, at, id, n, st, dr, grow, rp_min, L, n_div, o);
        unsigned long long wide = __ballot(n > kGrowWide && (threadIdx.x & (kLanes - 1)) == 0);
        for (; wide != 0ull; wide &= wide - 1ull) {
            const int l = __ffsll(static_cast<long long>(wide)) - 1;
            grow_one<64>(b, __shfl(at, l, 64), __shfl(id, l, 64), __shfl(n, l, 64), __shfl(st, l, 64), dr, grow, rp_min,
                         L, n_div, o);
        }
    }
}

// Aggregate::split's question (aggregat.cpp:553-584) for each aggregate of
// ids: are its spheres one connected set under the contact test
// (sphere_distances.cpp:81-90)?  One wave per aggregate of at most 64
// spheres: lane i builds sphere i's contact bits, and the set reached from
// sphere 0 grows by wave-wide ORs until it stops.  o_flag[wave] |= kGrowSplit when the
// aggregate falls apart, or when it has more than 64 spheres (left to the host).
__global__ __launch_bounds__(kBlock) void k_connected(DevBox b, const int *ids, int n_ids, double L, int *o_flag) {
    const int wave = static_cast<int>((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
    const int lane = static_cast<int>(threadIdx.x & 63);
    if (wave >= n_ids) return;
    const int id = ids[wave];
    const int n = b.acount[id];
    if (n <= 1) return;
    if (n > 64) {
        if (lane == 0) o_flag[wave] |= kGrowSplit;
        return;
    }
    const int st = b.astart[id];
    double x = 0.0, y = 0.0, z = 0.0, r = 0.0;
    if (lane < n) {
        const int s = b.members[st + lane];
        x = b.sx[s];
        y = b.sy[s];
        z = b.sz[s];
        r = b.sr[s];
    }
    unsigned long long adj = 0ull;
    for (int j = 0; j < n; ++j) {
        const double xj = __shfl(x, j, 64), yj = __shfl(y, j, 64), zj = __shfl(z, j, 64), rj = __shfl(r, j, 64);
        if (lane < n && contact(x, y, z, r, xj, yj, zj, rj, L)) adj |= 1ull << j;
    }
    const unsigned long long all = (n == 64) ? ~0ull : ((1ull << n) - 1ull);
    unsigned long long reached = 1ull;
    for (int it = 0; it < n; ++it) {
        unsigned long long mine = ((reached >> lane) & 1ull) ? adj : 0ull;
        unsigned lo = static_cast<unsigned>(mine), hi = static_cast<unsigned>(mine >> 32);
        for (int m = 1; m < 64; m <<= 1) {
            lo |= __shfl_xor(lo, m, 64);
            hi |= __shfl_xor(hi, m, 64);
        }
        const unsigned long long next = reached | (static_cast<unsigned long long>(hi) << 32) | lo;
        if (next == reached) break;
        reached = next;
    }
    if (lane == 0 && (reached & all) != all) o_flag[wave] |= kGrowSplit;
}

}  // namespace mcac_dev
