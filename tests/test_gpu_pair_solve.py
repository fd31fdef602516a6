"""Pair solve of the survivors (solve_tile): the contact found equals, bit for
bit, the smallest of the exact swept-sphere distances over every sphere pair
(swept_sphere_batch, itself checked against the oracle), the first pair in
(i, j) order where two are equal.  Sizes at the edges of the mover and sphere
tiles, moves up to and past the range of the pre-test, a direction that is not
of unit length (no pre-test) and spheres stored one box length away."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def make_box(sizes, L, rng, shift):
    import mcac_amd
    xyz, rel, r, pos, rcm, rmax, vol_a, surf_a = [], [], [], [], [], [], [], []
    for n in sizes:
        ri = rng.uniform(0.8, 1.6, n) * 1e-8
        pi = rng.normal(size=(n, 3)) * 2.2e-8 * n ** 0.4
        com = rng.uniform(0, L, 3)
        vi = 4 / 3 * np.pi * ri ** 3
        p0 = pi - (vi[:, None] * pi).sum(0) / vi.sum() + com
        xyz.append(p0 + shift * L * rng.integers(-1, 2, 3))
        rel.append(p0 - p0[0])
        rcm.append(com - p0[0])
        r.append(ri)
        pos.append(com)
        rmax.append((np.linalg.norm(p0 - com, axis=1) + ri).max() * (1 + 1e-12))
        vol_a.append(vi.sum())
        surf_a.append((4 * np.pi * ri ** 2).sum())
    xyz, rel, r = np.concatenate(xyz), np.concatenate(rel), np.concatenate(r)
    sph = dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=4 / 3 * np.pi * r ** 3, surf=4 * np.pi * r ** 2,
               rx=rel[:, 0], ry=rel[:, 1], rz=rel[:, 2])
    agg = dict(pos=np.array(pos), rcm=np.array(rcm), rmax=np.array(rmax), volume=np.array(vol_a),
               surface=np.array(surf_a), count=np.array(sizes, np.int64), members=np.arange(len(r)))
    box = mcac_amd.Box(L, 4, len(r), len(sizes))
    box.upload(sph, agg)
    return box, xyz, r, max(rmax)


@pytest.mark.parametrize("sizes", [(1, 1, 1), (2, 3, 1), (5, 1, 64), (64, 63, 65), (65, 257, 2), (511, 40, 7),
                                   (512, 255, 256), (513, 256, 90), (130, 600, 129)])
@pytest.mark.parametrize("reach,scale,shift", [(0.1, 1.0, 0), (0.44, 1.0, 1), (0.8, 1.0, 0), (1.3, 1.0, 0),
                                               (0.2, 1.01, 0), (0.0, 1.0, 0)])
def test_contact_is_the_least_pair(sizes, reach, scale, shift):
    import mcac_amd
    print(f"case: sizes {sizes}, move {reach} L, |dir| {scale}, shift {shift}", flush=True)
    L = 1.5e-6
    rng = np.random.default_rng([sum(sizes), int(100 * reach), int(100 * scale), shift])
    found = 0
    for _ in range(3):
        box, xyz, r, rmax = make_box(sizes, L, rng, shift)
        first = np.concatenate([[0], np.cumsum(sizes)])
        for q in range(4):
            if q % 2:  # towards a sphere of another aggregate
                d = xyz[rng.integers(sizes[0], sum(sizes))] - xyz[rng.integers(sizes[0])]
                d -= L * np.round(d / L)
            else:
                d = rng.normal(size=3)
            d *= scale / np.linalg.norm(d)
            lpm = reach * L
            got = box.next_contact(0, d, lpm, rmax)
            best = (np.inf, -1, -1)
            # a survivor's bounding distance is below the move (aggregat_list.cpp:510-532): none at a zero move
            for k in range(1, len(sizes) if lpm > 0 else 1):
                i, j = np.meshgrid(np.arange(sizes[0]), np.arange(first[k], first[k + 1]), indexing="ij")
                i, j = i.ravel(), j.ravel()
                dist = mcac_amd.swept_sphere_batch(xyz[i], r[i], xyz[j], r[j], np.tile(d, (len(i), 1)),
                                                   np.full(len(i), lpm), L)
                w = int(np.argmin(dist))  # the first of equal minima, in (i, j) order
                if dist[w] < best[0]:
                    best = (float(dist[w]), int(i[w]), int(j[w]))
                elif dist[w] == best[0] and best[0] < np.inf:
                    best = (best[0], None, None)  # equal over two aggregates: their order decides
            assert got["distance"] == best[0]
            if best[0] < np.inf and best[1] is not None:
                assert (got["moving_sphere"], got["other_sphere"]) == best[1:]
                found += 1
        box.close()
    sys.stdout.flush()
    if reach > 0.9:  # past the largest distance of nearest images
        assert found > 0
