"""Merges of more spheres than one workgroup holds, at the edges of their tiles:
every value bit for bit against the sums taken in order, twice on one box (the
second merge finds the first one's scratch cleared)."""
import math

import numpy as np
import pytest

import oracle_lib
from test_gpu_merge_sizes import chain, expected

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [2e-5, 1e-4])  # in the large box rounding may part the spheres again: no merge then
@pytest.mark.parametrize("close", [1.0, 0.2, 0.1])  # 0.1: more contacts of a sphere than its row holds
@pytest.mark.parametrize("na,nb", [(200, 57), (256, 256), (1, 512), (511, 2), (300, 341), (1100, 260)])
def test_large_merge_equals_sums_in_order(na, nb, close, L):
    import mcac_amd
    print(f"case: {na} + {nb} spheres, spacing {close}, box {L}", flush=True)
    rng = np.random.default_rng([na, nb, int(100 * close)])
    n, gap = na + nb, 3e-8
    r = rng.uniform(0.8, 1.4, n) * 1e-8
    a, b = chain(na, r[:na], rng, close), chain(nb, r[na:], rng, close)
    a0 = np.array([0.4, 0.5, 0.6]) * L
    i, j = int(np.argmax(a[:, 0])), int(np.argmin(b[:, 0]))
    b0 = a[i] + a0 + np.array([r[i] + r[na + j] + gap, 0.0, 0.0]) - b[j]
    xyz, rel = np.concatenate([a + a0, b + b0]), np.concatenate([a, b])
    vol, surf = 4 / 3 * math.pi * r ** 3, 4 * math.pi * r ** 2
    parts = [slice(0, na), slice(na, n)]
    rcm = np.array([(vol[s, None] * rel[s]).sum(0) / vol[s].sum() for s in parts])
    rmax = np.array([(np.linalg.norm(rel[s] - c, axis=1) + r[s]).max() for s, c in zip(parts, rcm)])
    v0 = expected(rel[:na], r[:na], vol[:na], surf[:na])
    box = mcac_amd.Box(L, 4, n, 2)
    for again in range(2):
        box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=vol, surf=surf, rx=rel[:, 0], ry=rel[:, 1],
                        rz=rel[:, 2]),
                   dict(pos=np.array([a0, b0]) + rcm, rcm=rcm, rmax=rmax,
                        volume=np.array([v0["volume"], vol[na:].sum()]),
                        surface=np.array([v0["surface"], surf[na:].sum()]), count=np.array([na, nb]),
                        members=np.arange(n)))
        hit = box.next_contact(1, [-1.0, 0.0, 0.0], 4 * gap, float(rmax.max()), move=True)
        assert hit["contact"] == 1
        sph = box.spheres()
        at = np.stack([sph["x"], sph["y"], sph["z"]], axis=1)
        ms, os_ = int(hit["moving_sphere"]), int(hit["other_sphere"])
        touch = oracle_lib.contact(at[ms], r[ms], at[os_], r[os_], L)
        got = box.merge(hit)
        assert got["merged"] == int(touch)
        if not touch:
            assert box.aggregates()["count"].tolist() == [na, nb]
            continue
        assert got["n"] == n
        sph = box.spheres()
        new = np.stack([sph["rx"], sph["ry"], sph["rz"]], axis=1)
        assert np.array_equal(new[:na], rel[:na])
        ref = expected(new, r, vol, surf)
        for k in ("volume", "surface", "radius_sum", "rmax", "rg", "overlapping", "coordination"):
            assert got[k] == ref[k], (again, k, got[k], ref[k])
        assert tuple(got["rcm"].tolist()) == ref["rcm"]
        assert np.array_equal(box.members(0), np.arange(n))
        agg = box.aggregates()
        assert agg["rmax"][0] == ref["rmax"] and agg["rg"][0] == ref["rg"]
    box.close()
