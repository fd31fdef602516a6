"""Merge of two aggregates in one workgroup at the edges of its waves, contact
words and contact list, against the reference's sums taken in its order in
Python floats (the same IEEE operations): every value bit for bit."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def chain(n, r, rng, close):
    """n spheres, each touching (or with close < 1 overlapping) the one before."""
    p, way = np.zeros((n, 3)), np.array([1.0, 0.0, 0.0])
    for i in range(1, n):
        way = way + 0.8 * rng.normal(size=3)
        way /= np.linalg.norm(way)
        p[i] = p[i - 1] + way * (r[i] + r[i - 1]) * close
    return p


def expected(rel, r, vol, surf):
    V = S = vx = vy = vz = sr = svr2 = 0.0
    for (x, y, z), ri, vi, si in zip(rel.tolist(), r.tolist(), vol.tolist(), surf.tolist()):
        V, S, sr = V + vi, S + si, sr + ri
        vx, vy, vz = vx + x * vi, vy + y * vi, vz + z * vi
        svr2 = svr2 + vi * (ri * ri)
    rcm = (vx / V, vy / V, vz / V)
    rmax, arg = 0.0, 0.0
    for (x, y, z), ri, vi in zip(rel.tolist(), r.tolist(), vol.tolist()):
        d0, d1, d2 = x - rcm[0], y - rcm[1], z - rcm[2]
        dc = math.sqrt(d0 * d0 + d1 * d1 + d2 * d2)
        rmax, arg = max(rmax, ri + dc), arg + vi * (dc * dc)
    over, inter = 0.0, 0
    q, rr = rel.tolist(), r.tolist()
    for i in range(len(q)):
        for j in range(i + 1, len(q)):
            d0, d1, d2 = q[i][0] - q[j][0], q[i][1] - q[j][1], q[i][2] - q[j][2]
            s2 = rr[i] + rr[j]
            d = math.sqrt(d0 * d0 + d1 * d1 + d2 * d2)
            if d <= (1. + 1e-10) * s2:
                over += 2.0 * ((s2 - d) / s2)
                inter += 2
    if inter:
        over /= float(inter)
    return dict(volume=V, surface=S, radius_sum=sr, rmax=rmax, rg=math.sqrt(abs((arg + 3. / 5. * svr2) / V)),
                overlapping=over, coordination=inter / float(len(q)) if inter else 0.0, rcm=rcm)


@pytest.mark.parametrize("close", [1.0, 0.2])  # 0.2: more contacts than the list in order holds
@pytest.mark.parametrize("na,nb", [(1, 1), (1, 30), (31, 1), (32, 1), (32, 33), (63, 2), (64, 64), (100, 93), (127, 129),
                                   (1, 255), (255, 1), (256, 1)])
def test_merge_equals_sums_in_order(na, nb, close):
    import mcac_amd
    print(f"case: {na} + {nb} spheres, spacing {close}", flush=True)
    rng = np.random.default_rng([na, nb, int(10 * close)])
    L = 2e-5
    r = rng.uniform(0.8, 1.4, na + nb) * 1e-8
    a, b = chain(na, r[:na], rng, close), chain(nb, r[na:], rng, close)
    a0 = np.array([5e-6, 6e-6, 7e-6])
    far = a[np.argmax(a[:, 0])] + a0  # the moving aggregate stops beside its outermost sphere
    i, j = int(np.argmax(a[:, 0])), int(np.argmin(b[:, 0]))
    gap = 3e-8
    b0 = far + np.array([r[i] + r[na + j] + gap, 0.0, 0.0]) - b[j]
    xyz = np.concatenate([a + a0, b + b0])
    rel = np.concatenate([a, b])
    vol, surf = 4 / 3 * math.pi * r ** 3, 4 * math.pi * r ** 2
    first = [slice(0, na), slice(na, na + nb)]
    rcm = np.array([(vol[s, None] * rel[s]).sum(0) / vol[s].sum() for s in first])
    pos = np.array([a0, b0]) + rcm
    rmax = np.array([(np.linalg.norm(rel[s] - c, axis=1) + r[s]).max() for s, c in zip(first, rcm)])
    box = mcac_amd.Box(L, 4, na + nb, 2)
    box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=vol, surf=surf, rx=rel[:, 0], ry=rel[:, 1],
                    rz=rel[:, 2]),
               dict(pos=pos, rcm=rcm, rmax=rmax, volume=np.array([vol[s].sum() for s in first]),
                    surface=np.array([surf[s].sum() for s in first]), count=np.array([na, nb]),
                    members=np.arange(na + nb)))
    # the volume and surface a merge continues are the uploaded ones: give it the ordered sums
    v0, s0 = expected(rel[:na], r[:na], vol[:na], surf[:na]), None
    box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=vol, surf=surf, rx=rel[:, 0], ry=rel[:, 1],
                    rz=rel[:, 2]),
               dict(pos=pos, rcm=rcm, rmax=rmax, volume=np.array([v0["volume"], vol[na:].sum()]),
                    surface=np.array([v0["surface"], surf[na:].sum()]), count=np.array([na, nb]),
                    members=np.arange(na + nb)))
    hit = box.next_contact(1, [-1.0, 0.0, 0.0], 4 * gap, float(rmax.max()), move=True)
    assert hit["contact"] == 1
    got = box.merge(hit)
    assert got["merged"] == 1 and got["n"] == na + nb
    sph = box.spheres()
    new = np.stack([sph["rx"], sph["ry"], sph["rz"]], axis=1)
    assert np.array_equal(new[:na], rel[:na])
    ref = expected(new, r, vol, surf)
    for k in ("volume", "surface", "radius_sum", "rmax", "rg", "overlapping", "coordination"):
        assert got[k] == ref[k], (k, got[k], ref[k])
    assert tuple(got["rcm"].tolist()) == ref["rcm"]
    assert np.array_equal(box.members(0), np.arange(na + nb))
    agg = box.aggregates()
    assert agg["count"].tolist() == [na + nb, 0] and agg["rmax"][0] == ref["rmax"] and agg["rg"][0] == ref["rg"]
    box.close()
