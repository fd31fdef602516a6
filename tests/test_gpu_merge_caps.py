"""Merges with spherical caps in one workgroup, at the edges of its waves and
contact words: the merge in a step's own launch and the one called after it
against the sequence of kernels over rows in memory, bit for bit."""
import math

import numpy as np
import pytest

from test_gpu_merge_sizes import chain

pytestmark = pytest.mark.gpu


def merged(na, nb, close, sequence, in_launch, monkeypatch):
    import mcac_amd
    monkeypatch.setenv("MCAC_FUSED_MERGE", "0" if sequence else "1")
    rng = np.random.default_rng([na, nb, int(10 * close)])
    n, L, gap = na + nb, 2e-5, 3e-8
    r = rng.uniform(0.8, 1.4, n) * 1e-8
    a, b = chain(na, r[:na], rng, close), chain(nb, r[na:], rng, close)
    a0 = np.array([5e-6, 6e-6, 7e-6])
    i, j = int(np.argmax(a[:, 0])), int(np.argmin(b[:, 0]))
    b0 = a[i] + a0 + np.array([r[i] + r[na + j] + gap, 0.0, 0.0]) - b[j]
    xyz, rel = np.concatenate([a + a0, b + b0]), np.concatenate([a, b])
    vol, surf = 4 / 3 * math.pi * r ** 3, 4 * math.pi * r ** 2
    parts = [slice(0, na), slice(na, n)]
    rcm = np.array([(vol[s, None] * rel[s]).sum(0) / vol[s].sum() for s in parts])
    rmax = np.array([(np.linalg.norm(rel[s] - c, axis=1) + r[s]).max() for s, c in zip(parts, rcm)])
    box = mcac_amd.Box(L, 4, n, 2, volsurf=1)
    box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=vol, surf=surf, rx=rel[:, 0], ry=rel[:, 1],
                    rz=rel[:, 2]),
               dict(pos=np.array([a0, b0]) + rcm, rcm=rcm, rmax=rmax, volume=np.array([vol[s].sum() for s in parts]),
                    surface=np.array([surf[s].sum() for s in parts]), count=np.array([na, nb]), members=np.arange(n)))
    if in_launch:
        assert mcac_amd.load_gpu().mcac_box_merge_in_launch(box.h, 1) == 0
        hit, _ = box.move_result(box.move_enqueue(1, [-1.0, 0.0, 0.0], 4 * gap, float(rmax.max())))
    else:
        hit = box.next_contact(1, [-1.0, 0.0, 0.0], 4 * gap, float(rmax.max()), move=True)
    assert hit["contact"] == 1
    try:
        got = box.merge(hit)
    except mcac_amd.MCACError as e:  # a sphere with more contacts than its row holds
        box.close()
        return str(e)
    out = (got, box.spheres(), box.aggregates(), box.members(0))
    box.close()
    return out


@pytest.mark.parametrize("close", [0.95, 0.55])
@pytest.mark.parametrize("na,nb", [(1, 1), (31, 1), (32, 1), (1, 32), (40, 25), (64, 64), (127, 129), (255, 1)])
@pytest.mark.parametrize("in_launch", [False, True])
def test_caps_merge_equals_the_kernel_sequence(na, nb, close, in_launch, monkeypatch):
    print(f"case: {na} + {nb} spheres, spacing {close}, in launch {in_launch}", flush=True)
    want = merged(na, nb, close, True, False, monkeypatch)
    got = merged(na, nb, close, False, in_launch, monkeypatch)
    if isinstance(want, str):  # refused by both
        assert got == want
        return
    assert want[0]["merged"] == 1
    for f in want[0].dtype.names:
        assert np.array_equal(got[0][f], want[0][f]), f
    for g, w in zip(got[1:3], want[1:3]):
        for f in w:
            assert np.array_equal(g[f], w[f]), f
    assert np.array_equal(got[3], want[3])
