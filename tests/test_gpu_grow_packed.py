"""Surface growth of many aggregates, several to a wave, against the form with a
wave for each (the same aggregates in parts): bit for bit."""
import ctypes
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 7, 8, 9, 16, 31, 32, 33, 64, 65, 130]


@pytest.mark.parametrize("grow", [1, 0])
@pytest.mark.parametrize("n,wide", [(8193, 12), (9001, 5), (8200, 9)])  # wide: aggregates take the first sizes so many
def test_packed_growth_equals_a_wave_each(n, wide, grow):
    import mcac_amd
    print(f"case: {n} aggregates, {wide} sizes, grow {grow}", flush=True)
    rng = np.random.default_rng([n, wide])
    count = np.where(rng.random(n) < 0.06, rng.choice(SIZES[:wide], n), rng.integers(1, 6, n))
    S = int(count.sum())
    owner = np.repeat(np.arange(n), count)
    side = 21
    at = np.stack([np.arange(n) // side ** 2, np.arange(n) // side % side, np.arange(n) % side], 1) * 1e-7 + 2e-8
    rel = rng.normal(size=(S, 3)) * 2e-9
    r = rng.uniform(0.8, 1.4, S) * 1e-9
    vol, surf = 4 / 3 * math.pi * r ** 3, 4 * math.pi * r ** 2
    xyz = at[owner] + rel
    ptr = lambda a: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
    lib, got = mcac_amd.load_gpu(), []
    for parts in ([np.arange(n)], [np.arange(n // 2), np.arange(n // 2, n)]):
        box = mcac_amd.Box(side * 1e-7, 6, S, n)
        box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=r, vol=vol, surf=surf, rx=rel[:, 0], ry=rel[:, 1],
                        rz=rel[:, 2]),
                   dict(pos=at, rcm=np.zeros((n, 3)), rmax=np.full(n, 1e-8), volume=np.bincount(owner, vol),
                        surface=np.bincount(owner, surf), count=count, members=np.arange(S)))
        out = np.zeros((5, n))
        flags = np.zeros(n, np.int32)
        for ids in parts:
            ids = np.ascontiguousarray(ids, np.int64)
            rc = lib.mcac_box_grow_ids(box.h, ids.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), ctypes.c_int64(len(ids)),
                                       ctypes.c_double(1e-11), grow, ctypes.c_double(0.85e-9), 0,
                                       *[ptr(out[k]) for k in range(5)],
                                       flags.ctypes.data_as(ctypes.POINTER(ctypes.c_int32)))
            assert rc == 0
        got.append((out, flags, {**box.spheres(), **box.radii()}, box.aggregates()))
        box.close()
    (o1, f1, s1, a1), (o2, f2, s2, a2) = got
    assert np.array_equal(o1, o2) and (o1[0] > 0).all()
    assert np.array_equal(f1, f2) and 0 < f1.sum() < n
    for x, y in ((s1, s2), (a1, a2)):
        for k in x:
            assert np.array_equal(x[k], y[k]), k
    for a in (0, int(np.argmax(count)), n - 1):  # a sum against the list order
        v = 0.0
        for q in np.nonzero(owner == a)[0]:
            v += float(s1["vol"][q])
        assert o1[0][a] == v
