"""A search with more survivors than candidate_capacity is refused
(MCAC_E_CAPACITY), with up to as many it is answered, whichever form takes it:
one block, several, or steps queued in one launch."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def row(n, spare, capacity):
    """A mover and n monomers along its way (all of them survivors); spare more, out of
    the way but in the visited cells, so that the window takes several blocks."""
    import mcac_amd
    L, r = 1e-5, 1e-8
    rng = np.random.default_rng([n, spare])
    pos = np.full((1 + n + spare, 3), 0.5 * L)
    pos[0, 0] = 0.1 * L
    pos[1:1 + n, 0] = 0.2 * L + 0.4 * L * (np.arange(n) + 0.5) / n
    pos[1:1 + n, 1] += r
    pos[1 + n:, 0] = rng.uniform(0.1 * L, 0.7 * L, spare)
    pos[1 + n:, 1] += rng.uniform(0.05 * L, 0.15 * L, spare)
    m = len(pos)
    one = np.ones(m)
    box = mcac_amd.Box(L, 2, m, m, candidate_capacity=capacity)
    box.upload(dict(x=pos[:, 0], y=pos[:, 1], z=pos[:, 2], r=r * one, vol=4.2e-24 * one, surf=1.3e-15 * one,
                    rx=0 * one, ry=0 * one, rz=0 * one),
               dict(pos=pos, rcm=np.zeros((m, 3)), rmax=r * one, volume=4.2e-24 * one, surface=1.3e-15 * one,
                    count=np.ones(m, np.int64), members=np.arange(m)))
    return box, 0.55 * L, r


@pytest.mark.parametrize("spare", [0, 3000])
@pytest.mark.parametrize("capacity", [1, 8, 40, 63, 64, 65, 100])
def test_survivors_past_the_capacity_are_refused(capacity, spare):
    import mcac_amd
    for n in (capacity, capacity + 1):
        print(f"case: {n} survivors, capacity {capacity}, {spare} others", flush=True)
        auto, lpm, r = row(n, spare, 0)
        want = auto.next_contact(0, [1.0, 0.0, 0.0], lpm, r)
        assert want["n_filtered"] == n and want["contact"] == 1
        box, _, _ = row(n, spare, capacity)
        if n > capacity:
            with pytest.raises(mcac_amd.MCACError, match="status 33"):
                box.next_contact(0, [1.0, 0.0, 0.0], lpm, r)
        else:
            got = box.next_contact(0, [1.0, 0.0, 0.0], lpm, r)
            for f in want.dtype.names:
                assert got[f] == want[f], f
        auto.close()
        box.close()


@pytest.mark.parametrize("capacity", [8, 40])
def test_queued_steps_past_the_capacity_are_refused(capacity):
    import mcac_amd
    print(f"case: steps in one launch, capacity {capacity}", flush=True)
    box, lpm, r = row(capacity + 1, 0, capacity)
    L = mcac_amd.load_gpu()
    aggs, t = np.array([1, 2, 0, 3]), (ctypes.c_uint64 * 4)()
    dirs, lpms = np.tile([0.0, 1.0, 0.0], 4), np.full(4, 1e-9)
    dirs[6:9], lpms[2] = [1.0, 0.0, 0.0], lpm
    aggs, dirs, lpms = aggs.astype(np.int64), np.ascontiguousarray(dirs), np.ascontiguousarray(lpms)
    L.mcac_move_enqueue_run.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_double),
                                        ctypes.POINTER(ctypes.c_double), ctypes.c_double, ctypes.c_int,
                                        ctypes.POINTER(ctypes.c_uint64)]
    assert L.mcac_move_enqueue_run(box.h, mcac_amd._ip(aggs), mcac_amd._dp(dirs), mcac_amd._dp(lpms), r, 4, t) == 0
    assert box.move_result(t[0])[0]["contact"] == 0 and box.move_result(t[1])[0]["contact"] == 0
    with pytest.raises(mcac_amd.MCACError, match="status 33"):
        box.move_result(t[2])
    assert box.move_result(t[3])[1] == 1
    box.close()
