"""Grouped moves of boxes whose spheres have grown (the host no longer knows where
their aggregates are) share launches, and give what the same moves give one at a
time, bit for bit; beside boxes that have not, and up to a move that is refused."""
import ctypes

import numpy as np
import pytest

from test_gpu_pair_solve import make_box
from test_gpu_steps_in_one_launch import enqueue

pytestmark = pytest.mark.gpu


def grow(L, m, box, dr):
    out = [np.zeros(box.n_aggs) for _ in range(5)]
    assert L.mcac_box_grow(box.h, ctypes.c_double(dr), *[m._dp(v) for v in out]) == 0


@pytest.mark.parametrize("sizes", [(1,) * 40, (1, 2, 1, 70, 3, 1), (130, 9, 131, 1, 4), (2,) * 600])
@pytest.mark.parametrize("k,n_boxes", [(1, 1), (1, 6), (2, 6), (8, 3), (8, 1)])
def test_grown_boxes_share_launches(sizes, k, n_boxes):
    import mcac_amd as m
    print(f"case: {n_boxes} boxes of {len(sizes)} aggregates, {k} moves each", flush=True)
    L, group = m.load_gpu(), ctypes.c_void_p()
    side = 6e-7 * len(sizes) ** (1 / 3)
    assert L.mcac_group_create(0, n_boxes, ctypes.byref(group)) == 0
    pairs, stats = [], np.zeros(3, np.int64)
    try:
        for i in range(n_boxes):
            made = [make_box(sizes, side, np.random.default_rng([len(sizes), i]), 0) for _ in range(2)]
            pairs.append((made[0][0], made[1][0], 1.1 * made[0][3]))
            assert L.mcac_group_add(group, made[0][0].h) == 0
        maxr = max(p[2] for p in pairs)
        rng = np.random.default_rng([k, n_boxes, len(sizes)])
        launches = 0
        for _ in range(3):
            for box, one, _ in pairs:
                for b in (box, one):
                    grow(L, m, b, 1e-10)
            aggs = rng.integers(0, min(len(sizes), 6), (n_boxes, k))
            dirs = rng.normal(size=(n_boxes, k, 3))
            dirs /= np.linalg.norm(dirs, axis=2)[..., None]
            lpm = rng.uniform(0.02, 0.2, (n_boxes, k)) * side
            t = enqueue(L, m, group, [p[0] for p in pairs for _ in range(k)], aggs.ravel(), dirs.reshape(-1, 3),
                        lpm.ravel(), maxr)
            assert L.mcac_group_stats(group, m._ip(stats)) == 0
            launches += k  # a move of each box a launch
            if n_boxes > 1:
                assert (stats[0], stats[1], stats[2]) == (launches, launches * n_boxes, 0)
            for i, (box, one, _) in enumerate(pairs):
                stopped = False
                for q in range(k):
                    got, skipped = box.move_result(t[i * k + q])
                    assert (skipped == 1) == stopped
                    if skipped == 1:
                        continue
                    ref = one.next_contact(int(aggs[i, q]), dirs[i, q], float(lpm[i, q]), maxr, move=True)
                    for f in ("distance", "move", "moving_sphere", "other_sphere", "other_agg", "contact", "n_query",
                              "n_filtered", "n_pairs"):
                        assert got[f] == ref[f], (q, f, got[f], ref[f])
                    stopped = bool(ref["contact"]) or skipped == 2
                if stopped:
                    box.release()
        for box, one, _ in pairs:
            for ga, gb in ((one.spheres(), box.spheres()), (one.aggregates(), box.aggregates())):
                for f in ga:
                    assert np.array_equal(ga[f], gb[f]), f
    finally:
        for box, one, _ in pairs:
            box.close()
            one.close()
        L.mcac_group_destroy(group)


@pytest.mark.parametrize("bad", [None, 2, 9, 13])
def test_grown_boxes_beside_others(bad):
    """Four boxes with four moves each, every other one grown: all run, or those before
    the move that is refused do."""
    import mcac_amd as m
    print(f"case: grown boxes beside others, refused move {bad}", flush=True)
    L, group, k, n = m.load_gpu(), ctypes.c_void_p(), 4, 30
    side = 2e-6
    assert L.mcac_group_create(0, 4, ctypes.byref(group)) == 0
    pairs = []
    for i in range(4):
        made = [make_box((1,) * n, side, np.random.default_rng(i), 0) for _ in range(2)]
        pairs.append((made[0][0], made[1][0], made[0][3]))
        assert L.mcac_group_add(group, made[0][0].h) == 0
        if i % 2:
            for b in pairs[-1][:2]:
                grow(L, m, b, 1e-10)
    maxr = 1.1 * max(p[2] for p in pairs)
    rng = np.random.default_rng(3)
    aggs = rng.integers(0, n, 4 * k)
    dirs = rng.normal(size=(4 * k, 3))
    dirs /= np.linalg.norm(dirs, axis=1)[:, None]
    lpm = np.full(4 * k, 1e-9)
    if bad is not None:
        aggs[bad] = n
    arr = (ctypes.c_void_p * (4 * k))(*[pairs[i // k][0].h for i in range(4 * k)])
    t = (ctypes.c_uint64 * (4 * k))()
    rc = L.mcac_move_enqueue_group(group, arr, m._ip(aggs), m._dp(dirs.ravel()), m._dp(lpm), m._dp(np.full(4 * k, maxr)),
                                   4 * k, t)
    assert rc == (0 if bad is None else 34)
    for i in range(4 * k if bad is None else bad):
        box, one, _ = pairs[i // k]
        got, skipped = box.move_result(t[i])
        assert skipped == 0
        ref = one.next_contact(int(aggs[i]), dirs[i], float(lpm[i]), maxr, move=True)
        assert got["distance"] == ref["distance"] and got["contact"] == ref["contact"] == 0
    for box, one, _ in pairs:
        if bad is not None:  # nothing else is in flight
            assert L.mcac_box_spare_moves(box.h) == 16
        for f, v in one.spheres().items():
            assert np.array_equal(v, box.spheres()[f]), f
        box.close()
        one.close()
    L.mcac_group_destroy(group)
