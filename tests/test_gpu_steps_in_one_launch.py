"""Several steps of a box in one launch (k_steps, k_steps_group) give what the
same moves give one at a time: contacts, skipped steps behind a contact, and
the positions left behind, bit for bit.  Few aggregates in a box, so that steps
of one launch meet movers that moved before them in it, and the same aggregate
moves several times."""
import ctypes

import numpy as np
import pytest

from test_gpu_pair_solve import make_box

pytestmark = pytest.mark.gpu


def enqueue(L, m, group, boxes, aggs, dirs, lpm, maxr):
    n = len(boxes)
    arr = (ctypes.c_void_p * n)(*[b.h.value if hasattr(b.h, "value") else b.h for b in boxes])
    t = (ctypes.c_uint64 * n)()
    aggs, lpm = np.asarray(aggs, np.int64), np.asarray(lpm, np.float64)
    dirs, maxr = np.ascontiguousarray(dirs, np.float64).ravel(), np.full(n, maxr)
    assert L.mcac_move_enqueue_group(group, arr, m._ip(aggs), m._dp(dirs), m._dp(lpm), m._dp(maxr), n, t) == 0
    return list(t)


@pytest.mark.parametrize("n_boxes", [1, 3])
@pytest.mark.parametrize("k", [1, 2, 7, 8])
@pytest.mark.parametrize("sizes", [(1,) * 5, (1, 2, 1, 70, 3, 1), (300, 5, 260, 1), (1,) * 300, (3,) * 700])
def test_launch_equals_single_moves(sizes, k, n_boxes):
    import mcac_amd as m
    print(f"case: {len(sizes)} aggregates of {max(sizes)}, {k} steps a launch, {n_boxes} boxes", flush=True)
    L = m.load_gpu()
    side = 6e-7 * len(sizes) ** (1 / 3)
    pairs, group = [], ctypes.c_void_p()
    assert L.mcac_group_create(0, n_boxes, ctypes.byref(group)) == 0
    contacts = moved_twice = 0
    try:
        for i in range(n_boxes):
            made = [make_box(sizes, side, np.random.default_rng([len(sizes), max(sizes), i]), 0) for _ in range(2)]
            pairs.append((made[0][0], made[1][0], made[0][3]))
            assert L.mcac_group_add(group, made[0][0].h) == 0
        rng = np.random.default_rng([k, n_boxes, len(sizes)])
        for _ in range(6):
            moves = []
            for i in range(n_boxes):
                a = rng.integers(0, min(len(sizes), 6), k)  # a few movers: some move again in the launch
                moved_twice += len(set(a.tolist())) < k
                d = rng.normal(size=(k, 3))
                d /= np.linalg.norm(d, axis=1)[:, None]
                moves.append((a, d, rng.uniform(0.02, 0.25, k) * side))
            t = enqueue(L, m, group, [pairs[i][0] for i in range(n_boxes) for _ in range(k)],
                        np.concatenate([v[0] for v in moves]), np.concatenate([v[1] for v in moves]),
                        np.concatenate([v[2] for v in moves]), max(p[2] for p in pairs))
            for i in range(n_boxes):
                box, one, _ = pairs[i]
                stopped = False
                for q in range(k):
                    got, skipped = box.move_result(t[i * k + q])
                    assert (skipped == 1) == stopped
                    if skipped == 1:
                        continue
                    ref = one.next_contact(int(moves[i][0][q]), moves[i][1][q], float(moves[i][2][q]),
                                           max(p[2] for p in pairs), move=True)
                    for f in ("distance", "move", "moving_sphere", "other_sphere", "other_agg", "contact", "n_query",
                              "n_filtered", "n_pairs"):
                        assert got[f] == ref[f], (q, f, got[f], ref[f])
                    if ref["contact"] or skipped == 2:
                        contacts += int(ref["contact"])
                        stopped = True
                if stopped:
                    box.release()
        for box, one, _ in pairs:
            for f, v in one.spheres().items():
                assert np.array_equal(v, box.spheres()[f]), f
            ga, gb = one.aggregates(), box.aggregates()
            for f in ga:
                assert np.array_equal(ga[f], gb[f]), f
    finally:
        for box, one, _ in pairs:
            box.close()
            one.close()
        L.mcac_group_destroy(group)
    print(f"  {contacts} contacts", flush=True)
    if k > 2:
        assert moved_twice > 0
