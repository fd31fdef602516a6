"""Contacts, merges and hand-overs inside a launch of several steps, and boxes
whose member pool was compacted, against the same moves one at a time (or on a
box with room in its pool), bit for bit."""
import ctypes
import functools

import numpy as np
import pytest

from test_gpu_merge_caps import merged
from test_gpu_pair_solve import make_box
from test_gpu_steps_in_one_launch import enqueue

pytestmark = pytest.mark.gpu

FIELDS = ("distance", "move", "moving_sphere", "other_sphere", "other_agg", "contact", "n_query", "n_filtered", "n_pairs")


def enqueue_run(m, box, aggs, dirs, lpm, maxr):
    L, n = m.load_gpu(), len(aggs)
    f = L.mcac_move_enqueue_run
    f.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int64), ctypes.POINTER(ctypes.c_double),
                  ctypes.POINTER(ctypes.c_double), ctypes.c_double, ctypes.c_int, ctypes.POINTER(ctypes.c_uint64)]
    t = (ctypes.c_uint64 * n)()
    assert f(box.h, m._ip(np.asarray(aggs, np.int64)), m._dp(np.ascontiguousarray(dirs, np.float64).ravel()),
             m._dp(np.asarray(lpm, np.float64)), maxr, n, t) == 0
    return list(t)


def same_state(a, b):
    for x, y in ((a.spheres(), b.spheres()), (a.aggregates(), b.aggregates())):
        for f in x:
            assert np.array_equal(x[f], y[f]), f


def read_run(box, one, t, aggs, dirs, lpm, maxr):
    """Results of a run in order against single moves; the contact (or None), its
    place in the run and whether a step was handed over."""
    hit, at, over, stopped = None, -1, False, False
    for q, ticket in enumerate(t):
        got, skipped = box.move_result(ticket)
        assert (skipped == 1) == stopped
        if skipped == 1:
            continue
        ref = one.next_contact(int(aggs[q]), dirs[q], float(lpm[q]), maxr, move=True)
        for f in FIELDS:
            assert got[f] == ref[f], (q, f, got[f], ref[f])
        if ref["contact"]:
            hit, at = (got, ref), q
        over = over or skipped == 2
        stopped = bool(ref["contact"]) or skipped == 2
    return hit, at, over


@pytest.mark.parametrize("volsurf", [0, 1])
@pytest.mark.parametrize("size", [1, 3])
def test_contacts_behind_moves_of_the_same_launch(size, volsurf, monkeypatch):
    import mcac_amd as m
    print(f"case: aggregates of {size}, method {volsurf}", flush=True)
    monkeypatch.setattr(m, "Box", functools.partial(m.Box, volsurf=volsurf))
    n, side = 120, 4e-6
    made = [make_box((size,) * n, side, np.random.default_rng([size]), 0) for _ in range(2)]
    box, one, maxr = made[0][0], made[1][0], 8 * made[0][3]
    assert m.load_gpu().mcac_box_merge_in_launch(box.h, 1) == 0
    rng = np.random.default_rng([size, volsurf, 1])
    contacts, late = 0, {"neither": 0, "mover": 0, "target": 0, "both": 0}
    for _ in range(48):
        agg = one.aggregates()
        alive = np.nonzero(agg["count"] > 0)[0]
        mover, target, *rest = rng.permutation(alive)[:6]
        kind = rng.choice(list(late))
        early = [int(rest[0])] + [int(v) for v, k in ((mover, "mover"), (target, "target")) if kind in (k, "both")]
        aggs = early + [int(mover)] + [int(v) for v in rest[: 7 - len(early)]]
        dirs = rng.normal(size=(len(aggs), 3))
        dirs /= np.linalg.norm(dirs, axis=1)[:, None]
        lpm = np.full(len(aggs), 2e-9)
        pos = agg["pos"].copy()
        for a, d in zip(early, dirs):
            pos[a] += 2e-9 * d
        way = pos[target] - pos[mover]
        way -= side * np.round(way / side)
        j = len(early)
        lpm[j] = np.linalg.norm(way)
        dirs[j] = way / lpm[j]
        t = enqueue_run(m, box, aggs, dirs, lpm, maxr)
        hit, at, _ = read_run(box, one, t, aggs, dirs, lpm, maxr)
        if hit is None:
            continue
        contacts += 1
        if at == j and hit[1]["other_agg"] == target:
            late[kind] += 1
        outcome = []
        for b, c in ((box, hit[0]), (one, hit[1])):
            try:
                outcome.append(b.merge(c))
            except m.MCACError as e:
                outcome.append(str(e))
        box.release()
        if isinstance(outcome[1], str):
            assert outcome[0] == outcome[1]
            break
        for f in outcome[1].dtype.names:
            assert np.array_equal(outcome[0][f], outcome[1][f]), f
    same_state(one, box)
    stats = box.stats()
    print(f"  {contacts} contacts, {late}, {stats}", flush=True)
    assert all(v > 0 for v in late.values())
    assert stats["inline_merges"] == contacts and stats["launched_merges"] == 0
    box.close()
    one.close()


def line_box(n, blocked):
    """A mover, three monomers out of the way and n pairs of spheres on both sides of
    its way: their bounding spheres are on it, the spheres are not; at its end a monomer."""
    import mcac_amd
    L, r, gap = 1e-5, 1e-8, 5e-8
    pos, xyz, rel, rcm, count = [], [], [], [], []

    def add(com, offsets):
        pos.append(com)
        count.append(len(offsets))
        for o in offsets:
            xyz.append(np.add(com, o))
            rel.append(np.subtract(o, offsets[0]))
        rcm.append(np.subtract([0, 0, 0], offsets[0]))

    y = 0.5 * L
    add([0.1 * L, y, y], [(0, 0, 0)])
    for k in range(3):
        add([0.2 * L, y + 0.2 * L, 0.2 * L * (k + 1)], [(0, 0, 0)])
    for k in range(n):
        add([0.2 * L + 0.3 * L * (k + 0.5) / n, y, y], [(0, -gap, 0), (0, gap, 0)])
    if blocked:
        add([0.53 * L, y, y], [(0, 0, 0)])
    xyz, rel, count = np.array(xyz), np.array(rel), np.array(count, np.int64)
    S, A, v, s = len(xyz), len(count), 4 / 3 * np.pi * r ** 3, 4 * np.pi * r ** 2
    box = mcac_amd.Box(L, 4, S, A)
    box.upload(dict(x=xyz[:, 0], y=xyz[:, 1], z=xyz[:, 2], r=np.full(S, r), vol=np.full(S, v), surf=np.full(S, s),
                    rx=rel[:, 0], ry=rel[:, 1], rz=rel[:, 2]),
               dict(pos=np.array(pos), rcm=np.array(rcm), rmax=np.where(count > 1, gap + r, r), volume=v * count,
                    surface=s * count, count=count, members=np.arange(S)))
    return box, L, gap + r


@pytest.mark.parametrize("blocked", [0, 1])
@pytest.mark.parametrize("n", [64, 65, 150])
@pytest.mark.parametrize("before", [0, 3])
def test_hand_over_behind_moves_of_the_same_launch(n, blocked, before):
    import mcac_amd as m
    print(f"case: {n} pairs on the way, blocked {blocked}, {before} steps before", flush=True)
    (box, L, maxr), (one, _, _) = line_box(n, blocked), line_box(n, blocked)
    box.set_auto_merge(True)
    aggs = [0, 1, 4][:before] + [0] + [2, 3]  # the mover and a pair of the way move first
    dirs = np.tile([0.0, 0.0, 1.0], (len(aggs), 1))
    lpm = np.full(len(aggs), 1e-9)
    dirs[before], lpm[before] = [1.0, 0.0, 0.0], 0.45 * L
    t = enqueue_run(m, box, aggs, dirs, lpm, maxr)
    hit, at, over = read_run(box, one, t, aggs, dirs, lpm, maxr)
    survivors = n + blocked
    assert box.stats()["handover"] == (1 if survivors > 64 else 0)
    assert (hit is not None) == bool(blocked) and over == (survivors > 64 and not blocked)
    if blocked:
        assert at == before
        a, b = box.merge(hit[0]), one.merge(hit[1])
        for f in b.dtype.names:
            assert np.array_equal(a[f], b[f]), f
        assert box.stats()["inline_merges"] == 1
        box.release()
    t = enqueue_run(m, box, aggs[:before] + [2, 3], dirs[: before + 2] * 0 + [0.0, 1.0, 0.0], lpm[:before + 2] * 0 + 1e-9, maxr)
    read_run(box, one, t, aggs[:before] + [2, 3], np.tile([0.0, 1.0, 0.0], (before + 2, 1)), np.full(before + 2, 1e-9), maxr)
    same_state(one, box)
    box.close()
    one.close()


@pytest.mark.parametrize("na,nb", [(1, 1), (32, 1), (64, 64), (255, 1)])
@pytest.mark.parametrize("close", [0.95, 0.55])
def test_caps_contacts_merge_in_the_launch(na, nb, close, monkeypatch):
    import mcac_amd
    print(f"case: {na} + {nb} spheres with caps, spacing {close}", flush=True)
    seen, shut = [], mcac_amd.Box.close

    def close_box(self):
        if getattr(self, "h", None):
            seen.append(self.stats())
        shut(self)

    monkeypatch.setattr(mcac_amd.Box, "close", close_box)
    merged(na, nb, close, False, True, monkeypatch)
    assert seen[0]["inline_merges"] == 1 and seen[0]["launched_merges"] == 0


@pytest.mark.parametrize("auto", [0, 1])
def test_a_compacted_pool_serves_every_form(auto, monkeypatch):
    import mcac_amd as m
    print(f"case: member pool compacted, merges in the launch {auto}", flush=True)
    L, group, n, side, k = m.load_gpu(), ctypes.c_void_p(), 150, 2.5e-6, 4
    plain = m.Box
    assert L.mcac_group_create(0, 2, ctypes.byref(group)) == 0
    boxes = []
    for pool in (n + 8, 0):
        monkeypatch.setattr(m, "Box", functools.partial(plain, member_pool=pool))
        made = make_box((1,) * n, side, np.random.default_rng(5), 0)
        boxes.append(made[0])
        boxes[-1].set_auto_merge(bool(auto))
    small, roomy = boxes
    maxr, rng, after = 20 * made[3], np.random.default_rng([auto, 9]), 0
    grouped = False
    for turn in range(60):
        agg = roomy.aggregates()
        alive = np.nonzero(agg["count"] > 0)[0]
        pick = rng.permutation(alive)[: k + 1]
        way = agg["pos"][pick[1:]] - agg["pos"][pick[:-1]]
        way -= side * np.round(way / side)
        lpm = np.linalg.norm(way, axis=1)
        dirs = way / lpm[:, None]
        a, b = (x.next_contact(int(pick[0]), dirs[1], float(lpm[1]), maxr) for x in boxes)
        for f in FIELDS:
            assert a[f] == b[f], f
        if turn == 20:
            for x in boxes:
                assert L.mcac_group_add(group, x.h) == 0
            grouped = True
        if grouped:
            t = enqueue(L, m, group, [small] * k + [roomy] * k, np.tile(pick[:k], 2), np.tile(dirs[:k], (2, 1)),
                        np.tile(lpm[:k], 2), maxr)
            tickets = [t[:k], t[k:]]
        else:
            tickets = [enqueue_run(m, x, pick[:k], dirs[:k], lpm[:k], maxr) for x in boxes]
        hits = [None, None]
        for q in range(k):
            (ga, sa), (gb, sb) = (x.move_result(tickets[i][q]) for i, x in enumerate(boxes))
            assert sa == sb
            if sa == 1:
                continue
            for f in FIELDS:
                assert ga[f] == gb[f], f
            if ga["contact"]:
                hits = [ga, gb]
        if hits[0] is not None:
            ra, rb = (x.merge(h) for x, h in zip(boxes, hits))
            for f in rb.dtype.names:
                assert np.array_equal(ra[f], rb[f]), f
            for x in boxes:
                x.release()
            after += small.stats()["pool_compactions"] > 0
    same_state(roomy, small)
    print(f"  {small.stats()}, {roomy.stats()}, {after} merges after it", flush=True)
    assert small.stats()["pool_compactions"] > 0 and roomy.stats()["pool_compactions"] == 0 and after > 10
    small.close()
    roomy.close()
    L.mcac_group_destroy(group)
