"""Launch shapes planned for a whole batch (csrc/launch_plan.cpp), host only."""
import ctypes as C

import numpy as np
import pytest

from spand_public_amd import _lib

PANEL, TRAIL, SPLIT = range(3)


def plan_getrf(sizes):
    L = _lib.lib()
    n = np.ascontiguousarray(sizes, dtype=np.int32)
    call = lambda out, rows: L.spand_plan_getrf(n.ctypes.data_as(C.c_void_p), C.c_int(len(n)),
                                                out.ctypes.data_as(C.c_void_p), C.c_int(rows))
    rows = call(np.zeros(7, np.int32), 0)
    out = np.zeros((max(rows, 1), 7), np.int32)
    assert call(out, rows) == rows
    return out[:rows]


def batch(kind):
    rng = np.random.default_rng(5)
    if kind == "cube128":  # as many pivots as the level-0 scaling of a 128^3 grid, sizes like its
        return np.minimum(1 + rng.geometric(0.03, 77949), 140)
    if kind == "square2048":
        return np.minimum(1 + rng.geometric(0.15, 97539), 60)
    if kind == "one large":  # a short pivot still inside a narrower first panel when the form changes
        return np.r_[4096, 1030, rng.integers(1, 40, 70000)]
    if kind == "form change":
        return np.r_[1030, 20, 17, 16, 9, 8, 1, 33, 32, 31]
    return np.r_[np.full(200000, 65), 512] if kind == "many" else np.array([1])


@pytest.mark.parametrize("kind", ["cube128", "square2048", "one large", "form change", "many", "single"])
def test_lu_launches_fit_the_device_and_cover_every_pivot(kind):
    n = np.sort(batch(kind))[::-1]
    plan = plan_getrf(n)
    done = np.zeros(len(n), np.int64)     # columns factored so far
    trailed = np.zeros(len(n), np.int64)  # panels whose other columns were updated
    split = np.zeros(len(n), np.int64)
    for kind_, kb, nb, first, count, per_task, threads in plan.tolist():
        # along x only, and HIP's bound on the work items of a launch
        assert count > 0 and per_task > 0 and count * per_task * threads < 2 ** 32
        assert threads % 64 == 0 and 64 <= threads <= 1024
        at = slice(first, first + count)
        if kind_ == PANEL:
            assert (done[at] == kb).all() and (n[at] > kb).all()
            assert threads * (32 // nb) >= (n[at] - kb).max()
            done[at] = np.minimum(kb + nb, n[at])
            trailed[at] += (n[at] <= nb) & (kb == 0)  # no other column
        elif kind_ == TRAIL:
            assert per_task * 8 >= n[at].max()
            trailed[at] += 1
        else:
            assert (per_task >= ((n[at] + 31) // 32) ** 2).all() and (done[at] == n[at]).all()
            split[at] += 1
    assert (done == n).all() and (split == 1).all()
    panels = np.zeros(len(n), np.int64)
    for row in plan[plan[:, 0] == PANEL]:
        panels[row[3]:row[3] + row[4]] += 1
    assert (trailed == panels).all()


def plan_slabs(nsub, steps, cap):
    L = _lib.lib()
    nsub, steps = (np.ascontiguousarray(v, dtype=np.int32) for v in (nsub, steps))
    chunks, place = np.zeros((4096, 4), np.int32), np.zeros((1 << 18, 2), np.int32)
    np_ = C.c_int()
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    k = L.spand_plan_slabs(p(nsub), p(steps), C.c_int(len(nsub)), C.c_int(cap), p(chunks), C.c_int(len(chunks)),
                           p(place), C.c_int(len(place)), C.byref(np_))
    assert k <= len(chunks) and np_.value <= len(place)
    return chunks[:k].tolist(), place[:np_.value]


@pytest.mark.parametrize("cap", [8, 20, 64, 1000, 2048])
@pytest.mark.parametrize("kind", ["single", "mixed", "ordinary", "long"])
def test_persistent_rrqr_slabs_are_placed_once_and_waiting_ones_marked(kind, cap):
    """Each cluster whole in one launch of at most cap workgroups, on one XCD (workgroup modulo 8)
    unless none holds it. A launch in which a cluster has several slabs is one whose workgroups
    wait for each other: it has to be marked, because they have to be resident together."""
    rng = np.random.default_rng(cap)
    nsub = {"single": np.ones(300, int), "mixed": rng.choice([1, 1, 1, 2], 200), "ordinary": rng.integers(1, 9, 500),
            "long": rng.integers(1, max(2, cap + 1), 40)}[kind]
    steps = rng.integers(0, 300, len(nsub))
    chunks, place = plan_slabs(nsub, steps, cap)
    if nsub.max() > cap:
        assert not chunks
        return
    seen, at = [], 0
    for first, count, nsteps, waits in chunks:
        assert first == at and 0 < count <= cap
        at += count
        rows = place[first:first + count]
        used = np.flatnonzero(rows[:, 0] >= 0)
        here = np.unique(rows[used, 0])
        for c in here:
            mine = used[rows[used, 0] == c]
            assert sorted(rows[mine, 1]) == list(range(nsub[c]))  # the whole cluster, each slab once
            assert nsub[c] > cap // 8 or len(set(mine % 8)) == 1
        assert nsteps == steps[here].max() and bool(waits) == bool((nsub[here] > 1).any())
        seen += list(here)
    assert at == len(place) and sorted(seen) == list(range(len(nsub)))


def test_a_cluster_longer_than_the_device_is_not_planned():
    assert plan_slabs([3, 65, 2], [1, 1, 1], 64)[0] == []
