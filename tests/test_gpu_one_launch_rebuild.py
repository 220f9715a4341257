"""The rebuild kernel's phases (binning, scan, scatter, sort, reorder in one
launch) where its work splits differently: part-filled and single workgroups,
more cells than a workgroup sums the prefix of by itself, cells of more than a
wave's members, workgroups that came too late to take part.

Every step rebuilds and reorders (zero skin, sort at every build), so each phase
hands over to the next many times before the final cells, in-cell order and
neighbour sets are held bit for bit to the oracle's at the final positions.
"""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import BeadsError, Engine

pytestmark = pytest.mark.gpu


def _final_state(w, steps):
    with Engine(w) as e:
        e.initialize(observables=False)
        e.advance(steps)
        plan = O.plan(w)
        st, cells, stats = e.state(), e.cells(plan.n_cells), e.stats()
        counts, lst = e.neighbors()
    assert stats.overflow == 0
    assert stats.build_count == steps + 1 and stats.reorder_count >= steps
    ref = O.cell_ids(w, positions=st["positions"])
    order, ref_counts, offsets = O.stable_cell_order(ref, plan.n_cells, st["positions"])
    np.testing.assert_array_equal(cells["cell_count"], ref_counts)
    np.testing.assert_array_equal(cells["cell_start"], offsets)
    np.testing.assert_array_equal(cells["cell_atoms"], order)
    assert sorted(st["tags"]) == list(range(1, w.n + 1))
    rc, rl, ovf = O.neighbor_lists(w, positions=st["positions"], tags=st["tags"], types=st["types"])
    assert not ovf
    np.testing.assert_array_equal(counts, rc)
    for i in range(0, w.n, max(1, w.n // 3000)):
        assert np.array_equal(np.sort(lst[:counts[i], i]), np.sort(rl[i, :rc[i]])), i


def _limit(e, members=256, join_ticks=3000, wait_polls=1 << 27):
    """How the workgroups of e's rebuilds meet from here on."""
    e._check(e.lib.beads_internal_rebuild_limits(e.handle, C.c_uint32(members),
                                                 C.c_int64(join_ticks), C.c_uint32(wait_polls)))


def _members(e):
    n = C.c_uint32()
    e._check(e.lib.beads_internal_rebuild_members(e.handle, C.byref(n)))
    return n.value


def _every_step(w):
    return w.with_(cutoff_buffer=0.0, sort_every_rebuild=1)


@pytest.mark.parametrize("n", [500, 1023, 1024, 1025, 5000])
def test_part_filled_workgroups(n):
    _final_state(_every_step(W.lj_box(n, 0.8, 1.0, seed=n)), 40)


def test_more_cells_than_one_prefix():
    w = _every_step(W.lj_box(20000, 0.05, 1.0, seed=2))
    assert O.plan(w).n_cells > 16384
    _final_state(w, 24)


@pytest.mark.parametrize("n,steps,cutoff", [(6000, 10, 5.0), (30000, 48, 5.0), (7000, 10, 6.0)])
def test_cells_of_more_than_a_wave(n, steps, cutoff):
    """One wave orders such a cell in chunks and runs of chunks, from entries that
    other workgroups scattered (at 30,000 beads over a hundred of them)."""
    w = _every_step(W.lj_box(n, 0.8, 1.0, seed=4, cutoff=cutoff)).with_(max_neighbors=1024)
    assert w.n / O.plan(w).n_cells > 64
    _final_state(w, steps)


@pytest.mark.parametrize("members,join_ticks", [(1, 3000), (2, 3000), (37, 3000), (256, 0)])
def test_rebuilds_that_part_of_the_grid_shares(members, join_ticks):
    """The list of a rebuild's workgroups closed before all are on it, as beside
    another stream's kernels (at a count, so that the split is known, and at
    once): those on it do the whole of every phase, reorders with listed terms
    among them, and the others leave."""
    w = _every_step(W.polymer_melt(n_chains=300, beads_per_chain=50, seed=7))
    assert O.plan(w).path != 0
    got = []
    for limits in ({}, dict(members=members, join_ticks=join_ticks)):
        with Engine(w) as e:
            e.initialize(observables=False)
            full = _members(e)
            _limit(e, **limits)
            e.advance(20, observables_on_last=True)  # a captured graph and single steps
            took = _members(e)
            st, cells, stats = e.state(), e.cells(O.plan(w).n_cells), e.stats()
            counts, lst = e.neighbors()
        assert stats.overflow == 0 and stats.build_count == 21 and stats.reorder_count >= 20
        assert full > 37
        if limits and join_ticks:  # closed at once: as many as had started
            assert took == members
        got.append((st, cells, counts, list(stats.pe),
                    np.where(np.arange(len(lst))[:, None] < counts[None], lst, 0)))
    (sa, ca, na, pa, la), (sb, cb, nb, pb, lb) = got
    for k in sa:
        assert np.array_equal(sa[k], sb[k]), k
    for k in ca:
        assert np.array_equal(ca[k], cb[k]), k
    assert np.array_equal(na, nb) and np.array_equal(la, lb) and pa == pb


def test_engines_rebuilding_side_by_side():
    """Several engines step on their own streams at once, each rebuilding every
    step: the result is that of the engine alone."""
    ws = [_every_step(W.lj_box(n, 0.8, 1.0, seed=n)) for n in (3000, 40000, 20000, 60000)]
    alone = []
    for w in ws:
        with Engine(w) as e:
            e.initialize(observables=False)
            e.advance(48)
            alone.append(e.state())
    engines = [Engine(w) for w in ws]
    try:
        for e in engines:
            e.initialize(observables=False)
        for _ in range(3):  # calls return at once, so the engines' steps overlap
            for e in engines:
                e.advance(16)
        for e, a in zip(engines, alone):
            s = e.state()
            assert e.stats().overflow == 0
            for k in ("positions", "velocities", "tags", "images"):
                assert np.array_equal(s[k], a[k]), k
    finally:
        for e in engines:
            e.close()


def test_a_stalled_rebuild_is_final():
    """A wait that passes its bound (here no poll at all, so that every kernel
    leaves at once) ends in an error of its own, and in the same error from
    then on: no later launch bins on counts that were not cleared, and a list
    overflow does not take its place."""
    w = _every_step(W.lj_box(20000, 0.8, 1.0, seed=8))
    with Engine(w) as e, Engine(w.with_(max_neighbors=1)) as over:
        for engine in (e, over):
            engine.initialize(observables=False)
            assert _members(engine) > 1
        assert over.stats().overflow == 1
        for engine in (e, over):
            _limit(engine, wait_polls=0)
            engine.advance(24)  # a captured graph and single steps
            for call in (engine.synchronize, engine.stats, engine.state,
                         lambda: engine.advance(1), lambda: engine.initialize(False),
                         engine.neighbors):
                with pytest.raises(BeadsError, match="lost each other"):
                    call()
    # Other engines are untouched.
    _final_state(_every_step(W.lj_box(5000, 0.8, 1.0, seed=9)), 8)
