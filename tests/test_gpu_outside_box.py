"""Atoms that the wrap leaves outside the box: a displacement of millions of box
lengths rounds by a good part of a cell, so the cell such an atom is clamped into
does not hold it and a wrapped cell says nothing about its image. Lists then are
what the scan of the 27 cells with a minimum image per candidate finds, in each
width of the build; sets and counts are held bit for bit to the oracle's."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import Engine
from gpu_cases import elongated_lj

pytestmark = pytest.mark.gpu


def _flying(w, count, seed, speed=4e9):
    """w with count atoms that a step carries millions of box lengths away."""
    rng = np.random.default_rng(seed)
    v = w.velocities.copy()
    fast = rng.choice(w.n, size=count, replace=False)
    v[fast] = (rng.standard_normal((count, 3)) * speed).astype(np.float32)
    return w.with_(velocities=v, cutoff_buffer=0.0, max_neighbors=256)


# 32, 16 and 4 lanes per atom; few atoms outside and many; a grid of 5 cells on
# two axes and one of 3.
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("make,count", [
    (lambda: W.lj_box(3000, 0.8, 1.0, seed=1), 200),
    (lambda: W.lj_box(3000, 0.8, 1.0, seed=2), 1000),
    (lambda: W.lj_box(40000, 0.8, 1.0, seed=3), 8000),
    (lambda: W.lj_box(110000, 0.8, 1.0, seed=4), 20000),
    (lambda: elongated_lj(3000, (14.1, 14.1, 18.9)), 400),
    (lambda: elongated_lj(3000, (8.5, 8.5, 51.9)), 400),
])
def test_lists_are_the_full_scans(make, count, half):
    w = _flying(make(), count, seed=count).with_(half_list=half)
    with Engine(w) as e:
        e.initialize(observables=False)
        e.advance(1)
        st, stats = e.state(), e.stats()
        counts, lst = e.neighbors()
    assert stats.overflow == 0 and stats.build_count == 2
    x = st["positions"]
    assert np.isfinite(x).all()
    assert ((x < w.box_bound[0]) | (x > w.box_bound[1])).any()
    rc, rl, ovf = O.neighbor_lists(w, positions=x, tags=st["tags"], types=st["types"])
    assert not ovf
    m = int(rc.max())
    want = np.where(np.arange(m)[None] < rc[:, None], rl[:, :m], 0xffffffff)
    if half:
        want = np.where(want > np.arange(w.n)[:, None], want, 0xffffffff)
    got = np.where(np.arange(m)[:, None] < counts[None], lst[:m], 0xffffffff)
    np.testing.assert_array_equal(counts, (want != 0xffffffff).sum(axis=1))
    assert np.array_equal(np.sort(got, axis=0).T, np.sort(want, axis=1))


def test_all_atoms_in_the_corner_cells():
    """Farther still, and the wrap leaves every atom far outside: the corner
    cells hold them all, and their members come in order of x."""
    w = _flying(W.lj_box(40000, 0.8, 1.0, seed=7), 40000, seed=7, speed=4e12)
    plan = O.plan(w)
    with Engine(w) as e:
        e.initialize(observables=False)
        e.advance(1)
        st, cells = e.state(), e.cells(plan.n_cells)
    ref = O.cell_ids(w, positions=st["positions"])
    order, counts, offsets = O.stable_cell_order(ref, plan.n_cells, st["positions"])
    assert counts.max() > 2000
    np.testing.assert_array_equal(cells["cell_count"], counts)
    np.testing.assert_array_equal(cells["cell_start"], offsets)
    np.testing.assert_array_equal(cells["cell_atoms"], order)
