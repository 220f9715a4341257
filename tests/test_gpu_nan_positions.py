"""Positions that are not numbers: every bead keeps one entry of the cell order,
so that no reorder loses a bead and no list entry is left from an earlier build.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import Engine

pytestmark = pytest.mark.gpu


def _check_cells(e, w):
    n_cells = O.plan(w).n_cells
    c = e.cells(n_cells)
    np.testing.assert_array_equal(np.sort(c["cell_atoms"]), np.arange(w.n))
    assert c["cell_count"].sum() == w.n
    np.testing.assert_array_equal(c["cell_of"][c["cell_atoms"]],
                                  np.repeat(np.arange(n_cells), c["cell_count"]))


# From the first frame on, when the arrays hold nothing yet; few, and so many that
# some cells pass 64 members.
@pytest.mark.parametrize("n,bad", [(3000, 1), (3000, 30), (20000, 5), (20000, 4000)])
def test_frames(n, bad):
    w = W.lj_box(n, 0.8, 1.0, seed=n).with_(max_neighbors=6000)
    x = w.positions.copy()
    rng = np.random.default_rng(bad)
    at = rng.choice(n, size=bad, replace=False)
    x[at, rng.integers(0, 3, bad)] = np.nan
    x[at[: bad // 3]] = np.nan
    with Engine(w) as e:
        for frame in (x, w.positions, x):
            p = torch.tensor(frame, device="cuda")
            e.frame_load(p.data_ptr(), reuse_list=False)
            _check_cells(e, w)


@pytest.mark.parametrize("make", [
    lambda: W.lj_box(3000, 0.8, 1.0, seed=5),
    lambda: W.polymer_melt(n_chains=80, beads_per_chain=50, seed=7)])
def test_dynamics_that_turn_to_nan(make):
    """Coincident beads: their force is 0 * inf, and NaN spreads by a cutoff a
    step through rebuilds that reorder every time."""
    w = make().with_(cutoff_buffer=0.0, sort_every_rebuild=1)
    x = w.positions.copy()
    x[1] = x[0]
    x[w.n // 2 + 1] = x[w.n // 2]
    w = w.with_(positions=x, exclusion_distance=0)
    with Engine(w) as e:
        e.initialize(observables=False)
        spread = []
        for _ in range(6):
            e.advance(2)
            st = e.state()
            _check_cells(e, w)
            assert sorted(st["tags"]) == list(range(1, w.n + 1))
            spread.append(int(np.isnan(st["positions"]).any(axis=1).sum()))
    assert spread[0] > 0
