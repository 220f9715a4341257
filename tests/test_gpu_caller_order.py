"""Beads in a caller's (spatially random) order on the GPU.

A wave of such beads meets up to 64 different cells, so the binning kernels
leave the shared-atomic loop and add lane by lane; and a frame far from the
last one raises the rebuild flag from every lane. Cells, in-cell order and
neighbour sets are decisions: the bar is bit-exactness against the oracle. A
frame's forces must equal those of an engine that never held another list
(the same kernel on the same list, so bit for bit).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import Engine

pytestmark = pytest.mark.gpu


def shuffled_lj(n: int, seed: int = 3) -> W.Workload:
    w = W.lj_box(n, 0.8, 1.0, seed=seed)
    order = np.random.default_rng(seed).permutation(n)
    return w.with_(positions=w.positions[order], velocities=w.velocities[order])


@pytest.mark.parametrize("n", [1000, 4097, 6400])  # part-filled and whole last waves
def test_cells_and_lists_of_shuffled_beads(n):
    w = shuffled_lj(n)
    plan = O.plan(w)
    assert plan.path != O.PATH_DIRECT
    with Engine(w) as e:
        e.initialize(observables=False)
        counts, lst = e.neighbors()
        cells = e.cells(plan.n_cells)
        st = e.state()
    ref = O.cell_ids(w, positions=st["positions"])
    order, ref_counts, offsets = O.stable_cell_order(ref, plan.n_cells, st["positions"])
    np.testing.assert_array_equal(cells["cell_of"], ref)
    np.testing.assert_array_equal(cells["cell_count"], ref_counts)
    np.testing.assert_array_equal(cells["cell_start"], offsets)
    np.testing.assert_array_equal(cells["cell_atoms"], order)
    rc, rl, _ = O.neighbor_lists(w, positions=st["positions"], tags=st["tags"], types=st["types"])
    np.testing.assert_array_equal(counts, rc)
    for i in range(n):
        assert np.array_equal(np.sort(lst[:counts[i], i]), np.sort(rl[i, :rc[i]])), i


@pytest.mark.parametrize("n", [1000, 4097])
@pytest.mark.parametrize("moved", ["all", "one"])
def test_frame_that_moved_rebuilds(n, moved):
    w = shuffled_lj(n)
    hi = w.box_bound[1]
    second = w.positions.copy()
    if moved == "all":
        second = np.mod(second + np.float32(1.7), hi).astype(np.float32)
    else:  # the last bead alone, past half the skin
        second[-1] = np.mod(second[-1] + np.float32(0.2), hi).astype(np.float32)
    second = np.where(second >= hi, np.float32(0), second)
    x = [torch.tensor(q, device="cuda") for q in (w.positions, second)]
    out = [torch.empty_like(x[0]) for _ in range(2)]
    with Engine(w) as e:
        e.frame_forces(x[0].data_ptr(), out[0].data_ptr())
        e.frame_forces(x[1].data_ptr(), out[0].data_ptr(), reuse_list=True)
        assert e.stats().build_count == 2
    with Engine(w) as e:
        e.frame_forces(x[1].data_ptr(), out[1].data_ptr())
    assert torch.equal(out[0], out[1])
