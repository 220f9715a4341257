"""A batch whose atoms fly: a displacement of millions of box lengths leaves
the wrapped position outside the box by its rounding, so the cell an atom is
put in says little about where its neighbours are. Lists then are what the scan
of the 27 cells finds; the phased build must find the same ones as the
persistent one, in the same order, so both modes agree bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from beads_amd import workloads as W
from beads_amd.capi import Batch

pytestmark = pytest.mark.gpu


def _flying(n: int, count: int, seed: int) -> W.Workload:
    w = W.lj_box(n, 0.8, 1.0, seed=seed)
    v = w.velocities.copy()
    rng = np.random.default_rng(seed)
    fast = rng.choice(n, size=count, replace=False)
    v[fast] = (rng.standard_normal((count, 3)) * 3e8).astype(np.float32)
    return w.with_(velocities=v)


@pytest.mark.parametrize("count", [40, 400])
def test_modes_agree_with_atoms_outside_the_box(count):
    # 5 cells per axis, 3 cells per axis
    ws = [_flying(3000, count, 1), _flying(700, count, 2)]
    got = []
    for config in (0, 3):  # persistent; phased with the same force shape
        with Batch(ws) as b:
            b.set_config(config)
            b.run(6)
            got.append([(b.state(r), b.stats(r).build_count) for r in range(len(ws))])
    outside = 0
    for (a, builds_a), (c, builds_c), w in zip(got[0], got[1], ws):
        assert builds_a == builds_c
        for k in ("positions", "velocities", "forces", "tags", "images"):
            assert np.array_equal(a[k], c[k], equal_nan=a[k].dtype.kind == "f"), k
        x = a["positions"]
        outside += int(((x < w.box_bound[0]) | (x > w.box_bound[1])).any(axis=1).sum())
    assert outside > 0
