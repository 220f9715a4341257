"""The force pass's three shapes (16, 8 and 4 lanes per atom) on both sides of
the sizes where one gives way to the next, with part-filled last workgroups:
forces of LJ pairs and every listed term within 1e-5 of the oracle's FP64 per
component (of max(|f|, f_rms)), energies and virials within 1e-5 of the summed
values, as the parity tests hold them.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import Engine

pytestmark = pytest.mark.gpu

RTOL = 1e-5


def _check(w):
    with Engine(w) as e:
        e.initialize(observables=True)
        st, stats = e.state(), e.stats()
    f_ref, obs = O.forces(w, positions=st["positions"], tags=st["tags"], types=st["types"])
    scale = np.sqrt(np.mean(f_ref ** 2))
    err = np.max(np.abs(st["forces"] - f_ref) / np.maximum(np.abs(f_ref), scale))
    assert err <= RTOL, err
    for q, term in enumerate(("pair", "bond", "angle", "dihedral")):
        ref_pe, ref_w = obs[f"{term}_pe"], obs[f"{term}_virial"]
        assert abs(stats.pe[q] - ref_pe) <= RTOL * max(1.0, abs(ref_pe)), term
        assert abs(stats.virial[q] - ref_w) <= RTOL * max(1.0, abs(ref_w)) + 1e-6 * w.n, term


# 1,200 chains of 10 are 12,000 beads, 4,000 are 40,000.
@pytest.mark.parametrize("chains", [57, 1200, 1201, 4000, 4001])
def test_melt(chains):
    _check(W.polymer_melt(n_chains=chains, beads_per_chain=10, seed=chains))


@pytest.mark.parametrize("n_types", [1, 4, 17])  # coefficients in registers, LDS, memory
@pytest.mark.parametrize("n", [12000, 12001, 40000, 40001])
def test_mixture(n, n_types):
    _check(W.lj_mixture(n=n, n_types=n_types, seed=n + n_types))
