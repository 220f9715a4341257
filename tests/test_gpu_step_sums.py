"""The kinetic energy a call leaves behind. Without a thermostat only a call's
last step forms it; that must hold for every way a call can end: single steps,
whole step graphs, graphs and single steps, with and without a rebuild in the
last step. The engine's FP64 sum of the stored binary32 velocities against the
oracle's: 1e-9 relative, the parity tests' bar."""

from __future__ import annotations

import pytest

import oracle as O
from beads_amd import workloads as W
from beads_amd.capi import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("berendsen", [False, True])
@pytest.mark.parametrize("check_every", [1, 10])
@pytest.mark.parametrize("half", [False, True])
def test_kinetic_energy_after_every_kind_of_call(berendsen, check_every, half):
    w = W.lj_box(1500, 0.8, 1.0, seed=8, berendsen=berendsen, check_every=check_every)
    with Engine(w.with_(half_list=half)) as e:
        e.initialize(observables=False)
        builds = 0
        for steps in (1, 15, 16, 17, 3, 20, 40, 41, 64):
            e.advance(steps)
            s, st = e.state(), e.stats()
            ke = O.kinetic_energy(s["velocities"], s["masses"])
            assert abs(st.ke - ke) <= 1e-9 * ke, steps
            builds = st.build_count
        assert builds > 3


def test_energies_on_the_last_step_only():
    w = W.lj_box(1500, 0.8, 1.0, seed=8)
    with Engine(w) as e:
        e.initialize(observables=True)
        e.advance(37, observables_on_last=True)
        s, st = e.state(), e.stats()
    f, obs = O.forces(w, positions=s["positions"], tags=s["tags"], types=s["types"])
    assert abs(st.pe[0] - obs["pair_pe"]) <= 1e-5 * abs(obs["pair_pe"])
    ke = O.kinetic_energy(s["velocities"], s["masses"])
    assert abs(st.ke - ke) <= 1e-9 * ke
