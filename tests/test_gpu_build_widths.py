"""The three widths of the neighbour build, at the atoms where the dispatch turns
from one to the next and on every grid that they treat differently.

Up to 12,000 atoms an atom is built by 32 lanes over its runs of cells, up to
100,000 by 16, above by four lanes over staged rows; x-boundary cells make two
runs of a row, grids
of fewer than five cells per axis take the minimum image per candidate, and
short axes have fewer rows. Lists are decisions: counts and sets are held bit
for bit to the oracle's.
"""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from beads_amd.capi import Engine
from gpu_cases import bonded_lattice, elongated_lj

pytestmark = pytest.mark.gpu


def _check(w):
    with Engine(w) as e:
        e.initialize(observables=False)
        st, stats = e.state(), e.stats()
        counts, lst = e.neighbors()
    assert stats.overflow == 0
    assert stats.mean_neighbors == counts.sum() / w.n
    rc, rl, ovf = O.neighbor_lists(w, positions=st["positions"], tags=st["tags"], types=st["types"])
    assert not ovf
    np.testing.assert_array_equal(counts, rc)
    m = int(counts.max())
    got = np.where(np.arange(m)[:, None] < counts[None], lst[:m], 0xffffffff)
    want = np.where(np.arange(m)[None] < rc[:, None], rl[:, :m], 0xffffffff)
    assert np.array_equal(np.sort(got, axis=0).T, np.sort(want, axis=1))


# 8,000 beads: the 32-lane build; 91,125: the 16-lane build; 125,000: the
# four-lane build.
@pytest.mark.parametrize("side", [20, 45, 50])
@pytest.mark.parametrize("kind,distance", [("chains", 1), ("chains", 3), ("stars", 2)])
def test_exclusion_variants_on_both_sides(side, kind, distance):
    _check(bonded_lattice(kind, distance, side=side).with_(max_neighbors=160))


# Edges of the dispatch on grids of 2 to 5 cells on the short axes (search
# cutoff 2.8), the long axis along x and along z.
@pytest.mark.parametrize("n", [12000, 12001, 100000, 100001])
@pytest.mark.parametrize("short", [5.7, 8.5, 11.3, 14.1])
@pytest.mark.parametrize("axis", [0, 2])
def test_grids_on_both_sides(n, short, axis):
    lengths = [short, short, short]
    lengths[axis] = n / 0.8 / short ** 2
    _check(elongated_lj(n, lengths).with_(max_neighbors=160))


# Whole (1,504) and part-filled workgroups of 8 atoms in the 32-lane build.
@pytest.mark.parametrize("n", [1500, 1504, 1505])
@pytest.mark.parametrize("half", [False, True])
def test_small_grids_and_half_lists(n, half):
    for short in (5.7, 8.5, 11.3, 14.1):
        w = elongated_lj(n, (max(5.7, n / 0.8 / short ** 2), short, short))
        w = w.with_(max_neighbors=192)
        if not half:
            _check(w)
        else:
            with Engine(w) as e, Engine(w.with_(half_list=True)) as h:
                e.initialize(observables=False)
                h.initialize(observables=False)
                (ca, la), (cb, lb) = e.neighbors(), h.neighbors()
            assert 2 * int(cb.sum()) == int(ca.sum())
            for i in range(n):
                want = np.sort(la[:ca[i], i])
                assert np.array_equal(np.sort(lb[:cb[i], i]), want[want > i]), i


# The half list's filter in the 16-lane and the four-lane build: what the full list
# holds above the atom's own slot.
@pytest.mark.parametrize("n", [12001, 100001])
def test_half_lists_of_larger_systems(n):
    w = elongated_lj(n, (n / 0.8 / 14.1 ** 2, 14.1, 14.1)).with_(max_neighbors=192)
    with Engine(w) as e, Engine(w.with_(half_list=True)) as h:
        e.initialize(observables=False)
        h.initialize(observables=False)
        (ca, la), (cb, lb) = e.neighbors(), h.neighbors()
    m = int(ca.max())
    full = np.where(np.arange(m)[:, None] < ca[None], la[:m], 0xffffffff)
    want = np.where(full > np.arange(n)[None], full, 0xffffffff)
    got = np.where(np.arange(m)[:, None] < cb[None], lb[:m], 0xffffffff)
    assert 2 * int(cb.sum()) == int(ca.sum())
    assert np.array_equal(np.sort(got, axis=0), np.sort(want, axis=0))
