"""Reading the state back: the single copy, the copy in pieces by several
threads, subsets of the fields and reads from several threads at once give back
exactly what the run was created with (before its first step nothing has touched
it)."""

from __future__ import annotations

import ctypes as C
import threading

import numpy as np
import pytest

from beads_amd import capi
from beads_amd import workloads as W

pytestmark = pytest.mark.gpu

FIELDS = ("positions", "velocities", "masses", "types", "tags", "molecule_ids", "images")


def _inputs(n: int) -> W.Workload:
    w = W.lj_box(n, 0.8, 1.0, seed=n)
    rng = np.random.default_rng(n)
    return w.with_(images=rng.integers(-5, 6, (n, 3)), tags=rng.permutation(n) + 1,
                   types=rng.integers(1, 4, n).astype(np.int32), lj_epsilon=np.ones((3, 3)),
                   lj_sigma=np.ones((3, 3)), masses=rng.uniform(1, 2, n).astype(np.float32),
                   molecule_ids=np.arange(1, n + 1))


# 64 bytes an atom in binary32, 104 in binary64: 65,536 and 40,329 atoms are the
# last in one copy; pieces of 1 MB are whole at 81,920, windows of 16 MB at
# 524,288.
@pytest.mark.parametrize("precision,n", [("single", 500), ("single", 65536), ("single", 65537),
                                         ("single", 81920), ("single", 131071),
                                         ("single", 524288), ("single", 524289),
                                         ("double", 40329), ("double", 40330)])
def test_state_is_what_went_in(precision, n):
    w = _inputs(n)
    if precision == "double":
        w = w.as_float64(jitter=1e-9)
    with capi.Engine(w, precision) as e:
        for _ in range(2):
            s = e.state()
            for k in FIELDS:
                assert np.array_equal(s[k], getattr(w, k)), k
            assert not s["forces"].any()


# Windows as small as they get where the card is full: a few and many, pieces
# that divide a window and pieces that do not, one piece a window.
@pytest.mark.parametrize("precision,n,window,piece", [
    ("single", 500, 1 << 14, 1 << 14), ("single", 700, 1 << 14, 1000),
    ("single", 20001, 1 << 14, 1 << 12), ("single", 20001, 100000, 1 << 20),
    ("double", 20001, 20000, 4096)])
def test_small_windows(precision, n, window, piece):
    w = _inputs(n)
    if precision == "double":
        w = w.as_float64(jitter=1e-9)
    with capi.Engine(w, precision) as e:
        e._check(e.lib.beads_internal_state_sizes(e.handle, C.c_uint64(0), C.c_uint64(window),
                                                  C.c_uint64(piece)))
        for _ in range(2):
            s = e.state()
            for k in FIELDS:
                assert np.array_equal(s[k], getattr(w, k)), k


@pytest.mark.parametrize("n", [500, 200000])
def test_reads_from_several_threads(n):
    w = _inputs(n)
    wrong = []
    with capi.Engine(w, "single") as e:
        def read(k):
            try:
                for _ in range(6):
                    s = e.state()
                    if not all(np.array_equal(s[f], getattr(w, f)) for f in FIELDS):
                        wrong.append(k)
            except Exception as x:  # noqa: BLE001
                wrong.append(x)
        threads = [threading.Thread(target=read, args=(k,)) for k in range(4)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert not wrong


@pytest.mark.parametrize("n", [500, 131071])
def test_subsets_of_fields(n):
    w = _inputs(n)
    with capi.Engine(w, "single") as e:
        for wanted in (("images",), ("types", "molecule_ids"), ("velocities", "tags"), ()):
            so = capi.StateOut()
            out = {}
            for k in wanted:
                a = np.zeros_like(getattr(w, k))
                out[k] = a
                field = dict(capi.StateOut._fields_)[k]
                setattr(so, k, C.cast(a.ctypes.data, field))
            assert e.lib.beads_engine_read_state(e.handle, C.byref(so)) == 0
            for k in wanted:
                assert np.array_equal(out[k], getattr(w, k)), k


def test_batch_states():
    ws = [_inputs(n) for n in (700, 70001, 1300)]
    with capi.Batch(ws) as b:
        for r, w in enumerate(ws):
            s = b.state(r)
            for k in ("positions", "velocities", "masses", "types", "tags", "images"):
                assert np.array_equal(s[k], getattr(w, k)), (r, k)
