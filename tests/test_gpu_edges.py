"""Calls that meet two limits of a build at once, or whose inputs change
between two calls, each against the oracle or the entry point that it varies.
"""
import ctypes

import numpy as np
import pytest
import torch

import nlhip
import oracle
from nlhip import _lib, workloads
from test_zz_no_alloc import _noalloc

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a).view(np.int64)


def _same(nl, ref, want_R=False):
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
    if want_R:
        assert np.array_equal(_bits(nl.R), _bits(ref.R))


def _cluster_with_far_windings(s, rc, m=60):
    """The last m atoms of s in the middle of one cell, the last two of them
    300 cells away to either side: their own pair, whose shift of 600 takes
    16-byte entries, is behind the end of both rows."""
    X = s.X.copy()
    L = np.diag(np.asarray(s.cell))
    edge = L / np.floor(L / rc)
    rng = np.random.default_rng(len(X))
    X[-m:] = (np.minimum(2.0, np.floor(L / rc) - 1) + 0.5) * edge + 0.4 * (rng.random((m, 3)) - 0.5)
    X[-2] += 300 * np.asarray(s.cell)[0]
    X[-1] -= 300 * np.asarray(s.cell)[0]
    return X


@pytest.mark.parametrize("want_R", [False, True])
@pytest.mark.parametrize("n", [3000, 20000, 270000])
def test_wide_entries_behind_short_rows(n, want_R):
    """Slot rows that are too short hide the pair that also needs wider
    entries: on a new handle, on one that knows this system's counts, and in
    the build that allocates nothing."""
    s = workloads.random_cubic(n, density=0.02, seed=n, cutoff=5.0)
    X = _cluster_with_far_windings(s, 5.0)
    print(f"wide behind short rows {n} {want_R}", flush=True)
    ref = oracle.neighbour_list(X, 5.0, s.cell, s.pbc, want_R=want_R, nthreads=8)
    assert np.abs(ref.S).max() == 600
    for warm in (0, 3):
        h = _lib.Handle()
        for _ in range(warm):
            nlhip.neighbour_list(s.X, 5.0, s.cell, s.pbc, want_R=want_R, handle=h)
        _same(nlhip.neighbour_list(X, 5.0, s.cell, s.pbc, want_R=want_R, handle=h), ref, want_R)
    if n <= 20000:
        st, P, out = _noalloc(X, s.cell, 5.0, s.pbc, want_R=want_R, cap=ref.npairs)
        assert st == _lib.NLH_OK, _lib.lib().nlh_last_error()
        assert P == ref.npairs
        for k in ("i", "j", "S", "first"):
            assert np.array_equal(out[k], getattr(ref, k)), k
        if want_R:
            assert np.array_equal(_bits(out["R"]), _bits(ref.R))


def test_wide_entries_behind_short_rows_of_a_batch():
    """The same in a fused batch of small systems, some of them ordinary."""
    systems = []
    for k in range(70):
        s = workloads.random_cubic(200 + k, density=0.02, seed=k, cutoff=5.0)
        X = _cluster_with_far_windings(s, 5.0) if k % 9 == 4 else s.X
        systems.append(workloads.System(X, s.cell, s.pbc, s.cutoff))
    print("wide behind short rows, batch", flush=True)
    got = nlhip.BatchBuilder().run(systems)
    for k, y in enumerate(systems):
        _same(got.pairlist(k), oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc))
