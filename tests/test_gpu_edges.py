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


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("n,density,moved", [(40, 0.05, 1.0), (3000, 0.05, 0.3), (3000, 0.01, 1.0), (20000, 0.05, 0.02)])
def test_lazy_queries_read_the_positions_as_they_are(n, density, moved, int_type, bits):
    """Device positions moved in place between the build and the queries: a
    range query sees for every atom what the one-atom query sees."""
    s = workloads.random_cubic(n, density=density, seed=n, cutoff=5.0, pbc=(True, n != 3000, True))
    X = torch.as_tensor(s.X).cuda()
    cl = nlhip.build_cell_list(X, 5.0, s.cell, s.pbc, int_type=int_type)
    print(f"lazy, moved {n} {moved} {bits}", flush=True)
    rng = np.random.default_rng(n)
    before = nlhip.neighbours_range(cl, 1, min(n, 500))
    Y = s.X + 0.4 * rng.standard_normal((n, 3)) * (rng.random((n, 1)) < moved)
    Y[::50] += np.asarray(s.cell)[0]
    X.copy_(torch.as_tensor(Y))
    torch.cuda.synchronize()
    first, m = 2, min(n - 1, 600)
    offs, j, R, S = nlhip.neighbours_range(cl, first, m)
    L, h = _lib.lib(), cl._handle
    dt = np.int32 if bits == 32 else np.int64
    for a in range(0, m, 1 if n < 1000 else 7):
        c = ctypes.c_int64()
        j1, R1, S1 = np.empty(4096, dt), np.empty((4096, 3)), np.empty((4096, 3), dt)
        _lib.check(L.nlh_neighbours(h.ptr, 0, first + a, 4096, j1.ctypes.data, R1.ctypes.data, S1.ctypes.data,
                                    ctypes.byref(c)))
        q, k = slice(offs[a], offs[a + 1]), c.value
        assert offs[a + 1] - offs[a] == k and np.array_equal(j[q], j1[:k]) and np.array_equal(S[q], S1[:k])
        assert np.array_equal(_bits(R[q]), _bits(R1[:k]))
    # and the positions as they were give the first answer again
    X.copy_(torch.as_tensor(s.X))
    torch.cuda.synchronize()
    for u, v in zip(nlhip.neighbours_range(cl, 1, min(n, 500)), before):
        assert np.array_equal(u, v)


@pytest.mark.parametrize("cells,square", [(56, 25.0), (34, 25.0), (56, 30.0)])
def test_cells_smaller_than_the_cutoff(cells, square):
    """A caller's own cell counts with a reach of one cell, and its own square of
    the cutoff: the 27 cells around an atom and no more, whatever the pair search
    shares between home cells."""
    n = 250000
    s = workloads.random_cubic(n, density=0.05, seed=1, cutoff=5.0)
    g = _lib.geometry(s.cell, 5.0, s.pbc, 4)
    for k in range(3):
        g.ncells[k], g.nxyz[k] = cells, 1
    g.ncells_total = cells ** 3
    g.cutoff_sq = square
    L, h, m = _lib.lib(), _lib.Handle(), ctypes.c_int64()
    print(f"cells {cells} {square}", flush=True)
    _lib.check(L.nlh_neighbour_list(h.ptr, s.X.ctypes.data, n, ctypes.byref(g), 0, ctypes.byref(m)))
    j, first, S = np.empty(m.value, np.int32), np.empty(n + 1, np.int32), np.empty((m.value, 3), np.int32)
    _lib.check(L.nlh_copy_pairlist(h.ptr, None, j.ctypes.data, S.ctypes.data, first.ctypes.data, None))
    for i in range(1, n + 1, 997):
        c, j1, S1 = ctypes.c_int64(), np.empty(256, np.int32), np.empty((256, 3), np.int32)
        _lib.check(L.nlh_neighbours(h.ptr, 0, i, 256, j1.ctypes.data, None, S1.ctypes.data, ctypes.byref(c)))
        a, b = first[i - 1] - 1, first[i] - 1
        assert b - a == c.value and np.array_equal(j[a:b], j1[:c.value]) and np.array_equal(S[a:b], S1[:c.value])


def _edge_batches():
    """name -> systems: units at their limits, systems without atoms, one beyond a
    unit, rows that overflow, atoms far outside open cells."""
    def cubes(sizes):
        out = []
        for k, n in enumerate(sizes):
            y = workloads.random_cubic(max(n, 1), density=0.05, seed=k, cutoff=3.5 + 0.1 * (k % 9))
            out.append(workloads.System(y.X[:n], y.cell, y.pbc, y.cutoff))
        return out

    rng = np.random.default_rng(8)
    clusters, far = [], []
    for k in range(66):
        n = [30, 300, 900][k % 3]
        cell = np.eye(3) * (6.0 if k % 3 == 0 else 40.0)
        X = rng.random((n, 3)) * 40.0
        X[-30:] = 20.0 + 0.5 * rng.random((30, 3))
        clusters.append(workloads.System(X, cell, (True, True, k % 2 == 0), 5.0))
        y = workloads.random_cubic(150 + k, density=0.05, seed=k, cutoff=4.0)
        pbc = (k % 2 == 0, k % 3 == 0, False)
        far.append(workloads.System(y.X + np.where(pbc, 0.0, [0.3, 17.0, 1e6][k % 3]) * y.cell[0][0], y.cell, pbc, 4.0))
    return {"full units": cubes([2048] * 64), "one large": cubes([1] * 700 + [2048]), "empty": cubes([2047, 1, 0, 1] * 20),
            "almost empty": cubes([0] * 70 + [3]), "beyond a unit": cubes([2049] + [5] * 70), "clusters": clusters,
            "far": far}


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("name", sorted(_edge_batches()))
def test_R_of_batches_at_their_edges(name, int_type, bits):
    """R of batches at the limits of the fused build, against the oracle bit for bit."""
    systems = _edge_batches()[name]
    print(f"R batch edges {name} {bits}", flush=True)
    got = nlhip.BatchBuilder(int_type=int_type).run(systems, want_R=True)
    for k, y in enumerate(systems):
        _same(got.pairlist(k), oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc, ti_bits=bits, want_R=True), True)
