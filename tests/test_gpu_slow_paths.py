"""Systems that leave the pair search's fast path: results against the oracle
at the edges of its other paths, and their times against an ordinary system's.
"""
import ctypes
import time

import numpy as np
import pytest
import torch

import nlhip
import oracle
from nlhip import _lib, workloads

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a).view(np.int64)


def _check(X, rc, cell, pbc, want_R=False):
    ref = oracle.neighbour_list(X, rc, cell, pbc, want_R=want_R, nthreads=8)
    nl = nlhip.neighbour_list(X, rc, cell, pbc, want_R=want_R)
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
    if want_R:
        assert np.array_equal(_bits(nl.R), _bits(ref.R))


def _time(X, rc, cell, pbc):
    """Median time of a build of device positions on a handle that knows them (us)."""
    L, h, m = _lib.lib(), _lib.Handle(), ctypes.c_int64()
    g = _lib.geometry(cell, rc, pbc, 4)
    D = torch.as_tensor(np.ascontiguousarray(X)).cuda()
    torch.cuda.synchronize()
    t = []
    for _ in range(30):
        t0 = time.perf_counter()
        _lib.check(L.nlh_neighbour_list(h.ptr, D.data_ptr(), len(X), ctypes.byref(g), _lib.NLH_X_DEVICE, ctypes.byref(m)))
        _lib.check(L.nlh_synchronize(h.ptr))
        t.append(time.perf_counter() - t0)
    return 1e6 * float(np.median(t[5:]))


def _time_batch(systems):
    """Median time of a rebuild of a batch of device positions (us)."""
    B = nlhip.BatchBuilder()
    X = np.concatenate([y.X for y in systems])
    D = torch.as_tensor(X).cuda()
    torch.cuda.synchronize()
    B.run(systems, X_device=D, copy=False)
    t = []
    for _ in range(30):
        t0 = time.perf_counter()
        B.rebuild(X, X_device=D, copy=False)
        _lib.check(_lib.lib().nlh_synchronize(B.handle.ptr))
        t.append(time.perf_counter() - t0)
    return 1e6 * float(np.median(t[5:]))


@pytest.mark.parametrize("reach", [1, 2])
@pytest.mark.parametrize("sizes", [(1, 1, 1), (47, 48, 49, 63, 64, 65), (96, 97, 144, 145, 0, 200), (3, 0, 0, 130, 7, 1)])
def test_cells_counted_from_global_memory(sizes, reach):
    """A row of cells of given sizes, dense enough or of a reach that takes
    them to the per-wave count: groups of home atoms up to a wave, shares of
    larger cells, more waves than cells."""
    rng = np.random.default_rng(sum(sizes))
    rc = 2.0 if reach == 1 else 2.9   # along z: one cell of 2.02
    cell = np.diag([len(sizes) * rc * 1.01, 2.0 * rc * 1.01, 2.02])
    parts = []
    for k, n in enumerate(sizes):
        for y in range(2):
            parts.append((np.array([k, y, 0]) + rng.random((n, 3))) * [rc * 1.01, rc * 1.01, 2.02])
    print(f"per-wave {sizes} {reach}", flush=True)
    for pbc in [(True, True, True), (False, True, True)]:
        _check(np.concatenate(parts), rc, cell, pbc, want_R=True)


def test_time_of_a_reach_of_two_cells():
    """A plate one cell thick with a reach of two across it (few cells, none of
    them in the LDS path): its bricks of one cell keep all their waves busy.
    It took twice an ordinary system's time, and takes 1.3 of it."""
    n = 3000
    s = workloads.random_cubic(n, density=0.05, seed=n, cutoff=5.0)
    L = (n / 0.05 / 6) ** 0.5
    y = workloads.random_in_cell(n, np.diag([6.0, L, L]), seed=n, cutoff=7.0)
    print("plate", flush=True)
    assert _time(y.X, 7.0, y.cell, (True,) * 3) < 1.65 * _time(s.X, 5.0, s.cell, (True,) * 3)


@pytest.mark.parametrize("n", [65, 3000, 40000])
@pytest.mark.parametrize("base", [(0, 0, 0), (200, -300, 400), (511, -512, 511)])
@pytest.mark.parametrize("spread", [0, 127, 128, 200, 254, 255, 256, 500])
def test_windings_of_a_brick(spread, base, n):
    """Atoms that drifted together by hundreds of cells, some of them apart by
    up to twice `spread`: the brick path as long as the windings of a brick span
    no more than its entries hold, and the paths beyond."""
    s = workloads.random_in_cell(n, np.array([[1.0, 0.1, 0.0], [0.2, 1.1, 0.1], [0.0, 0.1, 0.9]]) * (n / 0.05) ** (1 / 3),
                                 seed=n, cutoff=4.0)
    rng = np.random.default_rng(spread)
    w = rng.choice([-spread, 0, 0, spread], size=(n, 3)) + np.array(base) * (1 if spread < 300 else 0)
    print(f"brick windings {spread} {base} {n}", flush=True)
    _check(s.X + w.astype(float) @ s.cell, 4.0, s.cell, (True, True, True), want_R=n == 3000)


def test_time_of_positions_that_were_never_wrapped():
    """Positions hundreds of cells from the cell they are described in: twice an
    ordinary system's time it was, and is the same."""
    s = workloads.random_cubic(500000, density=0.05, seed=1, cutoff=5.0)
    print("drifted", flush=True)
    assert _time(s.X + 200 * np.asarray(s.cell).sum(0), 5.0, s.cell, s.pbc) < 1.5 * _time(s.X, 5.0, s.cell, s.pbc)


@pytest.mark.parametrize("n", [27000, 33000])
def test_time_of_a_dense_region(n):
    """Half of the atoms in an eighth of the cell: 1.2 of a uniform system's time,
    with bricks whose halos fit the LDS there (2.2 to 2.6 with the next larger ones)."""
    s = workloads.random_cubic(n, density=0.02, seed=n, cutoff=5.0)
    X, c = s.X.copy(), np.diag(np.asarray(s.cell)) / 2
    X[::2] = c + (X[::2] - c) * 0.5
    print(f"dense region {n}", flush=True)
    assert _time(X, 5.0, s.cell, s.pbc) < 1.7 * _time(s.X, 5.0, s.cell, s.pbc)


@pytest.mark.parametrize("off", [0.0, 30.0, 1e3, 1e5, -1e7])
@pytest.mark.parametrize("shell", [0.5, 1.0])
@pytest.mark.parametrize("eps", [0.0, 3e-16, 1e-7, -1e-7])
def test_crystals_far_from_an_open_cell(shell, eps, off):
    """Crystal slabs away from their cell along its open axis, the cutoff at a
    neighbour distance: single builds and a fused batch, where the home atoms'
    own position is the tests' centre."""
    rc = 3.61 * np.sqrt(shell) * (1.0 + eps)
    systems = []
    for k in range(66):
        X, cell = workloads.fcc(3.61, (2 + k % 3, 2 + k % 2, 1 + k % 4))
        systems.append(workloads.System(X + 0.1 + np.array([0.0, 0.0, off * (1 + k % 2)]), cell, (True, True, False), rc))
    X, cell = workloads.fcc(3.61, (14, 13, 2))
    print(f"far crystals {shell} {eps} {off}", flush=True)
    _check(X + np.array([0.1, 0.1, off]), rc, cell, (True, True, False), want_R=True)
    got = nlhip.BatchBuilder().run(systems)
    for k, y in enumerate(systems):
        ref = oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc)
        nl = got.pairlist(k)
        assert np.array_equal(nl.first, ref.first), k
        assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S), k


def test_time_of_a_sheet_far_from_its_cell():
    """A sheet one cell thick 1,000 A along its open axis from the cell: twice the
    time of one inside it was, and is the same."""
    L = (200000 / 0.05 / 10) ** 0.5
    s = workloads.random_in_cell(200000, np.diag([L, L, 10.0]), seed=1, cutoff=5.0)
    pbc = (True, True, False)
    print("sheet", flush=True)
    assert _time(s.X + [0.0, 0.0, 1000.0], 5.0, s.cell, pbc) < 1.5 * _time(s.X, 5.0, s.cell, pbc)


def test_time_of_a_batch_far_from_its_cells():
    """A fused batch 300 cells along its open axes from its cells: as long as 3
    cells away (it took six times as long)."""
    t = []
    for w in (3, 300):
        systems = []
        for k in range(200):
            s = workloads.random_cubic(500 + 7 * k, density=0.05, seed=k, cutoff=5.0)
            systems.append(workloads.System(s.X + [0.0, 0.0, w * s.cell[2][2]], s.cell, (True, True, False), 5.0))
        t.append(_time_batch(systems))
    print("far batch", t, flush=True)
    assert t[1] < 1.5 * t[0]

def _batch(nsys, lo, hi, move, seed):
    rng = np.random.default_rng(seed)
    out = []
    for k in range(nsys):
        n = int(rng.integers(lo, hi + 1))
        s = workloads.random_cubic(n, density=0.05, seed=seed + k, cutoff=4.0 + 0.5 * (k % 3))
        out.append(workloads.System(s.X + move(rng, k, n).astype(float) @ np.asarray(s.cell), s.cell,
                                    (True, k % 5 != 1, True), s.cutoff))
    return out


@pytest.mark.parametrize("want_R", [False, True])
@pytest.mark.parametrize("base", [0, 300, -511])
@pytest.mark.parametrize("spread", [1, 128, 251, 252, 253, 256])
def test_batch_windings_of_a_system(spread, base, want_R):
    """Systems of a fused batch that drifted by up to 511 cells, with atoms apart
    by one to twice `spread`, R included."""
    def move(rng, k, n):
        w = rng.choice([0, 0, spread if base <= 0 else -spread, -spread if base == 0 and k % 2 else 0], size=(n, 3))
        return w + base * (k % 3 != 2)
    print(f"batch windings {spread} {base} {want_R}", flush=True)
    systems = _batch(70, 1, 300, move, 17)
    got = nlhip.BatchBuilder().run(systems, want_R=want_R)
    for k, y in enumerate(systems):
        ref = oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc, want_R=want_R)
        nl = got.pairlist(k)
        assert np.array_equal(nl.first, ref.first), k
        assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S), k
        if want_R:
            assert np.array_equal(_bits(nl.R), _bits(ref.R)), k


def test_time_of_a_batch_that_was_never_wrapped():
    """A fused batch of drifted systems: twice an ordinary batch's time it was, and is the same."""
    t = [_time_batch(_batch(200, 500, 2000, lambda rng, k, n: np.full((n, 3), w), 5)) for w in (0, 200)]
    print("drifted batch", t, flush=True)
    assert t[1] < 1.5 * t[0]
