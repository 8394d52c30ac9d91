"""Size edges of the launch paths, each against the oracle bit for bit:
lazy range queries, scans, the pair search.
"""
import ctypes
import dataclasses

import numpy as np
import pytest
import torch

import nlhip
import oracle
from nlhip import _lib, workloads

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a).view(np.int64)


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("wind", [0, 3, 700])
def test_lazy_range_sizes(int_type, bits, wind):
    """Ranges of 1 atom to all of them, growing and shrinking on one handle
    (outputs that suffice and outputs that have to grow), with windings
    inside and beyond the packed range and a reach of 3 cells."""
    s = workloads.random_in_cell(700, [[11.0, 1.0, -0.5], [0.3, 12.0, 0.8], [-0.4, 0.2, 4.1]], seed=5, cutoff=5.0,
                                 pbc=(True, False, True))
    X = s.X.copy()
    X[::7] += wind * np.array(s.cell[0])
    X[3::11] -= wind * np.array(s.cell[2])
    ref = oracle.neighbour_list(X, s.cutoff, s.cell, s.pbc, ti_bits=bits, want_R=True)
    cl = nlhip.build_cell_list(X, s.cutoff, s.cell, s.pbc, int_type=int_type)
    for first, n in [(1, 1), (700, 1), (3, 4), (2, 5), (1, 700), (100, 64), (637, 64)]:
        print(f"lazy range {first} {n}", flush=True)
        offs, j, R, S = nlhip.neighbours_range(cl, first, n)
        a, b = ref.first[first - 1] - 1, ref.first[first - 1 + n] - 1
        assert np.array_equal(offs, ref.first[first - 1:first + n] - ref.first[first - 1])
        assert np.array_equal(j, ref.j[a:b]) and np.array_equal(S, ref.S[a:b])
        assert np.array_equal(_bits(R), _bits(ref.R[a:b]))


@pytest.mark.parametrize("n,rc", [(2047, 1.0), (2049, 1.0), (256 * 2048, 1.0), (256 * 2048 + 1, 1.0),
                                  (2048 * 2048 + 3, 1.0)])
def test_pair_scan_forms(n, rc):
    """Pair counts of 1 and 2 tiles, of 256 tiles (single pass in block order)
    and one more (by ticket), and of 2049 tiles (three kernels)."""
    s = workloads.random_cubic(n, density=0.8, seed=7, cutoff=rc)
    print(f"pair scan {n}", flush=True)
    ref = oracle.neighbour_list(s.X, rc, s.cell, s.pbc, nthreads=8)
    nl = nlhip.neighbour_list(s.X, rc, s.cell, s.pbc)
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)


def _check(X, rc, cell, pbc, int_type=np.int32):
    bits = 32 if int_type == np.int32 else 64
    ref = oracle.neighbour_list(X, rc, cell, pbc, ti_bits=bits, nthreads=8)
    nl = nlhip.neighbour_list(X, rc, cell, pbc, int_type=int_type)
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)


@pytest.mark.parametrize("reps", [(2, 2, 2), (3, 5, 4), (12, 11, 13)])
@pytest.mark.parametrize("shell", [0.5, 1.0, 1.5, 2.0])
@pytest.mark.parametrize("eps", [0.0, 3e-16, -3e-16, 1e-7, -1e-7])
def test_cutoff_on_a_shell(reps, shell, eps):
    """A perfect crystal with the cutoff at a neighbour distance, to the last
    bit and to about the 32-bit filter's error: every pair of that shell is
    decided by the 64-bit test."""
    X, cell = workloads.fcc(3.61, reps)
    rc = 3.61 * np.sqrt(shell) * (1.0 + eps)
    print(f"shell {reps} {shell} {eps}", flush=True)
    _check(X + 0.1, rc, cell, (True, True, True))


@pytest.mark.parametrize("n", [2, 63, 64, 65, 700, 3000, 30000])
@pytest.mark.parametrize("spread", [0, 1, 120, 140])
@pytest.mark.parametrize("pbc", [(True, True, True), (True, False, True), (False, False, False)])
def test_unwrapped_positions(n, spread, pbc):
    """Atoms each moved by its own lattice vector (up to `spread` cells, past
    the packed range of a brick at 140) or, along open axes, far outside the
    grid: 4-byte rows, 8-byte rows and the per-wave path."""
    s = workloads.random_in_cell(n, np.array([[1.0, 0.1, 0.0], [0.2, 1.1, 0.1], [0.0, 0.1, 0.9]]) * (n / 0.06) ** (1 / 3),
                                 seed=n, cutoff=4.0, pbc=pbc)
    rng = np.random.default_rng(n + spread)
    X = s.X + rng.integers(-spread, spread + 1, (n, 3)).astype(float) @ s.cell * (rng.random((n, 1)) < 0.3)
    print(f"unwrapped {n} {spread} {pbc}", flush=True)
    _check(X, 4.0, s.cell, pbc)


@pytest.mark.parametrize("ncells", [(1, 1, 1), (2, 1, 3), (3, 2, 1), (2, 2, 2), (4, 3, 5), (5, 5, 1), (7, 1, 2)])
@pytest.mark.parametrize("per_cell", [1, 6, 24, 70])
def test_small_grids_and_dense_cells(ncells, per_cell):
    """Grids of a few cells, each its own neighbour along the short axes, from
    one atom per cell to more than a wave of home atoms and several passes of
    candidates; the search split over the waves and over several workgroups."""
    rc = 3.0
    n = max(1, per_cell * int(np.prod(ncells)))
    cell = np.diag([(k + 0.2) * rc for k in ncells])
    s = workloads.random_in_cell(n, cell, seed=n, cutoff=rc)
    for pbc in [(True, True, True), (False, True, False)]:
        print(f"grid {ncells} {per_cell} {pbc}", flush=True)
        _check(s.X, rc, cell, pbc, np.int64)


@pytest.mark.parametrize("n", [40000, 1000000])
def test_rows_that_overflow(n):
    """A dense cluster whose atoms outgrow the estimated slot rows, among them
    the last rows of the buffer (the build grows them and counts again)."""
    s = workloads.random_cubic(n, density=0.02, seed=3, cutoff=5.0)
    X = s.X.copy()
    rng = np.random.default_rng(1)
    X[-40:] = X[100] + 0.9 * rng.random((40, 3))
    X[5000:5040] = X[4000] + 0.9 * rng.random((40, 3))
    _check(X, 5.0, s.cell, s.pbc)


def _same_R(nl, ref):
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
    assert np.array_equal(_bits(nl.R), _bits(ref.R))


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("n,density,wind", [(1, 0.05, 0), (7, 0.5, 0), (300, 0.05, 2), (5000, 0.001, 0), (5000, 0.05, 700),
                                            (262144, 0.004, 0), (262145, 0.004, 0), (262145, 0.004, 700)])
def test_R_in_the_fill(int_type, bits, n, density, wind):
    """R of lists with few pairs, of runs of atoms without any, of 4-byte,
    8-byte and 16-byte rows, below and above the size from which R is
    written in cell order."""
    s = workloads.random_cubic(n, density=density, seed=n, cutoff=5.0)
    X = s.X.copy()
    X[::5] += wind * np.asarray(s.cell)[0]
    print(f"R {n} {density} {wind}", flush=True)
    ref = oracle.neighbour_list(X, 5.0, s.cell, s.pbc, ti_bits=bits, want_R=True, nthreads=8)
    _same_R(nlhip.neighbour_list(X, 5.0, s.cell, s.pbc, int_type=int_type, want_R=True), ref)


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("sizes", [[3] * 300, [1, 0, 40, 2, 0, 0, 5] * 60, [700, 5000, 2]])
def test_R_in_the_fill_of_batches(int_type, bits, sizes):
    """Tiles of pairs that span several systems, each with its own cell."""
    systems = []
    for k, n in enumerate(sizes):
        y = workloads.random_cubic(max(n, 1), density=0.05, seed=k, cutoff=4.0 + 0.01 * (k % 7))
        systems.append(dataclasses.replace(y, X=y.X[:n]))
    print(f"R batch {len(sizes)} {bits}", flush=True)
    got = nlhip.BatchBuilder(int_type=int_type).run(systems, want_R=True)
    for k, y in enumerate(systems):
        ref = oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc, ti_bits=bits, want_R=True)
        _same_R(got.pairlist(k), ref)


@pytest.mark.parametrize("n", [100, 20000, 300000])
def test_R_after_the_positions_are_gone(n):
    """Device positions belong to the caller again once a build has returned:
    overwritten at once, and before a later materialisation, R is the same."""
    s = workloads.random_cubic(n, density=0.02, seed=n, cutoff=4.0)
    ref = nlhip.neighbour_list(s.X, 4.0, s.cell, s.pbc, want_R=True)
    print(f"R after {n}", flush=True)
    L = _lib.lib()
    side = torch.cuda.Stream()
    h = _lib.Handle()
    geom = _lib.geometry(s.cell, 4.0, s.pbc, 4)
    m = ctypes.c_int64()
    for step in range(4):
        X = torch.as_tensor(s.X).cuda()
        torch.cuda.synchronize()
        if step < 3:
            _lib.check(L.nlh_neighbour_list(h.ptr, X.data_ptr(), n, ctypes.byref(geom),
                                            _lib.NLH_X_DEVICE | _lib.NLH_WANT_R, ctypes.byref(m)))
        else:
            _lib.check(L.nlh_build_cell_list(h.ptr, X.data_ptr(), n, ctypes.byref(geom), _lib.NLH_X_DEVICE))
            _lib.check(L.nlh_synchronize(h.ptr))
        with torch.cuda.stream(side):
            X.fill_(float("nan"))
            side.synchronize()
        if step == 3:
            _lib.check(L.nlh_materialize(h.ptr, _lib.NLH_WANT_R, ctypes.byref(m)))
        R = np.empty((m.value, 3))
        _lib.check(L.nlh_copy_pairlist(h.ptr, None, None, None, None, R.ctypes.data))
        assert m.value == ref.npairs() and np.array_equal(_bits(R), _bits(ref.R))


def _check_batch(systems, int_type=np.int32, want_R=False):
    bits = 32 if int_type == np.int32 else 64
    got = nlhip.BatchBuilder(int_type=int_type).run(systems, want_R=want_R)
    for k, y in enumerate(systems):
        ref = oracle.neighbour_list(y.X, y.cutoff, y.cell, y.pbc, ti_bits=bits, want_R=want_R)
        nl = got.pairlist(k)
        assert np.array_equal(nl.first, ref.first), k
        assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S), k


@pytest.mark.parametrize("shell", [0.5, 1.0, 1.5])
@pytest.mark.parametrize("eps", [0.0, 3e-16, -3e-16, 1e-7, -1e-7])
@pytest.mark.parametrize("scale", [1.0, 1e-10, 1e6])
def test_batch_cutoff_on_a_shell(shell, eps, scale):
    """Perfect crystals with the cutoff at a neighbour distance, in units from
    metres to micrometres per metre: every pair of that shell is decided by
    the 64-bit test."""
    systems = []
    for k in range(70):
        X, cell = workloads.fcc(3.61, (1 + k % 3, 1 + k % 5, 1 + k % 4))
        systems.append(workloads.System((X + 0.1 * (k % 7)) * scale, cell * scale, (True, k % 2 == 0, True),
                                        3.61 * scale * np.sqrt(shell) * (1.0 + eps)))
    print(f"batch shell {shell} {eps} {scale}", flush=True)
    _check_batch(systems)


@pytest.mark.parametrize("wind", [0, 1, 128, 129, 300, 511, 512])
@pytest.mark.parametrize("pbc", [(True, True, True), (True, False, True), (False, False, False)])
def test_batch_windings_and_far_atoms(wind, pbc):
    """Atoms moved by lattice vectors: inside the packed differences, beyond
    them, and beyond the packed windings; along open axes they lie far
    outside the cell."""
    rng = np.random.default_rng(wind)
    systems = []
    for k in range(72):
        n = [1, 2, 7, 63, 64, 65, 200, 900][k % 8]
        cell = (np.eye(3) + 0.1 * rng.random((3, 3))) * (n / 0.06) ** (1 / 3) * (1.0, 1.0, 0.6 + 0.2 * (k % 5))
        X = rng.random((n, 3)) @ cell
        X += (rng.integers(-wind, wind + 1, (n, 3)) * (rng.random((n, 1)) < 0.2)) @ cell
        systems.append(workloads.System(X, cell, pbc, 3.0 + 0.3 * (k % 6)))
    print(f"batch windings {wind} {pbc}", flush=True)
    _check_batch(systems, np.int64 if wind % 2 else np.int32)


@pytest.mark.parametrize("sizes", [[2048] * 64, [1] * 700 + [2048], [2047, 1, 0, 1] * 20, [0] * 70 + [3], [2049] + [5] * 70])
def test_batch_unit_edges(sizes):
    """Units of one full system, of hundreds of atoms of their own system, of
    systems without atoms; one system beyond a unit (the general pipeline)."""
    systems = []
    for k, n in enumerate(sizes):
        y = workloads.random_cubic(max(n, 1), density=0.05, seed=k, cutoff=3.5 + 0.1 * (k % 9))
        systems.append(dataclasses.replace(y, X=y.X[:n]))
    print(f"batch units {len(sizes)}", flush=True)
    _check_batch(systems)


@pytest.mark.parametrize("n", [40, 400, 2000])
def test_batch_rows_that_overflow(n):
    """Clusters whose atoms outgrow the estimated slot rows by far, the last
    atoms of the batch among them, in cells whose images are neighbours too."""
    rng = np.random.default_rng(n)
    systems = []
    for k in range(66):
        cell = np.eye(3) * (6.0 if k % 3 == 0 else 40.0)
        X = rng.random((n if k % 3 else 20, 3)) * 40.0
        X[-min(n, 30):] = 20.0 + 0.5 * rng.random((len(X[-min(n, 30):]), 3))
        systems.append(workloads.System(X, cell, (True, True, k % 2 == 0), 5.0))
    print(f"batch overflow {n}", flush=True)
    _check_batch(systems)


@pytest.mark.parametrize("n", [50, 1200, 20000])
@pytest.mark.parametrize("shift", [0.25, 0.5, 30.0, 1e7])
@pytest.mark.parametrize("pbc", [(False, False, False), (True, True, False), (False, True, True)])
def test_open_axes_far_from_the_cell(n, shift, pbc):
    """Positions shifted against the cell by parts and multiples of it along
    open axes, so that edge cells hold atoms from far outside (up to all of
    them, more than a brick stages)."""
    if n == 20000 and sum(pbc) < 2 and shift > 0.25:
        pytest.skip("a few cells hold every atom: slow in the oracle")
    s = workloads.random_cubic(n, density=0.05, seed=n, cutoff=4.0)
    X = s.X - np.where(pbc, 0.0, shift) * np.diag(np.asarray(s.cell))
    print(f"open {n} {shift} {pbc}", flush=True)
    _check(X, 4.0, s.cell, pbc)


@pytest.mark.parametrize("n", [0, 1, 3, 500, 5000])
@pytest.mark.parametrize("int_type", [np.int32, np.int64])
@pytest.mark.parametrize("shift", [0, 1, 2, 3])
def test_copy_to_device_memory(n, int_type, shift):
    """Lists copied to device memory of any element alignment, all arrays and
    some, while the default stream still writes that memory."""
    s = workloads.random_cubic(max(n, 1), density=0.05, seed=n, cutoff=5.0)
    X = s.X[:n]
    ref = nlhip.neighbour_list(X, 5.0, s.cell, s.pbc, int_type=int_type, want_R=True)
    td = torch.int32 if int_type == np.int32 else torch.int64
    h = _lib.Handle()
    geom = _lib.geometry(s.cell, 5.0, s.pbc, 4 if int_type == np.int32 else 8)
    m = ctypes.c_int64()
    print(f"copy {n} {shift}", flush=True)
    L = _lib.lib()
    _lib.check(L.nlh_neighbour_list(h.ptr, X.ctypes.data, n, ctypes.byref(geom), _lib.NLH_WANT_R, ctypes.byref(m)))
    P = m.value
    for skip in [None, 0, 2, 4]:
        out = [torch.zeros(k + 8, dtype=t, device="cuda") for k, t in
               ((P, td), (P, td), (3 * P, td), (n + 1, td), (3 * P, torch.float64))]
        big = torch.empty(1 << 26, device="cuda")
        for _ in range(4):
            big.fill_(1.0)
        for o in out:
            o.fill_(-7)
        ptrs = [None if k == skip else o[shift:].data_ptr() for k, o in enumerate(out)]
        _lib.check(L.nlh_copy_pairlist(h.ptr, *ptrs))
        for k, (o, r) in enumerate(zip(out, (ref.i, ref.j, ref.S, ref.first, ref.R))):
            o, r = o.cpu().numpy(), np.asarray(r).reshape(-1)
            want = np.full(o.shape, -7, o.dtype)
            if k != skip:
                want[shift:shift + r.size] = r
            assert np.array_equal(o, want), (k, skip)


@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
@pytest.mark.parametrize("n,per_cell,wind", [(1, 1.0, 0), (2, 0.001, 0), (1023, 6.0, 700), (1024, 0.25, 0), (1025, 0.2501, 3),
                                             (2047, 2047.0, 0), (2048, 0.5, 0), (2048, 0.49, 0), (2049, 0.5, 0),
                                             (4096, 4096.0, 1), (300, 300.0, 0), (5000, 5000.0, 2)])
def test_cell_list_sort_forms(n, per_cell, wind, int_type, bits):
    """The cell list of one system around the sizes (atoms, cells) up to which
    one workgroup sorts it, from empty cells to all atoms in one; a position
    that is none is refused in each form."""
    rc = 2.0
    cells = max(1, int(round(n / per_cell)))
    shape = (cells, 1, 1) if cells < 64 else (16, 16, max(1, cells // 256))
    cell = np.diag([(k + 0.01) * rc for k in shape])
    rng = np.random.default_rng(n)
    X = rng.random((n, 3)) @ cell
    X[::5] += wind * cell[0]
    print(f"sort {n} {shape} {wind}", flush=True)
    pbc = (True, True, True)
    cl = nlhip.build_cell_list(X, rc, cell, pbc, int_type=int_type)
    ids = oracle.cell_ids(X, rc, cell, pbc, ti_bits=bits)[0]
    perm = np.argsort(ids, kind="stable")
    assert np.array_equal(cl.perm, perm + 1) and np.array_equal(cl.cell_id, ids[perm])
    assert np.array_equal(cl.cell_offsets, np.searchsorted(ids[perm], np.arange(1, int(np.prod(shape)) + 2)) + 1)
    assert np.array_equal(cl.X, X[perm])
    if per_cell <= 10.0:
        _check(X, rc, cell, pbc, int_type)
    X[n // 2, 1] = np.nan
    with pytest.raises(nlhip.NLHInvalidError):
        nlhip.build_cell_list(X, rc, cell, pbc, int_type=int_type)


@pytest.mark.parametrize("n", [3900, 5300, 43690, 43691, 120000])
@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
def test_lists_in_host_memory(n, int_type, bits):
    """Positions and lists around the sizes from which several threads copy
    them, on one handle (threads and pinned memory kept) and a fresh one, and
    two handles at once from two threads."""
    import threading

    s = workloads.random_cubic(n, density=0.05, seed=n, cutoff=5.0)
    ref = oracle.neighbour_list(s.X, 5.0, s.cell, s.pbc, ti_bits=bits, want_R=True, nthreads=8)
    print(f"host list {n} {bits}", flush=True)
    bad = []

    def work():
        h = _lib.Handle()
        for want_R in (False, True, True):
            nl = nlhip.neighbour_list(s.X, 5.0, s.cell, s.pbc, int_type=int_type, want_R=want_R, handle=h)
            ok = (np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
                  and np.array_equal(nl.first, ref.first) and (not want_R or np.array_equal(_bits(nl.R), _bits(ref.R))))
            if not ok:
                bad.append(want_R)

    work()
    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


@pytest.mark.parametrize("n", [12288, 30000])
@pytest.mark.parametrize("int_type,bits", [(np.int32, 32), (np.int64, 64)])
def test_slot_rows_follow_the_last_builds(n, int_type, bits):
    """Repeated builds on one handle: a crystal whose rows shrink to its counts,
    atoms that outgrow them (4-byte rows, 8-byte rows of unwrapped atoms), 16-byte
    rows, another density and cutoff, and back."""
    X, cell = workloads.fcc(3.61, (15, 15, (n + 899) // 900))
    X, rng = X[:n], np.random.default_rng(n)
    pbc = (True, True, False)
    close = X.copy()
    close[-60:] = X[50] + rng.random((60, 3))
    moved = X.copy()
    moved[::4] += cell[0] * rng.integers(-3, 4, (len(X[::4]), 1))
    wide = X.copy()
    wide[::9] += 600 * cell[1]
    h = _lib.Handle()
    for k, (Y, rc) in enumerate([(X, 4.9), (X, 4.9), (X, 4.9), (moved, 4.9), (close, 4.9), (X, 4.9), (X, 6.0), (X, 4.9),
                                 (X * 0.9, 4.9), (wide, 4.9), (moved, 4.9), (X, 4.9)]):
        print(f"slot rows {n} {bits} {k}", flush=True)
        for want_R in ((False, True) if k in (2, 4) else (False,)):
            ref = oracle.neighbour_list(Y, rc, cell, pbc, ti_bits=bits, want_R=want_R, nthreads=8)
            nl = nlhip.neighbour_list(Y, rc, cell, pbc, int_type=int_type, want_R=want_R, handle=h)
            assert np.array_equal(nl.first, ref.first)
            assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
            if want_R:
                assert np.array_equal(_bits(nl.R), _bits(ref.R))
