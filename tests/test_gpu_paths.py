"""Size edges of the launch paths, each against the oracle bit for bit:
lazy range queries, scans.
"""
import numpy as np
import pytest

import nlhip
import oracle
from nlhip import workloads

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
