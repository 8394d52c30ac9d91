"""The pair scan where no block waits for another, and the scans of sizes
served in block order, by ticket and by three kernels.
"""
import ctypes as C
import os
import re

import numpy as np
import pytest
import torch

import nlhip
import oracle
from nlhip import _lib, workloads

HERE = os.path.dirname(os.path.abspath(__file__))
HEADER = os.path.join(HERE, "..", "neighbourlists.jl_amd", "csrc", "nlhip_internal.h")
LIB = os.path.join(HERE, "user_kernel", "libnlh_scan_help.so")
TILE = 2048


def _constants():
    """The integer constants of the header that the scans' sizes follow from."""
    k = {}
    for line in open(HEADER):
        m = re.match(r"constexpr (?:int|unsigned|int64_t|int32_t) (k\w+ = .*?);", line)
        for part in m.group(1).split(", k") if m else ():
            name, expr = (part if part.startswith("k") else "k" + part).split(" = ", 1)
            try:
                k[name] = int(eval(expr.replace("/", "//"), {}, k))
            except (NameError, SyntaxError):
                pass
    return k


def _stuck(tiles, launches, per_cu, cus=32, xcds=8):
    """Whether `launches` scans of `tiles` blocks in block order can wait for
    one another for ever: launch l's next block finds no place on XCD l mod m
    (an XCD starts a launch's blocks in order), and each such XCD is full of
    the other launches' blocks, all of which wait."""
    per_xcd = -(-tiles // xcds)
    for m in range(2, min(launches, xcds) + 1):
        if all(per_xcd * sum(1 for l in range(launches) if l % m != x) >= per_cu * cus for x in range(m)):
            return True
    return False


def test_block_order_is_for_scans_that_cannot_block_one_another():
    """Scans without tickets leave a place on every XCD free, with every
    hardware queue of several processes at one: three scans of 1,024 tiles
    would not."""
    k = _constants()
    assert _stuck(1024, 3, 5) and not _stuck(256, 4, 5) and _stuck(256, 8, 5)
    for limit, per_cu in ((8 * k["kBucketScanBlocksPerCu"], 8), (8 * k["kCellScanBlocksPerCu"], 5)):
        for queues in range(2, k["kHwQueues"] + 1):
            assert not _stuck(limit, queues, per_cu)
    assert k["kXcds"] == 8 and k["kXcdCus"] == 32 and k["kHwQueues"] >= 32


def _scan(counts, ti_bytes, reps):
    if not os.path.exists(LIB):
        raise RuntimeError(f"{LIB} is missing: run the package build first")
    L = C.CDLL(LIB)
    f = L.scan_help
    f.argtypes = [C.c_void_p, C.c_int64, C.c_int32, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p,
                  C.c_void_p, C.POINTER(C.c_int64)]
    n, words = len(counts), C.c_int64()
    f(None, n, ti_bytes, None, None, None, 0, None, None, C.byref(words))
    flags = np.where(np.arange(n) % 3 == 0, 1 << 30, 0).astype(np.int32)   # the slot-row format's bit
    c = torch.as_tensor(counts | flags).cuda()
    tiles = int(counts.sum()) // 256 + 2
    for _ in range(reps):
        off = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
        first = torch.full((n + 1,), -1, dtype=torch.int32 if ti_bytes == 4 else torch.int64, device="cuda")
        ta = torch.full((2 * tiles,), -1, dtype=torch.int32, device="cuda")
        status = torch.zeros(64, dtype=torch.int32, device="cuda")
        look = torch.full((words.value,), 1 << 40, dtype=torch.int64, device="cuda")
        torch.cuda.synchronize()
        assert f(c.data_ptr(), n, ti_bytes, off.data_ptr(), first.data_ptr(), ta.data_ptr(), tiles, status.data_ptr(),
                 look.data_ptr(), None) == 0
        want = np.concatenate([[0], np.cumsum(counts, dtype=np.int64)])
        assert np.array_equal(off.cpu().numpy(), want)
        assert np.array_equal(first.cpu().numpy(), want + 1)
        t0 = np.arange(0, want[-1], 256)
        owner = np.searchsorted(want, t0, side="right") - 1
        got = ta.cpu().numpy().reshape(-1, 2)[:len(t0)]
        assert np.array_equal(got[:, 0], owner) and np.array_equal(got[:, 1], t0 - want[owner])
        st = status[:2].cpu().numpy().view(np.int64)
        assert st[0] == want[-1] and int(status[2]) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("ti_bytes", [4, 8])
@pytest.mark.parametrize("n", [1, TILE, TILE + 1, 65 * TILE, 257 * TILE + 5, 1025 * TILE + 1, 2048 * TILE])
def test_pair_scan_that_helps_itself(n, ti_bytes):
    print(f"scan help {n} {ti_bytes}", flush=True)
    rng = np.random.default_rng(n)
    _scan(rng.integers(0, 40, n).astype(np.int32) * (rng.random(n) < 0.6), ti_bytes, 3)


@pytest.mark.gpu
@pytest.mark.parametrize("tiles,more", [(1, 1), (40, 0), (40, 1), (1024, 0), (1024, 1), (2048, 0), (2048, 1)])
def test_pair_scan_sizes(tiles, more):
    """Pair counts of as many tiles as one, as the sort scans take in block
    order, as a device holds at once, and as one kernel scans, and one more."""
    n = tiles * TILE + more
    s = workloads.random_cubic(n, density=0.5, seed=11, cutoff=1.0)
    print(f"pair scan {n}", flush=True)
    ref = oracle.neighbour_list(s.X, 1.0, s.cell, s.pbc, nthreads=8)
    nl = nlhip.neighbour_list(s.X, 1.0, s.cell, s.pbc)
    assert np.array_equal(nl.first, ref.first)
    assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(34, 60, 40), (34, 61, 40), (128, 128, 128), (128, 128, 129), (161, 161, 162)])
def test_cell_scan_sizes(cells):
    """The atomic sort's cell counts of as many tiles as go in block order, by
    ticket, up to 1,024 and beyond, and by three kernels."""
    cell = np.diag([(k + 0.01) * 1.0 for k in cells])
    s = workloads.random_in_cell(5000, cell, seed=3, cutoff=1.0)
    print(f"cell scan {cells}", flush=True)
    h = _lib.Handle()
    t = h.get_tuning()
    h.set_tuning(t.brick_atoms, t.fill_block, t.fill_pairs, t.count_block, cell_sort=1)
    for _ in range(2):
        nl = nlhip.neighbour_list(s.X, 1.0, s.cell, s.pbc, handle=h)
        ref = oracle.neighbour_list(s.X, 1.0, s.cell, s.pbc)
        assert np.array_equal(nl.first, ref.first)
        assert np.array_equal(nl.i, ref.i) and np.array_equal(nl.j, ref.j) and np.array_equal(nl.S, ref.S)
