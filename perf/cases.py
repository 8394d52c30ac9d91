"""Performance cases: the neighbour-list work a program asks of this package.

Five ways in, as programs use them:

  list   nlhip.neighbour_list on a CUDA tensor with a kept handle: a script or
         an MD loop in Python; the PairList comes back as tensors of its own
  build  nlh_neighbour_list through the C ABI with resident positions, the
         result read in place through nlh_pairlist_device: a host code (the
         Julia extension, a compiled MD code) that keeps its data on the GPU
  host   nlhip.neighbour_list on a numpy array: positions up, PairList down
  batch  BatchBuilder.rebuild of many small systems on resident positions,
         the result read in place: training and screening workloads
  lazy   build_cell_list, then the neighbours of a range of atoms
         (neighbours_range): analysis of part of a system

Systems: "cube" uniform atoms in a cube, "tri" uniform atoms in a sheared
cell, "fcc" a copper crystal (a = 3.61 A) jittered by 0.05 A, "slab" that
crystal in a sheared cell with 30 A of vacuum.  Density in atoms/A^3, cutoff
in A, float64 positions; "ti" is the index type (4 or 8 bytes).
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "neighbourlists.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import nlhip  # noqa: E402
from nlhip import _lib  # noqa: E402
from nlhip.batch import BatchBuilder  # noqa: E402

_A = 3.61   # copper lattice constant (A)
_BALL = 4.0 / 3.0 * math.pi


def _single(name, kind, system, n, **kw):
    case = {"name": name, "kind": kind, "system": system, "n": n, "rho": 0.05, "rc": 5.0, "pbc": "TTT", "ti": 4,
            "want_R": False, "query": 0}
    case.update(kw)
    return case


def listed():
    return [
        # the smallest calls: a crystal cell that is its own neighbour (two cells
        # across at most, images in every direction), e.g. phonon displacements
        _single("fcc_96", "list", "fcc", 96, reps=423),
        # the smallest size of the reference's published table: one small MD cell
        _single("cube_1k", "list", "cube", 1000),
        # the table's middle
        _single("cube_10k", "list", "cube", 10000),
        # an odd-sized sheared cell, open along one axis, with the vectors R and
        # 64-bit indices: input of a message-passing potential
        _single("tri_20k_R_i64", "list", "tri", 20011, rho=0.07, pbc="TTF", ti=8, want_R=True),
        # the headline: the table's largest size, one rebuild of an MD loop
        _single("cube_100k", "build", "cube", 100000),
        # the same call for a potential that reads R, at the largest served size
        _single("cube_200k_R", "build", "cube", 200000, want_R=True),
        # the largest single builds
        _single("cube_1M", "build", "cube", 1000000),
        _single("slab_1M", "build", "slab", 4 * 63 ** 3, pbc="TTF"),
        # numpy in, numpy out, at the headline size
        _single("host_100k", "host", "cube", 100000),
        # neighbours of a few thousand atoms of a larger system, no pair list
        _single("lazy_50k", "lazy", "cube", 50000, query=4096),
        # a training minibatch of small structures, rebuilt on new positions
        {"name": "batch_128", "kind": "batch", "nsys": 128, "nmin": 8, "nmax": 400, "mix": 7, "ti": 4},
        # screening: thousands of structures of uneven size in one call
        {"name": "batch_4096", "kind": "batch", "nsys": 4096, "nmin": 8, "nmax": 2048, "mix": 7, "ti": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["list", "list", "build", "build", "host", "batch", "lazy"])
    if kind == "batch":
        nsys = _log_uniform(rng, 64, 3000)
        return {"kind": kind, "nsys": nsys, "nmin": 8, "nmax": _log_uniform(rng, 100, 2000),
                "mix": rng.randrange(1, 1 << 30), "ti": rng.choice([4, 4, 8])}
    lo, hi = {"list": (100, 60000), "build": (20000, 700000), "host": (1000, 100000), "lazy": (5000, 200000)}[kind]
    n = _log_uniform(rng, lo, hi)
    pbc = "".join(rng.choice("TTTF") for _ in range(3))
    case = _single(None, kind, rng.choice(["cube", "tri"]), n, rho=round(rng.uniform(0.04, 0.09), 4),
                   rc=round(rng.uniform(4.0, 6.0), 3), pbc=pbc, ti=rng.choice([4, 4, 4, 8]))
    del case["name"]
    if kind == "lazy":
        case["query"] = rng.randrange(500, 5000)
    elif n <= 200000:
        case["want_R"] = rng.random() < 0.3
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

def _crystal(reps):
    basis = np.array([[0, 0, 0], [0, 0.5, 0.5], [0.5, 0, 0.5], [0.5, 0.5, 0]])
    g = np.stack(np.meshgrid(*(np.arange(r) for r in reps), indexing="ij"), -1).reshape(-1, 3)
    return (g[:, None, :] + basis[None, :, :]).reshape(-1, 3) * _A


def _sheared(d):
    return d * np.array([[1.0, 0.08, -0.11], [0.05, 1.0, 0.13], [-0.09, 0.04, 1.0]])


def _cell(case):
    """Cell matrix, rows the lattice vectors."""
    if case["system"] == "fcc":
        return np.diag([_A * r for r in _reps(case)])
    if case["system"] == "slab":
        k = round((case["n"] / 4) ** (1 / 3))
        return np.array([[k * _A, 0, 0], [round(0.3 * k) * _A, k * _A, 0], [0.2 * k * _A, 0, k * _A + 30.0]])
    d = (case["n"] / case["rho"]) ** (1 / 3)
    return _sheared(d) if case["system"] == "tri" else np.eye(3) * d


def _heights(cell):
    """Face-to-face heights of the cell."""
    vol = abs(np.dot(cell[:, 0], np.cross(cell[:, 1], cell[:, 2])))
    return vol / np.linalg.norm(np.cross(cell[[1, 2, 0]], cell[[2, 0, 1]]), axis=1)


def _reps(case):
    r = case["reps"]
    return r // 100, r // 10 % 10, r % 10


def _shuffled(rng, u, pbc, keep=None):
    """Fractional coordinates u from another origin along the periodic axes
    and in another order (the rows `keep` stay where they are as a set): the
    pairs are the same ones, between other atoms at other places."""
    u = u.copy()
    for k in range(3):
        if pbc[k]:
            u[:, k] = (u[:, k] + rng.random()) % 1.0
    if keep is None:
        return u[rng.permutation(len(u))]
    order = np.arange(len(u))
    inside = np.zeros(len(u), dtype=bool)
    inside[keep] = True
    order[inside] = rng.permutation(order[inside])
    order[~inside] = rng.permutation(order[~inside])
    return u[order]


def _positions(case, seed):
    """The case's configuration as `seed` places and orders it (its pair count
    is the case's, as a result of one size is what a caller can compare)."""
    rng, fixed = np.random.default_rng(seed), np.random.default_rng(case["n"])
    if case["system"] in ("fcc", "slab"):
        # in the order a crystal is written in, drifted by up to a lattice constant
        reps = _reps(case) if case["system"] == "fcc" else (round((case["n"] / 4) ** (1 / 3)),) * 3
        X = _crystal(reps)
        X = X + 0.05 * fixed.standard_normal(X.shape) + _A * rng.random(3) * np.array(_pbc(case))
        return np.roll(X, int(rng.integers(len(X))), axis=0)
    keep = slice(_query_first(case) - 1, _query_first(case) - 1 + case["query"]) if case["query"] else None
    return _shuffled(rng, fixed.random((case["n"], 3)), _pbc(case), keep) @ _cell(case)


def _pbc(case):
    return tuple(c == "T" for c in case["pbc"])


class _System:
    def __init__(self, X, cell, pbc, cutoff):
        self.X, self.cell, self.pbc, self.cutoff = X, cell, pbc, cutoff


def _batch_plan(case):
    """(atoms, cell, pbc, cutoff) of every system: sizes log-uniform, a tenth
    of them 1 to 4 atoms in a cell smaller than the cutoff."""
    rng = np.random.default_rng(case["mix"])
    out = []
    for _ in range(case["nsys"]):
        tiny = rng.random() < 0.1
        n = int(rng.integers(1, 5)) if tiny else int(round(math.exp(rng.uniform(math.log(case["nmin"]),
                                                                               math.log(case["nmax"])))))
        d = (n / rng.uniform(0.04, 0.09)) ** (1 / 3)
        cell = d * (np.eye(3) + (1 - np.eye(3)) * rng.uniform(-0.15, 0.15, (3, 3)))
        pbc = tuple(bool(b) for b in rng.random(3) < 0.5)
        out.append((n, cell, (True, True, True) if tiny else pbc, float(rng.uniform(4.0, 6.0))))
    return out


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "batch":
        rng, fixed = np.random.default_rng(seed), np.random.default_rng(case["mix"] + 1)
        systems = [_System(_shuffled(rng, fixed.random((n, 3)), pbc) @ cell, cell, pbc, rc)
                   for n, cell, pbc, rc in _batch_plan(case)]
        X = np.concatenate([s.X for s in systems])
        state["X"] = torch.from_numpy(X).cuda()
        state["X_host"] = X
        state["builder"] = BatchBuilder(np.int64 if case["ti"] == 8 else np.int32)
        torch.cuda.synchronize()
        state["builder"].run(systems, X_device=state["X"], copy=False)
        return state
    X, cell = _positions(case, seed), _cell(case)
    state.update(cell=cell, pbc=_pbc(case), int_type=np.int64 if case["ti"] == 8 else np.int32,
                 X=X if case["kind"] == "host" else torch.from_numpy(np.ascontiguousarray(X)).cuda(),
                 handle=_lib.Handle(), count=ctypes.c_int64())
    if case["kind"] == "build":
        state["geom"] = _lib.geometry(cell, case["rc"], state["pbc"], case["ti"])
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------

class _DeviceArray:
    """Memory of a build's handle, which the tensors made from it keep alive."""

    def __init__(self, handle, ptr, shape, typestr):
        self.handle = handle
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": typestr, "version": 3}


def _wrap(handle, ptr, shape, typestr):
    dtype = {"<i4": torch.int32, "<i8": torch.int64, "<f8": torch.float64}[typestr]
    if 0 in shape:
        return torch.empty(shape, dtype=dtype, device="cuda")
    return torch.as_tensor(_DeviceArray(handle, ptr, shape, typestr), device="cuda")


def _pairlist_in_place(handle, nfirst):
    v = _lib.PairListView()
    _lib.check(_lib.lib().nlh_pairlist_device(handle.ptr, ctypes.byref(v)), "pairlist")
    t = "<i8" if v.ti_bytes == 8 else "<i4"
    out = [_wrap(handle, v.i, (v.npairs,), t), _wrap(handle, v.j, (v.npairs,), t),
           _wrap(handle, v.S, (v.npairs, 3), t), _wrap(handle, v.first, (nfirst,), t)]
    if v.R:
        out.append(_wrap(handle, v.R, (v.npairs, 3), "<f8"))
    return out


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        b = state["builder"]
        b.rebuild(state["X_host"], X_device=state["X"], copy=False)
        po = np.zeros(case["nsys"] + 1, dtype=np.int64)
        _lib.check(_lib.lib().nlh_batch_pair_offsets(b.handle.ptr, po.ctypes.data_as(ctypes.POINTER(ctypes.c_int64))),
                   "pair offsets")
        return _pairlist_in_place(b.handle, state["X"].shape[0] + case["nsys"]) + [po]
    if kind == "build":
        flags = _lib.NLH_X_DEVICE | (_lib.NLH_WANT_R if case["want_R"] else 0)
        h, n = state["handle"], case["n"]
        _lib.check(_lib.lib().nlh_neighbour_list(h.ptr, state["X"].data_ptr(), n, ctypes.byref(state["geom"]), flags,
                                                 ctypes.byref(state["count"])), "neighbour_list")
        return _pairlist_in_place(h, n + 1)
    if kind == "lazy":
        cl = nlhip.build_cell_list(state["X"], case["rc"], state["cell"], state["pbc"], int_type=state["int_type"],
                                   handle=state["handle"])
        return list(nlhip.neighbours_range(cl, _query_first(case), case["query"]))
    nl = nlhip.neighbour_list(state["X"], case["rc"], state["cell"], state["pbc"], int_type=state["int_type"],
                              want_R=case["want_R"], handle=state["handle"])
    return [nl.i, nl.j, nl.S, nl.first] + ([nl.R] if case["want_R"] else [])


def _query_first(case):
    return max(1, (case["n"] - case["query"]) // 2)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _expected_pairs(n, cell, pbc, rc):
    """Uniform atoms: every atom sees its sphere, less the caps beyond open
    faces (0.375 rc / height of the sphere on average)."""
    share = 1.0
    for h, p in zip(_heights(cell), pbc):
        share *= 1.0 if p else max(1.0 - 0.375 * rc / h, min(1.0, 0.5 * h / rc))
    return n * n / abs(np.linalg.det(cell)) * _BALL * rc ** 3 * share


def work(case):
    """Positions read and the result written once; one distance (8 flops) per
    neighbour found and one cell (18 flops) per atom."""
    ti = case["ti"]
    if case["kind"] == "batch":
        plan = _batch_plan(case)
        n = sum(p[0] for p in plan)
        pairs = sum(_expected_pairs(*p) for p in plan)
        per_pair, extra = 5 * ti, ti * (n + case["nsys"]) + 8 * (case["nsys"] + 1)
        return {"bytes": float(24 * n + per_pair * pairs + extra), "flops": float(18 * n + 8 * pairs)}
    n = case["n"]
    if case["system"] in ("fcc", "slab"):
        pairs = 42.0 * n
    else:
        pairs = _expected_pairs(n, _cell(case), _pbc(case), case["rc"])
    if case["kind"] == "lazy":
        pairs *= case["query"] / n
        return {"bytes": float(24 * n + (4 * ti + 24) * pairs + 8 * (case["query"] + 1)),
                "flops": float(18 * n + 8 * pairs)}
    per_pair = 5 * ti + (24 if case["want_R"] else 0)
    return {"bytes": float(24 * n + per_pair * pairs + ti * (n + 1)), "flops": float(18 * n + 8 * pairs)}


# ---------------------------------------------------------------------------
# the computed numbers (R) in 64 bits
# ---------------------------------------------------------------------------

def _pair_vectors(X, cell, pbc, rc, lo, hi):
    """R of every pair of atoms lo <= i < hi, in the list's order: by i, then
    neighbour cell (z outermost, x innermost), then cell order."""
    n = X.shape[0]
    heights = _heights(cell)
    nc = np.maximum(np.floor(heights / rc).astype(np.int64), 1)
    reach = np.ceil(rc * (nc / heights)).astype(np.int64)
    inv = np.linalg.inv(cell)
    c = np.floor((X[:, :1] * inv[0] + X[:, 1:2] * inv[1] + X[:, 2:] * inv[2]) * nc).astype(np.int64)
    wind = np.zeros_like(c)
    for k in range(3):
        if pbc[k]:
            wind[:, k] = c[:, k] // nc[k]
            c[:, k] -= wind[:, k] * nc[k]
        else:
            c[:, k] = np.clip(c[:, k], 0, nc[k] - 1)
    cid = c[:, 0] + nc[0] * (c[:, 1] + nc[1] * c[:, 2])
    perm = np.argsort(cid, kind="stable")
    start = np.zeros(int(nc.prod()) + 1, dtype=np.int64)
    np.cumsum(np.bincount(cid, minlength=int(nc.prod())), out=start[1:])
    atoms = np.arange(lo, hi)
    ri, rR = [], []
    for dz in range(-reach[2], reach[2] + 1):
        for dy in range(-reach[1], reach[1] + 1):
            for dx in range(-reach[0], reach[0] + 1):
                a = c[lo:hi] + np.array([dx, dy, dz])
                ok = np.ones(hi - lo, dtype=bool)
                s = np.zeros_like(a)
                for k in range(3):
                    if pbc[k]:
                        s[:, k] = a[:, k] // nc[k]
                        a[:, k] -= s[:, k] * nc[k]
                    else:
                        ok &= (a[:, k] >= 0) & (a[:, k] < nc[k])
                i, a, s = atoms[ok], a[ok], s[ok]
                g = a[:, 0] + nc[0] * (a[:, 1] + nc[1] * a[:, 2])
                cnt = start[g + 1] - start[g]
                off = np.cumsum(cnt) - cnt
                q = np.arange(int(cnt.sum())) - np.repeat(off, cnt)
                j = perm[np.repeat(start[g], cnt) + q]
                s, i = np.repeat(s, cnt, axis=0), np.repeat(i, cnt)
                S = (s + wind[i] - wind[j]).astype(np.float64)
                R = (X[j] - X[i]) + ((cell[0] * S[:, :1] + cell[1] * S[:, 1:2]) + cell[2] * S[:, 2:])
                r2 = (R[:, 0] * R[:, 0] + R[:, 1] * R[:, 1]) + R[:, 2] * R[:, 2]
                hit = (r2 < rc * rc) & ~((i == j) & (s == 0).all(axis=1))
                ri.append(i[hit])
                rR.append(R[hit])
    order = np.argsort(np.concatenate(ri), kind="stable")
    return np.concatenate(rR)[order]


def exact(case, seed):
    """R; indices, shifts and offsets are whole numbers and have no other value."""
    if case["kind"] == "lazy":
        lo = _query_first(case) - 1
        R = _pair_vectors(_positions(case, seed), _cell(case), _pbc(case), case["rc"], lo, lo + case["query"])
        return [None, None, R, None]
    if not case.get("want_R") or case["n"] > 250000:
        return None
    R = _pair_vectors(_positions(case, seed), _cell(case), _pbc(case), case["rc"], 0, case["n"])
    return [None, None, None, None, R]
