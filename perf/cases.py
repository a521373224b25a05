"""Performance cases of the library: the calls that programs around an AMG solver make.

A case names a kind of call, an operator and its size.  Operators carry random
coefficients drawn from the seed: finite-volume diffusion operators with
log-normal conductivities (5-point in 2D, 7-point in 3D), the random 27-point
stencil and the lognormal irregular matrix of the benchmark.  Transfer
operators are smoothed aggregation, P = (I - 2/3 D^-1 A) P0 and R = P^T, over
2x2 / 2x2x2 / 3x3x3 blocks (partial blocks at the far faces of odd grids) or
random aggregates of 4 to 12 rows.  Every call uses the library's default
schedule, as a program does that does not tune.
"""
import functools
import json
import math
import random

import numpy as np
import torch

from sp3mm4amg_amd import lib
from sp3mm4amg_amd.amg import GraphVCycle
from sp3mm4amg_amd.csr import CSR

OMEGA = 2.0 / 3.0
DEV = "cuda" if torch.cuda.is_available() else "cpu"


def listed():
    return [
        # the coarse end of a hierarchy or a small 2D problem: latency and launches
        dict(name="rap_2d_64", kind="rap", op="5pt", nx=64, ny=64, nz=1, path="direct", precision="fp64"),
        # an ordinary 3D operator on a ragged grid
        dict(name="rap_3d_odd", kind="rap", op="7pt", nx=61, ny=47, nz=53, path="direct", precision="fp64"),
        # the finest level of a large 3D problem, the benchmark's own size
        dict(name="rap_3d_128", kind="rap", op="7pt", nx=128, ny=128, nz=128, path="direct", precision="fp64"),
        # finite elements on a ragged grid: wide rows, FP64
        dict(name="rap_27pt_odd", kind="rap", op="27pt", nx=41, ny=56, nz=37, path="direct", precision="fp64"),
        # the same kind of operator, large, FP32 operands with FP64 sums
        dict(name="rap_27pt_mixed64", kind="rap", op="27pt", nx=100, ny=100, nz=100, path="direct",
             precision="mixed64"),
        # two SpGEMMs with the intermediate kept in HBM, at the size of the reference's published group
        dict(name="pair_3d_80", kind="rap", op="7pt", nx=80, ny=80, nz=80, path="pair", precision="fp64"),
        # unstructured operator, random aggregates: a dense-ish coarse operator
        dict(name="rap_irregular", kind="rap", op="irregular", nx=60000, ny=1, nz=1, path="direct",
             precision="fp64"),
        # a time-stepping program: the matrix's values change, the whole hierarchy is recomputed
        dict(name="hier_update_96", kind="hier_update", op="7pt", nx=96, ny=96, nz=96, levels=5),
        # a program's first contact with a matrix: the hierarchy is set up level by level
        dict(name="hier_setup_odd", kind="hier_setup", op="7pt", nx=81, ny=66, nz=71, levels=3),
        # levels of a hierarchy and many small problems of uneven sizes in one graph launch
        dict(name="batch_mixed_sizes", kind="batch", op="7pt", nx=48, ny=48, nz=48, levels=4, count=16, lo=16, hi=256),
        # the consumer of a hierarchy: V(2,2) cycles on the finest level of the benchmark
        dict(name="vcycle_128", kind="vcycle", op="7pt", nx=128, ny=128, nz=128, levels=4, cycles=5),
        # the drop-in call of a Fortran program: 1-based host arrays in, host arrays out
        dict(name="host_merged_80", kind="host", op="7pt", nx=80, ny=80, nz=80),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["rap", "rap", "rap", "rap", "hier_update", "hier_setup", "batch", "vcycle", "host"])
    if kind == "rap":
        op = rng.choice(["5pt", "7pt", "7pt", "27pt", "irregular"])
        path = "pair" if op != "irregular" and rng.random() < 0.25 else "direct"
        prec = "mixed64" if path == "direct" and op != "irregular" and rng.random() < 0.25 else "fp64"
        if op == "5pt":
            dims = [_log(rng, 48, 1024), _log(rng, 48, 1024), 1]
        elif op == "7pt":
            dims = [_log(rng, 16, 120) for _ in range(3)]
        elif op == "27pt":
            dims = [_log(rng, 16, 90) for _ in range(3)]
        else:
            dims = [_log(rng, 4000, 60000), 1, 1]
        return dict(kind="rap", op=op, nx=dims[0], ny=dims[1], nz=dims[2], path=path, precision=prec)
    if kind == "batch":
        n = _log(rng, 16, 48)
        return dict(kind="batch", op="7pt", nx=n, ny=n, nz=n, levels=rng.randint(2, 3), count=rng.randint(4, 16),
                    lo=16, hi=rng.randint(64, 256))
    lo, hi = {"hier_update": (24, 96), "hier_setup": (24, 80), "vcycle": (32, 120), "host": (16, 80)}[kind]
    dims = [_log(rng, lo, hi) for _ in range(3)]
    case = dict(kind=kind, op="7pt", nx=dims[0], ny=dims[1], nz=dims[2])
    if kind != "host":
        case["levels"] = rng.randint(2, 4)
    if kind == "vcycle":
        case["cycles"] = rng.randint(2, 5)
    return case


# ---------------------------------------------------------------------------
# operators, in torch (int64 CSR, float64 values)
# ---------------------------------------------------------------------------
class _Mat:
    def __init__(self, M, N, rp, col, val):
        self.M, self.N, self.rp, self.col, self.val = int(M), int(N), rp, col, val

    @property
    def nnz(self):
        return self.col.numel()

    def lengths(self):
        return self.rp[1:] - self.rp[:-1]

    def rows(self):
        return torch.repeat_interleave(torch.arange(self.M, device=self.col.device), self.lengths())


def _offsets(counts):
    rp = torch.zeros(counts.numel() + 1, dtype=torch.int64, device=counts.device)
    torch.cumsum(counts, 0, out=rp[1:])
    return rp


def _from_coo(M, N, r, c, v):
    """Sorted CSR; entries on one place are added."""
    key, order = torch.sort(r * N + c, stable=True)
    ukey, inv, _ = torch.unique_consecutive(key, return_inverse=True, return_counts=True)
    val = torch.zeros(ukey.numel(), dtype=torch.float64, device=v.device).index_add_(0, inv, v[order])
    row = ukey // N
    return _Mat(M, N, _offsets(torch.bincount(row, minlength=M)), ukey - row * N, val)


def _expand(A, B, e0, e1):
    """The products of A's entries e0..e1 with the rows of B they select: (entry, position in B)."""
    k = A.col[e0:e1]
    n = B.lengths()[k]
    e = torch.repeat_interleave(torch.arange(e0, e1, device=k.device), n)
    first = torch.cumsum(n, 0) - n
    pos = torch.arange(e.numel(), device=k.device) - first[e - e0] + B.rp[A.col[e]]
    return e, pos


def _mul(A, B, chunk=1 << 26):
    """A*B, structural entries kept, in slabs of rows of about `chunk` products."""
    work = _offsets(B.lengths()[A.col])[A.rp]
    rows, rp_h = A.rows(), A.rp.tolist() if work[-1] > chunk else None
    parts, r0 = [], 0
    while r0 < A.M:
        r1 = A.M if rp_h is None else min(A.M, max(r0 + 1, int(torch.searchsorted(work, work[r0] + chunk, right=True)) - 1))
        e0, e1 = (0, A.nnz) if rp_h is None else (rp_h[r0], rp_h[r1])
        e, pos = _expand(A, B, e0, e1)
        parts.append(_from_coo(r1 - r0, B.N, rows[e] - r0, B.col[pos], A.val[e] * B.val[pos]))
        r0 = r1
    if len(parts) == 1:
        return parts[0]
    return _Mat(A.M, B.N, _offsets(torch.cat([p.lengths() for p in parts])), torch.cat([p.col for p in parts]),
                torch.cat([p.val for p in parts]))


def _transpose(A):
    c, order = torch.sort(A.col, stable=True)
    return _Mat(A.N, A.M, _offsets(torch.bincount(c, minlength=A.N)), A.rows()[order], A.val[order])


def _stencil(dims, full):
    """Neighbour lists of the star or box stencil on a grid: (columns, inside), one column per offset, columns rising."""
    nx, ny, nz = dims
    i = torch.arange(nx * ny * nz, device=DEV)
    x, y, z = i % nx, (i // nx) % ny, i // (nx * ny)
    cols, inside, offs = [], [], []
    for dz in (-1, 0, 1) if nz > 1 else (0,):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if not full and abs(dx) + abs(dy) + abs(dz) > 1:
                    continue
                offs.append((dx, dy, dz))
                cols.append(i + dx + nx * (dy + ny * dz))
                inside.append((x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0) & (z + dz < nz))
    return torch.stack(cols, 1), torch.stack(inside, 1), offs


def _operator(case, seed, op=None, dims=None):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    op = op or case["op"]
    dims = dims or (case["nx"], case["ny"], case["nz"])
    M = dims[0] * dims[1] * dims[2]
    if op == "irregular":  # lognormal row lengths, uniform columns (the size's own pattern); values in [-1, 1)
        h = torch.Generator(device=DEV)
        h.manual_seed(M)
        cnt = torch.exp(2.5 + torch.randn(M, generator=h, device=DEV, dtype=torch.float64)).round().clamp(1, 4096).long()
        r = torch.repeat_interleave(torch.arange(M, device=DEV), cnt)
        c = torch.randint(0, M, (r.numel(),), generator=h, device=DEV)
        d = torch.arange(M, device=DEV)
        key = torch.unique(torch.cat([r * M + c, d * M + d]))
        val = torch.rand(key.numel(), generator=g, device=DEV, dtype=torch.float64) * 2 - 1
        row = key // M
        return _Mat(M, M, _offsets(torch.bincount(row, minlength=M)), key - row * M, val)
    cols, inside, offs = _stencil(dims, op == "27pt")
    S, center = len(offs), len(offs) // 2
    val = torch.zeros(M, S, dtype=torch.float64, device=DEV)
    if op == "27pt":  # Uniform[0.5, 1.5) couplings, made symmetric; dominant diagonal
        u = torch.rand(M, S, generator=g, device=DEV, dtype=torch.float64) + 0.5
    else:  # conductivities of the cells, harmonic-like mean on the faces
        k = torch.exp(0.5 * torch.randn(M, generator=g, device=DEV, dtype=torch.float64))
    other = cols.clamp(0, M - 1)
    for s in range(S):
        if s != center:
            j = other[:, s]
            val[:, s] = -0.5 * (u[:, s] + u[j, S - 1 - s]) if op == "27pt" else -torch.sqrt(k * torch.where(inside[:, s], k[j], k))
    if op == "27pt":
        val[:, center] = -1.001 * torch.where(inside, val, torch.zeros_like(val)).sum(1)
    else:
        val[:, center] = -val.sum(1)  # the faces of the boundary stay on the diagonal
    return _Mat(M, M, _offsets(inside.sum(1)), cols[inside], val[inside])


def _block(op):
    return 3 if op == "27pt" else 2


def _aggregates(op, dims):
    """(aggregate of every row, number, coarse grid)"""
    if op == "irregular":
        n = dims[0]
        g = np.random.Generator(np.random.PCG64(n))
        ends = np.cumsum(g.integers(4, 13, size=n // 4 + 2))
        agg = np.empty(n, np.int64)
        agg[g.permutation(n)] = np.searchsorted(ends, np.arange(n), side="right")
        return torch.from_numpy(agg).to(DEV), int(agg.max()) + 1, None
    b = _block(op)
    c = tuple(-(-d // b) for d in dims)
    i = torch.arange(dims[0] * dims[1] * dims[2], device=DEV)
    x, y, z = i % dims[0], (i // dims[0]) % dims[1], i // (dims[0] * dims[1])
    return x // b + c[0] * (y // b + c[1] * (z // b)), c[0] * c[1] * c[2], c


def _prolongator(A, agg, nagg, absdiag):
    rows = A.rows()
    at = A.col == rows
    d = torch.zeros(A.M, dtype=torch.float64, device=A.val.device)
    d[rows[at]] = A.val[at]
    d = d.abs() + 1.0 if absdiag else d
    s = -(OMEGA / d)[rows] * A.val
    s[at] += 1.0
    return _from_coo(A.M, nagg, rows, agg[A.col], s)


def _level(A, op, dims):
    agg, nagg, cdims = _aggregates(op, dims)
    P = _prolongator(A, agg, nagg, op == "irregular")
    return _transpose(P), A, P, cdims


def _chain(A, op, dims, levels):
    """[(R, A, P)] level by level and the coarsest operator."""
    out = []
    for _ in range(levels):
        R, A, P, dims = _level(A, op, dims)
        out.append((R, A, P))
        A = _mul(R, _mul(A, P))
    return out, A


def _triples(case, seed):
    """The products of a batch: the levels of a hierarchy, then 2D problems of uneven sizes."""
    levels, _ = _chain(_operator(case, seed), case["op"], (case["nx"], case["ny"], case["nz"]), case["levels"])
    sides = random.Random(case["count"] * 1000 + case["hi"])
    for i in range(case["count"]):
        n = sides.randint(case["lo"], case["hi"])
        R, A, P, _ = _level(_operator(case, seed * 64 + i + 1, "5pt", (n, n, 1)), "5pt", (n, n, 1))
        levels.append((R, A, P))
    return levels


def _triple(case, seed):
    dims = (case["nx"], case["ny"], case["nz"])
    R, A, P, _ = _level(_operator(case, seed), case["op"], dims)
    if case.get("precision") == "mixed64":
        for m in (R, A, P):
            m.val = m.val.float().double()
    return R, A, P


# ---------------------------------------------------------------------------
# the library's side
# ---------------------------------------------------------------------------
class _Ptr:
    def __init__(self, t):
        self.ptr = t.data_ptr()


class _View:
    """A device array of the library for torch; holds what owns it."""

    def __init__(self, ptr, n, kind, owner):
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": kind, "data": (ptr, False), "version": 2}
        self.owner = owner


def _tensors(m):
    """The arrays of a device matrix, without a copy."""
    d = m.d
    return {"rp": torch.as_tensor(_View(d.rp, d.M + 1, "<i8", m), device="cuda"),
            "col": torch.as_tensor(_View(d.col, d.nnz, "<i4", m), device="cuda"),
            "val": torch.as_tensor(_View(d.val, d.nnz, "<f8", m), device="cuda")}


def _to_library(m, vtype=lib.F64):
    val = m.val.float() if vtype == lib.F32 else m.val
    torch.cuda.synchronize()
    return lib.DeviceCSR.import_device(m.M, m.N, m.nnz, _Ptr(m.rp), _Ptr(m.col), _Ptr(val), vtype)


def _aggs(case):
    dims, out = (case["nx"], case["ny"], case["nz"]), []
    for _ in range(case["levels"]):
        agg, nagg, dims = _aggregates(case["op"], dims)
        out.append((agg.cpu().numpy(), nagg))
    return out


class _HostResult:
    """The matrix that a drop-in call returned; freed with the last array over it."""

    def __init__(self, p):
        self.p = p

    def __del__(self):
        lib.lib().freeSpmat(self.p)

    def array(self, p, n, kind):
        class View:
            __array_interface__ = {"shape": (int(n),), "typestr": kind, "version": 3,
                                   "data": (lib.C.cast(p, lib.C.c_void_p).value, False)}
        view = View()
        view.owner = self
        return np.asarray(view)


def prepare(case, seed):
    kind, s = case["kind"], {"case": case}
    if kind == "rap":
        s["ops"] = [_to_library(m, lib.F32 if case["precision"] == "mixed64" else lib.F64) for m in _triple(case, seed)]
        s["path"] = lib.PAIR if case["path"] == "pair" else lib.DIRECT
        s["precision"] = lib.MIXED64 if case["precision"] == "mixed64" else lib.FP64
    elif kind == "batch":
        s["ops"] = [[_to_library(m) for m in ms] for ms in zip(*_triples(case, seed))]
        s["batch"] = lib.Batch(*s["ops"], graph=True)
    elif kind == "host":
        ms = [CSR(m.M, m.N, m.rp.cpu().numpy(), m.col.cpu().numpy(), m.val.cpu().numpy()) for m in _triple(case, seed)]
        s["ops"] = [lib.HostSpmat(m, base=1) for m in ms]
        s["config"] = lib.default_config()
    else:
        s["A"] = _to_library(_operator(case, seed))
        s["aggs"] = _aggs(case)
        if kind == "hier_update":
            s["hier"] = lib.Hierarchy(s["A"], s["aggs"], graph=True)
            s["out"] = [[_tensors(m) for m in s["hier"].level(l)] for l in range(case["levels"])]
        elif kind == "vcycle":
            s["levels"], s["coarse"] = lib.hierarchy_device(s["A"], s["aggs"])
            s["solver"] = GraphVCycle(s["levels"], s["coarse"])
            g = np.random.Generator(np.random.PCG64(int(seed)))
            s["b"] = lib.DeviceArray.from_numpy(g.uniform(-1.0, 1.0, s["A"].d.M))
            s["x"] = lib.DeviceArray(s["A"].d.M)
            s["xt"] = torch.as_tensor(_View(s["x"].ptr, s["x"].n, "<f8", s["x"]), device="cuda")
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rap":
        out, _ = lib.rap(*s["ops"], path=s["path"], precision=s["precision"])
        return _tensors(out)
    if kind == "batch":
        s["batch"].run()
        return [_tensors(s["batch"].result(i)) for i in range(s["batch"].count)]
    if kind == "hier_update":
        s["hier"].update()
        return s["out"]
    if kind == "hier_setup":
        levels, coarse = lib.hierarchy_device(s["A"], s["aggs"])
        return [[_tensors(m) for m in ((R, P) if l == 0 else (R, A, P))] for l, (R, A, P) in enumerate(levels)] + [_tensors(coarse)]
    if kind == "vcycle":
        lib.axpby(0.0, None, 0.0, s["x"])
        _, hist, _ = _solve(s["solver"], s["b"], s["x"], case["cycles"])
        return {"x": s["xt"], "hist": hist}
    # a Fortran program's call: sp3mmRowByRowMerged_1 on host arrays
    L, C = lib.lib(), lib.C
    r, a, p = (C.byref(m.s) for m in s["ops"])
    got = L.sp3mmRowByRowMerged_1(r, a, p, C.byref(s["config"]), None)
    if not got:
        raise RuntimeError("sp3mmRowByRowMerged_1 failed: " + lib.last_error())
    m, res = got.contents, _HostResult(got)
    return {"rp": res.array(m.IRP, m.M + 1, "<i8"), "col": res.array(m.JA, m.NZ, "<i8"),
            "val": res.array(m.AS, m.NZ, "<f8")}


def _solve(solver, b, x, cycles):
    """A fixed number of cycles on device vectors (sp3mm_vcycle_solve, as a C program calls it)."""
    C = lib.C
    hist, k, ms = np.zeros(cycles + 1), C.c_int32(), C.c_double()
    if lib.lib().sp3mm_vcycle_solve(solver.h, b.ptr, x.ptr, 0.0, cycles, C.byref(k), hist.ctypes.data, C.byref(ms)):
        raise RuntimeError("sp3mm_vcycle_solve failed: " + lib.last_error())
    return k.value, hist, ms.value


# ---------------------------------------------------------------------------
# 64-bit results
# ---------------------------------------------------------------------------
def _values(m):
    return {"rp": None, "col": None, "val": m.val}


def _spmv(A, x):
    return torch.zeros(A.M, dtype=torch.float64, device=x.device).index_add_(0, A.rows(), A.val * x[A.col])


def _cycle(levels, coarse, l, b, x):
    def jacobi(A, x, sweeps):
        rows = A.rows()
        d = A.val[A.col == rows]
        for _ in range(sweeps):
            x = x + OMEGA * (b - _spmv(A, x)) / d
        return x

    if l == len(levels):
        return jacobi(coarse, x, 50)
    R, A, P = levels[l]
    x = jacobi(A, x, 2)
    rc = _spmv(R, b - _spmv(A, x))
    x = x + _spmv(P, _cycle(levels, coarse, l + 1, rc, torch.zeros_like(rc)))
    return jacobi(A, x, 2)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("rap", "host"):
        R, A, P = _triple(case, seed)
        return _values(_mul(R, _mul(A, P)))
    if kind == "batch":
        return [_values(_mul(R, _mul(A, P))) for R, A, P in _triples(case, seed)]
    levels, coarse = _chain(_operator(case, seed), case["op"], (case["nx"], case["ny"], case["nz"]), case["levels"])
    if kind == "hier_update":
        ops = [A for _, A, _ in levels[1:]] + [coarse]
        return [[_values(m) for m in (R, P, ops[l])] for l, (R, _, P) in enumerate(levels)]
    if kind == "hier_setup":
        return [[_values(m) for m in ((R, P) if l == 0 else (R, A, P))] for l, (R, A, P) in enumerate(levels)] + [_values(coarse)]
    g = np.random.Generator(np.random.PCG64(int(seed)))
    b = torch.from_numpy(g.uniform(-1.0, 1.0, levels[0][1].M)).to(DEV)
    x, A = torch.zeros_like(b), levels[0][1]
    hist = [1.0]
    for _ in range(case["cycles"]):
        x = _cycle(levels, coarse, 0, b, x)
        hist.append(float((b - _spmv(A, x)).norm() / b.norm()))
    return {"x": x, "hist": np.array(hist)}


# ---------------------------------------------------------------------------
# bytes and operations
# ---------------------------------------------------------------------------
def _bytes(m, v=8, i=4, p=8):
    return m.nnz * (v + i) + (m.M + 1) * p


def _macs(A, B):
    return int(B.lengths()[A.col].sum())


def _product_work(R, A, P, v=8, i=4):
    """(bytes, multiply-adds, the product): operands read once, the result written once; the cheaper association's
    multiply-adds."""
    RA, AP = _mul(R, A), _mul(A, P)
    C = _mul(R, AP)
    macs = min(_macs(R, A) + _macs(RA, P), _macs(A, P) + _macs(R, AP))
    return sum(_bytes(m, v, i) for m in (R, A, P)) + _bytes(C, 8, i), macs, C


@functools.lru_cache(maxsize=None)
def _work(text):
    case = json.loads(text)
    kind = case["kind"]
    if kind in ("rap", "host"):
        v = 4 if case.get("precision") == "mixed64" else 8
        nbytes, macs, _ = _product_work(*_triple(case, 0), v=v, i=8 if kind == "host" else 4)
        return nbytes, 2 * macs
    if kind == "batch":  # the batch's results are copied out of it once more
        total = [0, 0]
        for R, A, P in _triples(case, 0):
            nbytes, macs, C = _product_work(R, A, P)
            total[0] += nbytes + 2 * _bytes(C)
            total[1] += 2 * macs
        return total
    levels, coarse = _chain(_operator(case, 0), case["op"], (case["nx"], case["ny"], case["nz"]), case["levels"])
    if kind == "vcycle":  # per cycle: every sweep, residual and transfer reads its matrix and vectors once
        nbytes = flops = 0
        for R, A, P in levels:  # four sweeps and a residual; restriction; prolongation
            nbytes += 5 * (_bytes(A, p=4) + 24 * A.M) + sum(_bytes(m, p=4) + 8 * m.N + 16 * m.M for m in (R, P))
            flops += 2 * (5 * A.nnz + R.nnz + P.nnz)
        A = levels[0][1]  # the residual whose norm ends a cycle
        nbytes += _bytes(A, p=4) + 24 * A.M + _bytes(coarse, p=4) + 16 * coarse.M
        return nbytes * case["cycles"], (flops + 2 * A.nnz + 100 * coarse.nnz) * case["cycles"]
    nbytes = flops = 0
    for l, (R, A, P) in enumerate(levels):  # P from A, R from P, then the product
        got, macs, C = _product_work(R, A, P)
        nbytes += (_bytes(A) if l == 0 else 0) + _bytes(P) + _bytes(R) + _bytes(C) + 8 * A.M
        flops += 2 * macs + 2 * A.nnz
    return nbytes, flops


def work(case):
    nbytes, flops = _work(json.dumps({k: v for k, v in case.items() if k != "name"}, sort_keys=True))
    return {"bytes": float(nbytes), "flops": float(flops)}
