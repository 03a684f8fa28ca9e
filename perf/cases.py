"""Performance cases of the engine: what its users run, through race_amd's public entry points.

A case names a workload and its sizes.  prepare() makes what a program holds
before it calls the engine (coloured handle, registered functions or batch,
device vectors), run() is one call sequence of such a program on its own HIP
stream, exact() the same results in float64 from plain torch / numpy
arithmetic on the same matrices, vectors and row order.

Workloads (the kinds are the engine's kernels):

  gs        one symmetric Gauss-Seidel step (forward and backward sweep) on a
            27-point grid, a smoother of a multigrid or a preconditioner
  color     RACE colouring of a matrix pattern, what every new mesh pays first
  kacz      one symmetric Kaczmarz step on a 7-point grid
  symmspmv  b += A x from the upper triangle of a coloured matrix
  spmv      b = A x on a graph Laplacian with hubs or a banded matrix, no schedule needed
  spmtv     b += A^T x
  mpk       the powers A x .. A^k x under RACE's level blocking
  batch     many matrices of both families at once: SymmSpMV and one symmetric Kaczmarz step
  refine    a linear solve: FP64 refinement around low-precision Gauss-Seidel sweeps
"""
import math

import numpy as np
import torch

import race_amd as R
from race_amd.interface import Batch

PREC = {"fp64": R.FP64, "fp32": R.FP32, "bf16": R.BF16}
SIZE = {"fp64": 8, "fp32": 4, "bf16": 2}
POINTS = {"7pt": 7, "27pt": 27}

_streams = {}


def _stream():
    """The program's own HIP stream (default priority), as an integer handle."""
    if "main" not in _streams:
        _streams["main"] = torch.cuda.Stream()
    return _streams["main"].cuda_stream


def listed():
    return [
        # the coarse grid of a multigrid cycle: launches and latency
        {"name": "gs-coarse", "kind": "gs", "grid": 14, "prec": "fp64"},
        # the engine's headline workload (bench.py's default)
        {"name": "gs-fine", "kind": "gs", "grid": 128, "prec": "fp64"},
        # colouring a mesh before its first sweep
        {"name": "color-mesh", "kind": "color", "pattern": "27pt", "grid": 72, "dist": 1, "rows_per_thread": 16},
        # row projections on an ordinary grid
        {"name": "kacz-grid", "kind": "kacz", "grid": 45, "prec": "fp64", "flow": False},
        # the 64^3 Laplacian product bench.py names
        {"name": "symm-grid", "kind": "symmspmv", "pattern": "7pt", "n": 262144, "prec": "fp64", "nrhs": 1},
        # a block of vectors (block Krylov, several right-hand sides) on a random banded matrix
        {"name": "symm-block", "kind": "symmspmv", "pattern": "banded", "n": 90001, "mean": 21, "prec": "fp32",
         "nrhs": 8},
        # a graph operator with hub rows: ragged row lengths
        {"name": "spmv-graph", "kind": "spmv", "pattern": "graph", "n": 150000, "mean": 20, "prec": "fp64", "nrhs": 1},
        # the transpose product of a least-squares or adjoint step, 16-bit values
        {"name": "spmtv-bf16", "kind": "spmtv", "pattern": "27pt", "n": 884736, "prec": "bf16", "nrhs": 1},
        # a Chebyshev / s-step Krylov basis on a large grid with the 256 MB blocking bench.py uses
        {"name": "mpk-large", "kind": "mpk", "pattern": "7pt", "grid": 192, "power": 8, "cache_mb": 256,
         "prec": "fp64", "highest": False},
        # a polynomial smoother on a small grid: only the last power is kept
        {"name": "mpk-small", "kind": "mpk", "pattern": "27pt", "grid": 33, "power": 5, "cache_mb": 4,
         "prec": "fp32", "highest": True},
        # many matrices of different size and structure in one program
        {"name": "batch", "kind": "batch", "count": 16, "n_lo": 2000, "n_hi": 40000, "prec": "fp32", "nrhs": 8},
        # a solve to 1e-10 with single-precision smoothing
        {"name": "refine-fp32", "kind": "refine", "grid": 56, "prec": "fp32", "sweeps": 4},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gs", "color", "kacz", "symmspmv", "spmv", "spmtv", "mpk", "batch", "refine"])
    prec = rng.choice(["fp64", "fp64", "fp32", "bf16"])
    if kind == "gs":
        return {"kind": kind, "grid": _log_int(rng, 10, 100), "prec": prec}
    if kind == "color":
        return {"kind": kind, "pattern": rng.choice(["7pt", "27pt"]), "grid": _log_int(rng, 12, 72),
                "dist": rng.choice([1, 2]), "rows_per_thread": rng.choice([16, 64, 256])}
    if kind == "kacz":
        return {"kind": kind, "grid": _log_int(rng, 10, 56), "prec": prec, "flow": rng.random() < 0.5}
    if kind in ("symmspmv", "spmv", "spmtv"):
        pattern = rng.choice(["7pt", "27pt", "banded", "graph"])
        case = {"kind": kind, "pattern": pattern, "prec": prec, "nrhs": rng.choice([1, 1, 2, 3, 8])}
        if pattern in POINTS:
            case["n"] = _log_int(rng, 12, 96) ** 3
        else:
            case["n"] = _log_int(rng, 2000, 200000)
            case["mean"] = rng.randint(5, 40)
        return case
    if kind == "mpk":
        pattern = rng.choice(["7pt", "27pt"])
        return {"kind": kind, "pattern": pattern, "grid": _log_int(rng, 16, 160 if pattern == "7pt" else 96),
                "power": rng.randint(2, 8), "cache_mb": rng.choice([4, 32, 256]), "prec": prec,
                "highest": rng.random() < 0.3}
    if kind == "batch":
        return {"kind": kind, "count": rng.randint(4, 16), "n_lo": 2000, "n_hi": _log_int(rng, 8000, 40000),
                "prec": rng.choice(["fp32", "fp64"]), "nrhs": rng.choice([1, 4, 8])}
    return {"kind": kind, "grid": _log_int(rng, 16, 56), "prec": prec, "sweeps": rng.choice([1, 2, 4])}


# ---------------------------------------------------------------------------
# matrices, made on the GPU
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _grid_pattern(points, g):
    """CRS pattern (rowPtr, row, col; columns ascending) of a g^3 grid stencil."""
    n = g * g * g
    idx = torch.arange(n, device="cuda")
    i, j, k = idx // (g * g), (idx // g) % g, idx % g
    offs = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)
            if points == 27 or abs(a) + abs(b) + abs(c) <= 1]
    off = torch.tensor([(a * g + b) * g + c for a, b, c in offs], device="cuda")
    ok = torch.stack([((i + a) >= 0) & ((i + a) < g) & ((j + b) >= 0) & ((j + b) < g) & ((k + c) >= 0) & ((k + c) < g)
                      for a, b, c in offs], 1)
    at = ok.nonzero()
    row = at[:, 0]
    return _row_ptr(ok.sum(1)), row, row + off[at[:, 1]]


def _row_ptr(lengths):
    rp = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=rp[1:])
    return rp


def _edges_pattern(n, a, b):
    """Symmetric CRS pattern with its diagonal from an edge list."""
    d = torch.arange(n, device="cuda")
    key = torch.unique(torch.cat([a * n + b, b * n + a, d * n + d]))
    row = key // n
    return _row_ptr(torch.bincount(row, minlength=n)), row, key % n


def _banded_pattern(n, mean, gen):
    """Random entries within 1 % of n around the diagonal."""
    bw, k = max(1, math.ceil(0.01 * n)), max(1, round((mean - 1) / 2))
    a = torch.arange(n, device="cuda").repeat_interleave(k)
    off = torch.randint(1, bw + 1, (n * k,), device="cuda", generator=gen)
    b = a + off * (2 * torch.randint(0, 2, (n * k,), device="cuda", generator=gen) - 1)
    ok = (b >= 0) & (b < n)
    return _edges_pattern(n, a[ok], b[ok])


def _graph_pattern(n, mean, gen):
    """Chung-Lu random graph, power-law exponent 2.3, expected degree at most 400."""
    w = torch.arange(1, n + 1, device="cuda", dtype=torch.float64) ** (-1.0 / 1.3)
    w *= mean * n / w.sum()
    w.clamp_(max=min(math.sqrt(mean * n), 400.0))
    cum = torch.cumsum(w, 0) / w.sum()
    m = int(mean * n / 2)
    u = torch.rand(2, m, device="cuda", dtype=torch.float64, generator=gen)
    at = torch.searchsorted(cum, u).clamp_(max=n - 1)
    place = torch.randperm(n, device="cuda", generator=gen)  # hubs spread over the numbering
    a, b = place[at[0]], place[at[1]]
    return _edges_pattern(n, a[a != b], b[a != b])


def _pattern(name, n, mean, gen):
    if name in POINTS:
        return _grid_pattern(POINTS[name], round(n ** (1 / 3)))
    return (_banded_pattern if name == "banded" else _graph_pattern)(n, mean, gen)


def _values(rp, row, col, gen, dominance=1.05):
    """A symmetric diagonally dominant operator with varying coefficients
    (multiples of 2^-22, so that their sums are exact in any order)."""
    n = rp.numel() - 1
    s = torch.randint(1 << 17, 1 << 21, (n,), device="cuda", generator=gen).double() * 2.0 ** -21
    off = torch.where(row == col, 0.0, -0.5 * (s[row] + s[col]))
    total = torch.zeros(n, device="cuda", dtype=torch.float64).index_add_(0, row, -off)
    return torch.where(row == col, dominance * total[row] + (total[row] == 0), off)


def _host(*tensors):
    return [t.to(torch.int32 if t.dtype == torch.int64 else t.dtype).cpu().numpy() for t in tensors]


def _permuted(rp, row, col, val, perm, inv):
    """The matrix in the engine's numbering, the diagonal first in each row."""
    perm, inv = (torch.from_numpy(v).cuda().long() for v in (perm, inv))
    length = (rp[1:] - rp[:-1])[perm]
    rp2 = _row_ptr(length)
    nnz = int(rp2[-1])
    row2 = torch.arange(perm.numel(), device="cuda").repeat_interleave(length)
    src = (rp[:-1][perm] - rp2[:-1])[row2] + torch.arange(nnz, device="cuda")
    return _diag_first(rp2, row2, inv[col[src]], val[src])


def _diag_first(rp, row, col, val):
    at = torch.arange(col.numel(), device="cuda")
    is_diag = row == col
    diag = torch.zeros(rp.numel() - 1, dtype=torch.int64, device="cuda")
    diag[row[is_diag]] = at[is_diag]
    to = torch.where(is_diag, rp[:-1][row], at + (at < diag[row]))
    c2, v2 = torch.empty_like(col), torch.empty_like(val)
    c2[to], v2[to] = col, val
    return rp, row, c2, v2


def _upper(rp, row, col, val):
    keep = col >= row
    return _row_ptr(torch.bincount(row[keep], minlength=rp.numel() - 1)), row[keep], col[keep], val[keep]


def _vec(n, prec, gen, nrhs=1):
    v = 2.0 * torch.rand(n * nrhs, device="cuda", dtype=torch.float64, generator=gen) - 1.0
    return v if prec == "fp64" else v.float()


def _stored(val, prec):
    """The values as the engine stores them, in float64."""
    return val if prec == "fp64" else val.float().double() if prec == "fp32" else val.float().bfloat16().double()


# ---------------------------------------------------------------------------
# the systems: handle, permuted matrix, vectors
# ---------------------------------------------------------------------------
def _colored(case, rp, col, n):
    """The engine's handle for a workload, coloured."""
    rp, col = _host(rp, col)
    kind = case["kind"]
    if kind in ("gs", "refine"):
        ce = R.Interface(n, max(1, n // 16), R.ONE, rp, col, symm_hint=True)
        ce.RACEColor()
    elif kind == "mpk":
        ce = R.Interface(n, 1, R.POWER, rp, col, symm_hint=True)
        ce.RACEColor(case["power"], case["cache_mb"] * 1e6)
    elif kind == "symmspmv":
        ce = R.Interface(n, max(1, min(1024, n // 4096)), R.TWO, rp, col, symm_hint=True)
        ce.RACEColor()
    elif kind in ("kacz", "batch"):
        ce = R.Interface(n, max(4, min(1024, n // 256)), R.TWO, rp, col, symm_hint=True)
        if case.get("flow"):
            ce.setOption("flow", 1)
        ce.RACEColor()
    else:  # products that need no schedule
        ce = R.Interface(n, 1, R.ONE, rp, col, symm_hint=True)
    return ce


def _system(case, pattern, n, mean, gen):
    """A handle and its matrix (rowPtr, row, col, val) in the engine's numbering."""
    rp, row, col = _pattern(pattern, n, mean, gen)
    val = _values(rp, row, col, gen)
    ce = _colored(case, rp, col, n)
    if case["kind"] in ("spmv", "spmtv"):
        return ce, _diag_first(rp, row, col, val)
    return ce, _permuted(rp, row, col, val, ce.getPerm(), ce.getInvPerm())


def _inputs(case, seed):
    """Handle(s), matrices and vectors of a case, from the seed."""
    gen, kind, prec = _gen(seed), case["kind"], case.get("prec")
    if kind == "batch":
        items = []
        for m in range(case["count"]):
            share = (m + 0.5) / case["count"]
            n = int(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** share)
            ce, A = _system(case, "banded" if m % 2 == 0 else "graph", n, 5 + (7 * m) % 36, gen)
            items.append((ce, A, [_vec(n, prec, gen, case["nrhs"]) for _ in range(4)]))
        return items
    pattern, n, mean = case.get("pattern", "7pt" if kind == "kacz" else "27pt"), case.get("n"), case.get("mean")
    n = n or case["grid"] ** 3
    ce, A = _system(case, pattern, n, mean, gen)
    if kind == "mpk":
        x = torch.zeros(2 if case["highest"] else case["power"] + 1, n, device="cuda",
                        dtype=torch.float64 if prec == "fp64" else torch.float32)
        x[0] = _vec(n, prec, gen)
        # a Chebyshev basis scales the operator to its spectral interval
        A = (A[0], A[1], A[2], A[3] / float(A[3].max()))
        return ce, A, [x]
    vec = "fp64" if kind == "refine" else prec
    return ce, A, [_vec(n, vec, gen, case.get("nrhs", 1)) for _ in range(2)]


def _register(ce, kind, A, x, b, prec, nrhs=1, power=1):
    rp, col, val = _host(A[0], A[2], A[3])
    return ce.registerDevice(kind, rp, col, val, x.data_ptr(), None if b is None else b.data_ptr(), nrhs=nrhs,
                             power=power, val_precision=PREC[prec], vec_precision=PREC["fp64" if prec == "fp64" else "fp32"])


def prepare(case, seed):
    kind, prec = case["kind"], case.get("prec")
    s = {"case": case, "stream": _stream()}
    if kind == "color":
        # the pattern of a mesh whose nodes the program has numbered its own way: shifted grid planes
        rp, row, col = _grid_pattern(POINTS[case["pattern"]], case["grid"])
        n = case["grid"] ** 3
        plane = case["grid"] ** 2
        shift = plane * (1 + int(seed) % max(1, case["grid"] - 1))
        order = (torch.arange(n, device="cuda") + shift) % n
        val = torch.zeros(col.numel(), device="cuda", dtype=torch.float32)
        rp, row, col, val = _permuted(rp, row, col, val, *_host(order, torch.argsort(order)))
        s["rp"], s["col"] = _host(rp, col)
        s["n"] = n
        return s
    if kind == "batch":
        symm = Batch(R.K_SYMMSPMV, PREC[prec], PREC[prec], case["nrhs"])
        kacz = Batch(R.K_KACZ, PREC[prec], PREC[prec], case["nrhs"])
        kacz.setOption("flow", 1)
        s["out"], s["keep"] = [], []
        for ce, A, (u, y, x, b) in _inputs(case, seed):
            rp, col, val = _host(*_upper(*A)[::2], _upper(*A)[3])
            symm.add(ce, rp, col, val, u.data_ptr(), y.data_ptr())
            rp, col, val = _host(A[0], A[2], A[3])
            kacz.add(ce, rp, col, val, x.data_ptr(), b.data_ptr())
            s["out"] += [y, x]
            s["keep"] += [u, b, ce]
        symm.useCandidate(7)  # 8 rows per chunk, sorted in windows of 32
        kacz.useCandidate(8)  # 512 threads, 256 rows, 4 lanes per row
        symm.build()
        kacz.build()
        s["symm"], s["kacz"] = symm, kacz
        return s
    ce, A, vecs = _inputs(case, seed)
    x, b = vecs[0], vecs[1] if len(vecs) > 1 else None
    s |= {"ce": ce, "x": x, "b": b}
    nrhs = case.get("nrhs", 1)
    if kind == "mpk":
        s["id"] = _register(ce, R.K_MPK_HIGHEST if case["highest"] else R.K_MPK, A, x, None, prec, power=case["power"])
    elif kind == "refine":
        wide = "fp64" if prec == "fp64" else "fp32"
        xi, bi = _vec(x.numel(), wide, _gen(0)), _vec(x.numel(), wide, _gen(0))
        inner = _register(ce, R.K_GS, A, xi, bi, prec)
        rp, col, val = _host(A[0], A[2], A[3])
        s["id"] = ce.registerRefinement(R.K_GS, rp, col, val, x.data_ptr(), b.data_ptr(), inner, case["sweeps"])
        s["keep"], s["guess"] = (xi, bi), x.clone()
    else:
        code = {"gs": R.K_GS, "kacz": R.K_KACZ, "symmspmv": R.K_SYMMSPMV, "spmv": R.K_SPMV, "spmtv": R.K_SPMTV}[kind]
        s["id"] = _register(ce, code, _upper(*A) if kind == "symmspmv" else A, x, b, prec, nrhs)
    return s


def run(s):
    kind, stream = s["case"]["kind"], s["stream"]
    if kind == "color":
        c = s["case"]
        ce = R.Interface(s["n"], max(1, s["n"] // c["rows_per_thread"]), R.ONE if c["dist"] == 1 else R.TWO, s["rp"],
                         s["col"], symm_hint=True)
        ce.RACEColor()
        return ce.getPerm(), ce.getInvPerm()
    if kind == "batch":
        s["symm"].executeAsync(stream=stream)
        s["kacz"].executeAsync(stream=stream)
        s["kacz"].executeAsync(rev=True, stream=stream)
        return s["out"]
    if kind in ("gs", "kacz"):
        s["ce"].executeAsync(s["id"], stream=stream)
        s["ce"].executeAsync(s["id"], rev=True, stream=stream)
        return s["x"]
    if kind == "refine":
        s["x"].copy_(s["guess"])
        torch.cuda.current_stream().synchronize()  # refine runs on the handle's own stream
        outer, sweeps, _ = s["ce"].refine(s["id"], 1e-10)
        return s["x"], outer, sweeps
    s["ce"].executeAsync(s["id"], stream=stream)
    return s["x"] if kind == "mpk" else s["b"]


def _nnz(pattern, n, mean):
    if pattern in POINTS:
        g = round(n ** (1 / 3))
        return (3 * g - 2) ** 3 if pattern == "27pt" else n + 6 * g * g * (g - 1)
    return n * mean


def work(case):
    """Bytes: each stored entry (value and 4-byte column) and row pointer once
    per pass over the matrix that the method needs, each vector read and
    written once.  SymmSpMV reads the upper triangle only; a symmetric sweep
    reads the matrix forward and backward; the powers read it once, as their
    blocking intends, and write every power kept.  Colouring reads the
    pattern and writes the two permutations."""
    kind, prec = case["kind"], case.get("prec")
    if kind == "batch":
        total = {"bytes": 0, "flops": 0}
        for m in range(case["count"]):
            n = int(case["n_lo"] * (case["n_hi"] / case["n_lo"]) ** ((m + 0.5) / case["count"]))
            nnz, e = n * (5 + (7 * m) % 36), SIZE[prec]
            k = case["nrhs"]
            total["bytes"] += (nnz + n) // 2 * (e + 4) + 4 * n + 3 * k * n * e
            total["bytes"] += 2 * (nnz * (e + 4) + 12 * n + 3 * k * n * e)
            total["flops"] += 2 * nnz * k + 8 * nnz * k
        return total
    pattern = case.get("pattern", "7pt" if kind == "kacz" else "27pt")
    n = case.get("n") or case["grid"] ** 3
    nnz = _nnz(pattern, n, case.get("mean", 0))
    if kind == "color":
        return {"bytes": 4 * (nnz + n + 1) + 8 * n, "flops": 0}
    e, v, k = SIZE[prec], SIZE["fp64" if prec == "fp64" else "fp32"], case.get("nrhs", 1)
    if kind in ("gs", "kacz"):
        per_row = 8 if kind == "kacz" else 0
        return {"bytes": 2 * (nnz * (e + 4) + n * (4 + per_row + 3 * v)), "flops": (4 if kind == "gs" else 8) * nnz}
    if kind == "symmspmv":
        return {"bytes": (nnz + n) // 2 * (e + 4) + 4 * n + 3 * k * n * v, "flops": 2 * nnz * k}
    if kind in ("spmv", "spmtv"):
        return {"bytes": nnz * (e + 4) + 4 * n + (2 if kind == "spmv" else 3) * k * n * v, "flops": 2 * nnz * k}
    if kind == "mpk":
        kept = 1 if case["highest"] else case["power"]
        return {"bytes": nnz * (e + 4) + 4 * n + (1 + kept) * n * v, "flops": 2 * nnz * case["power"]}
    # refine: the solve's steps follow from the operator; one step is one residual and its sweeps
    steps = 112 // case["sweeps"]
    sweep = 2 * (nnz * (e + 4) + n * (4 + 3 * v))
    residual = nnz * 12 + n * (4 + 24)
    return {"bytes": steps * (case["sweeps"] * sweep + residual), "flops": steps * nnz * (4 * case["sweeps"] + 2)}


# ---------------------------------------------------------------------------
# the results in float64
# ---------------------------------------------------------------------------
def _product(A, val, x, n):
    """A x for x of shape (nrhs, n)."""
    rp, row, col = A[:3]
    out = torch.zeros_like(x)
    for q in range(x.shape[0]):
        out[q].index_add_(0, row, val * x[q][col])
    return out


def _order(ce, rev):
    """Row numbers in the order of a sweep: the phases in turn, their leaves
    one after another (leaves of a phase are independent)."""
    _, lo, hi = ce.schedule(rev)
    parts = [np.arange(h - 1, l - 1, -1) if rev else np.arange(l, h) for l, h in zip(lo.tolist(), hi.tolist())]
    return np.concatenate(parts)


def _sweep_gs(ce, A, val, x, b, rev):
    """A Gauss-Seidel sweep: (D + L) y = b - U x with L the entries whose
    column comes earlier in the order; L's part by repeated substitution,
    which converges like the diagonal dominance."""
    rp, row, col = A[:3]
    n = rp.numel() - 1
    pos = torch.empty(n, dtype=torch.int64, device="cuda")
    pos[torch.from_numpy(_order(ce, rev)).cuda()] = torch.arange(n, device="cuda")
    earlier, diag = pos[col] < pos[row], torch.empty(n, device="cuda", dtype=torch.float64)
    diag[row[row == col]] = val[row == col]
    later = (~earlier) & (row != col)

    def times(mask, v):
        return torch.zeros_like(v).index_add_(0, row[mask], val[mask] * v[col[mask]])

    rhs = b - times(later, x)
    at, vals, cols = row[earlier], val[earlier], col[earlier]
    y = x.clone()
    for _ in range(400):
        z = (rhs - torch.zeros_like(y).index_add_(0, at, vals * y[cols])) / diag
        far = float((z - y).abs().max())
        y = z
        if far <= 1e-17 * float(z.abs().max()):
            break
    return y


def _sweep_kacz(ce, A, val, x, b, rev):
    """A Kaczmarz sweep row by row; x and b of shape (n, nrhs), changed in place."""
    rp, col, val = A[0].cpu().numpy(), A[2].cpu().numpy(), val.cpu().numpy()
    norm = np.add.reduceat(val * val, rp[:-1])
    for r in _order(ce, rev).tolist():
        lo, hi = rp[r], rp[r + 1]
        c, a = col[lo:hi], val[lo:hi]
        xc = x[c]
        x[c] = xc + np.outer(a, (b[r] - a @ xc) / norm[r])


def _solve(A, b):
    """A^-1 b by conjugate gradients, to rounding."""
    n = b.numel()
    x, r = torch.zeros_like(b), b.clone()
    p, rr = r.clone(), float(r @ r)
    first = rr
    for _ in range(2000):
        q = _product(A, A[3], p[None], n)[0]
        alpha = rr / float(p @ q)
        x, r = x + alpha * p, r - alpha * q
        old, rr = rr, float(r @ r)
        if rr <= 1e-30 * first:
            break
        p = r + (rr / old) * p
    return x


def exact(case, seed):
    kind, prec = case["kind"], case.get("prec")
    if kind == "color":
        return None  # whole numbers only
    if kind == "batch":
        out, k = [], case["nrhs"]
        for ce, A, (u, y, x, b) in _inputs(case, seed):
            n, val = A[0].numel() - 1, _stored(A[3], prec)
            out.append((y.double().view(k, n) + _product(A, val, u.double().view(k, n), n)).reshape(-1))
            xs, bs = (np.ascontiguousarray(t.double().view(k, n).T.cpu().numpy()) for t in (x, b))
            for rev in (False, True):
                _sweep_kacz(ce, A, val, xs, bs, rev)
            out.append(torch.from_numpy(np.ascontiguousarray(xs.T).reshape(-1)))
        return out
    ce, A, vecs = _inputs(case, seed)
    n, val = A[0].numel() - 1, _stored(A[3], prec)
    if kind == "mpk":
        x = vecs[0].double()
        for p in range(1, case["power"] + 1):
            to, frm = (p % 2, (p - 1) % 2) if case["highest"] else (p, p - 1)
            x[to] = _product(A, val, x[frm:frm + 1], n)[0]
        return x
    x, b = (v.double() for v in vecs)
    if kind == "gs":
        for rev in (False, True):
            x = _sweep_gs(ce, A, val, x, b, rev)
        return x
    if kind == "kacz":
        xs, bs = (v.view(1, n).T.cpu().numpy().copy() for v in (x, b))
        for rev in (False, True):
            _sweep_kacz(ce, A, val, xs, bs, rev)
        return torch.from_numpy(xs[:, 0].copy())
    if kind == "refine":
        # the iterate at a residual of 1e-10 is this near to the solution
        return _solve(A, b), None, None
    k = case["nrhs"]
    got = _product(A, val, x.view(k, n), n).reshape(-1)
    return got if kind == "spmv" else b + got
