"""The calls that the library is timed on: CSR SpMV, SpMVOp and SpMMOp as programs make them.

A case is a dict of plain values:

  api      which entry point, and what a program keeps between calls
             plan     CsrSpMV: descriptors, workspace and Preprocess kept, run() per product
             mv       torch.mv(csr, x): everything set up in each call (int64 indices, as torch builds them)
             once     spmv_npu(...): the same on explicit arrays, with op, alpha and beta
             spmvop   SpMVOp (compensated sums): the plan kept, run() per product
             spmm     SpMMOp (CSR times dense): the plan kept, run() per product
  pattern  stencil   5-point Laplacian on a grid of ``grid`` x ``grid`` points
           fixed     ``mean`` uniform sorted columns in every row
           poisson   Poisson(``mean``) uniform sorted columns per row, a tenth of the rows empty
           zipf      heavy-tailed row lengths (P(L >= l) ~ 1/l, at most 200,000) scaled to ``mean``
           half      the dense-block pattern of the SpMMOp perf table: about half of the places taken
  rows, cols, mean, n (SpMMOp: columns of B), dtype, op, alpha, beta, index (type of the row offsets)

Values are U(-1,1) in fp32 and complex64 and N(0,1) in 16 bits; x, y, B and C are U(-1,1).
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "ops-sparse_amd"))

import ops_sparse  # noqa: E402
from ops_sparse import CsrSpMV, SpMMOp, SpMVOp, spmv_npu  # noqa: E402
from ops_sparse._lib import Operation, SpMVOpAlg  # noqa: E402

_DTYPE = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16, "i8": torch.int8, "c64": torch.complex64}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2, "i8": 1, "c64": 8}
_OP = {"N": Operation.NON_TRANSPOSE, "T": Operation.TRANSPOSE, "H": Operation.CONJUGATE_TRANSPOSE}
_ZIPF_CAP = 200000


def _case(name, api, pattern, rows, cols, mean, dtype="f32", op="N", alpha=1.0, beta=0.0, index="i32", n=1):
    c = dict(api=api, pattern=pattern, rows=rows, cols=cols, mean=mean, dtype=dtype, op=op, alpha=alpha, beta=beta,
             index=index, n=n)
    return dict(c, name=name) if name else c


def _stencil(name, api, grid, dtype="f32", op="N", alpha=1.5, beta=0.5, n=1):
    return _case(name, api, "stencil", grid * grid, grid * grid, 5, dtype, op, alpha, beta, "i32", n)


def listed():
    return [
        # a small system solved iteratively: the launch and its latency count
        _case("small_f32", "plan", "fixed", 4096, 4096, 41),
        # a PDE solver's inner product on a structured grid
        _stencil("stencil_f32", "plan", 2048),
        # a web or social graph: PageRank and its like, rows from one entry to 200,000
        _case("zipf_f32", "plan", "zipf", 8388608, 8388608, 16),
        # the largest: a sparse 16-bit model layer or graph of half a billion entries, 64-bit row offsets
        _case("random_f16_i64", "plan", "fixed", 16777216, 16777216, 32, "f16", index="i64"),
        # least squares, adjoints: the transposed product of an unstructured matrix, minus what y holds
        _case("poisson_f32_T", "plan", "poisson", 2097152, 2097152, 12, "f32", "T", 1.0, -1.0),
        # the backward of a sparse 16-bit layer, a ragged rectangular matrix
        _case("random_bf16_T", "plan", "poisson", 1500007, 1200011, 20, "bf16", "T"),
        # Krylov methods on a complex grid operator: the conjugate transpose
        _stencil("stencil_c64_H", "plan", 1501, "c64", "H"),
        # a torch program that multiplies by a CSR tensor once: set-up and product in one call
        _case("mv_f32", "mv", "poisson", 500009, 500009, 16, index="i64"),
        # the same for a transposed product on explicit arrays
        _case("once_f32_T", "once", "poisson", 1000003, 1000003, 12, "f32", "T", 1.0, -1.0),
        # residuals that have to be exact to the last bits: compensated sums, the plan kept
        _case("spmvop_f32", "spmvop", "poisson", 2097152, 2097152, 12, "f32", "N", -1.0, 1.0),
        # the largest shape of the SpMMOp perf table: half-dense blocks times a wide matrix
        _case("spmm_half_f16", "spmm", "half", 2048, 128, 64, "f16", n=2048),
        # a grid operator times a block of vectors (block Krylov methods, several right-hand sides)
        _stencil("spmm_stencil_x16", "spmm", 2048, n=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("stencil", "random", "random", "random_T", "random_T", "mv", "once", "spmvop", "spmm", "spmm"))
    if kind == "stencil":
        dtype, op = rng.choice((("f32", "N"), ("f32", "T"), ("f16", "N"), ("bf16", "N"), ("i8", "N"), ("c64", "N"),
                                ("c64", "H")))
        scal = (2.0, 1.0) if dtype == "i8" else (1.5, 0.5)
        return _stencil(None, "plan", _log(rng, 128, 2048), dtype, op, *scal)
    rows = _log(rng, 4096, 4194304)
    cols = max(4096, int(rows * rng.uniform(0.6, 1.6)))
    mean = rng.randint(8, 40) if rows > 32768 else rng.randint(8, 64)
    pattern = rng.choice(("fixed", "poisson", "poisson", "zipf"))
    if kind == "random":
        return _case(None, "plan", pattern, rows, cols, mean, rng.choice(("f32", "f16", "bf16")),
                     beta=rng.choice((0.0, 0.5)), index=rng.choice(("i32", "i64")))
    if kind == "random_T":
        return _case(None, "plan", pattern, rows, cols, mean, rng.choice(("f32", "f16", "bf16")), "T",
                     beta=rng.choice((0.0, -1.0)))
    small = _log(rng, 4096, 1048576)
    if kind == "mv":
        return _case(None, "mv", pattern, small, small, mean, rng.choice(("f32", "f32", "f16")), index="i64")
    if kind == "once":
        return _case(None, "once", pattern, small, max(4096, int(small * rng.uniform(0.6, 1.6))), mean, "f32",
                     rng.choice(("N", "T", "T")), 1.0, rng.choice((0.0, -1.0)))
    if kind == "spmvop":
        return _case(None, "spmvop", rng.choice(("fixed", "poisson")), rows, cols, min(mean, 24), "f32", "N", -1.0, 1.0)
    if rng.random() < 0.35:  # dense blocks: rows and columns of the perf table's range
        return _case(None, "spmm", "half", rng.randint(512, 4096), rng.randint(32, 256), 0,
                     rng.choice(("f32", "f16")), n=rng.randint(64, 512) * 4)
    if rng.random() < 0.5:
        return _stencil(None, "spmm", _log(rng, 128, 1536), n=rng.choice((4, 8, 16, 24, 32, 33)))
    return _case(None, "spmm", "poisson", small, small, 12, rng.choice(("f32", "f16")), n=rng.choice((16, 32, 64, 100)))


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _uniform(shape, g, dtype):
    if dtype == "i8":
        return torch.randint(-5, 6, shape, generator=g, device="cuda", dtype=torch.int8)
    if dtype == "c64":
        return torch.view_as_complex(torch.rand(*shape, 2, generator=g, device="cuda") * 2 - 1)
    return (torch.rand(shape, generator=g, device="cuda") * 2 - 1).to(_DTYPE[dtype])


def _lengths(case, g):
    rows, mean = case["rows"], case["mean"]
    if case["pattern"] == "poisson":
        lens = torch.poisson(torch.full((rows,), float(mean), device="cuda"), generator=g)
        lens[torch.rand(rows, generator=g, device="cuda") < 0.1] = 0
        return lens.to(torch.int64)
    cap = min(_ZIPF_CAP, case["cols"])
    z = (1.0 / (1.0 - torch.rand(rows, generator=g, device="cuda", dtype=torch.float64))).floor_()
    u = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    lo, hi = 0.0, 64.0 * mean
    for _ in range(40):  # the scale at which the capped lengths have the mean asked for
        mid = 0.5 * (lo + hi)
        if float((z * mid + u).floor_().clamp_(max=cap).sum()) < mean * rows:
            lo = mid
        else:
            hi = mid
    return (z * hi + u).floor_().clamp_(max=cap).to(torch.int64)


def _pattern(case, g):
    """(row offsets, columns) on the GPU, columns sorted in each row."""
    rows, cols = case["rows"], case["cols"]
    off = torch.int64 if case["index"] == "i64" else torch.int32
    if case["pattern"] == "stencil":
        n = math.isqrt(rows)
        idx = torch.arange(rows, device="cuda")
        i, j = idx // n, idx % n
        ok = torch.stack([i > 0, j > 0, i >= 0, j < n - 1, i < n - 1], dim=1)
        col = torch.stack([idx - n, idx - 1, idx, idx + 1, idx + n], dim=1)[ok].to(torch.int32)
        lens = ok.sum(dim=1)
    elif case["pattern"] == "half":
        r, c = torch.arange(rows, device="cuda") % 100, torch.arange(cols, device="cuda") % 100
        shift = int(torch.randint(0, 100, (1,), generator=g, device="cuda"))
        ok = (r[:, None] * 7 + c[None, :] * 13 + shift) % 100 < 50
        col = ok.nonzero()[:, 1].to(torch.int32)
        lens = ok.sum(dim=1)
    elif case["pattern"] == "fixed":
        col = torch.randint(0, cols, (rows, case["mean"]), generator=g, device="cuda", dtype=torch.int32)
        col = torch.sort(col, dim=1).values.reshape(-1)
        return torch.arange(0, rows * case["mean"] + 1, case["mean"], device="cuda", dtype=off), col
    else:
        lens = _lengths(case, g)
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"), lens)
        key = row.mul_(cols).add_(torch.randint(0, cols, (row.numel(),), generator=g, device="cuda"))
        col = torch.sort(key).values.remainder_(cols).to(torch.int32)
    ptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lens, 0, out=ptr[1:])
    return ptr.to(off), col


def _inputs(case, seed):
    g = _gen(seed)
    dt, t = case["dtype"], _DTYPE[case["dtype"]]
    ptr, col = _pattern(case, g)
    nnz, rows, cols = col.numel(), case["rows"], case["cols"]
    if case["pattern"] == "stencil":
        row = torch.repeat_interleave(torch.arange(rows, device="cuda", dtype=torch.int32), ptr.diff().to(torch.int64))
        val = torch.where(row == col, 4.0, -1.0).to(t)
        if dt == "c64":
            val = val + 0.25j * (row > col)
    elif dt in ("f16", "bf16") and case["api"] != "spmm":
        val = torch.randn(nnz, generator=g, device="cuda").to(t)
    else:
        val = _uniform((nnz,), g, dt)
    if case["api"] == "spmm":
        return ptr, col, val, _uniform((cols, case["n"]), g, dt), _uniform((rows, case["n"]), g, dt)
    xl, yl = (cols, rows) if case["op"] == "N" else (rows, cols)
    x, y = _uniform((xl,), g, dt), _uniform((yl,), g, dt)
    return ptr, col, val, x, y.to(torch.int32) if dt == "i8" else y


def prepare(case, seed):
    ptr, col, val, x, y = _inputs(case, seed)
    rows, cols, api = case["rows"], case["cols"], case["api"]
    s = dict(case=case, y=y)
    if api == "plan":
        s["plan"] = CsrSpMV(rows, cols, ptr, col, val, x, y, case["alpha"], case["beta"], op=_OP[case["op"]])
        s["plan"].preprocess()
    elif api == "mv":
        s["csr"] = torch.sparse_csr_tensor(ptr, col.to(torch.int64), val, (rows, cols))
        s["x"] = x
    elif api == "once":
        s["args"] = (ptr, col, val, x, y, case["alpha"], case["beta"], case["op"])
    elif api == "spmvop":
        s["z"] = torch.empty_like(y)
        s["plan"] = SpMVOp(rows, cols, ptr, col, val, x, y, s["z"], alg=SpMVOpAlg.ALG2)
    else:
        s["b"] = x
        s["plan"] = SpMMOp(rows, cols, ptr, col, val, x, y)
    return s


def run(state):
    case = state["case"]
    api = case["api"]
    if api == "plan":
        state["plan"].run()
        return state["y"]
    if api == "mv":
        return torch.mv(state["csr"], state["x"])
    if api == "once":
        return spmv_npu(*state["args"])
    if api == "spmvop":
        state["plan"].run(case["alpha"], case["beta"])
        return state["z"]
    state["plan"].run(state["b"], state["y"], case["alpha"], case["beta"])
    return state["y"]


def _nnz(case):
    rows, mean = case["rows"], case["mean"]
    if case["pattern"] == "stencil":
        return 5 * rows - 4 * math.isqrt(rows)
    if case["pattern"] == "half":
        return rows * case["cols"] // 2
    return int(rows * mean * (0.9 if case["pattern"] == "poisson" else 1.0))


def work(case):
    """Every array once: row offsets, columns and values, x (or B), y (or C) written, and read when beta != 0."""
    nnz, rows, cols, n, vb = _nnz(case), case["rows"], case["cols"], case["n"], _BYTES[case["dtype"]]
    ob = 4 if case["dtype"] == "i8" else vb
    xl, yl = (cols, rows) if case["op"] == "N" else (rows, cols)
    index = (8 if case["index"] == "i64" else 4) * (rows + 1) + (8 if case["api"] == "mv" else 4) * nnz
    return {"bytes": index + vb * nnz + vb * xl * n + ob * yl * n * (2 if case["beta"] != 0 else 1),
            "flops": (8 if case["dtype"] == "c64" else 2) * nnz * n}


def tolerance(case):
    """About four times the measured distance of the results from 64-bit ones: one rounding of the result for 16-bit
    types (2.1e-4 and 1.7e-3) and for compensated sums (2.5e-8), the roundings of a row's fp32 products and sums
    otherwise (6e-8 to 1.6e-7)."""
    if case["dtype"] == "i8":
        return "exact"
    if case["dtype"] in ("f16", "bf16"):
        return {"rel": 8e-4 if case["dtype"] == "f16" else 7e-3}
    return {"rel": 1e-7 if case["api"] == "spmvop" else 6e-7}


def exact(case, seed):
    ptr, col, val, x, y = _inputs(case, seed)
    rows, cols, n = case["rows"], case["cols"], case["n"]
    wide = torch.complex128 if case["dtype"] == "c64" else torch.int64 if case["dtype"] == "i8" else torch.float64
    alpha, beta = (int(case[k]) if case["dtype"] == "i8" else case[k] for k in ("alpha", "beta"))
    ptr = ptr.to(torch.int64)
    x = x.to(wide)
    acc = torch.zeros(y.shape, dtype=wide, device="cuda")
    step = max(1, (1 << 25) // n)  # entries at a time
    for lo in range(0, col.numel(), step):
        hi = min(lo + step, col.numel())
        c = col[lo:hi].to(torch.int64)
        r = torch.searchsorted(ptr, torch.arange(lo, hi, device="cuda"), right=True) - 1
        v = val[lo:hi].to(wide)
        if case["op"] == "H" and case["dtype"] == "c64":
            v = v.conj().resolve_conj()
        if case["op"] != "N":
            r, c = c, r
        acc.index_add_(0, r, v[:, None] * x[c] if case["api"] == "spmm" else v * x[c])
    out = alpha * acc
    if beta != 0:
        out = out + beta * y.to(wide)
    return out.clamp(-2**31, 2**31 - 1).to(torch.int32) if case["dtype"] == "i8" else out
