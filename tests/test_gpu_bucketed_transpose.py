"""GPU parity of the column-bucketed transpose (fp32 values, opA = T or H) through the C ABI.

Preprocess takes this path for fp32 transposes of at least 2^20 entries when
every bucket of columns fits pass 2's LDS; each test reads the choice from the
workspace header (staged_flag) so that a case meant for the bucketed kernels
cannot pass on the CSC kernels, and the other way round.
"""
import ctypes

import numpy as np
import pytest
import torch

from helpers import assert_close
from ops_sparse._lib import Operation, PointerMode
from ops_sparse.spmv import CsrSpMV
from ops_sparse import workloads as wl

pytestmark = pytest.mark.gpu

REGION_TARGET = 24576
REGION_CAP = 32768


def header(plan):
    h = np.frombuffer(plan.workspace[:192].cpu().numpy().tobytes(), dtype=np.uint64)
    return int(h[16] & 0xFFFFFFFF), int(h[16] >> 32), int(h[17])


def bucket_width(cols, nnz):
    target = REGION_TARGET * cols // nnz
    shift = 6
    while shift < 16 and (2 << shift) <= target:
        shift += 1
    return 1 << shift


def run(w, op=Operation.TRANSPOSE, preprocess=True, y0=None):
    y = (w.y0 if y0 is None else y0).clone()
    plan = CsrSpMV(w.rows, w.cols, w.row_ptr, w.col_ind, w.values, w.x, y, w.alpha, w.beta, op=op,
                   base=w.meta.get("base", 0))
    if preprocess:
        plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    return y, plan


def host(w):
    h = w.to("cpu")
    b = w.meta.get("base", 0)
    if b:
        h.col_ind = h.col_ind - b
        h.row_ptr = h.row_ptr - b
    return h


def transpose_workload(dev, rows, cols, mean, seed, base=0, rdtype=torch.int32, alpha=1.0, beta=2.0):
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    lengths = torch.poisson(torch.full((rows,), mean), generator=g).to(torch.int64)
    row_ptr, col = wl.csr_from_lengths(lengths, cols, g, "cpu", distinct=False)
    n = col.numel()
    vals = torch.rand(n, generator=g) * 2 - 1
    x = torch.rand(rows, generator=g) * 2 - 1
    y0 = torch.rand(cols, generator=g) * 2 - 1
    w = wl.Workload(f"bt_{rows}x{cols}", rows, cols, (row_ptr + base).to(rdtype), (col + base).to(torch.int32),
                    vals, x, y0, alpha, beta, trans="T", meta={"base": base})
    return w.to(dev)


def test_c5_takes_the_bucketed_path_and_matches_oracle(dev):
    w = wl.poisson_transpose().to(dev)
    y, plan = run(w)
    flag, buckets, tiles = header(plan)
    assert flag == 1, "c5's buckets fit the column pass's LDS: the bucketed kernels run"
    assert buckets == -(-w.cols // bucket_width(w.cols, w.nnz))
    assert_close(w.to("cpu"), y)
    # again from the same y: bit-identical (every column is summed in row order), on a new plan
    # (its first SpMV launches both kernel sets, which read the device flag) and on this plan
    # once Preprocess's choice has reached the host (only the bucketed kernels are launched)
    y3, _ = run(w)
    assert torch.equal(y.view(torch.int32), y3.view(torch.int32))
    first = y.clone()
    y.copy_(w.y0)
    plan.run()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int32), y.view(torch.int32))


def test_conjugate_transpose_int64_base1_beta0_ignores_nan_y(dev):
    w = transpose_workload(dev, rows=1 << 20, cols=3 << 18, mean=9.0, seed=5, base=1, rdtype=torch.int64,
                           alpha=-1.5, beta=0.0)
    y0 = torch.full((w.cols,), float("nan"), device=dev)
    y, plan = run(w, op=Operation.CONJUGATE_TRANSPOSE, y0=y0)
    assert header(plan)[0] == 1
    assert bool(torch.isfinite(y).all())
    assert_close(host(w), y)


def test_rectangular_device_scalars(dev):
    w = transpose_workload(dev, rows=3 << 20, cols=1 << 20, mean=2.0, seed=8, alpha=0.75, beta=-0.5)
    y = w.y0.clone()
    plan = CsrSpMV(w.rows, w.cols, w.row_ptr, w.col_ind, w.values, w.x, y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.handle.set_pointer_mode(PointerMode.DEVICE)
    da = torch.tensor([0.75], device=dev)
    db = torch.tensor([-0.5], device=dev)
    plan.alpha = type("P", (), {"ptr": ctypes.c_void_p(da.data_ptr())})()
    plan.beta = type("P", (), {"ptr": ctypes.c_void_p(db.data_ptr())})()
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    assert header(plan)[0] == 1
    assert_close(w.to("cpu"), y)


def test_a_giant_column_keeps_the_csc_kernels(dev):
    """One column holding more entries than pass 2's LDS: Preprocess keeps the CSC kernels."""
    w = transpose_workload(dev, rows=1 << 20, cols=1 << 20, mean=3.0, seed=9)
    col = w.col_ind.clone()
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    hot = torch.rand(col.numel(), generator=g, device=dev) < (2 * REGION_CAP) / col.numel()
    col[hot] = 12345
    w.col_ind = col
    y, plan = run(w)
    assert header(plan)[0] == 0
    assert_close(w.to("cpu"), y)


def test_entries_outside_the_rows_are_ignored(dev):
    """row_ptr[0] > 0: the leading entries belong to no row and must not reach y."""
    w = transpose_workload(dev, rows=1 << 20, cols=1 << 19, mean=4.0, seed=10)
    lead = 7
    w.row_ptr = w.row_ptr + lead
    w.col_ind = torch.cat([torch.arange(lead, dtype=torch.int32, device=dev), w.col_ind])
    w.values = torch.cat([torch.full((lead,), 1e6, device=dev), w.values])
    y, plan = run(w)
    assert header(plan)[0] == 1
    assert_close(w.to("cpu"), y)


def test_without_preprocess_runs_the_csc_kernels(dev):
    w = transpose_workload(dev, rows=1 << 20, cols=1 << 20, mean=6.0, seed=11)
    y, plan = run(w, preprocess=False)
    assert header(plan)[0] == 0
    assert_close(w.to("cpu"), y)


def banded_workload(dev, n=1536, beta=0.5, base=0):
    """A 5-point Laplacian (banded, long runs per tile) as a transpose workload."""
    w = wl.laplacian_2d(n=n)
    w = wl.Workload(w.name + "_T", w.rows, w.cols, (w.row_ptr + base).to(torch.int32),
                    (w.col_ind + base).to(torch.int32), w.values * (1.0 + 0.25 * torch.rand(w.nnz)),
                    w.x, w.y0, 1.5, beta, trans="T", meta={"base": base})
    return w.to(dev)


def test_banded_transpose_takes_the_one_pass_kernel(dev):
    """Long runs: Preprocess picks the one-pass banded column kernel, on its 16-bit copies (flag 4: every
    entry's row within 16 bits of its CSC block's first column, its CSR position within 16 bits of its CSC
    index); repeated runs are
    bit-identical on a new plan (every kernel set launched, gated on the device flag) and on this plan
    once the choice has reached the host (only the banded kernel launched)."""
    w = banded_workload(dev)
    assert w.nnz >= 1 << 20
    y, plan = run(w)
    assert header(plan)[0] == 4
    assert_close(w.to("cpu"), y)
    y3, _ = run(w)
    assert torch.equal(y.view(torch.int32), y3.view(torch.int32))
    first = y.clone()
    y.copy_(w.y0)
    plan.run()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int32), y.view(torch.int32))


def test_banded_conjugate_transpose_base1_beta0_ignores_nan_y(dev):
    w = banded_workload(dev, n=1100, beta=0.0, base=1)
    y0 = torch.full((w.cols,), float("nan"), device=dev)
    y, plan = run(w, op=Operation.CONJUGATE_TRANSPOSE, y0=y0)
    assert header(plan)[0] == 4
    assert bool(torch.isfinite(y).all())
    assert_close(host(w), y)


def test_banded_transpose_int64_offsets_keeps_the_csc_kernels(dev):
    """The one-pass banded kernel takes 32-bit row offsets: with int64 offsets Preprocess keeps the
    CSC kernels (flag 0) and the result is still right, on the first SpMV (every kernel set launched)
    and once the choice is on the host."""
    w = banded_workload(dev, n=1100)
    w.row_ptr = w.row_ptr.to(torch.int64)
    y, plan = run(w)
    assert header(plan)[0] == 0
    assert_close(w.to("cpu"), y)
    first = y.clone()
    y.copy_(w.y0)
    plan.run()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int32), y.view(torch.int32))


def test_banded_transpose_far_band_keeps_32_bit_streams(dev):
    """A Laplacian plus a band 40 000 columns off the diagonal: still banded (long runs, flag 2), but those
    entries' rows and positions are out of 16-bit reach, so the kernel streams the 32-bit arrays; the result
    is checked against the oracle and is bit-identical on a second run."""
    n = 1100
    m = n * n
    i = torch.arange(m, dtype=torch.int64)
    cols = [i - n, i - 1, i, i + 1, i + n, i + 40000]
    r = torch.cat([i] * len(cols))
    c = torch.cat(cols)
    ok = (c >= 0) & (c < m)
    r, c = r[ok], c[ok]
    order = torch.argsort(r * m + c)
    r, c = r[order], c[order]
    row_ptr = torch.zeros(m + 1, dtype=torch.int64)
    row_ptr[1:] = torch.cumsum(torch.bincount(r, minlength=m), 0)
    g = torch.Generator(device="cpu")
    g.manual_seed(12)
    vals = torch.rand(c.numel(), generator=g) * 2 - 1
    x = torch.rand(m, generator=g) * 2 - 1
    y0 = torch.rand(m, generator=g) * 2 - 1
    w = wl.Workload("laplace_far_T", m, m, row_ptr.to(torch.int32), c.to(torch.int32), vals, x, y0, 1.25, -0.5,
                    trans="T").to(dev)
    y, plan = run(w)
    flag, _, _ = header(plan)
    assert flag == 2
    assert_close(w.to("cpu"), y)
    first = y.clone()
    y.copy_(w.y0)
    plan.run()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int32), y.view(torch.int32))


@pytest.mark.parametrize("extra", [5000, 9000])
def test_banded_transpose_long_column_tasks(dev, extra):
    """A Laplacian plus one column holding `extra` more entries (rows within extra/2 of it): still the
    one-pass banded kernel on 16-bit copies (flag 4), with that column's block several chunks long, so
    it is summed by tasks whose partial sums are combined; checked against the oracle and bit-identical
    on a second run."""
    n = 1100
    m = n * n
    i = torch.arange(m, dtype=torch.int64)
    r = torch.cat([i] * 5)
    c = torch.cat([i - n, i - 1, i, i + 1, i + n])
    c0 = m // 2 + 17
    rr = torch.arange(c0 - extra // 2, c0 + extra // 2 + 1, dtype=torch.int64)
    r = torch.cat([r, rr])
    c = torch.cat([c, torch.full_like(rr, c0)])
    ok = (c >= 0) & (c < m)
    key = torch.unique(r[ok] * m + c[ok])
    r, c = key // m, key % m
    row_ptr = torch.zeros(m + 1, dtype=torch.int64)
    row_ptr[1:] = torch.cumsum(torch.bincount(r, minlength=m), 0)
    g = torch.Generator(device="cpu")
    g.manual_seed(extra)
    vals = torch.rand(c.numel(), generator=g) * 2 - 1
    x = torch.rand(m, generator=g) * 2 - 1
    y0 = torch.rand(m, generator=g) * 2 - 1
    w = wl.Workload("laplace_longcol_T", m, m, row_ptr.to(torch.int32), c.to(torch.int32), vals, x, y0, 0.75, 1.5,
                    trans="T").to(dev)
    y, plan = run(w)
    assert header(plan)[0] == 4
    assert_close(w.to("cpu"), y)
    first = y.clone()
    y.copy_(w.y0)
    plan.run()
    torch.cuda.synchronize()
    assert torch.equal(first.view(torch.int32), y.view(torch.int32))


@pytest.mark.parametrize("tail", [1, 2, 3, 5, 7, 8])
def test_entry_counts_of_every_remainder_mod_8(dev, tail):
    """nnz = 8q + tail (tail = 8: a multiple of 8): pass 2 reads each bucket's products and places
    by 16-byte loads from an 8-entry boundary, so the last bucket's final loads cross the end of the
    arrays at every offset; every column, the last (partial) bucket's included, must match the
    oracle."""
    w = transpose_workload(dev, rows=1 << 20, cols=(1 << 20) + 1237 * tail, mean=5.0, seed=20 + tail)
    keep = (w.nnz // 8 - 1) * 8 + tail
    drop = w.nnz - keep
    rp = w.row_ptr.clone()
    rp[-1] -= drop  # the last rows lose their final entries
    rp = torch.minimum(rp, rp[-1])
    w.row_ptr = rp
    w.col_ind = w.col_ind[:keep].contiguous()
    w.values = w.values[:keep].contiguous()
    assert w.nnz == keep and keep % 8 == tail % 8
    y, plan = run(w)
    assert header(plan)[0] == 1
    assert_close(w.to("cpu"), y)


def test_random_pattern_with_few_wide_buckets_takes_the_bucketed_kernels(dev):
    """2 M random entries over 1 M columns: the buckets are few and wide, so the tiles' runs are long
    (about 110 entries), but every tile has a run in every bucket: the pattern is scattered and the
    bucketed kernels take it (the one-pass banded kernel would gather every value from afar)."""
    w = transpose_workload(dev, rows=1 << 18, cols=1 << 20, mean=8.5, seed=31)
    assert w.nnz >= 1 << 21
    y, plan = run(w)
    flag, buckets, tiles = header(plan)
    assert flag == 1
    assert w.nnz / (buckets * tiles) > 64  # long runs, yet scattered
    assert_close(w.to("cpu"), y)


@pytest.mark.parametrize("seed", [41, 42])
def test_mixed_row_lengths_meet_the_middle_of_every_tile(dev, seed):
    """Rows of 0-120 entries (10% empty) with random columns: pass 1 spreads x and places the
    products half a tile at a time, so short rows, rows longer than 32 entries (spread by a wave)
    and empty rows meet the middle of the tile's entries, and runs cross the middle of its slots,
    at every offset.  Bit-identical on a second run."""
    rows, cols = 300_001, (1 << 20) + 77
    rng = np.random.default_rng(seed)
    lengths = torch.from_numpy(np.where(rng.random(rows) < 0.1, 0, rng.integers(1, 121, rows)).astype(np.int64))
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    row_ptr, col = wl.csr_from_lengths(lengths, cols, g, "cpu", distinct=False)
    n = col.numel()
    w = wl.Workload(f"bt_mixed_{seed}", rows, cols, row_ptr.to(torch.int32), col.to(torch.int32),
                    torch.rand(n, generator=g) * 2 - 1, torch.rand(rows, generator=g) * 2 - 1,
                    torch.rand(cols, generator=g) * 2 - 1, 0.75, -1.0, trans="T").to(dev)
    y, plan = run(w)
    assert header(plan)[0] == 1
    assert_close(w.to("cpu"), y)
    y2, _ = run(w)
    assert torch.equal(y.view(torch.int32), y2.view(torch.int32))


# rows, cols, mean: columns per bucket W and buckets S around the limits of the slot and place kernels
PLACE_CASES = [
    (600_000, 1 << 23, 4.0),  # W = 65536 (sorted in LDS), hyper-sparse columns
    (600_000, (1 << 22) + 65, 4.0),  # W = 32768, the last bucket 65 columns wide
    (1 << 20, (1 << 21) + 16383, 2.2),  # W = 16384, the last bucket one column short
    (1 << 20, (1 << 21) + 5, 4.0),  # W = 8192, the last bucket 5 columns wide
    (1 << 20, (1 << 20) + 2049, 4.5),  # W = 4096: two passes of 2048 columns, the last bucket 2049 columns wide
    (1 << 20, (1 << 20) + 4095, 6.5),  # W = 2048, a last bucket of 2047 columns
    (262_147, 8192, 8.5),  # W = 64, columns of about 270 entries
    (1 << 21, 1_800_001, 14.0),  # over 1400 buckets: the slot kernel's LDS beyond 64 KiB
]


@pytest.mark.parametrize("rows,cols,mean", PLACE_CASES)
@pytest.mark.parametrize("x_offset", [0, 1])
def test_columns_are_summed_in_row_order(dev, rows, cols, mean, x_offset):
    """Slots and places follow the entries' order: with alpha = 1 and beta = 0 every column of at most 64
    entries is the sequential fp32 sum of its products in row order, bit for bit (longer ones are summed
    by a wave).  x_offset = 1 binds an x that is only 4-byte aligned after Preprocess: the bucketed
    kernels keep the matrix, which has no CSC pattern to fall back to."""
    g = torch.Generator(device=dev)
    g.manual_seed(rows + cols)
    lengths = torch.poisson(torch.full((rows,), mean, device=dev), generator=g).to(torch.int64)
    row_ptr, col = wl.csr_from_lengths(lengths, cols, g, dev, distinct=False)
    vals = torch.rand(col.numel(), generator=g, device=dev) * 2 - 1
    xs = torch.rand(rows + 1, generator=g, device=dev) * 2 - 1
    y = torch.full((cols,), float("nan"), device=dev)
    plan = CsrSpMV(rows, cols, row_ptr.to(torch.int32), col, vals, xs[:rows], y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    x = xs[x_offset:x_offset + rows]
    plan._lib.aclsparseDnVecSetValues(plan.x.d, ctypes.c_void_p(x.data_ptr()))
    plan.run()
    torch.cuda.synchronize()
    flag, buckets, _ = header(plan)
    assert flag == 1 and buckets == -(-cols // bucket_width(cols, col.numel()))
    row = np.repeat(np.arange(rows), np.diff(row_ptr.cpu().numpy()))
    c, got = col.cpu().numpy(), y.cpu().numpy()
    prod = vals.cpu().numpy() * x.cpu().numpy()[row]
    want = np.zeros(cols, np.float32)
    np.add.at(want, c, prod)
    count = np.bincount(c, minlength=cols)
    short = count <= 64
    np.testing.assert_array_equal(got[short].view(np.uint32), (want[short] + 0.0).view(np.uint32))
    scale = np.bincount(c, weights=np.abs(prod), minlength=cols)
    exact = np.bincount(c, weights=prod.astype(np.float64), minlength=cols)
    assert np.all(np.abs(got - exact) <= 1e-5 * scale)


# entry counts around the CSC sort's smallest own sizes (2^17, with three digits 2^18, with four 3 * 2^17) and tile
# (16384) edges; columns of one to four digits
@pytest.mark.parametrize("nnz", [1, 1025, 131_071, 131_072, 131_073, 147_455, 147_457, 262_143, 262_145, 393_215,
                                 393_217])
@pytest.mark.parametrize("cols", [1, 255, 256, 70_000, 20_000_000])
@pytest.mark.parametrize("i64", [False, True])
def test_csc_sort_edges(dev, nnz, cols, i64):
    """Transposes below the bucketed path's size: the CSC kernels on the pattern the column sort leaves, with
    entries outside the columns ignored, against fp64 sums."""
    rng = np.random.default_rng(nnz * 7 + cols)
    rows = max(1, nnz // 3)
    row_ptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, rows - 1)), [nnz]])
    col = rng.integers(0, cols, nnz).astype(np.int32)
    col[::11] = np.where(np.arange(col[::11].size) % 2 == 0, cols, -1)  # outside the matrix
    val = rng.uniform(-1, 1, nnz).astype(np.float32)
    x = rng.uniform(-1, 1, rows).astype(np.float32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    y = torch.full((cols,), 0.5, device=dev)
    plan = CsrSpMV(rows, cols, d(row_ptr.astype(np.int64 if i64 else np.int32)), d(col), d(val), d(x), y, 2.0, -1.0,
                   op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    ok = (col >= 0) & (col < cols)
    prod = val.astype(np.float64) * x[np.repeat(np.arange(rows), np.diff(row_ptr))]
    want = 2.0 * np.bincount(col[ok], weights=prod[ok], minlength=cols) - 0.5
    scale = 2.0 * np.bincount(col[ok], weights=np.abs(prod[ok]), minlength=cols) + 0.5
    assert np.all(np.abs(y.cpu().numpy() - want) <= 1e-5 * scale)


@pytest.mark.parametrize("vdt,odt", [(torch.float16, torch.float16), (torch.float16, torch.float32),
                                     (torch.bfloat16, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("i64", [False, True])
@pytest.mark.parametrize("rows,cols,mean", [(1 << 20, (1 << 20) + 4095, 6.5), (300_001, 1 << 19, 9.3)])
def test_16_bit_values(dev, vdt, odt, i64, rows, cols, mean):
    """fp16 and bf16 values: fp32 products summed in row order and rounded once to y's type, bit for bit for
    columns of at most 64 entries (x two bytes off a 4-byte boundary, odd entry counts); beta != 0 within one
    rounding of the same sums."""
    g = torch.Generator(device=dev)
    g.manual_seed(rows + cols)
    lengths = torch.poisson(torch.full((rows,), mean, device=dev), generator=g).to(torch.int64)
    lengths[-1] += 1 - int(lengths.sum()) % 2
    row_ptr, col = wl.csr_from_lengths(lengths, cols, g, dev, distinct=False)
    assert col.numel() % 2 == 1
    vals = torch.randn(col.numel(), generator=g, device=dev).to(vdt)
    x = (torch.rand(rows + 1, generator=g, device=dev) * 2 - 1).to(vdt)[1:]
    rp = row_ptr.to(torch.int64 if i64 else torch.int32)
    y = torch.full((cols,), float("nan"), device=dev).to(odt)
    plan = CsrSpMV(rows, cols, rp, col, vals, x, y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    assert header(plan)[0] == 1
    row = np.repeat(np.arange(rows), np.diff(row_ptr.cpu().numpy()))
    c = col.cpu().numpy()
    prod = vals.float().cpu().numpy() * x.float().cpu().numpy()[row]
    acc = np.zeros(cols, np.float32)
    np.add.at(acc, c, prod)
    want = torch.from_numpy(acc + 0.0).to(odt)
    short = torch.from_numpy(np.bincount(c, minlength=cols) <= 64)
    bits = torch.int32 if odt == torch.float32 else torch.int16
    assert torch.equal(y.cpu()[short].view(bits), want[short].view(bits))
    y0 = (torch.rand(cols, generator=g, device=dev) * 2 - 1).to(odt)
    y2 = y0.clone()
    plan2 = CsrSpMV(rows, cols, rp, col, vals, x, y2, 0.5, -1.0, op=Operation.TRANSPOSE)
    plan2.preprocess()
    plan2.run()
    torch.cuda.synchronize()
    exact = 0.5 * np.bincount(c, weights=prod.astype(np.float64), minlength=cols) - y0.cpu().double().numpy()
    scale = 0.5 * np.bincount(c, weights=np.abs(prod), minlength=cols) + np.abs(y0.cpu().double().numpy())
    eps = {torch.float16: 2.0**-11, torch.bfloat16: 2.0**-8, torch.float32: 0.0}[odt]
    assert np.all(np.abs(y2.cpu().double().numpy() - exact) <= eps * np.abs(exact) + 1e-5 * scale + 1e-7)


def test_banded_16_bit_transpose_keeps_the_csc_kernels(dev):
    """The one-pass banded kernel is fp32's: a 16-bit Laplacian stays on the CSC kernels."""
    w = banded_workload(dev, n=1100)
    w.values, w.x, w.y0, w.out_dtype = w.values.half(), w.x.half(), w.y0.half(), torch.float16
    y, plan = run(w)
    assert header(plan)[0] == 0
    assert_close(w.to("cpu"), y)


# 40% of the entries in long rows; a row of 512 entries does not count as long, one of 513 does
@pytest.mark.parametrize("nnz,mean,long_row,flag", [(3_000_000, 2, 512, 1), (3_000_000, 2, 513, 0),
                                                    (4_000_000, 20, 4096, 1)])
def test_16_bit_values_with_long_rows(dev, nnz, mean, long_row, flag):
    """Long rows keep 16-bit transposes of few entries per row on the CSC kernels; either path's sums are within one
    rounding of 64-bit ones."""
    g = torch.Generator(device=dev)
    g.manual_seed(nnz + long_row)
    rows = cols = nnz // mean
    lengths = torch.zeros(rows, dtype=torch.int64, device=dev)
    many = torch.arange(2 * nnz // 5 // long_row, device=dev) * 317 % rows
    rest = nnz - many.numel() * long_row
    lengths += rest // rows
    lengths[: rest - int(lengths.sum())] += 1
    lengths[many] = long_row
    row_ptr, col = wl.csr_from_lengths(lengths, cols, g, dev, distinct=False)
    vals = torch.randn(col.numel(), generator=g, device=dev).half()
    x = (torch.rand(rows, generator=g, device=dev) * 2 - 1).half()
    y = torch.full((cols,), float("nan"), device=dev).half()
    plan = CsrSpMV(rows, cols, row_ptr.to(torch.int32), col, vals, x, y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    assert header(plan)[0] == flag
    prod = vals.double().cpu().numpy() * np.repeat(x.double().cpu().numpy(), lengths.cpu().numpy())
    c = col.cpu().numpy()
    exact = np.bincount(c, weights=prod, minlength=cols)
    scale = np.bincount(c, weights=np.abs(prod), minlength=cols)
    assert np.all(np.abs(y.double().cpu().numpy() - exact) <= 2.0**-11 * np.abs(exact) + 1e-5 * scale + 1e-7)


# the lines between the two kernels that write the column offsets (more columns than entries, or fewer than 2^20 of
# them), with columns crowded at either end, so that one entry is followed by almost all column starts
@pytest.mark.parametrize("nnz", [1, 1023, 1024, 5000, 140_000, (1 << 20) - 1, 1 << 20])
@pytest.mark.parametrize("more", [-1, 0, 1, 70_000])
@pytest.mark.parametrize("crowd", ["low", "high", "spread"])
@pytest.mark.parametrize("i64", [False, True])
def test_column_offsets_line(dev, nnz, more, crowd, i64):
    cols = nnz + more
    if cols < 1:
        pytest.skip("no columns")
    rng = np.random.default_rng(nnz + more)
    rows = nnz // 3 + 1
    row_ptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, rows - 1)), [nnz]])
    few = max(1, cols // 50)
    col = rng.integers(0, cols if crowd == "spread" else few, nnz).astype(np.int32)
    col = cols - 1 - col if crowd == "high" else col
    val, x = rng.uniform(-1, 1, nnz).astype(np.float32), rng.uniform(-1, 1, rows).astype(np.float32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    y = torch.full((cols,), float("nan"), device=dev)
    plan = CsrSpMV(rows, cols, d(row_ptr.astype(np.int64 if i64 else np.int32)), d(col.astype(np.int32)), d(val), d(x), y,
                   1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    prod = val.astype(np.float64) * x[np.repeat(np.arange(rows), np.diff(row_ptr))]
    want, scale = np.bincount(col, weights=prod, minlength=cols), np.bincount(col, weights=np.abs(prod), minlength=cols)
    assert np.all(np.abs(y.cpu().numpy() - want) <= 1e-5 * scale)


# rows and columns per entry on both sides of the line from which 16-bit transposes may take the bucketed kernels
@pytest.mark.parametrize("nnz,rows,cols,flag", [(1_200_000, 4_000_000, 4_000_000, 0), (2_097_151, 300_000, 300_000, 0),
                                                (2_110_000, 300_000, 300_000, 1), (2_200_000, 6_600_000, 300_000, 0),
                                                (2_200_000, 300_000, 6_600_000, 0), (4_400_000, 4_000_000, 300_000, 1)])
def test_16_bit_values_of_many_rows_and_columns(dev, nnz, rows, cols, flag):
    g = torch.Generator(device=dev)
    g.manual_seed(nnz + cols)
    row = torch.sort(torch.randint(0, rows, (nnz,), generator=g, device=dev)).values
    col = torch.randint(0, cols, (nnz,), generator=g, device=dev)
    row_ptr = torch.zeros(rows + 1, dtype=torch.int32, device=dev)
    row_ptr[1:] = torch.cumsum(torch.bincount(row, minlength=rows), 0)
    vals = torch.randn(nnz, generator=g, device=dev).bfloat16()
    x = (torch.rand(rows, generator=g, device=dev) * 2 - 1).bfloat16()
    y = torch.full((cols,), float("nan"), device=dev).bfloat16()
    plan = CsrSpMV(rows, cols, row_ptr, col.to(torch.int32), vals, x, y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    assert header(plan)[0] == flag
    prod = vals.double() * x.double()[row]
    want = torch.zeros(cols, dtype=torch.float64, device=dev).index_add_(0, col, prod)
    scale = torch.zeros(cols, dtype=torch.float64, device=dev).index_add_(0, col, prod.abs())
    assert bool(((y.double() - want).abs() <= 2.0**-8 * want.abs() + 1e-5 * scale + 1e-7).all())


# wide buckets (sorted in LDS) whose entries crowd in a few columns: one column of most of the bucket's entries at its
# start, middle or end, empty buckets, buckets of 1, 63, 64, 65 and the most entries that the kernels take
@pytest.mark.parametrize("width_bits", [13, 14, 15, 16])
def test_wide_buckets_with_crowded_columns(dev, width_bits):
    w = 1 << width_bits
    rng = np.random.default_rng(width_bits)
    counts = [32768, 0, 1, 63, 64, 65, 20000, 1024, 1025, 32767, 0, 5000] + [24000] * 90
    cols = w * (len(counts) - 1) + w // 2 + 3
    col = []
    for b, n in enumerate(counts):
        at = (0, w // 2, w - 1)[b % 3]
        many = np.full(n * 2 // 3, at) if b % 2 else np.zeros(0, np.int64)
        col.append(np.minimum(np.concatenate([many, rng.integers(0, w, n - len(many))]) + b * w, cols - 1))
    col = rng.permutation(np.concatenate(col)).astype(np.int32)
    nnz = len(col)
    assert bucket_width(cols, nnz) == w
    rows = nnz // 3
    row_ptr = np.concatenate([[0], np.sort(rng.integers(0, nnz + 1, rows - 1)), [nnz]])
    val, x = rng.uniform(-1, 1, nnz).astype(np.float32), rng.uniform(-1, 1, rows).astype(np.float32)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    y = torch.full((cols,), float("nan"), device=dev)
    plan = CsrSpMV(rows, cols, d(row_ptr.astype(np.int32)), d(col), d(val), d(x), y, 1.0, 0.0, op=Operation.TRANSPOSE)
    plan.preprocess()
    plan.run()
    torch.cuda.synchronize()
    assert header(plan)[0] == 1
    prod = val * x[np.repeat(np.arange(rows), np.diff(row_ptr))]
    got = y.cpu().numpy()
    want = np.zeros(cols, np.float32)
    np.add.at(want, col, prod)
    short = np.bincount(col, minlength=cols) <= 64
    np.testing.assert_array_equal(got[short].view(np.uint32), (want[short] + 0.0).view(np.uint32))
    exact = np.bincount(col, weights=prod.astype(np.float64), minlength=cols)
    assert np.all(np.abs(got - exact) <= 1e-5 * np.bincount(col, weights=np.abs(prod), minlength=cols))
