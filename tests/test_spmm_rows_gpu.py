"""The row kernel with wavefronts per row that follow each row's own length (``iex_spmm_sched``, family 11): forced on
every tile width and chunk budget, where the library picks it by itself, with a wrong histogram and with rows in another
order (both may cost time, never correctness), and the histogram kernel against numpy."""
import ctypes

import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib, workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import FP16_SUBNORMAL_HALF_STEP, assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops


def _histogram(row_offsets):
    lens = np.diff(row_offsets.astype(np.int64))
    return [int((lens > (64 << j)).sum()) for j in range(16)]


def test_histogram_kernel_counts_like_numpy(dev):
    for sparsity, m in ((0.7, 4096), (0.98, 4096), (0.9, 777)):
        c = W.config2_matrix(sparsity, m=m, k=4096, seed=5)
        ro = torch.from_numpy(c.row_offsets).to(dev)
        assert list(pyops._row_histogram_host(ro)) == _histogram(c.row_offsets)


def _call(c, dev, b_np, dtype, itype, flags, hist, batch=1, row_indices=None):
    ri, v, ro, ci = to_dev(c, dev, dtype, itype)
    if row_indices is not None:
        ri = torch.from_numpy(row_indices).to(dev)
    bt = torch.from_numpy(b_np).to(dev).to(dtype)
    out = torch.full((batch, c.m, b_np.shape[2]), float("nan"), device=dev, dtype=dtype)
    rc = _lib.load().iex_spmm_sched({torch.float32: _lib.F32, torch.float16: _lib.F16}[dtype], _lib.I16 if itype == torch.int16 else _lib.I32,
                                    flags, c.m, c.k, b_np.shape[2], c.nnz, ri.data_ptr(), v.data_ptr(), ro.data_ptr(), ci.data_ptr(),
                                    bt.data_ptr(), None, out.data_ptr(), torch.cuda.current_stream().cuda_stream, batch, None, 0,
                                    (ctypes.c_int * 16)(*hist) if hist is not None else None)
    assert rc == 0, _lib.last_error()
    return out


@pytest.mark.parametrize("n", [32, 64, 128, 256, 520])
@pytest.mark.parametrize("rounds_code", [0, 1, 3, 5])
def test_forced_on_every_tile_width_fp32(oracle, dev, n, rounds_code):
    c = W.config2_matrix(0.9, m=700, k=1024, seed=11)     # rows from 1 to several hundred nonzeros, a ragged last workgroup
    rng = np.random.default_rng(n)
    b_np = rng.standard_normal((2, c.k, n)).astype(np.float32)
    out = _call(c, dev, b_np, torch.float32, torch.int32, (11 << 16) | (rounds_code << 20), _histogram(c.row_offsets), batch=2)
    assert "spmm_rows_kernel" in _lib.last_kernels()
    want = oracle.spmm(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    assert_close(out.cpu().numpy(), want, scale, 1e-5, f"rows kernel n={n}")


@pytest.mark.parametrize("itype", [torch.int32, torch.int16])
def test_forced_fp16(oracle, dev, itype):
    c = W.config2_matrix(0.8, m=513, k=2048, seed=12)
    rng = np.random.default_rng(3)
    b_np = rng.standard_normal((1, c.k, 192)).astype(np.float32)
    out = _call(c, dev, b_np, torch.float16, itype, 11 << 16, _histogram(c.row_offsets))
    assert "spmm_rows_kernel" in _lib.last_kernels()
    v, b_r = rounded(c.values, torch.float16), rounded(b_np, torch.float16)
    want = oracle.spmm(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    assert_close(out.float().cpu().numpy(), want, scale, 1e-2, "rows kernel fp16", atol=FP16_SUBNORMAL_HALF_STEP)


def test_a_wrong_histogram_or_another_row_order_costs_time_only(oracle, dev):
    c = W.config2_matrix(0.95, m=1024, k=4096, seed=13)
    rng = np.random.default_rng(4)
    b_np = rng.standard_normal((1, c.k, 64)).astype(np.float32)
    want = oracle.spmm(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    for hist in ([0] * 16, [c.m] * 16, [c.m, c.m // 2, 3] + [0] * 13, [-5, 10 ** 9] + [0] * 14):
        out = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, hist)
        assert_close(out.cpu().numpy(), want, scale, 1e-5, f"histogram {hist[:3]}")
    identity = np.arange(c.m, dtype=np.int32)
    out = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, _histogram(c.row_offsets), row_indices=identity)
    assert_close(out.cpu().numpy(), want, scale, 1e-5, "rows in natural order")
    out = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, _histogram(c.row_offsets), row_indices=c.row_indices[::-1].copy())
    assert_close(out.cpu().numpy(), want, scale, 1e-5, "shortest rows first")


def test_repeated_calls_give_the_same_bits(dev):
    c = W.config2_matrix(0.98)
    b_np = W.config2_dense(128)
    a = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, _histogram(c.row_offsets))
    b = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, _histogram(c.row_offsets))
    assert torch.equal(a, b)


def test_picked_by_the_operator_on_the_sparsest_cells_of_the_sweep(oracle, dev):
    c = W.config2_matrix(0.98)
    ri, v, ro, ci = to_dev(c, dev)
    for n, expect in ((64, True), (128, True), (256, False)):
        b_np = W.config2_dense(n)
        out = ops.spmm_sputnik_reuse_weight(torch.from_numpy(b_np).to(dev), ri, v, ro, ci, c.m)
        assert ("spmm_rows_kernel" in _lib.last_kernels()) == expect, _lib.last_kernels()
        want = oracle.spmm(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
        scale = oracle.spmm_abs_scale(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
        assert_close(out.cpu().numpy(), want, scale, 1e-5, f"sweep cell 98 % n={n}")


@pytest.mark.parametrize("sparsity,n", [(0.98, 64), (0.9, 128), (0.7, 64)])
def test_order_of_rows_and_histogram_change_no_bit(dev, sparsity, n):
    """The operators promise that the order of row_indices is scheduling only.  Here it settles how many wavefronts a
    row has, but the row's sum is cut by the row's own length: a random order, the reverse order (the longest rows
    where one wavefront serves a row, the shortest where 16 do) and wrong histograms (every row long, no row long)
    give the bits of the sorted order with the true histogram."""
    c = W.config2_matrix(sparsity, m=2048, k=4096, seed=9)
    # a few very long rows, so that every class is there
    lens = np.diff(c.row_offsets).copy()
    lens[[5, 77, 1000]] = [4096, 2500, 1100]
    rng = np.random.default_rng(2)
    ro, ci = W.csr_from_row_lengths(rng, c.m, c.k, lens)
    c = W.CSR(c.m, c.k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    b_np = rng.standard_normal((1, c.k, n)).astype(np.float32)
    true_hist = _histogram(c.row_offsets)
    base = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, true_hist)
    assert "spmm_rows_kernel" in _lib.last_kernels()
    perm = rng.permutation(c.m).astype(np.int32)
    for order in (perm, c.row_indices[::-1].copy()):
        for hist in (true_hist, [c.m] * 16, [0] * 16, [c.m, c.m // 2, 7] + [0] * 13):
            got = _call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, hist, row_indices=order)
            assert torch.equal(got, base), (order[:4], hist[:4])
    for hist in ([c.m] * 16, [0] * 16):
        assert torch.equal(_call(c, dev, b_np, torch.float32, torch.int32, 11 << 16, hist), base)


@pytest.mark.parametrize("m,k,n,sparsity", [(2048, 1024, 64, 0.9), (4500, 600, 128, 0.9), (1100, 2000, 512, 0.85), (2100, 1500, 130, 0.95)])
def test_with_nothing_forced_the_histogram_settles_the_bits_and_the_order_does_not(oracle, dev, m, k, n, sparsity):
    """Several nonzeros per gather and one, whole vectors and ragged rows: another order of the rows changes no bit, another histogram (the rule may then cut
    the sums another way) or none at all leaves every row complete."""
    c = W.config2_matrix(sparsity, m=m, k=k, seed=21)
    rng = np.random.default_rng(22)
    b_np = rng.standard_normal((1, k, n)).astype(np.float32)
    want = oracle.spmm(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_np, c.row_indices, c.values, c.row_offsets, c.column_indices, c.m)
    true_hist = _histogram(c.row_offsets)
    for hist in (true_hist, [0] * 16, [m] * 16, [m, m // 2, 3] + [0] * 13, None):
        base = _call(c, dev, b_np, torch.float32, torch.int32, 0, hist)
        assert_close(base.cpu().numpy(), want, scale, 1e-5, f"histogram {hist and hist[:3]}")
        for order in (rng.permutation(m).astype(np.int32), c.row_indices[::-1].copy()):
            assert torch.equal(_call(c, dev, b_np, torch.float32, torch.int32, 0, hist, row_indices=order), base), hist and hist[:3]


def test_forcing_it_without_a_histogram_is_refused(dev):
    c = W.config2_matrix(0.9, m=64, k=256, seed=1)
    ri, v, ro, ci = to_dev(c, dev)
    b = torch.randn(1, c.k, 64, device=dev)
    out = torch.empty(1, c.m, 64, device=dev)
    rc = _lib.load().iex_spmm_ex(_lib.F32, _lib.I32, 11 << 16, c.m, c.k, 64, c.nnz, ri.data_ptr(), v.data_ptr(), ro.data_ptr(), ci.data_ptr(),
                                 b.data_ptr(), None, out.data_ptr(), torch.cuda.current_stream().cuda_stream, 1)
    assert rc == _lib.load().iex_spmm_ex.restype(-1) or rc == -1
    assert "histogram" in _lib.last_error()


@pytest.mark.parametrize("dtype,n", [(torch.float32, 32), (torch.float32, 64), (torch.float32, 100), (torch.float32, 256), (torch.float32, 130), (torch.float32, 301),
                                     (torch.float16, 64), (torch.float16, 128), (torch.float16, 200), (torch.float16, 520), (torch.float16, 259)])
@pytest.mark.parametrize("code", [1, 3, 15])                # more than 64 or 256 nonzeros are long, none is
def test_four_wavefronts_for_the_long_rows_only(oracle, dev, dtype, n, code):
    """Every tile width and rows of no whole vectors, empty rows, a ragged last workgroup; the order of the rows and a wrong histogram change no bit."""
    rng = np.random.default_rng(n + code)
    m, k = 205, 700
    lens = rng.integers(0, 90, m)
    lens[[3, 77, 150, 151]] = [700, 257, 65, 0]
    ro, ci = W.csr_from_row_lengths(rng, m, k, lens)
    c = W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    b_np = rng.standard_normal((2, k, n)).astype(np.float32)
    flags = (11 << 16) | (4 << 8) | (code << 20)
    hist = _histogram(c.row_offsets)
    out = _call(c, dev, b_np, dtype, torch.int32, flags, hist, batch=2)
    assert "spmm_rows_kernel4" in _lib.last_kernels()
    v, b_r = rounded(c.values, dtype), rounded(b_np, dtype)
    want = oracle.spmm(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    half = dtype == torch.float16   # 700 roundings of a sum, each 2^-24 of the magnitudes; fp16: the result's rounding too, 2^-11 of it or 2^-25
    assert_close(out.float().cpu().numpy(), want, scale, 2.0 ** -11 if half else 0.0, f"{dtype} n={n}", atol=700 * 2.0 ** -24 * scale + (2.0 ** -25 if half else 0.0))
    for order in (None, np.arange(m, dtype=np.int32), rng.permutation(m).astype(np.int32)):
        for h in (hist, [m] * 16, [0] * 16, [3, 2, 1] + [0] * 13, [-4] + [10 ** 9] * 15):
            assert torch.equal(_call(c, dev, b_np, dtype, torch.int32, flags, h, batch=2, row_indices=order), out), (h[:3], order is None)


@pytest.mark.parametrize("dtype,m,k,n,sparsity,even,kernel", [
    (torch.float32, 11008, 1000, 64, 0.95, True, "spmm_rows_kernel4"), (torch.float16, 11008, 1000, 64, 0.95, True, "8, 8, 1, 1"), (torch.float16, 6144, 512, 128, 0.9, False, "spmm_rows_kernel4"),
    (torch.float32, 4096, 1024, 512, 0.95, False, "spmm_rows_kernel4"), (torch.float32, 512, 1024, 512, 0.9, False, "spmm_rows_kernel<"), (torch.float32, 4096, 512, 256, 0.9, True, "64, 1, 1")])
def test_operator_takes_the_wavefronts_per_row_from_the_row_lengths(oracle, dev, dtype, m, k, n, sparsity, even, kernel):
    rng = np.random.default_rng(m + n)
    mean = k * (1 - sparsity)
    lens = np.full(m, int(mean)) if even else np.minimum(k, rng.geometric(1 / mean, m))
    ro, ci = W.csr_from_row_lengths(rng, m, k, lens)
    c = W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    ri, v, ro_t, ci_t = to_dev(c, dev, dtype)
    b_np = rng.standard_normal((1, k, n)).astype(np.float32)
    b = torch.from_numpy(b_np).to(dev).to(dtype)
    out = (ops.spmm_sputnik_reuse_weight if dtype == torch.float32 else ops.spmm_sputnik_reuse_weight_half)(b, ri, v, ro_t, ci_t, m)
    assert kernel in _lib.last_kernels(), _lib.last_kernels()
    v, b_r = rounded(c.values, dtype), rounded(b_np, dtype)
    want = oracle.spmm(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    scale = oracle.spmm_abs_scale(b_r, c.row_indices, v, c.row_offsets, c.column_indices, c.m)
    half = dtype == torch.float16
    assert_close(out.float().cpu().numpy(), want, scale, 2.0 ** -11 if half else 0.0, kernel, atol=float(lens.max()) * 2.0 ** -24 * scale + (2.0 ** -25 if half else 0.0))
