"""The dense products behind the sparse operators at shapes of no whole vectors, and A given as (K, M)."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import RTOL, assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu
DTYPES = [torch.float16, torch.bfloat16]
CODE = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _normal(rng, *shape):
    return rng.standard_normal(shape).astype(np.float32)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("tile", [0, 5, 8, 9, 10, 13, 14])
@pytest.mark.parametrize("mnk", [(304, 520, 200), (136, 136, 9), (264, 264, 1001), (8, 8, 129)])
def test_gemm_with_a_as_k_by_m(oracle, dev, dtype, tile, mnk):
    M, N, K = mnk
    rng = np.random.default_rng(K)
    a, b = _normal(rng, K, M), _normal(rng, K, N)
    at, bt = (torch.from_numpy(x).to(dev).to(dtype) for x in (a, b))
    out = torch.full((M, N), float("nan"), dtype=dtype, device=dev)
    lib = _lib.load()
    need = lib.iex_gemm_workspace_bytes(CODE[dtype], 2 | (tile << 4), M, N, K, 1)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
    rc = lib.iex_gemm_ws(CODE[dtype], 2 | (tile << 4), M, N, K, at.data_ptr(), bt.data_ptr(), out.data_ptr(), 1, 0, 0, 0,
                         torch.cuda.current_stream().cuda_stream, ws.data_ptr(), need)
    if tile == 14 and K < 64 * 2:
        assert rc != 0
        return
    _lib.check(rc)
    ar, br = rounded(a, dtype), rounded(b, dtype)
    assert_close(out.float().cpu().numpy(), oracle.gemm(np.ascontiguousarray(ar.T), br), np.abs(ar.T) @ np.abs(br), RTOL[dtype], f"{mnk} tile {tile}")


def _pattern(rng, m, k, dev, idtype, dtype):
    ro, ci = W.csr_from_row_lengths(rng, m, k, rng.integers(0, max(2, k // 4), m))
    csr = W.CSR(m, k, _normal(rng, ci.shape[0]), W.swizzle_from_offsets(ro), ro, ci)
    return csr, to_dev(csr, dev, dtype, idtype)


@pytest.mark.parametrize("dtype,idtype", [(torch.float16, torch.int16), (torch.float16, torch.int32), (torch.bfloat16, torch.int32)])
@pytest.mark.parametrize("m,k,n,batch", [(70, 45, 33, 1), (300, 129, 7, 2), (257, 1003, 264, 2), (129, 64, 521, 3), (65, 5000, 130, 1)])
def test_spmm_by_the_dense_form(oracle, dev, dtype, idtype, m, k, n, batch):
    rng = np.random.default_rng(m + k)
    csr, (ri, v, ro, ci) = _pattern(rng, m, k, dev, idtype, dtype)
    b = _normal(rng, batch, k, n)
    bias = _normal(rng, m)
    bt = torch.from_numpy(b).to(dev).to(dtype)
    kw = dict(per_batch_values=False, dtypes=(dtype,), allow_i16=True, force_variant=7)
    vr, br = rounded(csr.values, dtype), rounded(b, dtype)
    want = oracle.spmm(br, csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)
    scale = oracle.spmm_abs_scale(br, csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)
    got = pyops._spmm(bt, ri, v, ro, ci, m, accumulate=False, **kw)
    assert "csr_to_dense_kernel" in _lib.last_kernels()
    assert_close(got.float().cpu().numpy(), want, scale, RTOL[dtype], "plain")
    got = pyops._spmm(bt, ri, v, ro, ci, m, accumulate=False, bias=torch.from_numpy(bias).to(dev), relu=True, **kw)
    assert_close(got.float().cpu().numpy(), np.maximum(want + bias[None, :, None], 0), scale + np.abs(bias)[None, :, None], RTOL[dtype], "bias, relu")
    prev = rounded(_normal(rng, batch, m, n), dtype)
    got = pyops._spmm(bt, ri, v, ro, ci, m, accumulate=True, out=torch.from_numpy(prev).to(dev).to(dtype), **kw)
    assert_close(got.float().cpu().numpy(), want + prev, scale + np.abs(prev), RTOL[dtype], "accumulate")
    # A^T * dense from the same arrays
    g = _normal(rng, m, n)
    gt = torch.from_numpy(g).to(dev).to(dtype)
    out = torch.full((k, n), float("nan"), dtype=dtype, device=dev)
    lib = _lib.load()
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=dev)
    _lib.check(lib.iex_spmm_transposed(CODE[dtype], 1 if idtype == torch.int16 else 0, m, k, n, csr.nnz, v.data_ptr(), ro.data_ptr(), ci.data_ptr(),
                                       gt.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream, ws.data_ptr(), ws.numel()))
    ro_t, ci_t, perm = oracle.csr_transpose(m, k, csr.row_offsets, csr.column_indices)
    args = (rounded(g, dtype)[None], W.swizzle_from_offsets(ro_t), vr[perm], ro_t, ci_t, k)
    assert_close(out.float().cpu().numpy(), oracle.spmm(*args)[0], oracle.spmm_abs_scale(*args)[0], RTOL[dtype], "transposed")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("m,n,k,batch", [(70, 45, 33, 1), (300, 129, 7, 2), (257, 1003, 264, 2), (129, 64, 521, 3)])
def test_sddmm_by_the_dense_product(oracle, dev, dtype, m, n, k, batch):
    rng = np.random.default_rng(m + k)
    csr, (ri, _, ro, ci) = _pattern(rng, m, n, dev, torch.int32, dtype)
    a, b = _normal(rng, batch, m, k), _normal(rng, batch, n, k)
    got = pyops._sddmm(torch.from_numpy(a).to(dev).to(dtype), torch.from_numpy(b).to(dev).to(dtype), ri, ro, ci, sum_over_batch=False, dtypes=(dtype,),
                       force_variant=7)
    assert "sample_dense_kernel" in _lib.last_kernels()
    ar, br = rounded(a, dtype), rounded(b, dtype)
    args = (csr.row_indices, csr.row_offsets, csr.column_indices)
    scale = np.stack([oracle.sddmm_abs_scale(ar[z:z + 1], br[z:z + 1], *args) for z in range(batch)])
    assert_close(got.float().cpu().numpy(), oracle.sddmm(ar, br, *args, sum_over_batch=False), scale, RTOL[dtype], "sampled")


@pytest.mark.parametrize("layout", [0, 1, 2])      # B (K,N), B (N,K), A (K,M)
@pytest.mark.parametrize("tile,mnk", [(0, (1000, 200, 4104)), (14, (72, 136, 1160)), (12, (264, 264, 104)), (13, (264, 264, 72)), (15, (136, 264, 72))])
def test_operands_that_end_where_their_memory_does(oracle, dev, layout, tile, mnk):
    """K with a tail, in parts and whole, on operands that are the last bytes of a memory block of their own."""
    if tile == 12 and layout == 2:
        pytest.skip("K in halves has no A as (K, M)")
    M, N, K = mnk
    rng = np.random.default_rng(M + K)
    a, b = _normal(rng, M, K), _normal(rng, K, N)

    def at_the_end(x):
        block = torch.full((12 << 20,), float("nan"), dtype=torch.bfloat16, device=dev)      # (24 MiB: a segment of its own)
        view = block[block.numel() - x.size:].view(x.shape)
        view.copy_(torch.from_numpy(np.ascontiguousarray(x)).bfloat16())
        return view

    at, bt = at_the_end(a.T if layout == 2 else a), at_the_end(b.T if layout == 1 else b)
    out = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device=dev)
    lib = _lib.load()
    code = layout | (tile << 4)
    need = lib.iex_gemm_workspace_bytes(_lib.BF16, code, M, N, K, 1)
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
    _lib.check(lib.iex_gemm_ws(_lib.BF16, code, M, N, K, at.data_ptr(), bt.data_ptr(), out.data_ptr(), 1, 0, 0, 0, torch.cuda.current_stream().cuda_stream,
                               ws.data_ptr(), need))
    assert ("parts" in _lib.last_kernels()) == (tile in (0, 14))
    ar, br = rounded(a, torch.bfloat16), rounded(b, torch.bfloat16)
    assert_close(out.float().cpu().numpy(), oracle.gemm(ar, br), np.abs(ar) @ np.abs(br), RTOL[torch.bfloat16], f"{mnk} tile {tile} layout {layout}")
