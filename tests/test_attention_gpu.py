"""Dense attention on feature-major operands and the products with an auxiliary operand, against float64."""
import numpy as np
import pytest
import torch

import intrasm_engine_amd  # noqa: F401
from intrasm_engine_amd import _iex_host, _lib
from intrasm_engine_amd import workloads as W
from _util import RTOL, assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,d,seqs,length", [(2, 64, 1, 8), (3, 128, 2, 64), (2, 128, 3, 72), (1, 64, 2, 136), (2, 128, 1, 200), (8, 64, 2, 512)])
def test_attention(dev, dtype, heads, d, seqs, length):
    g = torch.Generator(dev).manual_seed(length)
    q, k, v = (torch.randn(heads * d, seqs * length, device=dev, generator=g).to(dtype) for _ in range(3))
    q = q * 2          # (scores of some spread: the running maximum moves)
    scale = d ** -0.5
    out = _iex_host.attention(q, k, v, heads, seqs, scale)
    assert "attention_kernel" in _lib.last_kernels() and out.shape == q.shape
    split = lambda t: t.double().cpu().view(heads, d, seqs, length).permute(2, 0, 3, 1)
    Q, K, V = split(q), split(k), split(v)
    p = torch.softmax(torch.matmul(Q, K.transpose(-1, -2).contiguous()) * scale, dim=-1)
    want = torch.matmul(p, V.contiguous()).permute(1, 3, 0, 2).reshape(heads * d, seqs * length)
    bound = torch.matmul(p, V.abs().contiguous()).permute(1, 3, 0, 2).reshape(heads * d, seqs * length)
    assert_close(out.float().cpu().numpy(), want.numpy(), bound.numpy() * 10, RTOL[dtype], "attention")


def test_attention_steps_aside(dev):
    x = torch.randn(3 * 32, 16, device=dev).half()
    assert _iex_host.attention(x, x, x, 3, 1, 0.1) is None          # heads of 32
    x = torch.randn(64, 12, device=dev).half()
    assert _iex_host.attention(x, x, x, 1, 1, 0.1) is None          # 12 tokens


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,k,n,dense", [(96, 64, 33, False), (640, 512, 200, True), (1000, 1024, 520, True), (513, 640, 264, True)])
def test_product_with_an_auxiliary_operand(oracle, dev, dtype, m, k, n, dense):
    rng = np.random.default_rng(m)
    ro, ci = W.csr_from_row_lengths(rng, m, k, np.full(m, k // 2 if dense else 5))
    csr = W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32) * 0.1, W.swizzle_from_offsets(ro), ro, ci)
    ri, v, ro, ci = to_dev(csr, dev, dtype)
    x, aux = rng.standard_normal((k, n)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    xr, ar, vr = rounded(x, dtype), rounded(aux, dtype).astype(np.float64), rounded(csr.values, dtype)
    base = oracle.spmm(xr[None], csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)[0]
    scale = oracle.spmm_abs_scale(xr[None], csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)[0]
    silu = ar / (1 + np.exp(-ar))
    xt, at = torch.from_numpy(x).to(dev).to(dtype), torch.from_numpy(aux).to(dev).to(dtype)
    for mode, want, bound in ((1, base + ar, scale + np.abs(ar)), (2, base * silu, scale * np.abs(silu) + 1e-3)):
        got = _iex_host.spmm_with(xt, ri, v, ro, ci, m, at, mode)
        assert ("combine_kernel" in _lib.last_kernels()) != ("csr_to_dense_kernel" in _lib.last_kernels())
        # (without an epilogue of its own the product is rounded before it is combined: twice the type's half step)
        assert_close(got.float().cpu().numpy(), want, 5 * bound, RTOL[dtype], f"mode {mode}")


@pytest.mark.parametrize("offset", [1, 2, 4])
def test_auxiliary_operand_at_any_alignment(dev, offset):
    """The other operand as a slice that starts 2, 4 or 8 bytes past an aligned address: the same bits as from a copy of it."""
    m, k, n = 640, 512, 264
    ro, ci = W.csr_from_row_lengths(np.random.default_rng(1), m, k, np.full(m, k // 2))
    csr = W.CSR(m, k, np.random.default_rng(2).standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    ri, v, ro, ci = to_dev(csr, dev, torch.float16)
    x = torch.randn(k, n, device=dev).half()
    flat = torch.randn(m * n + 8, device=dev).half()
    aux = flat[offset:offset + m * n].view(m, n)
    assert aux.data_ptr() % 16 == 2 * offset
    for mode in (1, 2):
        got = _iex_host.spmm_with(x, ri, v, ro, ci, m, aux, mode)
        assert "csr_to_dense_kernel" in _lib.last_kernels()
        assert torch.equal(got, _iex_host.spmm_with(x, ri, v, ro, ci, m, aux.clone(), mode))
