"""Infinities and NaN in the attention kernels: what a query does not attend to leaves no trace in its row, what it attends
to shows as it does in the plain formula, entry by entry in float64."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.pytorch.sparse_attention import sparse_attention
from _util import rounded

pytestmark = pytest.mark.gpu
# (as in test_sparse_attention_kernel_gpu.py: rounding of probabilities and results; fp32 sums of up to 333 products)
TOL = {torch.float16: 2e-3, torch.bfloat16: 1e-2, torch.float32: 1e-5}
DTYPES = list(TOL)


def _rows(mask, q, k, v, scale):
    out = np.zeros_like(q)
    with np.errstate(all="ignore"):
        for i in range(mask.shape[0]):
            j = np.flatnonzero(mask[i])
            if j.size == 0:
                continue
            s = np.einsum("hd,hjd->hj", q[:, i], k[:, j]) * scale
            p = np.exp(s - s.max(axis=1, keepdims=True))
            p /= p.sum(axis=1, keepdims=True)
            out[:, i] = (p[:, :, None] * v[:, j]).sum(axis=1)
    return out


def _check(dev, mask, q, k, v, dtype, scale=None):
    ro, ci, _ = W.csr_from_mask(mask)
    t = lambda a: torch.from_numpy(a).to(dev)
    got = sparse_attention(*(t(x).to(dtype) for x in (q, k, v)), t(W.swizzle_from_offsets(ro)), t(ro), t(ci), scale).float().cpu().numpy()
    assert "sparse_attention_kernel" in _lib.last_kernels()
    want = _rows(mask, *(rounded(x, dtype).astype(np.float64) for x in (q, k, v)), scale or 1.0 / np.sqrt(q.shape[2]))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    endless = np.isinf(want)
    assert np.array_equal(np.isinf(got), endless) and np.array_equal(got[endless], want[endless])
    rest = np.isfinite(want)
    assert np.linalg.norm(got[rest] - want[rest]) <= TOL[dtype] * np.linalg.norm(want[rest])
    return want


def _mask(tokens, band, extra, rng):
    """A causal band and scattered entries: tiles on the matrix cores, and lists."""
    away = np.arange(tokens)[:, None] - np.arange(tokens)[None, :]
    mask = (away >= 0) & (away < band)
    if extra:
        np.put_along_axis(mask, rng.integers(0, tokens, (tokens, extra)), True, axis=1)
    return mask


# (heads: wavefronts that share queries, and four wavefronts of queries per workgroup)
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads, d, band, extra", [(2, 64, 64, 0), (2, 32, 50, 9), (1, 128, 70, 5), (110, 64, 64, 3), (110, 32, 64, 0), (110, 128, 40, 2), (3, 64, 1, 11)])
def test_values_of_other_tokens_do_not_leak(dev, dtype, heads, d, band, extra):
    tokens, rng = 333, np.random.default_rng(d + band)
    mask = _mask(tokens, band, extra, rng)
    mask[:, [0, 70, 71, 200]] = False           # nobody looks at them ...
    mask[[2, 90, 210, 332], [0, 70, 71, 200]] = True     # ... but one row each
    mask[150] = False
    q, k, v = (rng.standard_normal((heads, tokens, d)).astype(np.float32) for _ in range(3))
    v[:, 0], v[:, 70], v[:, 71, ::2] = -np.inf, np.inf, np.nan
    k[:, 200], v[:, 200] = np.nan, np.nan
    want = _check(dev, mask, q, k, v, dtype)
    assert np.isfinite(want[:, [1, 3, 89, 91, 209, 331]]).all() and not want[:, 150].any()
    assert np.isinf(want[:, [2, 90]]).all() and np.isnan(want[:, [210], ::2]).all() and np.isnan(want[:, 332]).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("heads, extra", [(2, 0), (110, 4)])
def test_scores_below_any_mark(dev, dtype, heads, extra):
    """Every score of half the rows lies far below -1e30; scaled they are ordinary."""
    tokens, d, rng = 200, 64, np.random.default_rng(3)
    mask = _mask(tokens, 64, extra, rng)
    q, k, v = (rng.standard_normal((heads, tokens, d)).astype(np.float32) for _ in range(3))
    q, k = np.abs(q) * np.float32(1e16), np.abs(k) * np.float32(1e16)
    q[:, ::2] *= -1
    _check(dev, mask, q, k, v, dtype, scale=1e-33)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("heads, extra", [(2, 0), (2, 6), (110, 3)])
def test_infinite_scores(dev, dtype, heads, extra):
    tokens, d, rng = 200, 64, np.random.default_rng(4)
    mask = _mask(tokens, 64, extra, rng)
    mask[:, [100, 101]] = False
    mask[10], mask[11], mask[12] = False, False, False
    mask[10, 100], mask[11, [3, 100]], mask[12, [3, 101]] = True, True, True
    q, k, v = (rng.standard_normal((heads, tokens, d)).astype(np.float32) for _ in range(3))
    q = np.abs(q) + np.float32(0.1)
    k[:, 100], k[:, 101] = -np.inf, np.inf
    want = _check(dev, mask, q, k, v, dtype)
    assert np.isnan(want[:, [10, 12]]).all() and np.isfinite(want[:, 11]).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("d, length", [(64, 8), (128, 72), (64, 136), (128, 200), (64, 64)])
def test_dense_attention_with_infinite_values(dev, dtype, d, length):
    """Infinities in v show as infinities in their sequence, head and feature, also at the last keys of a length off the tile."""
    from intrasm_engine_amd import _iex_host
    heads, seqs, g = 2, 2, torch.Generator(dev).manual_seed(length)
    q, k, v = (torch.randn(heads * d, seqs * length, device=dev, generator=g).to(dtype) for _ in range(3))
    v[3, length - 1], v[d + 5, length - 8], v[7, 2 * length - 1] = np.inf, -np.inf, np.nan
    scale = d ** -0.5
    out = _iex_host.attention(q, k, v, heads, seqs, scale)
    assert "attention_kernel" in _lib.last_kernels()
    split = lambda t: t.double().cpu().view(heads, d, seqs, length).permute(2, 0, 3, 1)
    Q, K, V = split(q), split(k), split(v)
    p = torch.softmax(torch.matmul(Q, K.transpose(-1, -2).contiguous()) * scale, dim=-1)
    want = (p[..., None] * V[:, :, None]).sum(dim=3).permute(1, 3, 0, 2).reshape(heads * d, seqs * length).numpy()
    got = out.float().cpu().numpy()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any()
    endless = np.isinf(want)
    assert np.array_equal(np.isinf(got), endless) and np.array_equal(got[endless], want[endless]) and endless.any()
    rest = np.isfinite(want)
    assert np.linalg.norm(got[rest] - want[rest]) <= TOL[dtype] * np.linalg.norm(want[rest])
