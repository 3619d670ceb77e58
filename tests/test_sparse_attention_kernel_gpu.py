"""Sparse attention in one kernel: against dense masked attention in float64, at the edges of its tiles and lists."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.pytorch.sparse_attention import sparse_attention
from _util import rounded

pytestmark = pytest.mark.gpu


def _mask(tokens, band, extra, rng):
    i = np.arange(tokens)
    mask = np.abs(i[:, None] - i[None, :]) < band
    if extra:
        np.put_along_axis(mask, rng.integers(0, tokens, (tokens, extra)), True, axis=1)
    return mask


def _reference(mask, q, k, v):
    s = np.where(mask[None], np.einsum("htd,hsd->hts", q, k) / np.sqrt(q.shape[2]), -np.inf)
    top = s.max(axis=-1, keepdims=True)
    p = np.where(mask[None], np.exp(s - np.where(np.isfinite(top), top, 0.0)), 0.0)
    total = p.sum(axis=-1, keepdims=True)
    return np.divide(p, total, out=np.zeros_like(p), where=total > 0) @ v


@pytest.mark.parametrize("dtype, tol", [(torch.float16, 2e-3), (torch.bfloat16, 1e-2), (torch.float32, 1e-5)])
@pytest.mark.parametrize("heads, tokens, d, band, extra", [
    (1, 1, 64, 1, 0),            # one query, one key
    (2, 129, 32, 40, 0),         # a row past a block of rows, keys past a tile
    (3, 200, 128, 1, 3),         # no dense tile: lists only, shorter than a step of them
    (2, 333, 64, 30, 21),        # both, lists over several steps
    (40, 513, 32, 64, 9),        # four wavefronts of queries per workgroup
    (170, 130, 128, 64, 0)])
def test_against_dense_masked_attention(dev, dtype, tol, heads, tokens, d, band, extra):
    rng = np.random.default_rng(tokens)
    mask = _mask(tokens, band, extra, rng)
    if tokens > 100:
        mask[[0, 63, tokens - 1]] = False          # rows without entries
        mask[64:70, :] = True                      # rows that are full
    ro, ci, _ = W.csr_from_mask(mask)
    ri = W.swizzle_from_offsets(ro)
    q, k, v = (rng.standard_normal((heads, tokens, d)).astype(np.float32) for _ in range(3))
    k[:, tokens // 2] *= 20                        # a key that takes over late
    t = lambda a: torch.from_numpy(a).to(dev)
    ri, ro, ci = t(ri), t(ro), t(ci)
    operands = [t(x).to(dtype) for x in (q, k, v)]
    out = sparse_attention(*operands, ri, ro, ci)
    assert "sparse_attention_kernel" in _lib.last_kernels()
    want = _reference(mask, *(rounded(x, dtype).astype(np.float64) for x in (q, k, v)))
    got = out.float().cpu().numpy()
    assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
    assert not got[:, ~mask.any(axis=1)].any()
    assert torch.equal(out, sparse_attention(*operands, ri, ro, ci))


@pytest.mark.parametrize("dtype, tol", [(torch.bfloat16, 1e-2), (torch.float32, 1e-5)])
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("tokens, group, corner", [(31, 0, 3), (160, 1, 80), (161, 4, 230), (420, 12, 300)])
def test_lists_beside_tiles_that_few_rows_have(dev, dtype, tol, d, tokens, group, corner):
    """Few heads (the entries outside dense tiles go to wavefronts of their own): rows with lists and tiles of which one group of 32 rows has entries, on either
    side of the number that makes a tile dense, the last block of rows among them."""
    rng = np.random.default_rng(tokens + d)
    mask = _mask(tokens, 1, 5, rng)
    first = min(group * 32, tokens - 1)
    block = mask[first:first + 32, :64]
    block.flat[rng.permutation(block.size)[:corner]] = True
    ro, ci, _ = W.csr_from_mask(mask)
    t = lambda a: torch.from_numpy(a).to(dev)
    ri, ro, ci = t(W.swizzle_from_offsets(ro)), t(ro), t(ci)
    q, k, v = (rng.standard_normal((3, tokens, d)).astype(np.float32) for _ in range(3))
    out = sparse_attention(*(t(x).to(dtype) for x in (q, k, v)), ri, ro, ci)
    assert "sparse_attention_kernel" in _lib.last_kernels() and ", 1, " in _lib.last_kernels()
    want = _reference(mask, *(rounded(x, dtype).astype(np.float64) for x in (q, k, v)))
    assert np.linalg.norm(out.float().cpu().numpy() - want) <= tol * np.linalg.norm(want)


@pytest.mark.parametrize("dtype, tol", [(torch.float16, 2e-3), (torch.float32, 1e-5)])
def test_tiles_that_a_launch_takes_one_way_or_the_other(dev, dtype, tol):
    """About 245 entries a tile, between the two limits of 16-bit tables: one mask, launches of either kind and heads of all sizes; an infinity stays with the rows
    that attend to it."""
    rng = np.random.default_rng(11)
    tokens = 533
    mask = _mask(tokens, 8, 16, rng)
    mask[100:130] = _mask(tokens, 8, 0, rng)[100:130]     # rows without scattered entries among them
    ro, ci, _ = W.csr_from_mask(mask)
    t = lambda a: torch.from_numpy(a).to(dev)
    ri, ro, ci = t(W.swizzle_from_offsets(ro)), t(ro), t(ci)
    for heads, d, wide in ((64, 128, True), (2, 128, False), (64, 64, True), (2, 64, False), (2, 32, False)):
        q, k, v = (rng.standard_normal((2, tokens, d)).astype(np.float32) for _ in range(3))
        operands = [t(x).to(dtype).repeat(heads // 2, 1, 1) for x in (q, k, v)]
        out = sparse_attention(*operands, ri, ro, ci)
        assert f", {d}, {4 if wide else 1}, " in _lib.last_kernels(), _lib.last_kernels()
        want = _reference(mask, *(rounded(x, dtype).astype(np.float64) for x in (q, k, v)))
        assert np.linalg.norm(out[-2:].float().cpu().numpy() - want) <= tol * np.linalg.norm(want)
        assert torch.equal(out[:2], out[-2:])
        operands[2][:, 300, 3] = float("inf")
        odd = sparse_attention(*operands, ri, ro, ci)
        assert torch.equal(odd[-1].isfinite().all(dim=1), t(~mask[:, 300]))
        rest = ~mask[:, 300]
        assert np.linalg.norm(odd[-1].float().cpu().numpy()[rest] - want[-1][rest]) <= tol * np.linalg.norm(want[-1][rest])


def test_tables_follow_the_mask(dev):
    """A mask changed in place is looked at again; one that nobody may look at, and columns in another order, go by three kernels."""
    from intrasm_engine_amd.pytorch import ops as pyops
    rng = np.random.default_rng(5)
    mask = _mask(200, 20, 2, rng)
    t = lambda a: torch.from_numpy(a).to(dev)
    ro, ci, _ = (t(x) if x is not None else x for x in W.csr_from_mask(mask))
    ri = t(W.swizzle_from_offsets(ro.cpu().numpy()))
    q, k, v = (torch.randn(2, 200, 64, device=dev) for _ in range(3))
    before = sparse_attention(q, k, v, ri, ro, ci)
    shifted = (ci + 1) % 200
    order = torch.argsort(torch.repeat_interleave(torch.arange(200, device=dev), (ro[1:] - ro[:-1]).long()) * 200 + shifted)
    ci.copy_(shifted[order])
    after = sparse_attention(q, k, v, ri, ro, ci)
    assert "sparse_attention_kernel" in _lib.last_kernels() and not torch.allclose(before, after, atol=1e-3)
    rolled = sparse_attention(q, k.roll(-1, 1).contiguous(), v.roll(-1, 1).contiguous(), ri, ro, t(W.csr_from_mask(mask)[1]))
    assert torch.allclose(after, rolled, atol=1e-4)
    unmeasured = ci.clone()
    pyops.mark_canonical(ro, unmeasured, 200, measure=False)
    assert torch.allclose(sparse_attention(q, k, v, ri, ro, unmeasured), after, atol=1e-4)
    assert "sparse_attention_kernel" not in _lib.last_kernels()
    first = ci[ro[:-1].long()].clone()
    backwards = ci.clone()
    backwards[ro[:-1].long()], backwards[ro[:-1].long() + 1] = ci[ro[:-1].long() + 1], first
    assert torch.allclose(sparse_attention(q, k, v, ri, ro, backwards), after, atol=1e-4)
    assert "sparse_attention_kernel" not in _lib.last_kernels()
