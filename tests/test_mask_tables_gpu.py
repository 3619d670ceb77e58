"""What is derived from a pattern and kept with it, against everything that can come between: a capture, a change in
place, another stream, another thread."""
import threading

import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from intrasm_engine_amd.pytorch.cpp_extensions.cuda_graph_constructor import TorchCUDAGraphConstructor
from intrasm_engine_amd.pytorch.sparse_attention import sparse_attention
from _util import to_dev

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops


def _arrays(tokens, band, dev, shift=0):
    """A band and a scattered entry per row; the same number of entries per row whatever the shift."""
    i = np.arange(tokens)
    mask = (i[None, :] - i[:, None]) % tokens < band
    mask[i, (i + band + 7 + shift) % tokens] = True
    ro, ci, _ = W.csr_from_mask(mask)
    t = lambda a: torch.from_numpy(a).to(dev)
    return t(W.swizzle_from_offsets(ro)), t(ro), t(ci)


def _operands(dev, heads, tokens, d, dtype, seed=0):
    g = torch.Generator(dev).manual_seed(seed)
    return tuple(torch.randn(heads, tokens, d, device=dev, generator=g).to(dtype) for _ in range(3))


def _captured(fn):
    constructor = TorchCUDAGraphConstructor()
    with constructor.get_primary_stream():
        with constructor:
            out = fn()
    constructor.instantiate_graph_exec()
    return constructor, out


def _clutter(dev, nbytes):
    """Memory of that size, handed out before, overwritten (zeros: tables of an empty mask)."""
    return [torch.zeros(nbytes, dtype=torch.uint8, device=dev) for _ in range(4)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
def test_replays_work_on_the_mask_as_it_was_captured(dev, dtype):
    """... whatever becomes of its arrays, and of the tables that later calls replace."""
    tokens = 520
    ri, ro, ci = _arrays(tokens, 70, dev)
    first = _arrays(tokens, 70, dev)
    q, k, v = _operands(dev, 3, tokens, 64, dtype)
    sparse_attention(q, k, v, ri, ro, ci)
    constructor, out = _captured(lambda: sparse_attention(q, k, v, ri, ro, ci))
    assert "sparse_attention_kernel" in _lib.last_kernels()
    nbytes = _lib.load().iex_mask_tables_bytes(tokens, tokens, ci.numel())
    for it in range(5):
        if it:
            ci.copy_(_arrays(tokens, 70, dev, shift=11 * it)[2])
            for x, new in zip((q, k, v), _operands(dev, 3, tokens, 64, dtype, seed=it)):
                x.copy_(new)
        if it == 4:
            ro.zero_()
        if it in (1, 3):                        # (2, 4: changed, and only replayed)
            other = sparse_attention(q, k, v, ri, ro, ci)
            assert torch.equal(other, sparse_attention(q, k, v, *_arrays(tokens, 70, dev, shift=11 * it)))
        keep = _clutter(dev, nbytes)
        torch.cuda.synchronize()
        constructor.execute_graph()
        constructor.synchronize()
        assert torch.equal(out, sparse_attention(q, k, v, *first)), it
        assert "sparse_attention_kernel" in _lib.last_kernels() and not any(x.any() for x in keep)
    constructor.destroy_graph_exec()


@pytest.mark.parametrize("heads, tokens, band, dtype", [(3, 520, 70, torch.float16), (3, 520, 70, torch.float32), (8, 2048, 300, torch.float16)])
def test_replays_follow_a_mask_that_nobody_may_look_at(dev, heads, tokens, band, dtype):
    """(2048: the kernels for masks with structure, with tables written at every replay)"""
    ri, ro, ci = _arrays(tokens, band, dev)
    pyops.mark_canonical(ro, ci, tokens, measure=False)
    q, k, v = _operands(dev, heads, tokens, 64, dtype)
    constructor, out = _captured(lambda: sparse_attention(q, k, v, ri, ro, ci))
    for it in range(4):
        if it:
            ci.copy_(_arrays(tokens, band, dev, shift=11 * it)[2])
        torch.cuda.synchronize()
        constructor.execute_graph()
        constructor.synchronize()
        want = sparse_attention(q, k, v, *_arrays(tokens, band, dev, shift=11 * it))
        assert torch.allclose(out.float(), want.float(), atol=1e-2 if dtype == torch.float16 else 1e-4), it
    constructor.destroy_graph_exec()


def test_a_capture_that_comes_first_settles_calls_like_it_only(dev):
    tokens = 300
    ri, ro, ci = _arrays(tokens, 40, dev)
    pyops.prepare_pattern(ro, ci, tokens)
    q, k, v = _operands(dev, 2, tokens, 64, torch.float16)
    constructor, out = _captured(lambda: sparse_attention(q, k, v, ri, ro, ci))
    assert "sparse_attention_kernel" not in _lib.last_kernels()
    constructor.execute_graph()
    constructor.synchronize()
    for _ in range(2):
        assert torch.equal(out, sparse_attention(q, k, v, ri, ro, ci)) and "sparse_attention_kernel" not in _lib.last_kernels()
    constructor.destroy_graph_exec()
    for dtype, d in ((torch.float32, 64), (torch.bfloat16, 64), (torch.float16, 32)):
        sparse_attention(*_operands(dev, 2, tokens, d, dtype), ri, ro, ci)
        assert "sparse_attention_kernel" in _lib.last_kernels(), (dtype, d)
    sparse_attention(q, k, v, ri, ro, ci)
    assert "sparse_attention_kernel" not in _lib.last_kernels()
    assert pyops.prepare_mask(q, ro, ci)
    got = sparse_attention(q, k, v, ri, ro, ci)
    assert "sparse_attention_kernel" in _lib.last_kernels() and torch.allclose(got.float(), out.float(), atol=1e-2)


def test_no_tables_for_calls_that_do_not_use_them(dev):
    tokens = 200
    ri, ro, ci = _arrays(tokens, 30, dev)
    q, k, v = _operands(dev, 2, tokens, 64, torch.float16)
    want = sparse_attention(q, k, v, *_arrays(tokens, 30, dev))
    flat = torch.empty(q.numel() + 1, dtype=q.dtype, device=dev)
    off = flat[1:].view_as(q)                   # not 16-byte aligned
    off.copy_(q)
    for call in (lambda: sparse_attention(off, k, v, ri, ro, ci), lambda: sparse_attention(q.clone().requires_grad_(), k, v, ri, ro, ci),
                 lambda: sparse_attention(q, k, v, ri, ro, ci, return_probs=True)[0]):
        assert torch.allclose(call().detach().float(), want.float(), atol=1e-2)
        assert "_iex_mask_tables" not in ci.__dict__


def test_tables_outlive_their_mask_on_another_stream(dev):
    """The mask's tensor goes while a call on another stream has not run yet: its tables' memory is not handed out before."""
    tokens = 1024
    ri, ro, ci = _arrays(tokens, 90, dev)
    q, k, v = _operands(dev, 4, tokens, 64, torch.float16)
    want = sparse_attention(q, k, v, ri, ro, ci)
    nbytes = _lib.load().iex_mask_tables_bytes(tokens, tokens, ci.numel())
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)
        out = sparse_attention(q, k, v, ri, ro, ci)
    assert "sparse_attention_kernel" in _lib.last_kernels()
    del ci
    keep = _clutter(dev, nbytes)
    torch.cuda.synchronize()
    assert torch.equal(out, want) and len(keep) == 4


def test_a_captured_product_keeps_the_tables_it_reads(dev):
    """A product of a mask with structure, captured: the tables of the pattern that it reads survive later calls' new ones."""
    pattern, q_np, *_ = W.config3(tokens=2048, heads=8, band=128, extra=8)
    ri, _, ro, ci = to_dev(pattern, dev)
    q, k, _ = _operands(dev, 8, 2048, 64, torch.float16)
    want = ops.sddmm_sputnik_half(q, k, ri, ro, ci)
    assert "sddmm_mfma_kernel" in _lib.last_kernels()
    constructor, out = _captured(lambda: ops.sddmm_sputnik_half(q, k, ri, ro, ci))
    before = ci.__dict__["_iex_csr"][7]
    nbytes = before.numel()
    assert any(t is before for t in ci.__dict__["_iex_recorded"])
    del before
    ci.add_(0)                                  # (another version: looked at again, with tables of its own)
    assert torch.equal(ops.sddmm_sputnik_half(q, k, ri, ro, ci), want)
    assert not any(t is ci.__dict__["_iex_csr"][7] for t in ci.__dict__["_iex_recorded"])
    for _ in range(3):
        keep = _clutter(dev, nbytes)
        out.zero_()
        torch.cuda.synchronize()
        constructor.execute_graph()
        constructor.synchronize()
        assert torch.equal(out, want) and not any(x.any() for x in keep)
    constructor.destroy_graph_exec()


def test_operators_from_several_threads_and_streams(dev):
    a = W.config2_matrix(0.9, m=512, k=512)
    ri, values, ro, ci = to_dev(a, dev)
    b = torch.randn(1, 512, 64, device=dev)
    mri, mro, mci = _arrays(600, 50, dev)       # (nobody has looked at this one: several threads do at once)
    q, k, v = _operands(dev, 2, 600, 64, torch.float16)
    want = ops.spmm_sputnik_reuse_weight(b, ri, values, ro, ci, 512), sparse_attention(q, k, v, *_arrays(600, 50, dev))
    torch.cuda.synchronize()
    wrong = []

    def work():
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for _ in range(20):
                got = ops.spmm_sputnik_reuse_weight(b, ri, values, ro, ci, 512), sparse_attention(q, k, v, mri, mro, mci)
                stream.synchronize()
                if not all(torch.equal(x, y) for x, y in zip(got, want)):
                    wrong.append(got)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
