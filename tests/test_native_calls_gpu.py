"""The operators' native calls: the small kernels behind them, and when they step aside for the Python functions."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import to_dev

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("n", [1, 3, 4, 1023, 1025, 4096])
def test_gather_values(dev, dtype, n):
    values = torch.randn(n, device=dev).to(dtype)
    index = torch.randperm(n, device=dev)
    out = torch.empty_like(values)
    _lib.check(_lib.load().iex_gather_values(values.element_size(), n, values.data_ptr(), index.data_ptr(), out.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, values[index])


def test_long_inner_dimension_keeps_the_dense_product(dev):
    """A pruned weight of attention's size that has been looked at: no structure, so not the kernel for masks with
    structure, and a long k is still sampled from a dense product."""
    m, n, k = 8192, 4096, 1024
    ro, ci = W.csr_from_row_lengths(np.random.default_rng(1), m, n, np.full(m, n // 10))
    ri, _, ro, ci = to_dev(W.CSR(m, n, np.ones(ci.shape[0], np.float32), W.swizzle_from_offsets(ro), ro, ci), dev)
    assert pyops.prepare_pattern(ro, ci, n) == 0 and pyops._known_dense_share(ro, ci, n) < 0.5
    a, b = torch.randn(1, m, k, device=dev).half(), torch.randn(1, n, k, device=dev).half()
    out = ops.sddmm_sputnik_half(a, b, ri, ro, ci)
    assert "sample_dense_kernel" in _lib.last_kernels()
    assert torch.equal(out, pyops.sddmm_sputnik_half(a, b, ri, ro, ci))


def test_notes_follow_the_tensors(dev):
    """What is known about a pattern holds for its two index tensors as they are: in-place changes and other pairings are
    looked at again, and forced kernels reach the operators."""
    a = W.config2_matrix(0.9, m=256, k=256)
    ri, v, ro, ci = to_dev(a, dev)
    b = torch.randn(1, 256, 64, device=dev)
    want = ops.spmm_sputnik_reuse_weight(b, ri, v, ro, ci, 256)
    assert torch.equal(ops.spmm_sputnik_reuse_weight(b, ri, v, ro.clone(), ci, 256), want)
    with pyops.kernel_params(spmm={"force_variant": 1, "force_wpr": 1}):
        ops.spmm_sputnik_reuse_weight(b, ri, v, ro, ci, 256)
        assert "spmm_kernel" in _lib.last_kernels()
    start, end = int(ro[5]), int(ro[6])
    ci[start:end] = ci[start:end].flip(0)       # no longer ascending: same product, other kernels
    v[start:end] = v[start:end].flip(0)
    got = ops.spmm_sputnik_reuse_weight(b, ri, v, ro, ci, 256)
    assert torch.allclose(got, want, rtol=1e-5, atol=1e-6) and pyops._csr_status(ro, ci, 256) == _lib.CSR_NOT_ASCENDING
    ci[start] = 256
    with pytest.raises(RuntimeError, match="every column index must lie in"):
        ops.spmm_sputnik_reuse_weight(b, ri, v, ro, ci, 256)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_gather_values_outside_the_values_is_nan(dev, dtype):
    n = 1027
    values = torch.randn(n, device=dev).to(dtype)
    index = torch.randperm(n, device=dev)
    wrong = [0, 513, 1023, 1024, n - 1]
    index[wrong] = torch.tensor([n, -1, 1 << 40, -(1 << 62), n + 5], device=dev)
    out = torch.zeros_like(values)
    _lib.check(_lib.load().iex_gather_values(values.element_size(), n, values.data_ptr(), index.data_ptr(), out.data_ptr(),
                                             torch.cuda.current_stream().cuda_stream))
    good = torch.ones(n, dtype=torch.bool, device=dev)
    good[wrong] = False
    assert out[wrong].isnan().all() and torch.equal(out[good], values[index[good]])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_training_step_with_a_permutation_that_is_a_slice(dev, dtype):
    """The permutation of the transpose as part of a larger tensor: 8-byte aligned only."""
    from intrasm_engine_amd.pytorch.cpp_extensions.layers_and_funcs.sputnik import spmm
    from intrasm_engine_amd.pytorch.utils import transpose_info
    a = W.config2_matrix(0.9, m=300, k=200)
    ri, v, ro, ci = to_dev(a, dev, dtype)
    info = transpose_info(300, 200, ro, ci)
    larger = torch.cat([torch.zeros(1, dtype=torch.int64, device=dev), info[3]])
    b, grad = torch.randn(200, 17, device=dev).to(dtype), torch.randn(300, 17, device=dev).to(dtype)
    got = []
    for perm in (info[3], larger[1:]):
        b.requires_grad_(), v.requires_grad_()
        out = spmm(b, ri, v, ro, ci, 300, (*info[:3], perm))
        got.append(torch.autograd.grad(out, (b, v), grad))
    assert larger[1:].data_ptr() % 16 == 8
    assert all(torch.equal(x, y) for x, y in zip(*got))
