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
