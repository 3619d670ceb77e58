"""The few-columns SpMM kernel where its last column tile changes kind: vectors that are left, single columns beyond them."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib, workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("k", [64, 65])    # two vectors per lane; one
@pytest.mark.parametrize("extra", [0, 1, 63, 64, 65, 255, 256, 257, 320, 321])   # columns beyond one vector per lane (fp32; fp16: twice as many)
def test_last_column_tile(oracle, dev, dtype, k, extra):
    vec = 4 if dtype == torch.float32 else 8
    n = 64 * vec + (extra if vec == 4 else 2 * extra - (extra == 63))
    rng = np.random.default_rng(n)
    m = 75
    mask = rng.random((m, k)) < 0.15
    mask[3] = False
    mask[4] = True                 # more than eight nonzeros, rows that end anywhere in a step of eight
    ro, ci, _ = W.csr_from_mask(mask)
    ri = W.swizzle_from_offsets(ro)
    values = rng.standard_normal((2, ci.shape[0])).astype(np.float32)
    b = rng.standard_normal((2, k, n)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    with pyops.kernel_params(spmm={"force_variant": 8}):
        out = ops.spmm_sputnik_batched_values(t(b).to(dtype), t(ri), t(values).to(dtype), t(ro), t(ci), m)
    assert "spmm_smallk_kernel" in _lib.last_kernels()
    for z in range(2):
        args = rounded(b[z:z + 1], dtype), ri, rounded(values[z], dtype), ro, ci, m
        assert_close(out[z].float().cpu().numpy(), oracle.spmm(*args)[0], oracle.spmm_abs_scale(*args)[0], 1e-5 if vec == 4 else 1e-2, f"n={n} k={k}")
