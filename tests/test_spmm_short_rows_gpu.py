"""The row kernel with several nonzeros per gather: what is left of a share after whole windows, and rows short and many enough
for windows of four gathers."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib, workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("wpr", [1, 4])
@pytest.mark.parametrize("n", [8, 64, 128, 256])          # 8 (or 2) to 2 (or 1) nonzeros per gather
@pytest.mark.parametrize("m", [66, 4133])                 # few rows, and (four wavefronts on each) more than are resident
def test_shares_of_every_length(oracle, dev, dtype, wpr, n, m):
    rng = np.random.default_rng(n + m)
    k = 300
    lens = np.arange(m) % 66 if m > 66 else np.concatenate([np.arange(58), [63, 64, 65, 127, 128, 129, 255, 299]])   # one by one through a window
    lens = rng.permutation(lens)
    ro, ci = W.csr_from_row_lengths(rng, m, k, lens)
    csr = W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    b_np = rng.standard_normal((1, k, n)).astype(np.float32)
    ri, v, ro_t, ci_t = to_dev(csr, dev, dtype)
    b = torch.from_numpy(b_np).to(dev).to(dtype)
    out = pyops._spmm(b, ri, v, ro_t, ci_t, m, per_batch_values=False, accumulate=False, dtypes=(dtype,), allow_i16=False, force_variant=1, force_wpr=wpr)
    assert (", true>" in _lib.last_kernels()) == (m > 66 and wpr == 4 and (n < 256 or dtype != torch.float32)), _lib.last_kernels()
    b_r, v_r = rounded(b_np, dtype), rounded(csr.values, dtype)
    want = oracle.spmm(b_r, csr.row_indices, v_r, csr.row_offsets, csr.column_indices, m)
    scale = oracle.spmm_abs_scale(b_r, csr.row_indices, v_r, csr.row_offsets, csr.column_indices, m)
    # at most 300 roundings of a sum, each 2^-24 of the magnitudes; fp16: the result's rounding, 2^-11 of it or, below 2^-14, 2^-25
    half = dtype == torch.float16
    assert_close(out.float().cpu().numpy(), want, scale, 2.0 ** -11 if half else 0.0, f"{dtype} {m} x {n}, {wpr}",
                 atol=300 * 2.0 ** -24 * scale + (2.0 ** -25 if half else 0.0))
