"""The GEMM tiles by two groups of wavefronts in alternating phases: every operand layout at the edges of their stages."""
import numpy as np
import pytest
import torch

from _util import assert_close, rounded

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("layout", [0, 1, 2])   # B as (K, N), B as (N, K), A as (K, M)
@pytest.mark.parametrize("tile", [13, 15, 16])  # 256 x 256 in phases of 32 k, 128 x 256 in phases of 64, 192 x 256 in phases of 32
@pytest.mark.parametrize("mnk", [(8, 8, 8), (128, 256, 64), (136, 264, 72), (256, 256, 96), (264, 520, 192), (72, 1000, 1032)])
def test_layouts_at_the_edges_of_the_stages(oracle, dev, dtype, layout, tile, mnk):
    """One, two, three phases and more, the last one whole or with 8 k; tiles of which one row of chunks exists."""
    from intrasm_engine_amd import _lib
    M, N, K = mnk
    if tile == 16 and layout == 2:
        pytest.skip("a (K, M) operand has no rows of 192")
    rng = np.random.default_rng(M + K)
    a_np, b_np = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    a, b = torch.from_numpy(a_np).to(dev).to(dtype), torch.from_numpy(b_np).to(dev).to(dtype)
    a, b = a.t().contiguous() if layout == 2 else a, b.t().contiguous() if layout == 1 else b
    out = torch.full((M, N), float("nan"), device=dev, dtype=dtype)
    rc = _lib.load().iex_gemm(_lib.BF16 if dtype == torch.bfloat16 else _lib.F16, layout | (tile << 4), M, N, K, a.data_ptr(), b.data_ptr(), out.data_ptr(),
                              1, 0, 0, 0, torch.cuda.current_stream().cuda_stream)
    assert rc == 0, _lib.last_error()
    a_r, b_r = rounded(a_np, dtype), rounded(b_np, dtype)
    assert_close(out.float().cpu().numpy(), oracle.gemm(a_r, b_r), oracle.gemm(np.abs(a_r), np.abs(b_r)), 1e-2, f"tile {tile} layout {layout} {mnk}")
