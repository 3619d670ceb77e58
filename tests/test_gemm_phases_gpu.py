"""The GEMM tiles by two groups of wavefronts in alternating phases: every operand layout at the edges of their stages."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from _util import RTOL, assert_close, rounded

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


@pytest.mark.parametrize("tile", [5, 9, 13, 15, 16])
@pytest.mark.parametrize("M,N", [(255, 256), (257, 248), (193, 264), (1, 8), (256, 512)])
def test_stores_end_where_the_output_does(oracle, dev, tile, M, N):
    """Rows of whole vectors are stored without branches, by buffer stores that drop what lies outside: every entry of both batch
    entries is written and nothing around them."""
    rng = np.random.default_rng(M + N)
    a, b = (rng.standard_normal(s).astype(np.float32) for s in ((2, M, 72), (2, 72, N)))
    at, bt = (torch.from_numpy(x).to(dev).bfloat16() for x in (a, b))
    around = torch.full((4 * 256 * 512 + 2 * M * N,), 7.0, dtype=torch.bfloat16, device=dev)
    out = around[2 * 256 * 512:][:2 * M * N].view(2, M, N)
    out.fill_(float("nan"))
    lib = _lib.load()
    _lib.check(lib.iex_gemm(_lib.BF16, tile << 4, M, N, 72, at.data_ptr(), bt.data_ptr(), out.data_ptr(), 2, M * 72, 72 * N, M * N,
                            torch.cuda.current_stream().cuda_stream))
    for z in range(2):
        ar, br = rounded(a[z], torch.bfloat16), rounded(b[z], torch.bfloat16)
        assert_close(out[z].float().cpu().numpy(), oracle.gemm(ar, br), np.abs(ar) @ np.abs(br), RTOL[torch.bfloat16], f"{M} x {N} tile {tile}")
    rest = torch.cat([around[:2 * 256 * 512], around[2 * 256 * 512 + 2 * M * N:]])
    assert bool((rest == 7.0).all())
