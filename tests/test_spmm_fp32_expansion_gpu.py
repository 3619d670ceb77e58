"""The fp32 matrix-core SpMM's expansion: a chunk of 128 columns takes what a row has in it, however it lies against the
windows of 64 nonzeros that a wavefront holds."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib, workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from _util import assert_close, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arrangement", [4, 6])           # tiles of 32 and of 16 rows
@pytest.mark.parametrize("m,k", [(33, 8), (16, 127), (40, 128), (17, 129), (70, 1000)])
@pytest.mark.parametrize("filler", [0.02, 0.6])           # one window per row; rows dense enough for two
def test_runs_at_the_edges_of_the_windows(oracle, dev, arrangement, m, k, filler):
    rng = np.random.default_rng(m + k)
    mask = rng.random((m, k)) < filler
    for r, run in enumerate((0, 1, 63, 64, 65, 127, 128, 129, 64, 65)):      # so many adjacent columns, from a chunk's start or off it
        first = 0 if r < 8 else min(100, max(k - run, 0))
        mask[r % m] = False
        mask[r % m, first:first + run] = True
    mask[m - 1] = True                                                       # the arrays end with a full row
    lens = mask.sum(1)
    ro = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    ci = np.nonzero(mask)[1].astype(np.int32)
    csr = W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)
    b_np = rng.standard_normal((2, k, 132)).astype(np.float32)
    ri, v, ro_t, ci_t = to_dev(csr, dev)
    out = pyops._spmm(torch.from_numpy(b_np).to(dev), ri, v, ro_t, ci_t, m, per_batch_values=False, accumulate=False, dtypes=(torch.float32,),
                      allow_i16=False, force_variant=5, force_nt=arrangement)
    want = oracle.spmm(b_np, csr.row_indices, csr.values, csr.row_offsets, csr.column_indices, m)
    scale = oracle.spmm_abs_scale(b_np, csr.row_indices, csr.values, csr.row_offsets, csr.column_indices, m)
    # at most k roundings of a sum, each 2^-24 of it: k * 6e-8 of the sum of magnitudes
    assert_close(out.cpu().numpy(), want, scale, max(k, 16) * 6e-8, f"arrangement {arrangement} {m} x {k}")


@pytest.mark.parametrize("m,k,n,density", [(72, 300, 1 << 22, 0.5),            # 5 GB of the dense operand
                                           (32776, 32768, 128, 1.0)])          # 2^30 nonzeros and a few
def test_beyond_a_buffers_reach(dev, m, k, n, density):
    """Operands whose byte offsets take more than 32 bits stay with the matrix cores, and both ends of them are read."""
    gen = torch.Generator(dev).manual_seed(m)
    rows = torch.rand(m, k, device=dev, generator=gen) < density if density < 1 else None
    ro = torch.cat([torch.zeros(1, device=dev, dtype=torch.int64), rows.sum(1).cumsum(0) if rows is not None else torch.arange(1, m + 1, device=dev) * k]).int()
    ci = rows.nonzero()[:, 1].int() if rows is not None else torch.arange(k, device=dev, dtype=torch.int32).repeat(m)
    v = torch.randn(ci.numel(), device=dev, generator=gen)
    a = torch.zeros(m, k, device=dev).masked_scatter_(rows, v) if rows is not None else v.view(m, k)
    b = torch.randn(1, k, n, device=dev, generator=gen)
    ri = torch.arange(m, device=dev, dtype=torch.int32)
    out = torch.empty(1, m, n, device=dev)
    rc = _lib.load().iex_spmm_ex(_lib.F32, _lib.I32, 0, m, k, n, ci.numel(), ri.data_ptr(), v.data_ptr(), ro.data_ptr(), ci.data_ptr(), b.data_ptr(),
                                 None, out.data_ptr(), torch.cuda.current_stream().cuda_stream, 1)
    _lib.check(rc, "spmm")
    assert "spmm_mfma_f32_kernel" in _lib.last_kernels()
    for columns in (slice(0, 128), slice(n // 2, n // 2 + 128), slice(n - 128, n)):
        part = b[0, :, columns].double()
        want = torch.cat([r.double() @ part for r in a.split(1024)])
        scale = torch.cat([r.double().abs() @ part.abs() for r in a.split(1024)])
        # at most k roundings of a sum, each 2^-24 of it
        assert bool(((out[0, :, columns].double() - want).abs() <= k * 6e-8 * scale).all())
    del a, b, out, v, ci, rows
    torch.cuda.empty_cache()
