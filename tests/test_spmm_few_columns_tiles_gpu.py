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


@pytest.mark.parametrize("k", [1, 31, 64, 128])
@pytest.mark.parametrize("n,offset", [(257, 0), (272, 1), (481, 3), (511, 0), (513, 0), (543, 2), (785, 0), (1055, 1), (2049, 0)])
def test_whole_lines_by_one_wavefront(oracle, dev, n, offset, k):
    """fp32 rows that start anywhere in a line: from one tile of edges to several middle ones, an output at any alignment, rows
    without nonzeros, more nonzeros per wavefront than it holds at once; every entry is written, with the row kernel's bits, and nothing around
    the output."""
    rng = np.random.default_rng(n + k)
    m, batch = 150, 2
    mask = rng.random((m, k)) < min(0.5, 4.0 / k)
    mask[3] = False
    mask[4] = True
    mask[0, 0] = True
    ro, ci, _ = W.csr_from_mask(mask)
    ri = W.swizzle_from_offsets(ro)
    values = rng.standard_normal((batch, ci.shape[0])).astype(np.float32)
    b = rng.standard_normal((batch, k, n)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    around = torch.full((4096 + batch * m * n + 4096,), 7.0, device=dev)
    out = around[4096 + offset:][:batch * m * n].view(batch, m, n)
    out.fill_(float("nan"))
    common = dict(per_batch_values=True, accumulate=False, dtypes=(torch.float32,), allow_i16=False)
    pyops._spmm(t(b), t(ri), t(values), t(ro), t(ci), m, out=out, force_variant=8, **common)
    assert "spmm_smallk_kernel_lines" in _lib.last_kernels()
    for z in range(batch):
        args = b[z:z + 1], ri, values[z], ro, ci, m
        assert_close(out[z].cpu().numpy(), oracle.spmm(*args)[0], oracle.spmm_abs_scale(*args)[0], 1e-5, f"n={n} k={k}")
    assert torch.equal(out, pyops._spmm(t(b), t(ri), t(values), t(ro), t(ci), m, force_variant=1, force_wpr=1, **common))
    assert bool((around[:4096 + offset] == 7.0).all()) and bool((around[4096 + offset + batch * m * n:] == 7.0).all())


def test_more_nonzeros_than_a_wavefront_holds(oracle, dev):
    """Rows whose nonzeros cross the 512 that are loaded together, and more than 63 rows per wavefront."""
    rng = np.random.default_rng(9)
    m, k, n, batch = 4000, 40, 300, 60
    mask = rng.random((m, k)) < 0.15
    mask[700:760] = True
    ro, ci, _ = W.csr_from_mask(mask)
    ri = W.swizzle_from_offsets(ro)
    values, b = rng.standard_normal(ci.shape[0]).astype(np.float32), rng.standard_normal((1, k, n)).astype(np.float32)
    t = lambda a: torch.from_numpy(a).to(dev)
    for width in (300, 304):      # by lines, by vectors
        bz = t(np.repeat(np.pad(b, ((0, 0), (0, 0), (0, width - 300))), batch, axis=0))
        vz = t(np.repeat(values[None], batch, axis=0))
        with pyops.kernel_params(spmm={"force_variant": 8}):
            out = ops.spmm_sputnik_batched_values(bz, t(ri), vz, t(ro), t(ci), m)
        assert ("lines" in _lib.last_kernels()) == (width == 300)
        assert_close(out[-1, :, :300].cpu().numpy(), oracle.spmm(b, ri, values, ro, ci, m)[0], oracle.spmm_abs_scale(b, ri, values, ro, ci, m)[0], 1e-5, "long")
        assert torch.equal(out[0], out[-1])
