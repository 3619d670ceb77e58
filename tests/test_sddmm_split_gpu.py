"""The fp32 sampled product by three bf16 parts of every entry (variant 12): against the oracle at the edges of its tiles, planes and
parts of k, its error against 64 bits beside the gather kernel's, infinities and NaN, entries outside the range of the parts,
where the library takes it."""
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd.pytorch import ops as pyops
from intrasm_engine_amd.pytorch.utils import dense_to_sparse
from _util import assert_close

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops


def operands(m, n, k, density, batch=1, seed=0):
    g = torch.Generator("cuda").manual_seed(seed)
    mask = (torch.rand(m, n, device="cuda", generator=g) < density).float()
    mask[0] = 1
    if m > 2:
        mask[m // 2] = 0
    _, row_indices, row_offsets, columns = dense_to_sparse(mask)
    return (torch.randn(batch, m, k, device="cuda", generator=g), torch.randn(batch, n, k, device="cuda", generator=g), row_indices, row_offsets, columns)


def sampled(args, variant=0, **kw):
    return pyops._sddmm(*args, sum_over_batch=True, dtypes=(torch.float32,), force_variant=variant, **kw).view(-1)


def error(got, args):
    lhs, rhs, _, row_offsets, columns = args
    rows = torch.repeat_interleave(torch.arange(lhs.shape[1], device="cuda"), (row_offsets[1:] - row_offsets[:-1]).long())
    want = torch.matmul(lhs.double(), rhs.double().transpose(1, 2).contiguous()).sum(0)[rows, columns.long()]
    return float((got.double() - want).norm() / want.norm())


# (m, n, k, density, batch): edges of the 128 x 128 tile, of steps of 32 k, one part of k and several
@pytest.mark.parametrize("m,n,k,density,batch", [(1, 1, 1, 1.0, 1), (3, 5, 31, 0.5, 2), (127, 128, 32, 0.3, 1), (128, 127, 33, 0.3, 3), (129, 257, 64, 0.2, 1),
                                                 (300, 130, 1000, 0.2, 1), (515, 700, 2049, 0.1, 1), (70, 3000, 100, 0.1, 4), (3000, 131, 193, 0.1, 4)])
def test_against_the_oracle(oracle, m, n, k, density, batch):
    args = operands(m, n, k, density, batch)
    got = sampled(args, 12)
    assert "gemm_split_kernel" in _lib.last_kernels()
    lhs, rhs, ri, ro, ci = (t.cpu().numpy() for t in args)
    assert_close(got.cpu().numpy(), oracle.sddmm(lhs, rhs, ri, ro, ci), oracle.sddmm_abs_scale(lhs, rhs, ri, ro, ci), 1e-5, f"{m}x{n}x{k}")
    # (six of nine products of parts, what is left out below 2^-26 of a product; sums of a few terms are exact either way)
    assert error(got, args) <= max(1.05 * error(sampled(args, 1), args), 8e-8)


@pytest.mark.parametrize("what", [float("inf"), float("nan"), 3.4e38])
@pytest.mark.parametrize("where", ["lhs", "rhs", "both"])
def test_infinities_and_nan_as_in_the_dot_product(what, where):
    args = operands(300, 260, 500, 0.2, 2, seed=2)
    if where != "rhs":
        args[0][1, 7, 3] = what
    if where != "lhs":
        args[1][0, 40, 9] = what
    got, want = sampled(args, 12), sampled(args, 1)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert float((got - want)[fine].double().norm() / want[fine].double().norm()) < 1e-6


@pytest.mark.parametrize("of_lhs,of_rhs", [(1e-30, 1.0), (1.0, 1e-35), (1e-20, 1e-15), (1e25, 1e10), (1e-25, 1e20)])
def test_entries_outside_the_range_of_the_parts(of_lhs, of_rhs):
    lhs, rhs, *pattern = operands(200, 150, 300, 0.2, seed=4)
    args = (lhs * of_lhs, rhs * of_rhs, *pattern)
    assert error(sampled(args, 12), args) <= max(1.05 * error(sampled(args, 1), args), 8e-8)


@pytest.mark.parametrize("of_lhs,of_rhs", [(-126, 0), (0, -126), (-64, -64)])
def test_rows_of_widely_different_scales(of_lhs, of_rhs):
    lhs, rhs, *pattern = operands(128, 130, 300, 0.5, seed=11)
    down = lambda rows, least: torch.exp2(-(torch.arange(rows, device="cuda").double() * 2).clamp(max=-least))[:, None].float()
    args = (lhs * down(128, of_lhs), rhs * down(130, of_rhs), *pattern)
    row_offsets, columns = pattern[1:]
    rows = torch.repeat_interleave(torch.arange(128, device="cuda"), (row_offsets[1:] - row_offsets[:-1]).long())
    pick = lambda x, y: torch.matmul(x[0].double(), y[0].double().t().contiguous())[rows, columns.long()]
    exact, scale = pick(args[0], args[1]), pick(args[0].abs(), args[1].abs())
    fine = scale >= 2.0 ** -120
    of = lambda x: float(((x.double() - exact).abs() / scale)[fine].max())
    # (2^-24 for each of 300 terms, were they all to add up)
    assert of(sampled(args, 12)) <= max(1.05 * of(sampled(args, 1)), 2.0 ** -22)


@pytest.mark.parametrize("what", [float("inf"), float("nan")])
@pytest.mark.parametrize("of_lhs,of_rhs", [(1e-36, 1.0), (1.0, 1e-36), (1e-20, 1e-15), (1e25, 1e10)])
def test_an_infinity_beside_entries_outside_the_range(what, of_lhs, of_rhs):
    """The finite scores are the dot products themselves, as where there is no infinity."""
    lhs, rhs, *pattern = operands(200, 150, 300, 0.2, seed=4)
    clean = (lhs * of_lhs, rhs * of_rhs, *pattern)
    args = (clean[0].clone(), clean[1].clone(), *pattern)
    args[0][0, 7, 3] = what
    args[1][0, 40, 9] = what
    got, want = sampled(args, 12), sampled(args, 1)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    _, _, _, row_offsets, columns = clean
    rows = torch.repeat_interleave(torch.arange(200, device="cuda"), (row_offsets[1:] - row_offsets[:-1]).long())
    exact = torch.matmul(clean[0][0].double(), clean[1][0].double().t().contiguous())[rows, columns.long()][fine]
    of = lambda x: float((x[fine].double() - exact).norm() / exact.norm())
    # (two fp32 chains over the same 300 terms, cut differently)
    assert of(got) <= max(1.5 * of(want), 1.2e-7)


# a wavefront and a workgroup to a row, rows of one score, of no whole eights and of several hundred; k of no whole vectors, below and beyond four vectors a lane
@pytest.mark.parametrize("m,n,k,density,batch", [(5, 3, 1, 1.0, 1), (33, 70, 3, 0.4, 2), (40, 90, 31, 0.3, 1), (130, 600, 130, 0.5, 1), (300, 40, 257, 0.3, 3), (70, 1500, 300, 0.6, 2)])
def test_scores_computed_one_by_one(oracle, m, n, k, density, batch):
    """All of them (operands outside the range of the parts), or a row's and a column's (an infinity), as the dot products themselves."""
    lhs, rhs, *pattern = operands(m, n, k, density, batch, seed=12)
    args = (lhs * 1e-30, rhs * 1e-4, *pattern)
    lhs_np, rhs_np, ri, ro, ci = (t.cpu().numpy() for t in args)
    assert_close(sampled(args, 12).cpu().numpy(), oracle.sddmm(lhs_np, rhs_np, ri, ro, ci), oracle.sddmm_abs_scale(lhs_np, rhs_np, ri, ro, ci), 1e-5, f"{m}x{n}x{k}")
    assert "split_sample_kernel" in _lib.last_kernels()
    lhs[-1, m - 1, k - 1] = float("inf")
    rhs[0, n - 1, 0] = float("-inf")
    args = (lhs, rhs, *pattern)
    got, want = sampled(args, 12), sampled(args, 1)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf()) and torch.equal(got[want.isinf()], want[want.isinf()])
    fine = want.isfinite()
    assert not fine.any() or float((got - want)[fine].double().norm() / want[fine].double().norm()) < 1e-6


def test_where_it_is_taken_and_where_not():
    args = operands(2000, 1500, 700, 0.2, seed=5)
    lhs, rhs, row_indices, row_offsets, columns = args
    native = lambda: ops.sddmm_sputnik_atomic_upd_weight(lhs, rhs, row_indices, row_offsets, columns)
    taken = native()
    assert "gemm_split_kernel" in _lib.last_kernels() and torch.equal(taken.view(-1), sampled(args, 12)) and torch.equal(taken, native())
    sampled(args, no_workspace=True)
    assert "split" not in _lib.last_kernels()
    kind = lambda flags: _lib.load().iex_sddmm_workspace_kind(_lib.F32, flags, 2000, 700, 1500, columns.numel(), 1)
    assert kind(_lib.SDDMM_PAD_OPERANDS | _lib.SDDMM_SUM_OVER_BATCH) == 12 and kind(_lib.SDDMM_SUM_OVER_BATCH) == 0
    assert kind(_lib.SDDMM_PAD_OPERANDS | _lib.SDDMM_ACCUMULATE) == 0
    # columns in any order are served: the scores are picked by column
    order = torch.cat([torch.arange(a, b, device="cuda").flip(0) for a, b in zip(row_offsets[:-1].tolist(), row_offsets[1:].tolist())])
    backwards = (lhs, rhs, row_indices, row_offsets, columns[order].contiguous())
    assert torch.equal(sampled(backwards, 12), taken.view(-1)[order])


def test_training_step_in_fp32():
    """Forward and both gradients by parts, and replayed from a graph: against 64 bits."""
    from intrasm_engine_amd.pytorch.cpp_extensions.layers_and_funcs.sputnik import spmm as trainable
    from intrasm_engine_amd.pytorch.utils import transpose_info
    m, k, n = 2100, 1700, 900
    g = torch.Generator("cuda").manual_seed(8)
    w = torch.randn(m, k, device="cuda", generator=g) * (torch.rand(m, k, device="cuda", generator=g) < 0.2)
    values, row_indices, row_offsets, columns = dense_to_sparse(w)
    b = torch.randn(k, n, device="cuda", generator=g).requires_grad_()
    values.requires_grad_()
    gradient = torch.randn(m, n, device="cuda", generator=g)
    out = trainable(b, row_indices, values, row_offsets, columns, m, transpose_info(m, k, row_offsets, columns))
    assert "gemm_split_kernel" in _lib.last_kernels()
    grad_b, grad_v = torch.autograd.grad(out, (b, values), gradient)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), (row_offsets[1:] - row_offsets[:-1]).long())
    for got, want in ((out, w.double() @ b.double()), (grad_b, w.double().T.contiguous() @ gradient.double()),
                      (grad_v, (gradient.double() @ b.double().T.contiguous())[rows, columns.long()])):
        assert float((got.double() - want).norm() / want.norm()) < 1.5e-7
