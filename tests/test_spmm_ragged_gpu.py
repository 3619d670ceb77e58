"""Narrow outputs whose rows are no whole vectors (spmm_ragged.hip): several nonzeros per gather at element alignment, against the oracle at
the widths where the number of lanes per nonzero changes, by one wavefront a row and by four, and which rows get how many."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib
from intrasm_engine_amd.pytorch import ops as pyops
from intrasm_engine_amd.pytorch.utils import dense_to_sparse, to_int16_indices
from _util import RTOL, assert_close, rounded

pytestmark = pytest.mark.gpu


def operands(m, k, n, density, dtype, uneven=False, batch=1):
    g = torch.Generator("cuda").manual_seed(m + n)
    share = torch.full((m, 1), density, device="cuda")
    if uneven:
        share = (density * 2 * torch.rand(m, 1, device="cuda", generator=g)).clamp(max=1)
        share[::97] = min(1.0, 8 * density)
    w = torch.randn(m, k, device="cuda", generator=g) * (torch.rand(m, k, device="cuda", generator=g) < share)
    w[m // 2] = 0
    return dense_to_sparse(w.to(dtype)), torch.randn(batch, k, n, device="cuda", generator=g).to(dtype)


# (m, k, density, uneven) to either number of wavefronts
SHAPES = {1: (3000, 200, 0.3, False), 4: (300, 900, 0.4, False), -4: (1500, 900, 0.2, True)}


@pytest.mark.parametrize("waves", SHAPES)
@pytest.mark.parametrize("dtype,index,n", [(torch.float32, torch.int32, n) for n in (5, 7, 31, 33, 63, 65, 127)] +
                         [(torch.float16, torch.int32, n) for n in (9, 63, 65, 127, 129, 255)] + [(torch.float16, torch.int16, 14), (torch.bfloat16, torch.int32, 100)])
def test_against_the_oracle(oracle, dtype, index, n, waves):
    m, k, density, uneven = SHAPES[waves]
    batch = 2 if n == 33 else 1
    (values, row_indices, row_offsets, columns), b = operands(m, k, n, density, dtype, uneven, batch)
    c = to_int16_indices(columns, k) if index == torch.int16 else columns
    pyops.prepare_pattern(row_offsets, c, k)
    got = pyops._spmm(b, row_indices, values, row_offsets, c, m, per_batch_values=False, accumulate=False, dtypes=(dtype,), allow_i16=True, no_workspace=True)
    kernel = _lib.last_kernels()
    two_per_gather = n > 256 // values.element_size()
    if waves == 1 or not two_per_gather:
        lanes = 8 if n <= 8 * 16 // values.element_size() else 16 if n <= 256 // values.element_size() else 32
        assert "spmm_ragged_narrow_kernel" in kernel and f", {lanes}, {abs(waves)}," in kernel, kernel
    v, ri, ro, ci = (t.float().cpu().numpy() if t.is_floating_point() else t.cpu().numpy() for t in (values, row_indices, row_offsets, columns))
    x = b.float().cpu().numpy()
    want, scale = oracle.spmm(x, ri, v, ro, ci, m), oracle.spmm_abs_scale(x, ri, v, ro, ci, m)
    assert_close(got.float().cpu().numpy(), want, scale, RTOL[dtype], f"n = {n}, {kernel}")
    # nothing is written beside the output: rows end where the next one begins
    room = torch.full((batch * m * n + 64,), 7.0, device="cuda", dtype=dtype)
    out = room[32:32 + batch * m * n].view(batch, m, n)
    pyops._spmm(b, row_indices, values, row_offsets, c, m, per_batch_values=False, accumulate=False, dtypes=(dtype,), allow_i16=True, no_workspace=True, out=out)
    assert torch.equal(out, got) and (room[:32] == 7).all() and (room[-32:] == 7).all()


def test_what_stays_with_one_nonzero_per_gather():
    for m, k, n, density, uneven in ((1000, 300, 33, 0.3, False), (3000, 100, 33, 0.1, False), (1000, 300, 33, 0.2, True), (500, 900, 101, 0.4, False)):
        (values, row_indices, row_offsets, columns), b = operands(m, k, n, density, torch.float32, uneven)
        pyops.prepare_pattern(row_offsets, columns, k)
        call = lambda **kw: pyops._spmm(b, row_indices, values, row_offsets, columns, m, per_batch_values=False, accumulate=False, dtypes=(torch.float32,), allow_i16=False, no_workspace=True, **kw)
        call()
        assert "ragged_narrow" not in _lib.last_kernels()
        call(force_wpr=4)
        assert "ragged_narrow" not in _lib.last_kernels()


@pytest.mark.parametrize("m,k,n,density,dense_form", [(1500, 4000, 315, 0.15, True), (1500, 300, 315, 0.15, False), (2000, 5000, 67, 0.25, True), (2600, 3100, 26, 0.18, False)])
def test_rows_at_element_alignment_count_in_the_choice_of_the_dense_form(oracle, m, k, n, density, dense_form):
    (values, row_indices, row_offsets, columns), b = operands(m, k, n, density, torch.float16)
    got = torch.ops.iex_ops.spmm_sputnik_reuse_weight_half(b, row_indices, values, row_offsets, columns, m)
    assert ("csr_to_dense" in _lib.last_kernels()) == dense_form, _lib.last_kernels()
    v, ri, ro, ci = (t.float().cpu().numpy() if t.is_floating_point() else t.cpu().numpy() for t in (values, row_indices, row_offsets, columns))
    x = b.float().cpu().numpy()
    assert_close(got.float().cpu().numpy(), oracle.spmm(x, ri, v, ro, ci, m), oracle.spmm_abs_scale(x, ri, v, ro, ci, m), 1e-2, f"{m} x {k} x {n}")
