"""The fp32 product by three bf16 parts of every entry (family 12): against the oracle at the edges of its tiles, planes and parts of k,
its error against 64 bits beside the row kernel's, infinities and NaN, entries outside the range of the parts, where the
library takes it, and what it does without room."""
import numpy as np
import pytest
import torch

from intrasm_engine_amd import _lib, workloads as W
from intrasm_engine_amd.pytorch import ops as pyops
from intrasm_engine_amd.pytorch.utils import dense_to_sparse
from _util import assert_close

pytestmark = pytest.mark.gpu
ops = torch.ops.iex_ops
FORCED = {"force_variant": 12}


def operands(m, k, n, density, batch=1, seed=0, dev="cuda"):
    g = torch.Generator(dev).manual_seed(seed)
    w = torch.randn(m, k, device=dev, generator=g) * (torch.rand(m, k, device=dev, generator=g) < density)
    if m > 2:
        w[m // 2] = 0                                              # an empty row
        w[0] = torch.randn(k, device=dev, generator=g)             # a full one
    return w, dense_to_sparse(w), torch.randn(batch, k, n, device=dev, generator=g)


def product(csr, b, m, variant=0, **kw):
    values, row_indices, row_offsets, columns = csr
    return pyops._spmm(b, row_indices, values, row_offsets, columns, m, per_batch_values=False, accumulate=False, dtypes=(torch.float32,),
                       allow_i16=False, force_variant=variant, **kw)


def error(got, w, b):
    want = torch.matmul(w.double(), b.double())
    return float((got.double() - want).norm() / want.norm())


# (m, k, n, density, batch): edges of the 128 x 128 tile, of steps of 32 k, of the 4096 columns that a row is assembled in, of chunks of 8
@pytest.mark.parametrize("m,k,n,density,batch", [(1, 1, 4, 1.0, 1), (3, 31, 5, 0.5, 1), (127, 32, 128, 0.3, 1), (128, 33, 129, 0.3, 2), (129, 96, 127, 0.2, 1),
                                                 (257, 2049, 131, 0.1, 1), (70, 2048, 260, 0.1, 3), (130, 2047, 9, 0.05, 1), (515, 4100, 256, 0.2, 1),
                                                 (4100, 200, 40, 0.3, 1), (60, 4064, 16, 0.2, 1), (60, 4095, 20, 0.2, 1), (60, 4096, 12, 0.2, 1), (60, 4097, 16, 0.2, 2), (20, 8193, 8, 0.1, 1), (9000, 64, 136, 0.2, 1), (300, 12000, 300, 0.02, 1)])
def test_against_the_oracle(oracle, m, k, n, density, batch):
    w, csr, b = operands(m, k, n, density, batch)
    got = product(csr, b, m, 12)
    assert "gemm_split_kernel" in _lib.last_kernels()
    v, ri, ro, ci = (t.cpu().numpy() for t in csr)
    want = oracle.spmm(b.cpu().numpy(), ri, v, ro, ci, m)
    scale = oracle.spmm_abs_scale(b.cpu().numpy(), ri, v, ro, ci, m)
    assert_close(got.cpu().numpy(), want, scale, 1e-5, f"{m}x{k}x{n}")
    # six of nine products of parts: what is left out is below 2^-26 of a product (middle * low twice, 2^-9 * 2^-18 each), sums are fp32's
    assert error(got, w, b) <= max(1.05 * error(product(csr, b, m, 1), w, b), 1.2e-7)


@pytest.mark.parametrize("m,k,n", [(256, 512, 192), (515, 4100, 256)])     # K in one part and in several: the epilogue and the kernel behind it
def test_bias_and_relu(m, k, n):
    w, csr, b = operands(m, k, n, 0.2)
    bias = torch.randn(m, device="cuda")
    got = product(csr, b, m, 12, bias=bias, relu=True)
    want = (torch.matmul(w.double(), b[0].double()) + bias.double()[:, None]).relu()
    assert float((got[0].double() - want).norm() / want.norm()) < 1e-6


def test_entries_are_exact():
    """One nonzero of 1 per row: the result is the dense operand's entry, all 24 bits of it."""
    m, k, n = 200, 320, 136
    w = torch.zeros(m, k, device="cuda")
    w[torch.arange(m), torch.arange(m) + 3] = 1.0
    b = torch.randn(1, k, n, device="cuda") * torch.exp2(torch.randint(-60, 30, (1, k, n), device="cuda").float())
    b[0, 3, 0] = 1.0
    got = product(dense_to_sparse(w), b, m, 12)
    assert "gemm_split_kernel" in _lib.last_kernels() and torch.equal(got[0], b[0, 3:3 + m])


@pytest.mark.parametrize("where", ["dense", "values", "both", "dense, no nonzero there"])
@pytest.mark.parametrize("what", [float("inf"), float("nan"), 3.4e38])
def test_infinities_and_nan_stay_where_the_row_kernel_leaves_them(where, what):
    m, k, n = 300, 700, 200
    w, _, b = operands(m, k, n, 0.2, seed=3)
    if "no nonzero" in where:
        w[:, 17] = 0
    if where != "values":
        b[0, 17, 5] = what
    if where in ("values", "both"):
        w[9, 40] = what
    csr = dense_to_sparse(w)
    got, want = product(csr, b, m, 12), product(csr, b, m, 1)
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    fine = want.isfinite()
    assert float((got - want)[fine].double().norm() / want[fine].double().norm()) < 1e-6
    if "no nonzero" in where:
        assert got.isfinite().all()


@pytest.mark.parametrize("of_values,of_dense", [(1e-30, 1.0), (1.0, 1e-35), (1e-20, 1e-15), (1e25, 1e10), (1e-25, 1e20)])
def test_entries_outside_the_range_of_the_parts(of_values, of_dense):
    m, k, n = 200, 300, 150
    w, _, b = operands(m, k, n, 0.2, seed=4)
    w, b = w * of_values, b * of_dense
    csr = dense_to_sparse(w)
    got, want = product(csr, b, m, 12), product(csr, b, m, 1)
    assert error(got, w, b) <= max(1.05 * error(want, w, b), 1.2e-7)


# (2-norms; rows of up to seven nonzeros are a chain as in the row kernel, longer ones gain by parts: 8 5.3e-8 / 5.4e-8, 32 6.2e-8 / 6.7e-8, 256 7.1e-8 / 1.5e-7.  Bound: the norm of
# 512 x 512 roundings is known to 1 / sqrt(2 * 512 * 512) = 1.4e-3 of itself, seven times that)
@pytest.mark.parametrize("per_row", [1, 2, 5, 7, 8, 16, 32, 128, 800])
def test_error_beside_the_row_kernels_by_the_length_of_rows(per_row):
    m, k, n = 512, 2048, 512
    g = torch.Generator("cuda").manual_seed(per_row)
    w = torch.zeros(m, k, device="cuda")
    w.scatter_(1, torch.rand(m, k, device="cuda", generator=g).argsort(1)[:, :per_row], torch.randn(m, per_row, device="cuda", generator=g))
    b = torch.randn(1, k, n, device="cuda", generator=g)
    csr = dense_to_sparse(w)
    by_parts, by_rows = error(product(csr, b, m, 12), w, b), error(product(csr, b, m, 1), w, b)
    assert by_parts <= 1.01 * by_rows, (by_parts, by_rows)


# (K in one part and in several; last chunks of one, two and three columns; more than a wavefront's columns)
@pytest.mark.parametrize("m,k,n,batch", [(200, 320, 133, 2), (130, 4100, 262, 1), (70, 64, 4, 3), (300, 96, 519, 1), (9000, 64, 12, 1)])
def test_rows_of_one_nonzero_are_rounded_once(m, k, n, batch):
    w, _, b = operands(m, k, n, 0.2, batch, seed=15)
    w[1::3] = 0
    w[torch.arange(1, m, 3), torch.randint(0, k, (len(range(1, m, 3)),))] = torch.randn(len(range(1, m, 3)), device="cuda")
    csr, bias = dense_to_sparse(w), torch.randn(m, device="cuda")
    got, want = product(csr, b, m, 12), torch.matmul(w.double(), b.double())
    assert "gemm_split_kernel" in _lib.last_kernels()
    one = (csr[2][1:] - csr[2][:-1] == 1).nonzero().view(-1)
    assert len(one) >= m // 3 and torch.equal(got[:, one], want[:, one].float())
    assert error(got, w, b) < 1.2e-7
    with_bias = product(csr, b[:1].contiguous(), m, 12, bias=bias, relu=True)
    assert torch.equal(with_bias[:, one], (want[:1, one].float() + bias[one, None]).relu())


@pytest.mark.parametrize("of_rows,of_columns", [(-126, 0), (0, -126), (-64, -64), (-110, 0)])
def test_rows_and_columns_of_widely_different_scales(of_rows, of_columns):
    """Every row and column from 1 down to 2^of_rows and 2^of_columns in steps of two powers: each result beside its own row's and column's scale."""
    m, k, n = 128, 320, 128
    w, _, b = operands(m, k, n, 0.3, seed=10)
    w *= torch.exp2(-(torch.arange(m, device="cuda").double() * 2).clamp(max=-of_rows))[:, None].float()
    b *= torch.exp2(-(torch.arange(n, device="cuda").double() * 2).clamp(max=-of_columns)).float()
    csr = dense_to_sparse(w)
    got, want, exact = product(csr, b, m, 12)[0], product(csr, b, m, 1)[0], w.double() @ b[0].double()
    # in fp32's normal range, each within rounding of the sum of its magnitudes: 2^-24 for each of some 100 terms, were they all to add up
    scale = w.double().abs() @ b[0].double().abs()
    fine = scale >= 2.0 ** -120
    of = lambda x: float(((x.double() - exact).abs() / scale)[fine].max())
    assert of(got) <= max(1.05 * of(want), 2.0 ** -22)


def test_stored_zeros_beside_entries_that_round_to_an_infinity():
    m, k, n = 130, 64, 40
    w, csr, b = operands(m, k, n, 0.3, seed=9)
    csr = (torch.zeros_like(csr[0]), *csr[1:])
    b[0, 3, 7] = 3.4e38
    got = product(csr, b, m, 12)
    assert "gemm_split_kernel" in _lib.last_kernels() and not got.any()


def test_where_it_is_taken_and_where_not():
    w, csr, b = operands(2048, 2048, 512, 0.2, seed=5)
    values, row_indices, row_offsets, columns = csr
    native = lambda: ops.spmm_sputnik_reuse_weight(b, row_indices, values, row_offsets, columns, 2048)
    taken = native()
    assert "gemm_split_kernel" in _lib.last_kernels()
    assert torch.equal(taken, product(csr, b, 2048, 12)) and torch.equal(taken, native())
    plain = product(csr, b, 2048, no_workspace=True)
    assert "split" not in _lib.last_kernels() and float((taken - plain).norm() / plain.norm()) < 2e-6
    with pyops.kernel_params(spmm={"beside_gather_kernel": True}):
        native()
        assert "split" not in _lib.last_kernels()
    # columns in any order, values per batch entry, accumulation: the kernels that take them
    size = lambda flags: _lib.load().iex_spmm_workspace_kind(_lib.F32, _lib.I32, flags | _lib.SPMM_PAD_OPERANDS, 2048, 2048, 512, columns.numel(), 1)
    assert size(0) == 12 and [size(f) for f in (_lib.SPMM_ANY_COLUMN_ORDER, _lib.SPMM_PER_BATCH_VALUES, _lib.SPMM_ACCUMULATE)] == [0, 0, 0]
    # unaligned operands are served
    shifted = torch.empty(b.numel() + 1, device="cuda")[1:].view_as(b).copy_(b)
    assert torch.equal(ops.spmm_sputnik_reuse_weight(shifted, row_indices, values, row_offsets, columns, 2048), taken)


def test_a_batch_in_groups():
    """The workspace does not grow with the batch: groups of entries share the room, the last one smaller; an infinity sends its own group to the row kernel."""
    m, k, n, batch = 256, 8192, 4096, 6              # planes of an entry: 201 MB, so two at a time
    w, csr, b = operands(m, k, n, 0.2, batch, seed=13)
    size = lambda batch: _lib.load().iex_spmm_workspace_bytes(_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS | 12 << 16, m, k, n, csr[0].numel(), batch)
    assert size(2) == size(6) == size(5000) > size(1)
    b[3, 5, 7] = float("inf")
    got = product(csr, b, m, 12)
    assert _lib.last_kernels().count("gemm_split_kernel") == 3
    for z in (0, 1, 4, 5):
        assert error(got[z], w, b[z]) < 1.2e-7
    assert torch.equal(got[3:4].isfinite(), product(csr, b[3:4].contiguous(), m, 1).isfinite())
    uneven = product(csr, b[2:5].contiguous(), m, 12)     # two and one
    assert torch.equal(uneven[2], got[4]) and error(uneven[2], w, b[4]) < 1.2e-7


def test_no_more_workspace_than_its_bound():
    size = lambda m, k, n, batch=1: _lib.load().iex_spmm_workspace_bytes(_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS | 12 << 16, m, k, n, m * k // 5, batch)
    of_sddmm = lambda m, n, k: _lib.load().iex_sddmm_workspace_bytes(_lib.F32, _lib.SDDMM_PAD_OPERANDS | 12 << 16, m, k, n, m * n // 5, 1)
    most = 4 << 30
    for shape in ((4096, 4096, 4096, 64), (4096, 4096, 2048, 384), (11008, 4096, 8192, 64), (20000, 20000, 512)):
        assert 0 < size(*shape) <= most
    assert size(26000, 26000, 4096) == 0 and 0 < of_sddmm(11008, 4096, 32768) <= most and of_sddmm(30000, 30000, 16384) == 0


def test_without_memory_for_the_workspace():
    """Where the allocator has none left for it, the operators run on the kernels that take none, as they did before there were parts."""
    m, k, n = 6144, 8192, 512
    w, csr, b = operands(m, k, n, 0.2, seed=14)
    values, row_indices, row_offsets, columns = csr
    lhs, rhs = torch.randn(1, m, n, device="cuda"), torch.randn(1, k, n, device="cuda")
    calls = {"native spmm": lambda: ops.spmm_sputnik_reuse_weight(b, row_indices, values, row_offsets, columns, m), "spmm": lambda: product(csr, b, m),
             "native sddmm": lambda: ops.sddmm_sputnik_atomic_upd_weight(lhs, rhs, row_indices, row_offsets, columns),
             "sddmm": lambda: pyops._sddmm(lhs, rhs, row_indices, row_offsets, columns, sum_over_batch=True, dtypes=(torch.float32,))}
    want = {}
    for name, call in calls.items():
        want[name] = call().cpu()
        assert "gemm_split_kernel" in _lib.last_kernels(), name
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    held = []
    try:   # everything taken in pieces, one of them left for the results: nowhere room for the 360 MB of planes
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (256 << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            while len(held) < 1000:
                held.append(torch.empty(48 << 20, dtype=torch.uint8, device="cuda"))
        held.pop()
        for name, call in calls.items():
            got = call()
            assert "split" not in _lib.last_kernels(), name
            assert float((got.cpu() - want[name]).norm() / want[name].norm()) < 2e-6, name
            del got
        with pytest.raises(torch.OutOfMemoryError):
            product(csr, b, m, 12)
    finally:
        held.clear()
        torch.cuda.set_per_process_memory_fraction(1.0)


def test_captured_and_replayed_between_other_work():
    w, csr, b = operands(1500, 2100, 600, 0.25, seed=6)
    values, row_indices, row_offsets, columns = csr
    call = lambda: ops.spmm_sputnik_reuse_weight(b, row_indices, values, row_offsets, columns, 1500)
    call()
    assert "gemm_split_kernel" in _lib.last_kernels()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call()
    for seed in range(3):
        b.copy_(torch.randn(b.shape, device="cuda", generator=torch.Generator("cuda").manual_seed(seed)))
        if seed == 1:
            b[0, 0, 0] = float("inf")
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out.nan_to_num(7.0), call().nan_to_num(7.0))


def test_static_scratch_too_small_for_the_parts(dev):
    """iex_spmm_static holds 96 MB: an fp32 call whose parts need more runs on the other families, as it did."""
    m, k, n = 4096, 4096, 512
    w, csr, b = operands(m, k, n, 0.2, seed=7)
    values, row_indices, row_offsets, columns = csr
    lib, out = _lib.load(), torch.empty(1, m, n, device="cuda")
    assert lib.iex_spmm_workspace_bytes(_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS, m, k, n, columns.numel(), 1) > lib.iex_spmm_static_scratch_bytes()
    _lib.check(lib.iex_spmm_static(_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS, m, k, n, columns.numel(), row_indices.data_ptr(), values.data_ptr(), row_offsets.data_ptr(),
                                   columns.data_ptr(), b.data_ptr(), None, out.data_ptr(), torch.cuda.current_stream().cuda_stream, 1), "static")
    assert "split" not in _lib.last_kernels() and error(out, w, b) < 2e-6


def test_static_scratch_is_not_for_parts_that_it_would_hold(dev):
    """iex_spmm_static's array is shared by all calls on the GPU.  fp32 calls never used it: programs may run them side by side."""
    m, k, n = 2048, 2048, 512
    w, csr, b = operands(m, k, n, 0.2, seed=7)
    values, row_indices, row_offsets, columns = csr
    lib, out, want = _lib.load(), torch.empty(1, m, n, device="cuda"), torch.empty(1, m, n, device="cuda")
    assert 0 < lib.iex_spmm_workspace_bytes(_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS, m, k, n, columns.numel(), 1) <= lib.iex_spmm_static_scratch_bytes()
    args = lambda out: (_lib.F32, _lib.I32, _lib.SPMM_PAD_OPERANDS, m, k, n, columns.numel(), row_indices.data_ptr(), values.data_ptr(), row_offsets.data_ptr(),
                        columns.data_ptr(), b.data_ptr(), None, out.data_ptr(), torch.cuda.current_stream().cuda_stream, 1)
    _lib.check(lib.iex_spmm_static(*args(out)), "static")
    assert "split" not in _lib.last_kernels() and error(out, w, b) < 2e-6
    _lib.check(lib.iex_spmm_ex(*args(want)), "plain")
    assert torch.equal(out, want)
