"""A sparse 16-bit weight laid out once (dense form, two-of-four form with spilled entries) and multiplied by what was laid out: every
kind at the edges of tiles, phases and spill blocks, against the oracle; when a form may stand for the CSR arrays."""
import ctypes
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from intrasm_engine_amd import _iex_host, _lib
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.decoder_layer import SparseDecoderLayer
from intrasm_engine_amd.pytorch import ops as pyops
from _util import RTOL, assert_close, rounded, to_dev

pytestmark = pytest.mark.gpu
CODE = {torch.float16: _lib.F16, torch.bfloat16: _lib.BF16}


def _two_four(rng, m, k):
    """Two of every four neighbouring columns (one of them, or none, in some groups)."""
    keep = np.zeros((m, (k + 3) // 4, 4), bool)
    order = rng.random(keep.shape).argsort(axis=2)
    np.put_along_axis(keep, order[:, :, :2], True, axis=2)
    keep &= rng.random(keep.shape) < 0.9
    return keep.reshape(m, -1)[:, :k]


def _csr(rng, m, k, density):
    mask = _two_four(rng, m, k) if density == "2:4" else rng.random((m, k)) < density
    mask[0, :min(k, 7)] = True           # (at least three entries; a row that spills)
    if m > 2:
        mask[2] = False
    ro = np.concatenate([[0], np.cumsum(mask.sum(axis=1))]).astype(np.int32)
    ci = np.nonzero(mask)[1].astype(np.int32)
    return W.CSR(m, k, rng.standard_normal(ci.shape[0]).astype(np.float32), W.swizzle_from_offsets(ro), ro, ci)


def _spilled_phases(csr, half):
    """What iex_form_measure counts, from the definition: columns with entries beyond the first two of their group, per block of rows."""
    phases = []
    for r0 in range(0, csr.m, half):
        cols = set()
        for r in range(r0, min(r0 + half, csr.m)):
            c = csr.column_indices[csr.row_offsets[r]:csr.row_offsets[r + 1]]
            cols.update(c[2:][c[2:] // 4 == c[:-2] // 4].tolist())
        phases.append((len(cols) + 31) // 32)
    return sum(phases), max(phases)


@pytest.mark.parametrize("dtype,idtype", [(torch.float16, torch.int16), (torch.bfloat16, torch.int32)])
@pytest.mark.parametrize("m,k,n,density", [(1, 7, 8, 1.0), (127, 64, 256, "2:4"), (300, 200, 264, 0.3), (257, 129, 520, 0.5), (193, 1000, 40, 0.1),
                                           (385, 65, 248, 0.05), (130, 260, 264, 1.0), (640, 4100, 264, 0.1)])
def test_every_kind(oracle, dev, dtype, idtype, m, k, n, density):
    rng = np.random.default_rng(m + k)
    csr = _csr(rng, m, k, density)
    _, v, ro, ci = to_dev(csr, dev, dtype, idtype)
    x, aux = rng.standard_normal((k, n)).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    xt, at = (torch.from_numpy(t).to(dev).to(dtype) for t in (x, aux))
    vr, xr, ar = rounded(csr.values, dtype), rounded(x, dtype), rounded(aux, dtype).astype(np.float64)
    base = oracle.spmm(xr[None], csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)[0]
    scale = oracle.spmm_abs_scale(xr[None], csr.row_indices, vr, csr.row_offsets, csr.column_indices, m)[0]
    silu = ar / (1 + np.exp(-ar))
    lib, it, nnz, stream = _lib.load(), 1 if idtype == torch.int16 else 0, ci.numel(), torch.cuda.current_stream().cuda_stream
    scratch = torch.empty(lib.iex_form_scratch_bytes(m, k), dtype=torch.uint8, device=dev)
    counts = torch.zeros(6, dtype=torch.int32, device=dev)
    _lib.check(lib.iex_form_measure(it, m, k, nnz, ro.data_ptr(), ci.data_ptr(), scratch.data_ptr(), scratch.numel(), counts.data_ptr(), stream))
    counts = counts.tolist()
    for i, half in enumerate((64, 96, 128)):
        assert (counts[i], counts[3 + i]) == _spilled_phases(csr, half)
    for i, kind in enumerate((0, 128, 192, 256)):
        room = counts[2 + i] if kind else 0
        form = torch.full((lib.iex_form_bytes(kind, m, k, room),), 0xff, dtype=torch.uint8, device=dev)      # (NaN where nothing is written)
        _lib.check(lib.iex_form_build(it, kind, m, k, nnz, ro.data_ptr(), ci.data_ptr(), v.data_ptr(), room, form.data_ptr(), form.numel(),
                                      scratch.data_ptr(), scratch.numel(), stream))
        need = lib.iex_form_product_workspace_bytes(kind, m, k, n)
        ws = torch.empty(max(need, 1), dtype=torch.uint8, device=dev)
        for mode, want, bound in ((0, base, scale), (1, base + ar, scale + np.abs(ar)), (2, base * silu, scale * np.abs(silu) + 1e-3)):
            out = torch.full((m, n), float("nan"), dtype=dtype, device=dev)
            _lib.check(lib.iex_form_product(CODE[dtype], kind, m, k, n, room, form.data_ptr(), xt.data_ptr(), at.data_ptr() if mode else None, mode,
                                            out.data_ptr(), ws.data_ptr(), need, stream))
            assert ("two_four_kernel" in _lib.last_kernels()) == (kind > 0)
            assert_close(out.float().cpu().numpy(), want, 5 * bound, RTOL[dtype], f"kind {kind} mode {mode}")


def test_values_that_mark_an_empty_place_and_infinities(dev):
    """Every bit pattern is a value; an infinity a row refers to shows as itself in that row."""
    m, k, n = 130, 128, 256
    rng = np.random.default_rng(1)
    csr = _csr(rng, m, k, "2:4")
    _, v, ro, ci = to_dev(csr, dev, torch.float16)
    x = torch.randn(k, n, device=dev).half()
    x[5, 3] = float("inf")
    v[torch.nonzero(ci == 9)[0]] = float("nan")
    form = pyops.WeightForm(v, ro, ci, m, k)
    dense = torch.zeros(m, k, device=dev, dtype=torch.float64)
    rows = torch.repeat_interleave(torch.arange(m, device=dev), ro.long().diff())
    dense[rows, ci.long()] = v.double()
    refers = dense[:, 5] != 0
    lib, kinds = _lib.load(), form._form.kinds
    assert kinds & 1
    for kind in (128, 256):
        counts = torch.zeros(6, dtype=torch.int32, device=dev)
        scratch = torch.empty(lib.iex_form_scratch_bytes(m, k), dtype=torch.uint8, device=dev)
        stream = torch.cuda.current_stream().cuda_stream
        _lib.check(lib.iex_form_measure(0, m, k, ci.numel(), ro.data_ptr(), ci.data_ptr(), scratch.data_ptr(), scratch.numel(), counts.data_ptr(), stream))
        room = counts.tolist()[2 + (kind // 64 - 1)]
        memory = torch.empty(lib.iex_form_bytes(kind, m, k, room), dtype=torch.uint8, device=dev)
        _lib.check(lib.iex_form_build(0, kind, m, k, ci.numel(), ro.data_ptr(), ci.data_ptr(), v.data_ptr(), room, memory.data_ptr(), memory.numel(),
                                      scratch.data_ptr(), scratch.numel(), stream))
        out = torch.empty(m, n, device=dev, dtype=torch.float16)
        _lib.check(lib.iex_form_product(_lib.F16, kind, m, k, n, room, memory.data_ptr(), x.data_ptr(), None, 0, out.data_ptr(), None, 0, stream))
        with_nan = dense.isnan().any(dim=1)
        assert bool(out[with_nan].isnan().all())
        assert bool(out[refers & ~with_nan][:, 3].isinf().all())
        others = torch.ones(n, dtype=torch.bool, device=dev)
        others[3] = False
        want = (torch.nan_to_num(dense) @ torch.nan_to_num(x.double(), posinf=0.0))[~with_nan][:, others]
        assert torch.allclose(out[~with_nan][:, others].double(), want, rtol=1e-2, atol=1e-1)


@pytest.mark.parametrize("dtype,idtype", [(torch.float16, torch.int16), (torch.bfloat16, torch.int32)])
@pytest.mark.parametrize("m,k,n,kind", [(1024, 4096, 8192, 128), (1536, 4096, 6144, 192), (2048, 4096, 6144, 256)])
def test_a_weight_with_spill_kept_and_captured(dev, dtype, idtype, m, k, n, kind):
    """A two-of-four weight some of whose groups hold more: kept, laid out by every replay, and after values and columns were written in place so
    that every row spills half of its entries."""
    rng = np.random.default_rng(kind)
    mask = _two_four(rng, m, k) | (rng.random((m, k)) < 5e-4)
    mask[5] = False
    ro_np = np.concatenate([[0], np.cumsum(mask.sum(1))]).astype(np.int32)
    csr = W.CSR(m, k, rng.standard_normal(ro_np[-1]).astype(np.float32), W.swizzle_from_offsets(ro_np), ro_np, np.nonzero(mask)[1].astype(np.int32))
    _, v, ro, ci = to_dev(csr, dev, dtype, idtype)
    x = torch.randn(k, n, device=dev, generator=torch.Generator(dev).manual_seed(kind)).to(dtype)
    rows = torch.repeat_interleave(torch.arange(m, device=dev), (ro[1:] - ro[:-1]).long())

    def close(out):
        a = torch.zeros(m, k, device=dev)
        a[rows, ci.long()] = v.float()
        want, scale = a.double() @ x.double(), a.abs() @ x.float().abs()
        # the result's rounding, and at most k roundings of a sum in fp32, each 2^-24 of the magnitudes
        return bool(((out.double() - want).abs() <= (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * want.abs() + k * 2.0 ** -24 * scale).all())

    form = pyops.WeightForm(v, ro, ci, m, k)
    kept = form.product(x)
    assert f"two_four_kernel<{'f16' if dtype == torch.float16 else 'bf16'}> ({kind} x" in _lib.last_kernels()
    assert close(kept)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        replayed = form.product(x)
    assert f"({kind} x" in _lib.last_kernels()
    for _ in range(3):
        replayed.zero_()
        graph.replay()
        assert torch.equal(replayed, kept) and torch.equal(form.product(x), kept)
    lens = np.diff(ro_np)
    first = rng.integers(0, k - lens + 1)                    # every row's entries side by side, from some column on
    ci.copy_(torch.from_numpy(np.concatenate([np.arange(f, f + c) for f, c in zip(first, lens)])).to(dev))
    v.mul_(-0.5)
    assert not form.is_of(v, ro, ci) and form.serve(v, ro, ci, x, None, 0) is False
    for _ in range(3):
        replayed.zero_()
        graph.replay()
        assert close(replayed)
    again = pyops.WeightForm(v, ro, ci, m, k)
    out = again.product(x)
    assert out is None or close(out)


def _layer(dev, hidden=256, mlp=512, seed=0, **options):
    rng = np.random.default_rng(seed)
    weights = {}
    for name, (m, k) in {**{x: (hidden, hidden) for x in "qkvo"}, "gate": (mlp, hidden), "up": (mlp, hidden), "down": (hidden, mlp)}.items():
        csr = _csr(rng, m, k, "2:4" if len(name) == 1 else 0.2)
        weights[name] = W.CSR(m, k, csr.values * 0.05, csr.row_indices, csr.row_offsets, csr.column_indices)
    return SparseDecoderLayer(weights, hidden, hidden // 64, mlp, dev, **options)


def test_layer_by_forms_follows_its_weights(dev):
    """By what was laid out and by the operators: the same result up to rounding, also after a weight was changed in place or replaced;
    replays of a captured call give the same bits and follow the weights, too; a kernel_params block and a gradient keep to the operators."""
    layer = _layer(dev)
    x = torch.randn(256, 1024, device=dev).half()

    def by_operators():
        with pyops.kernel_params(gemm={"tile": 13}):
            return layer.forward(x, 2)

    first = layer.forward(x, 2)
    assert torch.allclose(first.float(), by_operators().float(), rtol=2e-2, atol=2e-2)
    layer.w["q"][1].mul_(3.0)
    ri, v, ro, ci, m = layer.w["down"]
    layer.w["down"] = (ri, v * 0.5, ro, ci, m)
    second = layer.forward(x, 2)
    assert not torch.allclose(second.float(), first.float(), rtol=2e-2, atol=2e-2)
    assert torch.allclose(second.float(), by_operators().float(), rtol=2e-2, atol=2e-2)
    assert torch.equal(layer.forward(x, 2), second)
    assert layer._by_form("q", x.clone().requires_grad_()) is None and layer._by_form("q", x[:, :1021].contiguous()) is None
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer.forward(x, 2)
    for factor in (1.0, 0.25, 2.0):
        layer.w["gate"][1].mul_(factor)
        graph.replay()
        assert torch.equal(out, layer.forward(x, 2))


def _by_operators(layer, x, call=None):
    with pyops.kernel_params(gemm={"tile": 13}):
        return layer.forward(x, 2) if call is None else call("q", x)


def _follows(layer, x):
    """The layer's result is that of the operators on the weights as they are now, and another than before."""
    got, want = layer.forward(x, 2).float(), _by_operators(layer, x).float()
    return bool((got - want).norm() < 2e-3 * want.norm())


def test_projections_where_the_dispatcher_is_followed(dev):
    """A form serves calls past the dispatcher: not where a transform has wrapped the operand, or somebody follows the operators called."""
    layer = _layer(dev)
    xs = torch.randn(3, 256, 1024, device=dev).half()
    want = torch.stack([_by_operators(layer, x, layer.proj) for x in xs])
    assert layer._by_form("q", xs[0]) is not None
    assert torch.equal(torch.vmap(lambda x: layer.proj("q", x))(xs), want)
    assert torch.equal(torch.func.jvp(lambda x: layer.proj("q", x), (xs[0],), (xs[1],))[0], want[0])

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, function, types, args=(), kwargs=None):
            seen.append(str(function))
            return function(*args, **(kwargs or {}))

    seen = []
    with Names():
        out = layer.proj("q", xs[0])
    assert torch.equal(out, want[0]) and any("spmm_sputnik_reuse_weight_half" in name for name in seen)
    traced = torch.jit.trace(lambda x: layer.proj("q", x), xs[0], check_trace=False)
    assert torch.equal(traced(xs[1]), want[1])


def test_layer_under_inference_mode_follows_its_weights(dev):
    """Built, changed in place and given replaced weights under inference mode, where tensors count no changes: a relative error of 3e-2
    where a weight is stale, of 1e-4 (fp16 results rounded after sums in another order) where not."""
    with torch.inference_mode():
        layer = _layer(dev)
        x = torch.randn(256, 1024, device=dev).half()
        assert _follows(layer, x) and layer._by_form("q", x) is not None
        layer.w["q"][1].mul_(3.0)
        layer.w["down"][1].mul_(0.1)
        assert _follows(layer, x)
        ri, v, ro, ci, m = layer.w["down"]
        layer.w["down"] = (ri, v * 10.0, ro, ci, m)
        assert layer.w["down"][1].is_inference() and _follows(layer, x)
        layer.w["down"][1].mul_(0.1)
        assert _follows(layer, x) and layer._by_form("down", torch.randn(512, 1024, device=dev).half()) is None
        form = pyops.WeightForm(layer.w["down"][1], ro, ci, m, 512)
        assert not form.is_of(layer.w["down"][1], ro, ci)
    layer.w["q"][1].mul_(0.5)
    assert _follows(layer, x)


def test_writes_that_no_counter_shows(dev):
    """Through .data and by a replayed graph, values and patterns: followed after lay_out_weights, and without it by a layer that keeps
    no forms."""
    layer, plain = _layer(dev), _layer(dev, keep_forms=False)
    x = torch.randn(256, 1024, device=dev).half()
    assert _follows(plain, x) and plain._by_form("q", x) is None
    for it in (layer, plain):
        it.w["down"][1].data.mul_(0.1)
    assert _follows(plain, x)
    layer.lay_out_weights(["down"])
    assert _follows(layer, x) and layer._by_form("q", x) is not None
    assert torch.allclose(plain.forward(x, 2).float(), layer.forward(x, 2).float(), rtol=2e-2, atol=2e-2)
    for it in (layer, plain):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            it.w["gate"][1].mul_(3.0)
        seen = it.w["gate"][1]._version        # (the counter shows the recording, not the replay)
        it.forward(x, 2)
        graph.replay()
        assert it.w["gate"][1]._version == seen
    assert _follows(plain, x)
    layer.lay_out_weights()
    assert _follows(layer, x)
    # a pattern: the columns of every row in reverse, with them the values (same matrix, no canonical CSR)
    ri, v, ro, ci, m = layer.w["up"]
    order = torch.cat([torch.arange(e - 1, s - 1, -1) for s, e in zip(ro.tolist()[:-1], ro.tolist()[1:])]).to(dev)
    before = layer.forward(x, 2)
    ci.data.copy_(ci[order].clone())
    v.data.copy_(v[order].clone())
    layer.lay_out_weights(["up"])
    assert layer._by_form("up", x) is None and _follows(layer, x)
    assert torch.allclose(layer.forward(x, 2).float(), before.float(), rtol=2e-2, atol=2e-2)
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        with pytest.raises(RuntimeError):
            layer.lay_out_weights()


def test_a_replaced_weight_on_another_stream(dev):
    """A weight is replaced while a pass on another stream has not run yet: the memory of what was laid out is not handed out before."""
    layer = _layer(dev)
    x = torch.randn(256, 1024, device=dev).half()
    want = layer.proj("q", x)
    assert layer._by_form("q", x) is not None
    sizes = [_lib.load().iex_form_bytes(kind, 256, 256, room) for kind in pyops.WeightForm.KINDS for room in range(3)]
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200_000_000)
        out = layer.proj("q", x)
    ri, v, ro, ci, m = layer.w["q"]
    layer.w["q"] = (ri, v * 3.0, ro, ci, m)
    layer.proj("q", x)
    keep = [torch.zeros(n, dtype=torch.uint8, device=dev) for n in sizes for _ in range(4)]
    torch.cuda.synchronize()
    assert torch.equal(out, want) and len(keep) == 48


def test_a_form_is_laid_out_by_the_first_product_that_takes_it(dev):
    """Not before, no other kind, and without a read back to the host once the pattern is known; products on another stream wait for it."""
    layer = _layer(dev)
    x = torch.randn(256, 1024, device=dev).half()
    laid_out = lambda: [form._form.laid_out for form in layer._forms.values()]
    assert laid_out() == [0] * 7
    want = layer.forward(x, 2)
    before = laid_out()
    assert all(bin(bits).count("1") == 1 for bits in before)
    layer.forward(x, 2)
    assert laid_out() == before
    side = torch.cuda.Stream()
    torch.cuda.set_sync_debug_mode("error")
    try:
        for w in layer.w.values():
            w[1].mul_(1.0)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            torch.cuda._sleep(50_000_000)
            first = layer.forward(x, 2)
        second = layer.forward(x, 2)                  # (laid out on the other stream, which has not run yet)
    finally:
        torch.cuda.set_sync_debug_mode("default")
    torch.cuda.synchronize()
    assert torch.equal(first, want) and torch.equal(second, want)


def test_a_form_takes_other_values_of_its_pattern(dev):
    """Changed in place or other tensors, in turn and from two threads; nothing else is taken."""
    layer = _layer(dev)
    _, v, ro, ci, m = layer.w["gate"]
    form = pyops.WeightForm(v, ro, ci, m, 256)
    x = torch.randn(256, 1024, device=dev).half()
    weights = [v, v * 2, v * -0.5]
    want = [pyops.WeightForm(w, ro, ci, m, 256).product(x) for w in weights]
    for i in (1, 2, 0, 0, 1):
        assert torch.equal(form.serve(weights[i], ro, ci, x, None, 0), want[i]) and form.is_of(weights[i], ro, ci)
    v.mul_(2)                                    # (and back: exact)
    assert torch.equal(form.serve(v, ro, ci, x, None, 0), want[1])
    v.mul_(0.5)
    other = v.clone()
    with torch.cuda.graph(torch.cuda.CUDAGraph()):
        assert form.serve(other, ro, ci, x, None, 0) is False
    with torch.inference_mode():
        assert form.serve(v.clone(), ro, ci, x, None, 0) is False
    assert form.serve(v[1:], ro, ci, x, None, 0) is False and form.serve(v.bfloat16(), ro, ci, x, None, 0) is False
    assert form.serve(v, ro.clone(), ci, x, None, 0) is False and form.serve(v, ro, ci.clone(), x, None, 0) is False
    assert torch.equal(form.serve(v, ro, ci, x, None, 0), want[0])

    def many(stream):
        with torch.cuda.stream(stream):
            return [form.serve(v, ro, ci, x, None, 0) for _ in range(50)]

    torch.cuda.synchronize()
    with ThreadPoolExecutor(2) as pool:
        outs = [out for outs in pool.map(many, (torch.cuda.Stream(), torch.cuda.Stream())) for out in outs]
    torch.cuda.synchronize()
    assert len(outs) == 100 and all(torch.equal(out, want[0]) for out in outs)


def test_forms_are_refused_on_the_host(dev):
    lib = _lib.load()
    one = torch.zeros(1024, dtype=torch.int32, device=dev)
    at = one.data_ptr()
    assert lib.iex_form_bytes(64, 256, 256, 0) == 0 and lib.iex_form_bytes(256, 256, 70000, 0) == 0 and lib.iex_form_bytes(0, 1 << 16, 1 << 16, 0) == 0
    assert lib.iex_form_build(0, 256, 256, 256, 2, at, at, at, 0, at, 1 << 30, at, 1 << 30, None) != 0             # two nonzeros
    assert lib.iex_form_build(0, 256, 256, 256, 5, at, at, at, 0, at, 16, at, 1 << 30, None) != 0                  # no room
    assert lib.iex_form_product(_lib.F16, 256, 256, 256, 12, 0, at, at, None, 0, at, None, 0, None) != 0           # n off 8
    assert lib.iex_form_product(_lib.F32, 256, 256, 256, 16, 0, at, at, None, 0, at, None, 0, None) != 0
    assert lib.iex_form_choose(15, 256, 256, 0, 100, (ctypes.c_int * 3)()) == -1
    fp32 = torch.zeros(8, device=dev)
    assert pyops.WeightForm(fp32, one[:2], one[:8], 1, 16).product(torch.zeros(16, 8, device=dev)) is None
