"""What a user of the framework has it do, as cases that can be timed one by one.

Eight kinds of work, each through the public entry points: the two sparse products on their own, products with values
per batch entry, sparse attention, training steps of a sparse and of a dense layer, a sparse and a dense product side
by side on two branches of one graph, and a whole decoder layer.  ``listed()`` names twelve of them, ``draw()`` gives
more of the same ranges.
"""
import math

import numpy as np
import torch

from intrasm_engine_amd import interleaving as IL
from intrasm_engine_amd import workloads as W
from intrasm_engine_amd.decoder_layer import SparseDecoderLayer
from intrasm_engine_amd.pytorch.cpp_extensions.layers_and_funcs.sputnik import spmm as trainable_spmm
from intrasm_engine_amd.pytorch.cpp_extensions.layers_and_funcs.torch import linear as trainable_linear
from intrasm_engine_amd.pytorch.sparse_attention import sparse_attention
from intrasm_engine_amd.pytorch.utils import dense_to_sparse, to_int16_indices, transpose_info

ops = torch.ops.iex_ops
DTYPES = {"fp32": torch.float32, "fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one sparse product of a small layer: the smallest call, where latency and launches are what counts
        {"name": "spmm_fp32_1024", "kind": "spmm", "dtype": "fp32", "index": "int32", "m": 1024, "k": 1024, "n": 256, "sparsity": 0.90,
         "rows": "equal"},
        # ... of a 4096 x 4096 weight with rows of very different lengths: a cell of the benchmark's sweep
        {"name": "spmm_fp32_4096", "kind": "spmm", "dtype": "fp32", "index": "int32", "m": 4096, "k": 4096, "n": 256, "sparsity": 0.80,
         "rows": "geometric"},
        # ... the same sweep in half precision with 16-bit indices, at another width and sparsity
        {"name": "spmm_fp16_4096", "kind": "spmm", "dtype": "fp16", "index": "int16", "m": 4096, "k": 4096, "n": 128, "sparsity": 0.90,
         "rows": "geometric"},
        # the sampled product of the same small layer
        {"name": "sddmm_fp32_1024", "kind": "sddmm", "dtype": "fp32", "m": 1024, "n": 1024, "k": 64, "batch": 1, "sparsity": 0.90},
        # attention of one layer over a mask with a band and scattered columns
        {"name": "attention_fp16_4096", "kind": "attention", "dtype": "fp16", "heads": 16, "tokens": 4096, "d": 64, "band": 256, "extra": 32,
         "causal": False},
        # ... over a short prompt of no round length, with a causal window
        {"name": "attention_bf16_1000", "kind": "attention", "dtype": "bf16", "heads": 8, "tokens": 1000, "d": 64, "band": 256, "extra": 0,
         "causal": True},
        # values per batch entry and a wide output: a point of the vision-transformer sweep, rows of no round length
        {"name": "batched_fp32_785", "kind": "batched", "dtype": "fp32", "batch": 384, "m": 785, "k": 64, "sparsity": 0.90},
        # a training step (forward and both gradients) of a small sparse layer with odd sizes
        {"name": "train_fp32_1000", "kind": "train", "dtype": "fp32", "m": 1000, "k": 777, "n": 129, "sparsity": 0.90},
        # ... of a pruned 11008 x 4096 projection in half precision
        {"name": "train_fp16_11008", "kind": "train", "dtype": "fp16", "m": 11008, "k": 4096, "n": 2048, "sparsity": 0.90},
        # a training step of the dense companion layer
        {"name": "linear_bf16_4096", "kind": "linear", "dtype": "bf16", "tokens": 2048, "inner": 4096, "outer": 4096},
        # the sparse projection beside the dense one, recorded once and replayed: two branches of one graph
        {"name": "corun_11008", "kind": "corun", "m": 11008, "k": 4096, "n": 2048, "sparsity": 0.90, "gm": 4096, "gk": 4096},
        # the whole decoder layer, 16 sequences of 512 tokens: the largest
        {"name": "layer_4096", "kind": "layer", "hidden": 4096, "mlp": 11008, "seqs": 16, "length": 512},
    ]


def _between(rng, low, high, step=8):
    """A size, its logarithm spread over the range: half of them any whole number, half multiples of ``step``."""
    v = math.exp(rng.uniform(math.log(low), math.log(high)))
    if rng.random() < 0.5 and v >= 2 * step:
        return int(min(high, max(step, round(v / step) * step)))
    return int(min(high, max(low, round(v))))


def _multiple(rng, low, high, step):
    return int(max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))) / step) * step))


def draw(rng):
    kind = rng.choice(("spmm", "spmm", "sddmm", "attention", "batched", "train", "train", "linear", "corun", "layer"))
    if kind == "spmm":
        dtype = rng.choice(("fp32", "fp16", "bf16"))
        while True:
            c = {"kind": kind, "dtype": dtype, "index": rng.choice(("int16", "int32")) if dtype == "fp16" else "int32",
                 "m": _between(rng, 256, 11008), "k": _between(rng, 256, 11008), "n": _between(rng, 8, 2048),
                 "sparsity": round(rng.uniform(0.70, 0.98), 3), "rows": rng.choice(("equal", "geometric", "pruned"))}
            if c["m"] * c["k"] <= 11008 * 4096 and c["m"] * c["k"] * (1 - c["sparsity"]) * c["n"] <= 4e9:
                return c
    if kind == "sddmm":
        return {"kind": kind, "dtype": rng.choice(("fp32", "fp32", "fp16")), "m": _between(rng, 256, 4096), "n": _between(rng, 256, 4096),
                "k": _between(rng, 16, 256), "batch": rng.choice((1, 1, 2, 4)), "sparsity": round(rng.uniform(0.80, 0.98), 3)}
    if kind == "attention":
        return {"kind": kind, "dtype": rng.choice(("fp16", "bf16", "fp32")), "heads": rng.choice((4, 8, 12, 16, 32)), "tokens": _between(rng, 256, 4096),
                "d": rng.choice((32, 64, 64, 128)), "band": rng.choice((64, 128, 256, 512)), "extra": rng.choice((0, 16, 32)),
                "causal": rng.random() < 0.5}
    if kind == "batched":
        while True:
            c = {"kind": kind, "dtype": rng.choice(("fp32", "fp32", "fp16")), "batch": _between(rng, 8, 384), "m": _between(rng, 49, 3136),
                 "k": rng.choice((32, 64, 128)), "sparsity": round(rng.uniform(0.70, 0.99), 3)}
            if c["batch"] * c["m"] ** 2 <= 2.6e8:
                return c
    if kind == "train":
        while True:
            c = {"kind": kind, "dtype": rng.choice(("fp32", "fp16", "bf16")), "m": _between(rng, 256, 11008), "k": _between(rng, 256, 11008),
                 "n": _between(rng, 16, 2048), "sparsity": round(rng.uniform(0.80, 0.98), 3)}
            if c["m"] * c["k"] <= 11008 * 4096 and c["m"] * c["k"] * (1 - c["sparsity"]) * c["n"] <= 2e9:
                return c
    if kind == "linear":
        return {"kind": kind, "dtype": rng.choice(("bf16", "fp16")), "tokens": _multiple(rng, 16, 4096, 8), "inner": _multiple(rng, 256, 8192, 8),
                "outer": _multiple(rng, 256, 8192, 8)}
    if kind == "corun":
        return {"kind": kind, "m": _multiple(rng, 1024, 11008, 8), "k": _multiple(rng, 1024, 4096, 8), "n": _multiple(rng, 128, 2048, 8),
                "sparsity": round(rng.uniform(0.80, 0.95), 3), "gm": _multiple(rng, 1024, 4096, 8), "gk": _multiple(rng, 1024, 4096, 8)}
    hidden = rng.choice((512, 1024, 2048, 4096))
    return {"kind": "layer", "hidden": hidden, "mlp": hidden // 16 * 43, "seqs": rng.choice((1, 2, 4, 8, 16)), "length": _multiple(rng, 64, 512, 8)}


# ---------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _mask(g, m, k, sparsity, rows):
    """Which entries of an m x k matrix are stored: the same number in every row, or row lengths that follow a geometric
    distribution."""
    keys = torch.rand(m, k, device="cuda", generator=g)
    mean = max(1.0, k * (1 - sparsity))
    if rows == "equal":
        lengths = torch.full((m,), round(mean), device="cuda")
    else:
        u = torch.rand(m, device="cuda", generator=g).clamp_(1e-6, 1 - 1e-6)
        lengths = (torch.log(u) / math.log1p(-1.0 / max(mean, 1.0001))).ceil().clamp_(1, k)
        lengths = (lengths * (mean * m / lengths.sum())).round().clamp_(1, k)
    last = keys.sort(dim=1).values.gather(1, lengths.long().clamp(1, k)[:, None] - 1)
    return keys <= last


def _largest(w, sparsity):
    """The matrix with all but its largest magnitudes set to zero (as many of them for every matrix of this size)."""
    flat = w.view(-1)
    keep = flat.abs().argsort(descending=True)[:_kept(w.shape[0], w.shape[1], sparsity)]
    return torch.zeros_like(flat).index_copy_(0, keep, flat[keep]).view_as(w)


def _kept(m, k, sparsity):
    return max(1, round(m * k * (1 - sparsity)))


def _weight(g, m, k, sparsity, rows, dtype):
    w = torch.randn(m, k, device="cuda", generator=g) * 0.02
    return (_largest(w, sparsity) if rows == "pruned" else w * _mask(g, m, k, sparsity, rows)).to(dtype)


def _two_four(g, m, k):
    """A weight of which the two largest of every four neighbours stay."""
    w = torch.randn(m, k // 4, 4, device="cuda", generator=g) * 0.02
    keep = torch.zeros_like(w).scatter_(2, w.abs().topk(2, dim=2).indices, 1.0)
    return (w * keep).view(m, k).half()


def _attention_mask(g, c):
    i = torch.arange(c["tokens"], device="cuda")
    away = i[:, None] - i[None, :]
    mask = (away >= 0) & (away < c["band"]) if c["causal"] else away.abs() < c["band"] // 2
    if c["extra"]:
        columns = torch.randint(0, c["tokens"], (c["tokens"], c["extra"]), device="cuda", generator=g)
        mask = mask.scatter(1, columns, True)
        if c["causal"]:
            mask &= away >= 0
    return mask


def _on_host(weight):
    """The weight as the decoder layer takes it: CSR arrays in host memory."""
    values, row_indices, row_offsets, column_indices = (t.cpu().numpy() for t in dense_to_sparse(weight))
    return W.CSR(weight.shape[0], weight.shape[1], values.astype(np.float32), row_indices, row_offsets, column_indices)


def prepare(case, seed):
    g, kind = _generator(seed), case["kind"]
    dtype = DTYPES[case.get("dtype", "fp16")]

    def normal(*shape, dtype=dtype):
        return torch.randn(*shape, device="cuda", generator=g).to(dtype)

    s = {"kind": kind}
    if kind == "spmm":
        s["m"] = case["m"]
        s["values"], s["row_indices"], s["row_offsets"], columns = dense_to_sparse(
            _weight(g, case["m"], case["k"], case["sparsity"], case["rows"], dtype))
        s["columns"] = to_int16_indices(columns, case["k"]) if case["index"] == "int16" else columns
        s["b"] = normal(1, case["k"], case["n"])
    elif kind == "sddmm":
        _, s["row_indices"], s["row_offsets"], s["columns"] = dense_to_sparse(
            _weight(g, case["m"], case["n"], case["sparsity"], "pruned", torch.float32))
        s["lhs"], s["rhs"] = normal(case["batch"], case["m"], case["k"]), normal(case["batch"], case["n"], case["k"])
        s["summed"] = case["dtype"] == "fp32"
    elif kind == "attention":
        _, s["row_indices"], s["row_offsets"], s["columns"] = dense_to_sparse(_attention_mask(g, case).float())
        s["q"], s["k"], s["v"] = (normal(case["heads"], case["tokens"], case["d"]) for _ in range(3))
    elif kind == "batched":
        s["m"] = case["m"]
        _, s["row_indices"], s["row_offsets"], s["columns"] = dense_to_sparse(
            _weight(g, case["m"], case["k"], case["sparsity"], "pruned", torch.float32))
        s["values"] = torch.rand(case["batch"], s["columns"].numel(), device="cuda", generator=g).to(dtype)
        s["b"] = torch.rand(case["batch"], case["k"], case["m"], device="cuda", generator=g).to(dtype)
    elif kind == "train":
        s["m"] = case["m"]
        s["values"], s["row_indices"], s["row_offsets"], s["columns"] = dense_to_sparse(
            _weight(g, case["m"], case["k"], case["sparsity"], "pruned", dtype))
        s["transposed"] = transpose_info(case["m"], case["k"], s["row_offsets"], s["columns"])
        s["b"] = normal(case["k"], case["n"]).requires_grad_()
        s["values"].requires_grad_()
        s["gradient"] = normal(case["m"], case["n"])
    elif kind == "linear":
        s["x"] = normal(case["tokens"], case["inner"]).requires_grad_()
        s["weight"] = (torch.randn(case["outer"], case["inner"], device="cuda", generator=g) * 0.02).to(dtype).requires_grad_()
        s["gradient"] = normal(case["tokens"], case["outer"])
    elif kind == "corun":
        values, row_indices, row_offsets, columns = dense_to_sparse(_weight(g, case["m"], case["k"], case["sparsity"], "pruned", torch.float16))
        columns = to_int16_indices(columns, case["k"])
        b = normal(1, case["k"], case["n"], dtype=torch.float16)
        ga, gb = normal(case["gm"], case["gk"], dtype=torch.bfloat16), normal(case["gk"], case["n"], dtype=torch.bfloat16)
        s["graph"], s["outputs"] = IL.capture_interleaved(
            [lambda: ops.spmm_sputnik_reuse_weight_half(b, row_indices, values, row_offsets, columns, case["m"])],
            [lambda: ops.gemm_mfma(ga, gb, False)])
        s["graph"].instantiate_graph_exec()
        s["inputs"] = (values, row_indices, row_offsets, columns, b, ga, gb)
    else:
        h, mlp = case["hidden"], case["mlp"]
        weights = {name: _on_host(_two_four(g, h, h)) for name in ("q", "k", "v", "o")}
        for name in ("gate", "up"):
            weights[name] = _on_host(_weight(g, mlp, h, 0.80, "pruned", torch.float16))
        weights["down"] = _on_host(_weight(g, h, mlp, 0.80, "pruned", torch.float16))
        s["layer"] = SparseDecoderLayer(weights, h, h // 128, mlp, torch.device("cuda", 0))
        s["seqs"] = case["seqs"]
        s["x"] = normal(h, case["seqs"] * case["length"]).relu_()
    return s


# ---------------------------------------------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "spmm":
        op = ops.spmm_sputnik_reuse_weight if s["b"].dtype == torch.float32 else ops.spmm_sputnik_reuse_weight_half
        return op(s["b"], s["row_indices"], s["values"], s["row_offsets"], s["columns"], s["m"])
    if kind == "sddmm":
        op = ops.sddmm_sputnik_atomic_upd_weight if s["summed"] else ops.sddmm_sputnik_half
        return op(s["lhs"], s["rhs"], s["row_indices"], s["row_offsets"], s["columns"])
    if kind == "attention":
        return sparse_attention(s["q"], s["k"], s["v"], s["row_indices"], s["row_offsets"], s["columns"])
    if kind == "batched":
        return ops.spmm_sputnik_batched_values(s["b"], s["row_indices"], s["values"], s["row_offsets"], s["columns"], s["m"])
    if kind == "train":
        out = trainable_spmm(s["b"], s["row_indices"], s["values"], s["row_offsets"], s["columns"], s["m"], s["transposed"])
        return (out, *torch.autograd.grad(out, (s["b"], s["values"]), s["gradient"]))
    if kind == "linear":
        out = trainable_linear(s["x"], s["weight"])
        return (out, *torch.autograd.grad(out, (s["x"], s["weight"]), s["gradient"]))
    if kind == "corun":
        s["graph"].execute_graph()
        return s["outputs"]
    return s["layer"].forward(s["x"], s["seqs"])


# ---------------------------------------------------------------------------------------------------- what a pass is
def _band_nonzeros(c):
    t, band = c["tokens"], min(c["band"], c["tokens"])
    if c["causal"]:
        inside = t * band - band * (band - 1) // 2
        return int(inside + 0.5 * t * c["extra"])
    half = min(band // 2, t)
    return int((2 * half - 1) * t - half * (half - 1) + t * c["extra"])


def work(case):
    kind = case["kind"]
    sv = 4 if case.get("dtype") == "fp32" else 2
    if kind == "spmm":
        nnz = _kept(case["m"], case["k"], case["sparsity"])
        return {"bytes": W.spmm_bytes(case["m"], case["k"], case["n"], nnz, 1, sv, 2 if case["index"] == "int16" else 4),
                "flops": W.spmm_flops(nnz, case["n"])}
    if kind == "sddmm":
        nnz = _kept(case["m"], case["n"], case["sparsity"])
        return {"bytes": W.sddmm_bytes(case["m"], case["k"], case["n"], nnz, case["batch"], sv, sv == 4),
                "flops": W.sddmm_flops(nnz, case["k"], case["batch"])}
    if kind == "attention":
        nnz = _band_nonzeros(case)
        return {"bytes": 4 * case["heads"] * case["tokens"] * case["d"] * sv + nnz * 4 + case["tokens"] * 8,
                "flops": 2 * W.spmm_flops(nnz, case["d"], case["heads"])}
    if kind == "batched":
        nnz = _kept(case["m"], case["k"], case["sparsity"])
        return {"bytes": W.spmm_bytes(case["m"], case["k"], case["m"], nnz, case["batch"], sv, 4, True),
                "flops": W.spmm_flops(nnz, case["m"], case["batch"])}
    if kind == "train":
        nnz = _kept(case["m"], case["k"], case["sparsity"])
        # values, their gradient and one set of indices; the activations, the output and a gradient of each
        return {"bytes": nnz * (2 * sv + 4) + (case["m"] + case["k"]) * 8 + 2 * (case["m"] + case["k"]) * case["n"] * sv,
                "flops": 3 * W.spmm_flops(nnz, case["n"])}
    if kind == "linear":
        t, i, o = case["tokens"], case["inner"], case["outer"]
        return {"bytes": 2 * (t * i + t * o + i * o) * sv, "flops": 3 * W.gemm_flops(t, o, i)}
    if kind == "corun":
        nnz = _kept(case["m"], case["k"], case["sparsity"])
        return {"bytes": W.spmm_bytes(case["m"], case["k"], case["n"], nnz, 1, 2, 2) + W.gemm_bytes(case["gm"], case["n"], case["gk"]),
                "flops": W.spmm_flops(nnz, case["n"]) + W.gemm_flops(case["gm"], case["n"], case["gk"])}
    h, mlp, tokens = case["hidden"], case["mlp"], case["seqs"] * case["length"]
    nnz = 4 * h * h // 2 + int(0.2 * 3 * h * mlp)
    return {"bytes": nnz * 4 + 2 * h * tokens * 2, "flops": W.spmm_flops(nnz, tokens) + 4 * tokens * case["length"] * h}


def tolerance(case):
    # 32-bit sums in another order; 16-bit results (and 16-bit values between two products) rounded once more or less
    return {"rel": 1e-5} if case.get("dtype") == "fp32" else {"rel": 1e-2}
