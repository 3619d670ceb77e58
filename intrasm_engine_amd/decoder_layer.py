"""One sparse transformer decoder layer of LLaMA-7B shape, built only from the operators of
this package -- the workload of benchmark configuration 5.

Every projection is ``W_csr @ X`` (SpMM) with activations stored feature-major
``(features, tokens)``; the attention reads and writes them as they are, scores and
probabilities in registers (heads of 64 or 128; else heads are split off and scores and
context are batched MFMA GEMMs around PyTorch's softmax).  Included element-wise steps,
done by the epilogues of the products before them: SiLU(gate) * up and the two residual
additions.  Not included (the configuration
names none of them): RoPE, normalisation layers, causal masking, KV cache.

Three ways to run the same arithmetic, mirroring how the reference's harness compares
"serialized" with "interleaved" (tests/test_interleaving.py:348-369, 434-476):

  serialized   everything captured on one stream of a ``TorchCUDAGraphConstructor``;
  multistream  the batch is split into two halves that are captured on two streams of one
               graph (two branches joined at the end), so the sparse projections of one half
               can overlap the dense attention of the other;
  fused        the same two halves on one stream; where attention runs as batched GEMMs (heads of
               other sizes than 64 and 128), each of them is launched together with a sparse
               projection of the other half through the horizontally fused kernel; where it is one
               kernel there is nothing to fuse, and the halves run one after the other.
"""
from __future__ import annotations

import math

import torch

from . import interleaving as IL
from . import _iex_host, _lib
from .pytorch import ops as _pyops
from .pytorch.cpp_extensions.cuda_graph_constructor import TorchCUDAGraphConstructor

ops = torch.ops.iex_ops


class SparseDecoderLayer:
    def __init__(self, weights: dict, hidden: int, heads: int, mlp: int, device, index_dtype=torch.int16, keep_forms: bool = True):
        """``weights``: name -> workloads.CSR for q, k, v, o (hidden x hidden), gate, up
        (mlp x hidden), down (hidden x mlp); values are cast to fp16.

        ``w`` holds them on the device: name -> (row_indices, values, row_offsets, column_indices, m).  Eager passes follow
        entries that are replaced and tensors changed by ordinary operations; for writes that no version counter shows
        (``.data``, a replayed graph, a kernel that was given the address) call :meth:`lay_out_weights` afterwards.
        ``keep_forms=False`` keeps no copy of the values (1 to 2 bytes a cell of every weight for each kind of layout that the
        widths at hand take, four at most): every pass then reads the CSR arrays through the operators."""
        self.hidden, self.heads, self.mlp = hidden, heads, mlp
        self.head_dim = hidden // heads
        self.device = device
        # whether the attention kernel serves these heads; the layer then has no dense product of its own, and the steps
        # after its sparse products go into their epilogues
        self._heads_fit = bool(_lib.load().iex_attention_fits(_lib.F16, self.head_dim, 8))
        self.w = {}
        for name, csr in weights.items():
            idt = index_dtype if csr.k <= 32768 else torch.int32
            # (tensors that count their changes, also where the layer is built under inference_mode())
            with torch.inference_mode(False):
                self.w[name] = (torch.from_numpy(csr.row_indices).to(device),
                                torch.from_numpy(csr.values).to(device).half(),
                                torch.from_numpy(csr.row_offsets).to(device),
                                torch.from_numpy(csr.column_indices).to(device).to(idt), csr.m)
        # the weights as the schedules multiply them, laid out by the first pass that takes them (a capture lays them out inside the graph)
        self._keep_forms = keep_forms
        self._forms = {}
        self.lay_out_weights()

    def _inner(self, name: str) -> int:
        return self.mlp if name == "down" else self.hidden

    def _lay_out(self, name: str) -> "_pyops.WeightForm":
        _, v, ro, ci, m = self.w[name]
        return _pyops.WeightForm(v, ro, ci, m, self._inner(name))

    def lay_out_weights(self, names=None) -> None:
        """Take the weights (``names``; all of them) as they are now, patterns included: what was known of them goes, the next
        pass lays them out.  Not under stream capture."""
        if torch.cuda.is_current_stream_capturing():
            raise RuntimeError("lay_out_weights: the current stream is being captured")
        for name in self.w if names is None else names:
            _, _, ro, ci, _ = self.w[name]
            # (looked at here: the layer's schedules run under capture, where a pattern nobody has looked at
            # keeps to the kernels that take columns in any order)
            _pyops.forget_pattern(ci)
            _pyops.prepare_pattern(ro, ci, self._inner(name), tables=False)
            if self._keep_forms:
                self._forms[name] = self._lay_out(name)

    # ---- building blocks ---------------------------------------------------------------
    def _by_form(self, name: str, x: torch.Tensor, other=None, mode: int = 0):
        """The product by what was laid out, of the weight as it is now; None where the operators have to serve it."""
        if not self._keep_forms:
            return None
        _, v, ro, ci, _ = self.w[name]
        out = self._forms[name].serve(v, ro, ci, x, other, mode)
        if out is False:
            if torch.cuda.is_current_stream_capturing() or any(t.is_inference() for t in (v, ro, ci)):
                return None
            form = self._forms[name] = self._lay_out(name)
            out = form.product(x, other, mode)
        return out

    def proj(self, name: str, x: torch.Tensor) -> torch.Tensor:
        """(k, tokens) -> (m, tokens)."""
        out = self._by_form(name, x)
        if out is not None:
            return out
        ri, v, ro, ci, m = self.w[name]
        return ops.spmm_sputnik_reuse_weight_half(x.unsqueeze(0), ri, v, ro, ci, m)[0]

    def _one_attention(self, length: int) -> bool:
        """Whether ``attention`` over sequences of ``length`` tokens is the one kernel: heads and length that it serves, and no
        :func:`ops.kernel_params` block that names the kernels of the products it stands for."""
        return self._heads_fit and not _pyops.kernels_forced() and bool(_lib.load().iex_attention_fits(_lib.F16, self.head_dim, length))

    def _proj_with(self, name: str, x: torch.Tensor, other: torch.Tensor, mode: int):
        """``proj`` combined with ``other`` before it is rounded: plus it (mode 1), times its SiLU (mode 2)."""
        out = self._by_form(name, x, other, mode) if self._heads_fit else None
        if out is not None:
            return out
        ri, v, ro, ci, m = self.w[name]
        out = _iex_host.spmm_with(x, ri, v, ro, ci, m, other, mode) if self._heads_fit else None
        if out is None:
            out = self.proj(name, x)
            out = other + out if mode == 1 else torch.nn.functional.silu(other) * out
        return out

    def _split_heads(self, t: torch.Tensor, seqs: int, scale: float = 1.0) -> torch.Tensor:
        """(hidden, seqs*L) feature-major -> (seqs*heads, L, head_dim), times ``scale`` in the same pass."""
        L = t.shape[1] // seqs
        src = t.view(self.heads, self.head_dim, seqs, L).permute(2, 0, 3, 1)
        out = torch.empty((seqs, self.heads, L, self.head_dim), dtype=t.dtype, device=t.device)
        if scale == 1.0:
            out.copy_(src)
        else:
            torch.mul(src, scale, out=out)
        return out.view(seqs * self.heads, L, self.head_dim)

    def _merge_heads(self, o: torch.Tensor, seqs: int) -> torch.Tensor:
        """(seqs*heads, L, head_dim) -> (hidden, seqs*L)."""
        L = o.shape[1]
        return o.view(seqs, self.heads, L, self.head_dim).permute(1, 3, 0, 2).contiguous().view(
            self.hidden, seqs * L)

    def _softmax(self, s: torch.Tensor) -> torch.Tensor:
        """Over keys; the scores arrive scaled (1/sqrt(d) is folded into Q where the heads are split),
        so this is one pass: fp16 in, fp32 inside the kernel, fp16 out."""
        return torch.softmax(s, dim=-1)

    def _split_qkv(self, q, k, v, seqs: int):
        return (self._split_heads(q, seqs, 1.0 / math.sqrt(self.head_dim)), self._split_heads(k, seqs),
                self._split_heads(v, seqs))

    def attention(self, q, k, v, seqs: int) -> torch.Tensor:
        out = _iex_host.attention(q, k, v, self.heads, seqs, 1.0 / math.sqrt(self.head_dim)) if self._heads_fit else None
        if out is not None:
            return out
        Q, K, V = self._split_qkv(q, k, v, seqs)
        P = self._softmax(ops.gemm_mfma(Q, K, True))      # (B, L, L)
        return self._merge_heads(ops.gemm_mfma(P, V, False), seqs)

    def mlp_block(self, h: torch.Tensor) -> torch.Tensor:
        return self._proj_with("down", self._proj_with("up", h, self.proj("gate", h), 2), h, 1)

    def forward(self, x: torch.Tensor, seqs: int) -> torch.Tensor:
        """x: (hidden, seqs*L) fp16, contiguous -> same shape."""
        q, k, v = self.proj("q", x), self.proj("k", x), self.proj("v", x)
        h = self._proj_with("o", self.attention(q, k, v, seqs), x, 1)
        return self.mlp_block(h)

    # ---- fused schedule over two half-batches ----------------------------------------------
    def _fused(self, name: str, x: torch.Tensor, ga: torch.Tensor, gb: torch.Tensor, trans_b: bool, group):
        ri, v, ro, ci, m = self.w[name]
        out, c = ops.fused_spmm_gemm(x.unsqueeze(0), ri, v, ro, ci, m, ga, gb, trans_b, group)
        return out[0], c

    def forward_fused(self, xa: torch.Tensor, xb: torch.Tensor, seqs_half: int, group=None):
        """Halves a and b of the batch; the dense GEMMs of one half ride along with sparse
        projections of the other half, in the order that ``group`` names.  Where attention is one kernel there are none, and
        the halves go one after the other whatever ``group`` is (16 x 512 tokens, hidden 4096: 4.4 ms by fused launches before
        that kernel, 2.8 now)."""
        if self._one_attention(xa.shape[1] // seqs_half):
            return self.forward(xa, seqs_half), self.forward(xb, seqs_half)
        qa, ka, va = self.proj("q", xa), self.proj("k", xa), self.proj("v", xa)
        Qa, Ka, Va = self._split_qkv(qa, ka, va, seqs_half)
        qb, Sa = self._fused("q", xb, Qa, Ka, True, group)              # b.q  ||  a.QK^T
        Pa = self._softmax(Sa)
        kb, Oa = self._fused("k", xb, Pa, Va, False, group)             # b.k  ||  a.PV
        vb = self.proj("v", xb)
        Qb, Kb, Vb = self._split_qkv(qb, kb, vb, seqs_half)
        oa, Sb = self._fused("o", self._merge_heads(Oa, seqs_half), Qb, Kb, True, group)   # a.o  ||  b.QK^T
        ha = xa + oa
        Pb = self._softmax(Sb)
        ga, Ob = self._fused("gate", ha, Pb, Vb, False, group)          # a.gate  ||  b.PV
        acta = torch.nn.functional.silu(ga) * self.proj("up", ha)
        ya = ha + self.proj("down", acta)
        hb = xb + self.proj("o", self._merge_heads(Ob, seqs_half))
        return ya, self.mlp_block(hb)

    # ---- the three timed variants --------------------------------------------------------
    def capture_serialized(self, x: torch.Tensor, seqs: int):
        return IL.capture_serialized([lambda: self.forward(x, seqs)])

    def capture_multistream(self, xa: torch.Tensor, xb: torch.Tensor, seqs_half: int):
        return IL.capture_interleaved([lambda: self.forward(xa, seqs_half)], [lambda: self.forward(xb, seqs_half)])

    def capture_fused(self, xa: torch.Tensor, xb: torch.Tensor, seqs_half: int, group=None):
        return IL.capture_serialized([lambda: self.forward_fused(xa, xb, seqs_half, group)])
