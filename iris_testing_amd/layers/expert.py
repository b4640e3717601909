"""Expert compute with the reference's ``expert`` signature (layers/expert.py:6-66), plus the full
expert MLP the workloads define (Linear-act-Linear, SwiGLU, fp8) which the reference lacks.
"""
from __future__ import annotations

import weakref
from dataclasses import dataclass, field
from typing import Optional

import torch

from .. import _lib as L
from .. import ops
from ..utils import _assert_cuda_int32


# Re-tiled copies of weight tensors the operator has seen (None: seen once, not re-tiled yet), keyed on the tensor's storage and version counter, so that
# a weight that did not change between calls is re-tiled once, not on every call (the re-tiling reads and writes the
# whole tensor).  Entries die with their tensors (weak references); an in-place update bumps the version and re-tiles.
# While a stream is being captured nothing here changes and nothing from here is used: a re-tiling that was only recorded has not
# happened for the next eager call or the next graph, a copy dropped after an update would be freed under the graph, and a graph
# that holds an optimizer's update has to read the weights it left.  A captured call multiplies with the tensors as they are.
_PACKED = {}


def _pack_key(kind: str, w: torch.Tensor, w_up: Optional[torch.Tensor]):
    return (kind, w.data_ptr(), w._version, None if w_up is None else (w_up.data_ptr(), w_up._version), tuple(w.shape), w.dtype, w.device)


def _drop_packs(kind: str, w: torch.Tensor) -> None:
    for k in [k for k, v in _PACKED.items() if v[0]() is None or (v[0]() is w and k[0] == kind)]:
        del _PACKED[k]


def _cached_pack(kind: str, w: torch.Tensor, w_up: Optional[torch.Tensor], build) -> torch.Tensor:
    if L.capturing():
        return build(w, w_up)
    key = _pack_key(kind, w, w_up)
    hit = _PACKED.get(key)
    if hit is not None and hit[0]() is w:
        return hit[1]
    _drop_packs(kind, w)
    packed = build(w, w_up)
    _PACKED[key] = (weakref.ref(w), packed)
    return packed


def _weights_for(w: torch.Tensor, rows: int):
    """(weights, layout) for the forward GEMM on `rows` rows.  The first call with a weight -- or with what an in-place update made of
    it -- multiplies with the tensor as it is (see ExpertWeights.train_weights), the second one, if nothing has changed by
    then, re-tiles it."""
    if L.capturing():
        return w, L.W_RAW
    key = _pack_key("N", w, None)
    hit = _PACKED.get(key)
    if hit is None or hit[0]() is not w:
        _drop_packs("N", w)
        raw = rows < 4096 * w.shape[0] and w.data_ptr() % 16 == 0
        _PACKED[key] = hit = (weakref.ref(w), None if raw else ops.prepack_weights(w))
        if raw:
            return w, L.W_RAW
    elif hit[1] is None:
        _PACKED[key] = hit = (hit[0], ops.prepack_weights(w))
    return hit[1], L.W_TILED


def _packed_weights_t(w: torch.Tensor, w_up: Optional[torch.Tensor] = None) -> torch.Tensor:
    """Re-tiled w^T (with w_up: of the pair, in the fused gate/up column order) for d tokens = d out @ w^T."""
    return _cached_pack("T", w, w_up, ops.prepack_weights_transposed)


def _grouped_gemm_t(do: torch.Tensor, weights: torch.Tensor, cnt: torch.Tensor) -> torch.Tensor:
    """d tokens[rows of g] = do[rows of g] @ weights[g]^T; rows past sum(cnt) are zero."""
    E_l, K, N = weights.shape
    if do.dtype == torch.float32:
        return ops.grouped_gemm(do, ops.transpose_weights_f32(weights.contiguous()), cnt)
    S = do.shape[0]
    # (no whole stages of the reduction; worth a re-tiled copy; or not where the kernel's loads can start)
    if N % 64 or K % 8 or ((S >= 4096 * E_l or weights.data_ptr() % 16) and not L.capturing()):
        out = torch.zeros((S, K), dtype=do.dtype, device=do.device)
        if S:
            ops.grouped_gemm_mapped(do, None, _packed_weights_t(weights), cnt, S, K, "none", out, part_ws=_part_ws(do.device, 2 * N))
        return out
    return ops.expert_forward(do, weights.contiguous(), L.W_RAW_T, cnt, K, _part_ws(do.device, 2 * N))


def _part_ws(device, k_bytes: int = L.MOE_SPLIT_MIN_K_BYTES) -> Optional[torch.Tensor]:
    """Partial-sum workspace for the K split of GEMMs of few tiles, for one call (none where its longest rows, k_bytes of K, are too short to
    be cut): launches that may overlap must not share it, and under capture it has to belong to the graph.  (8 MB of the
    caching allocator's, which costs the host what a lookup did.)"""
    return ops.gemm_part_workspace(device) if k_bytes >= L.MOE_SPLIT_MIN_K_BYTES else None


def _grouped_gemm(tokens: torch.Tensor, weights: torch.Tensor, cnt: torch.Tensor) -> torch.Tensor:
    """out[rows of g] = tokens[rows of g] @ weights[g]; rows past sum(cnt) are zero."""
    if tokens.dtype != torch.bfloat16 or weights.shape[1] % 64 or weights.shape[2] % 8:  # (what the MFMA kernel covers)
        return ops.grouped_gemm(tokens, weights, cnt)
    w, layout = _weights_for(weights, tokens.shape[0])
    return ops.expert_forward(tokens, w, layout, cnt, weights.shape[2], _part_ws(tokens.device, 2 * weights.shape[1]))


class Expert(torch.autograd.Function):

    @staticmethod
    def forward(ctx, tokens, weights, local_expert_cnt, aggregrate_exp_cnt):
        """tokens [S,H], weights [E_local,H,F], local_expert_cnt [E_local] int32, total expert count
        (unused by the math, kept for the signature) -> [S,F] (layers/expert.py:20-29,43,60)."""
        assert tokens.is_cuda, "tokens must be CUDA"
        _assert_cuda_int32(local_expert_cnt, "local_expert_cnt")
        assert weights.shape[0] == local_expert_cnt.numel(), "one row count per local expert"
        ctx.save_for_backward(tokens, weights, local_expert_cnt)
        return _grouped_gemm(ops.aligned16(tokens.contiguous()), weights.contiguous(), local_expert_cnt.contiguous())

    @staticmethod
    def backward(ctx, do):
        """Gradients of out[rows of g] = tokens[rows of g] @ weights[g] (not implemented in the reference,
        layers/expert.py:62-64), both as grouped launches over all experts:
          d tokens[rows of g] = do[rows of g] @ weights[g]^T        the grouped GEMM over the transposed, re-tiled weights
          d weights[g]        = tokens[rows of g]^T @ do[rows of g]  the grouped GEMM in its weight-gradient mode: the
                                                                      reduction runs over the expert's (ragged) rows
        Rows past the counted total get a zero gradient, experts without rows a zero weight gradient."""
        tokens, weights, cnt = ctx.saved_tensors
        do = ops.aligned16(do.contiguous())
        cnt = cnt.contiguous()
        d_tokens = _grouped_gemm_t(do, weights, cnt)
        d_weights = ops.grouped_gemm_dw(tokens.contiguous(), do, cnt)
        return d_tokens, d_weights, None, None


expert = Expert.apply


@dataclass
class ExpertWeights:
    """Weights of the local experts, prepared once for the kernels.

    act in {"gelu","silu"}: y = act(x W1) W2.  act == "swiglu": y = (silu(x Wg) * (x Wu)) Wd.
    bf16: re-tiled for the MFMA kernels; fp32: reference layout; fp8: e4m3 codes + per-channel scales.
    """
    act: str
    hidden: int
    ffn: int
    e_local: int
    dtype: torch.dtype
    w1: torch.Tensor
    w2: torch.Tensor
    w_up: Optional[torch.Tensor] = None
    scales: Optional[tuple] = None  # fp8: (sg, su, sd)
    # the tensors prepare() was given, in the reference layout: (w1, w2, w_up); the backward pass differentiates with
    # respect to them and multiplies with them as they are
    raw: Optional[tuple] = field(default=None, repr=False)
    # version counters of the raw tensors when w1 / w2 / w_up were last derived from them (refresh() compares)
    raw_versions: Optional[tuple] = field(default=None, repr=False)
    seen_versions: Optional[tuple] = field(default=None, repr=False)  # ... when train_weights() last looked at them
    copies: tuple = field(default=(None, None, None), repr=False)  # those of w1, w2, w_up that are copies made here

    @staticmethod
    def _derive(raw, copies=(None, None, None)):
        """((w1, w2, w_up) as the kernels take them, the copies among them), from the tensors in the reference layout; ``copies``:
        those made before, which are written again."""
        w1, w2, w_up = (None if t is None else t.detach() for t in raw)
        if w1.dtype == torch.float32:
            copies = tuple(None if t is None or t.is_contiguous() else t.contiguous() if c is None else c.copy_(t)
                           for t, c in zip((w1, w2, w_up), copies))
            return tuple(t if c is None else c for t, c in zip((w1, w2, w_up), copies)), copies
        copies = (ops.prepack_weights(w1.contiguous(), None if w_up is None else w_up.contiguous(), out=copies[0]),
                  ops.prepack_weights(w2.contiguous(), out=copies[1]), None)
        return copies, copies

    @staticmethod
    def _versions(raw):
        return tuple(None if t is None else t._version for t in raw)

    @classmethod
    def prepare(cls, act: str, w1: torch.Tensor, w2: torch.Tensor, w_up: Optional[torch.Tensor] = None):
        e_l, H, F = w1.shape
        raw = (w1, w2, w_up)
        (p1, p2, pu), copies = cls._derive(raw)
        return cls(act, H, F, e_l, w1.dtype, p1, p2, pu, raw=raw, raw_versions=cls._versions(raw), copies=copies)

    def refresh(self) -> "ExpertWeights":
        """Derive the kernels' copies again if a tensor prepare() was given has been updated in place since (an optimizer
        step): the forward pass would otherwise multiply with the weights of before the update while the backward pass,
        which takes the tensors as they are, uses the new ones.  The copies stay where they are (a captured step holds their
        addresses).  Under capture the derivation is recorded, to happen on every replay, and not counted as done."""
        if self.raw is not None and self._versions(self.raw) != self.raw_versions:
            now = self._versions(self.raw)
            (self.w1, self.w2, self.w_up), self.copies = self._derive(self.raw, self.copies)
            if not L.capturing():
                self.raw_versions = now
        return self

    def train_weights(self, rows: int):
        """(layout, w1, w_up, w2) for the forward pass of a bf16 training step on `rows` rows.  Weights that an optimizer has updated
        since they were re-tiled are taken as they are if the rows per expert are few: the GEMMs read the reference layout at 0.88 to
        0.96 of the rate, which costs more than re-tiling (reading and writing every weight in either direction) from some 4000
        rows per expert on.  If they are still the same on the next call, they are re-tiled after all.  A captured call takes them as
        they are (see _PACKED): its replays may come after updates that nobody on the host sees."""
        if L.capturing():
            w1, w2, w_up = (None if t is None else t.detach().contiguous() for t in self.raw)
            return L.W_RAW, w1, w_up, w2
        now = self._versions(self.raw)
        if now != self.raw_versions:
            if now != self.seen_versions and rows < 4096 * self.e_local and all(t is None or (t.is_contiguous() and t.data_ptr() % 16 == 0) for t in self.raw):
                self.seen_versions = now
                return L.W_RAW, self.raw[0], self.raw[2], self.raw[1]
            self.refresh()
        return L.W_TILED, self.w1, None, self.w2

    @classmethod
    def prepare_fp8(cls, wg_q, sg, wu_q, su, wd_q, sd):
        """e4m3 codes (uint8) [E_l,H,F] x2 and [E_l,F,H] with fp32 per-output-channel scales."""
        e_l, H, F = wg_q.shape
        p1 = ops.prepack_weights_fp8(wg_q.contiguous(), wu_q.contiguous())
        p2 = ops.prepack_weights_fp8(wd_q.contiguous())
        return cls("swiglu", H, F, e_l, torch.uint8, p1, p2, None, (sg.contiguous(), su.contiguous(), sd.contiguous()))


class ExpertMLP(torch.autograd.Function):
    """y = act(x W1) W2, or (silu(x Wg) * (x Wu)) Wd, on expert-major rows, with its gradients (the reference defines
    neither the MLP nor a backward).  Inputs that autograd sees: tokens and the weight tensors ``prepare`` was given."""

    @staticmethod
    def forward(ctx, tokens, cnt, ew, w1, w2, w_up):
        tokens = ops.aligned16(tokens.contiguous())
        S, F = tokens.shape[0], ew.ffn
        a1 = None
        if tokens.dtype == torch.bfloat16 and ew.act != "none" and S:
            # the first GEMM also keeps what it feeds to the activation: the backward pass would otherwise run it again
            weights = ew.train_weights(S)
            ctx.raw = weights[0] == L.W_RAW
            out, hidden, a1 = ops.mlp_train_forward(tokens, cnt, ew.act, *weights, F, part_ws=_part_ws(tokens.device, 2 * max(ew.hidden, F)))
        else:
            ew.refresh()
            hidden = torch.empty((S, F), dtype=tokens.dtype, device=tokens.device)
            out = ops.grouped_mlp(tokens, cnt, ew.act, ew.w1, ew.w2, ew.w_up, F=F, hidden_ws=hidden,
                                  part_ws=_part_ws(tokens.device, 2 * max(ew.hidden, F)))
        ctx.save_for_backward(tokens, hidden, cnt, w1, w2, w_up, a1)
        ctx.ew = ew
        return out

    @staticmethod
    def backward(ctx, dy):
        """With a1 the pre-activations (bf16: kept by the forward's first GEMM; fp32: recomputed):
          d h  = dy @ W2^T          d W2 = h^T @ dy            (per expert, ragged rows as the reduction dimension)
          d a1 = d h * act'(a1)     (SwiGLU: d g = d h * u * silu'(g), d u = d h * silu(g))
          d x  = d a1 @ W1^T        d W1 = x^T @ d a1          (SwiGLU: both halves in one launch each)"""
        tokens, hidden, cnt, w1, w2, w_up, a1 = ctx.saved_tensors
        ew = ctx.ew
        dy = ops.aligned16(dy.contiguous())
        S, H, F = tokens.shape[0], ew.hidden, ew.ffn
        swiglu = ew.act == "swiglu"
        if tokens.dtype == torch.float32:
            if swiglu:
                raise NotImplementedError("expert_mlp backward: fp32 SwiGLU (the fp32 path serves the GELU / SiLU plumbing workload)")
            dh = ops.grouped_gemm(dy, ops.transpose_weights_f32(w2.contiguous()), cnt)
            dw2 = ops.grouped_gemm_dw(hidden, dy, cnt)
            a1 = ops.grouped_gemm(tokens, w1.contiguous(), cnt)
            da1 = ops.mlp_act_backward(a1, dh, ew.act)
            dx = ops.grouped_gemm(da1, ops.transpose_weights_f32(w1.contiguous()), cnt)
            dw1 = ops.grouped_gemm_dw(tokens, da1, cnt)
            return dx, None, None, dw1, dw2, None
        ws = _part_ws(tokens.device, 2 * max(H, 2 * F if swiglu else F))
        if a1 is not None:
            if ctx.raw or L.capturing():
                weights = (L.W_RAW_T, w1.contiguous(), None if w_up is None else w_up.contiguous(), w2.contiguous())
            else:
                weights = (L.W_TILED, _packed_weights_t(w1, w_up), None, _packed_weights_t(w2))
            dx, dw1, dw2, dw_up = ops.mlp_train_backward(tokens, hidden, a1, dy, cnt, ew.act, *weights, part_ws=ws)
            return dx, None, None, dw1, dw2, dw_up
        NP = 2 * F if swiglu else F
        dh = torch.zeros((S, F), dtype=dy.dtype, device=dy.device)
        dx = torch.zeros((S, H), dtype=dy.dtype, device=dy.device)
        if S:
            ops.grouped_gemm_mapped(dy, None, _packed_weights_t(w2), cnt, S, F, "none", dh, part_ws=ws)
        ew.refresh()
        a1 = torch.zeros((S, NP), dtype=dy.dtype, device=dy.device)  # (no rows, or an MLP without an activation)
        if S:
            ops.grouped_gemm_mapped(tokens, None, ew.w1, cnt, S, NP, "none", a1, part_ws=ws)
        dw2 = ops.grouped_gemm_dw(hidden, dy, cnt)
        da1 = ops.mlp_act_backward(a1, dh, ew.act)
        if S:
            ops.grouped_gemm_mapped(da1, None, _packed_weights_t(w1, w_up), cnt, S, H, "none", dx, part_ws=ws)
        dw1 = ops.grouped_gemm_dw(tokens, da1, cnt, split_F=F if swiglu else 0)
        if swiglu:
            return dx, None, None, dw1[..., :F], dw2, dw1[..., F:]
        return dx, None, None, dw1, dw2, None


def expert_mlp(tokens: torch.Tensor, weights: ExpertWeights, local_expert_cnt: torch.Tensor) -> torch.Tensor:
    """Full expert MLP on expert-major rows -> [S,H]."""
    assert tokens.is_cuda, "tokens must be CUDA"
    _assert_cuda_int32(local_expert_cnt, "local_expert_cnt")
    if weights.dtype == torch.uint8:
        sg, su, sd = weights.scales
        return ops.grouped_mlp_fp8(ops.aligned16(tokens.contiguous()), local_expert_cnt, weights.ffn, weights.w1, sg, su, weights.w2, sd,
                                   part_ws=_part_ws(tokens.device, max(weights.hidden, weights.ffn)))
    raw = weights.raw
    if torch.is_grad_enabled() and raw is not None and (tokens.requires_grad or any(t is not None and t.requires_grad for t in raw)):
        return ExpertMLP.apply(tokens, local_expert_cnt.contiguous(), weights, raw[0], raw[1], raw[2])
    weights.refresh()
    return ops.grouped_mlp(ops.aligned16(tokens.contiguous()), local_expert_cnt, weights.act, weights.w1, weights.w2, weights.w_up,
                           F=weights.ffn, part_ws=_part_ws(tokens.device, 2 * max(weights.hidden, weights.ffn)))
