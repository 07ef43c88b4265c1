"""Recurrent mixers whose state is one decayed matrix per head, written with scalar gates.

Per token and head, with query q and key k (``key_dim`` each), value v (``value_dim``) and two
scalars a (how much of the old state stays) and b (how strongly the token is written):

    S <- a S;   u = b (v - [delta] S^T k);   S <- S + k u^T;   o = S^T q

so the read-out sees the token's own write.

* ``gated_delta`` (the gated delta rule): [delta] is on. q and k come from ``num_kv_heads`` groups
  (head h reads group h // (num_heads / num_kv_heads)); q, k and v pass a short causal convolution
  over time per channel (``conv_taps`` taps, the last one the current token's, zeros before the
  start) and SiLU; q and k are then made unit vectors, x / sqrt(sum(x^2) + unit_eps), q also times
  key_dim^-1/2. b = sigmoid(W_b h) and a = exp(-exp(A_log) * softplus(W_a h + dt_bias)) per head.
  o is divided by its root mean square per head, multiplied by a weight of ``value_dim`` numbers
  that the heads share and by silu(W_g h).
* ``mlstm`` (the matrix memory of the xLSTM): [delta] is off. q = W_q h * key_dim^-1/2. With the log
  input gate i = cap tanh((W_i h + b_i) / cap), the log forget gate
  f = logsigmoid(cap tanh((W_f h + b_f) / cap)) and a running maximum m (0 at the start),
  m' = max(f + m, i), the scalars are a = exp(f + m - m'), b = exp(i - m'). A normaliser n (the same
  recurrence on k alone) is kept as one more column of S, fed with the value 1, and
  o <- o / (max(|n . q|, exp(-m')) + denom_eps). o is then divided by its root mean square per head,
  multiplied by a weight over all heads' channels and by sigmoid(W_g h).

* ``channel_delta`` (the gated delta rule with a decay per key channel): as ``gated_delta``, but a is a vector over
  the key channels, S <- diag(a) S, a = exp(-exp(A_log) * softplus(W_a2 (W_a1 h) + dt_bias)) per head and channel
  (A_log per head), and o, after its norm, is multiplied by sigmoid(W_g2 (W_g1 h)).
* ``constant_decay`` (lightning attention): [delta] is off, a is a constant per head and b = 1; q, k and v are SiLU of
  their projections. All heads' o together are divided by their root mean square, multiplied by a weight over all
  channels and by sigmoid(W_g h).

* ``gated_linear`` (gated linear attention): [delta] is off, b = 1, a is a vector over the key channels, S <- diag(a) S with
  a = sigmoid(z)^(1 / tau), z = W_a2 (W_a1 h) + bias per head and channel; q = W_q h * key_dim^-1/2, k and v are plain
  projections. o is divided by its root mean square per head, multiplied by a weight of ``value_dim`` numbers that the
  heads share and by silu(W_g h); ``out_scale`` is a constant on the result.

All keep S as float32 [heads, columns, key_dim] per request (a head's matrix column by column),
zero at a request's start; the convolution's last ``conv_taps - 1`` inputs (activation type) and the
running maximum (float32 [heads]) are state too. Gates, unit vectors and the recurrence are float32
whatever the activation type. All projections of the mixer's input are one packed product.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, Optional, Sequence, Tuple

import torch

from ..engine.step import most_units
from ..kernels.ops import RowSums
from .base import Mixer, PartSpec, Runtime, TensorDecl, register_mixer


# In a step that brings short requests too both paths run, one behind the other (a scan of up to 127 tokens, 28 us, and the
# chunks' two kernels, 20 us and more), where the scan alone takes 0.22 us a token of the longest. So such a step takes the
# chunks only for longer requests (us, 16 heads of 64, the scan alone / both paths: requests of 400, 300 and 150 tokens
# beside 17 single ones, general rule 100 / 77, per-head decay 94 / 64, sum 86 / 51, channel decays 97 / 65; of 230, 176 and
# 90 tokens 63 / 69, 58 / 66, 54 / 53, 59 / 67).
CHUNKS_BESIDE_SHORT = 384
# ... and a recording that has to serve any cut, in classes large enough to hold them.
CHUNKS_BESIDE_SHORT_CLASS = 1024


# A scan takes the time of its longest request, however many requests and heads walk beside it, until they fill the chip; the
# chunks' kernels write, read and multiply matrices for every chunk and head, so their time grows with both. What the two
# take (us, by key channels): a token of the longest request scanned; the chunks' two kernels, and a token of the longest
# there; nanoseconds a token and head there. Fitted to 18 cuts of 128 to 8,192 tokens, for 16 and 64 heads: the smaller of
# the two was chosen to within 3 % of the scan everywhere and missed up to 18 % of the chunks' gain where the two are close.
# Measured, scan / chunks: 64 requests of 128 tokens, 16 heads of 64, general rule 198 / 405, per-head decay 141 / 278, sum
# 140 / 168, channel decays 151 / 285; four of 512, 64 heads 235 / 361, 171 / 236, 167 / 151, 167 / 247; one of 2,048,
# 64 heads 450 / 342, 476 / 216, 411 / 155, 474 / 230; 16 of 256, 16 heads of 128 442 / 548, 237 / 512, 227 / 225, 274 / 525.
# (Since then the walk along the chunks takes 37 us instead of 57 at 2,048 tokens, the general rule's chunks 52 instead of 67 and the vectors'
# kernels in front of them, 15 to 29 us, are gone where no request is scanned: the line lies on the scan's side of where the two meet now.)
_SCAN_TOKEN = {64: 0.22, 128: 0.32}
_CHUNKS_ONCE = {64: (18.0, 0.013), 128: (29.0, 0.018)}
_CHUNKS_TOKEN_HEAD = {"delta": {64: 2.4, 128: 7.6}, "gated": {64: 1.55, 128: 7.0}, "channel": {64: 1.6, 128: 7.1},
                      "sum": {64: 1.0, 128: 3.1}}


def _chunk_tokens_worth(rule: str, heads: int, dk: int, dv: int, longest: int, longest_scanned: int = 0) -> float:
    """Up to how many tokens, in all the requests that go in chunks, the chunks (and a scan of the others beside them) take
    less time than a scan of all."""
    once, token = _CHUNKS_ONCE[dk]
    if longest_scanned:
        once += 3.0 + _SCAN_TOKEN[dk] * longest_scanned
    return ((_SCAN_TOKEN[dk] - token) * longest - once) * 1e3 / (_CHUNKS_TOKEN_HEAD[rule][dk] * heads * (dk + dv) / (2 * dk))


def _paths(ops, rule: str, heads: int, dk: int, dv: int, lens: Sequence[int]) -> Tuple[bool, bool]:
    """Whether the requests of many tokens go in chunks, and whether any requests are scanned."""
    line = ops.delta_chunk_line()
    longest, scanned = max(lens, default=0), max((q for q in lens if q < line), default=0)
    if longest < (CHUNKS_BESIDE_SHORT if scanned else line) or not ops.delta_chunks_serve(rule, dk, dv) \
            or sum(q for q in lens if q >= line) > _chunk_tokens_worth(rule, heads, dk, dv, longest, scanned):
        return False, True
    return True, scanned > 0


def recurrence(rt: Runtime, ctx, rule: str, n: int, heads: int, dk: int, dv: int, raw: torch.Tensor, scan, chunks, *operands) -> None:
    """A mixer's recurrence over the step's rows into ``raw``: requests of many tokens as products over chunks of tokens
    (``chunks``, None: not in this engine), the others, and heads of sizes these do not take, token by token (``scan``)."""
    in_chunks, scanned = step_paths(rt, ctx, rule, heads, dk, dv) if chunks is not None else (False, True)
    if not in_chunks:
        scan(*operands, raw)
        return
    chunks(*operands, *step_chunk_scratch(rt, ctx, rule, n, heads, dk, dv), raw)
    if scanned:
        scan(*operands, raw, below=rt.ops.delta_chunk_line())


def step_paths(rt: Runtime, ctx, rule: str, heads: int, dk: int, dv: int) -> Tuple[bool, bool]:
    """Whether the step's requests of many tokens go in chunks, and whether any requests are scanned."""
    ops, plan = rt.ops, ctx.attention_plan
    if plan is None:
        return False, True
    if plan.bound is None or plan.path_lens:
        return _paths(ops, rule, heads, dk, dv, plan.q_lens if plan.bound is None else plan.path_lens)
    line = ops.delta_chunk_line()
    short = plan.has_short(line)
    in_chunks = plan.has_long(CHUNKS_BESIDE_SHORT_CLASS if short else line) and ops.delta_chunks_serve(rule, dk, dv)
    return in_chunks, short or not in_chunks


def step_chunk_scratch(rt: Runtime, ctx, rule: str, n: int, heads: int, dk: int, dv: int):
    units = ctx.attention_plan.units(rt.ops.delta_chunk_tokens(), rt.ops.delta_chunk_line())
    return _chunk_scratch(rt.workspace, rule, n, heads, dk, dv, units)


def _chunk_scratch(ws, rule: str, n: int, heads: int, dk: int, dv: int, units: int):
    return (ws.get("mstate.chunk_maps", (units, heads) + ((dk, dk) if rule != "sum" else ()), torch.float32),
            ws.get("mstate.chunks", (units, heads, dv, dk), torch.float32),
            ws.get("mstate.chunk_queries", (n, heads, dk), torch.float32))


class ChunkedRecurrence(Mixer):
    """A mixer that calls ``recurrence``."""
    recurrence_sizes: Tuple[str, int, int, int]          # the rule, heads, key channels, columns

    def chunks(self, entry):
        """``entry`` (the products over chunks), or None in float32: there every sum's order depends on the request alone,
        not on how it is cut or what else is in the step, and which requests go in chunks depends on both."""
        return None if self.rt.dtype == torch.float32 else entry

    def step_path(self, lens: Sequence[int], starts: Sequence[int]):
        return None if self.chunks(self) is None else _paths(self.rt.ops, *self.recurrence_sizes, lens)

    def vectors(self, n: int) -> Tuple[torch.Tensor, ...]:
        """Scratch for the float vectors of ``n`` rows that a scan, and the chunks beside one, read. A step whose requests all go in chunks may
        do without."""
        raise NotImplementedError

    def reserve(self, tokens: int, seqs: int) -> None:
        (rule, heads, dk, dv), ops = self.recurrence_sizes, self.rt.ops
        self.vectors(tokens)
        line = ops.delta_chunk_line()
        if self.chunks(rule) is not None and tokens >= line and ops.delta_chunks_serve(rule, dk, dv):
            most = min(tokens, int(_chunk_tokens_worth(rule, heads, dk, dv, min(tokens, self.rt.max_positions))))
            if most >= line:
                _chunk_scratch(self.rt.workspace, rule, tokens, heads, dk, dv, most_units(most, seqs, ops.delta_chunk_tokens(), line))


def _pack(tensors: Dict[str, torch.Tensor], names, hidden: int, what: str):
    dtypes = {tensors[p].dtype for p in names}
    if len(dtypes) != 1:
        raise ValueError(f"{what}: the projections are stored in different dtypes {dtypes}; cannot pack them")
    blocks = [tensors[p] for p in names]
    rows = sum(b.shape[0] for b in blocks)
    pad = (-rows) % 8             # rows of the packed product keep a pitch of a multiple of 8 elements
    if pad:
        blocks.append(torch.zeros((pad, hidden), dtype=blocks[0].dtype, device=blocks[0].device))
    return torch.cat(blocks, dim=0).contiguous()


@dataclass(frozen=True)
class GatedDeltaSpec(PartSpec):
    kind = "gated_delta"
    hidden_size: int = 0
    num_heads: int = 0
    num_kv_heads: int = 0
    key_dim: int = 0
    value_dim: int = 0
    conv_taps: int = 1                  # 1: no convolution (a single tap still scales each channel)
    unit_eps: float = 1e-6              # inside the root of a query's or key's length
    out_norm_eps: float = 1e-6          # of the per-head RMS of the output

    @property
    def conv_channels(self) -> int:
        return 2 * self.num_kv_heads * self.key_dim + self.num_heads * self.value_dim


@register_mixer(GatedDeltaSpec.kind)
class GatedDelta(ChunkedRecurrence):
    spec_class = GatedDeltaSpec
    PACKED = ("q", "k", "v", "g", "b", "a")

    @classmethod
    def tensors(cls, spec: GatedDeltaSpec) -> Dict[str, TensorDecl]:
        hid, qk, vd = spec.hidden_size, spec.num_kv_heads * spec.key_dim, spec.num_heads * spec.value_dim
        t = {"q": TensorDecl((qk, hid)), "k": TensorDecl((qk, hid)), "v": TensorDecl((vd, hid)), "g": TensorDecl((vd, hid)),
             "b": TensorDecl((spec.num_heads, hid)), "a": TensorDecl((spec.num_heads, hid)),
             "q_conv": TensorDecl((qk, spec.conv_taps)), "k_conv": TensorDecl((qk, spec.conv_taps)),
             "v_conv": TensorDecl((vd, spec.conv_taps)),
             "A_log": TensorDecl((spec.num_heads,), init="zeros_normal"),
             "dt_bias": TensorDecl((spec.num_heads,), init="zeros_normal"),
             "norm": TensorDecl((spec.value_dim,), init="ones_normal"),
             "o": TensorDecl((hid, vd))}
        return t

    @classmethod
    def state_shapes(cls, spec: GatedDeltaSpec):
        shapes = {"state": ((spec.num_heads, spec.value_dim, spec.key_dim), torch.float32)}
        if spec.conv_taps > 1:
            shapes["conv"] = ((spec.conv_taps - 1, spec.conv_channels), None)      # the activation type
        return shapes

    def __init__(self, spec: GatedDeltaSpec, tensors: Dict[str, torch.Tensor], rt: Runtime, position: Optional[object] = None):
        if min(spec.num_heads, spec.num_kv_heads, spec.key_dim, spec.value_dim, spec.conv_taps) < 1 \
                or spec.num_heads % spec.num_kv_heads:
            raise ValueError(f"gated delta rule: bad sizes {spec}")
        self.spec, self.rt = spec, rt
        self.recurrence_sizes = ("gated", spec.num_heads, spec.key_dim, spec.value_dim)
        self.w_packed = _pack(tensors, self.PACKED, spec.hidden_size, "gated delta rule")
        self.width = self.w_packed.shape[0]
        self.gate_offset = spec.conv_channels
        self.conv_w = torch.cat([tensors["q_conv"], tensors["k_conv"], tensors["v_conv"]], dim=0).contiguous()
        self.a_log = tensors["A_log"].to(self.conv_w.dtype).contiguous()
        self.dt_bias = tensors["dt_bias"].to(self.conv_w.dtype).contiguous()
        self.norm, self.w_o = tensors["norm"].to(self.conv_w.dtype).contiguous(), tensors["o"]

    def vectors(self, n: int):
        spec, ws = self.spec, self.rt.workspace
        return (ws.get("mstate.qk", (n, spec.num_kv_heads, 2, spec.key_dim), torch.float32),
                ws.get("mstate.vals", (n, spec.num_heads, spec.value_dim), torch.float32))

    def forward(self, x: torch.Tensor, ctx, call: int) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, H, G, dk, dv = x.shape[0], spec.num_heads, spec.num_kv_heads, spec.key_dim, spec.value_dim
        packed = ws.get("mstate.packed", (n, self.width), rt.dtype)
        ops.gemm(x, self.w_packed, packed)
        gated = ws.get("mstate.gated", (n, H * dv), rt.dtype)
        y = ws.get("mixer.out", (n, spec.hidden_size), rt.dtype)
        plan = ctx.attention_plan
        # every request brings one token: everything between the two products as one kernel
        if plan is not None and plan.decode_only and ops.state_step(
                True, packed, H, G, dk, dv, self.norm, spec.out_norm_eps, ctx.state(call), ctx.token_seq, ctx.cu_seqlens,
                ctx.state_slots, ctx.n_seqs, gated, taps=spec.conv_taps, conv_w=self.conv_w, a_log=self.a_log,
                dt_bias=self.dt_bias, conv_state=ctx.state(call, "conv") if spec.conv_taps > 1 else None,
                unit_eps=spec.unit_eps):
            return ops.gemm(gated, self.w_o, y, defer_sum=True) or y
        conv_state = ctx.state(call, "conv") if spec.conv_taps > 1 else None
        gates = ws.get("mstate.gates", (n, H, 4), torch.float32)
        raw = ws.get("mstate.raw", (n, H, dv), torch.float32)
        if (self.chunks(ops.state_chunks) is not None and step_paths(rt, ctx, "gated", H, dk, dv) == (True, False)
                and ops.delta_chunks_conv_serve(packed, dk, dv, spec.conv_taps, self.conv_w, self.dt_bias, conv_state)):
            ops.delta_chunks_conv("gated", packed, 2 * G * dk + 2 * H * dv, H, G, dk, dv, spec.conv_taps, self.conv_w, self.a_log, self.dt_bias,
                                  conv_state, spec.unit_eps, None, ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs,
                                  *step_chunk_scratch(rt, ctx, "gated", n, H, dk, dv), raw)
        else:
            qk, vals = self.vectors(n)
            ops.gated_delta_prepare(packed, H, G, dk, dv, spec.conv_taps, self.conv_w, self.a_log, self.dt_bias, conv_state, spec.unit_eps,
                                    ctx.token_seq, ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, qk, vals, gates)
            recurrence(rt, ctx, "gated", n, H, dk, dv, raw, ops.state_scan, self.chunks(ops.state_chunks), qk, vals, gates,
                       ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, H, G, dk, dv, True)
        ops.state_finish(raw, gates, packed, self.gate_offset, self.norm, H, dv, spec.out_norm_eps, ctx.token_seq, gated,
                         shared_weight=True, silu_gate=True)
        return ops.gemm(gated, self.w_o, y, defer_sum=True) or y


@dataclass(frozen=True)
class MLSTMSpec(PartSpec):
    kind = "mlstm"
    hidden_size: int = 0
    num_heads: int = 0
    key_dim: int = 0
    value_dim: int = 0
    gate_cap: float = 15.0              # both gates' pre-activations are squashed into (-cap, cap)
    denom_eps: float = 1e-6             # added to the denominator
    out_norm_eps: float = 1e-6          # of the per-head RMS of the output


@register_mixer(MLSTMSpec.kind)
class MLSTM(ChunkedRecurrence):
    spec_class = MLSTMSpec
    PACKED = ("q", "k", "v", "g", "i", "f")

    @classmethod
    def tensors(cls, spec: MLSTMSpec) -> Dict[str, TensorDecl]:
        hid, qk, vd = spec.hidden_size, spec.num_heads * spec.key_dim, spec.num_heads * spec.value_dim
        return {"q": TensorDecl((qk, hid)), "k": TensorDecl((qk, hid)), "v": TensorDecl((vd, hid)), "g": TensorDecl((vd, hid)),
                "i": TensorDecl((spec.num_heads, hid)), "f": TensorDecl((spec.num_heads, hid)),
                "i_bias": TensorDecl((spec.num_heads,), init="zeros_normal"),
                "f_bias": TensorDecl((spec.num_heads,), init="zeros_normal"),
                "norm": TensorDecl((vd,), init="ones_normal"), "o": TensorDecl((hid, vd))}

    @classmethod
    def state_shapes(cls, spec: MLSTMSpec):
        # the matrix with the normaliser as its last column; the running maximum
        return {"state": ((spec.num_heads, spec.value_dim + 1, spec.key_dim), torch.float32),
                "max": ((spec.num_heads,), torch.float32)}

    def __init__(self, spec: MLSTMSpec, tensors: Dict[str, torch.Tensor], rt: Runtime, position: Optional[object] = None):
        if min(spec.num_heads, spec.key_dim, spec.value_dim) < 1 or not spec.gate_cap > 0:
            raise ValueError(f"mlstm: bad sizes {spec}")
        self.spec, self.rt = spec, rt
        self.recurrence_sizes = ("sum", spec.num_heads, spec.key_dim, spec.value_dim + 1)
        self.w_packed = _pack(tensors, self.PACKED, spec.hidden_size, "mlstm")
        self.width = self.w_packed.shape[0]
        self.gate_offset = spec.num_heads * (2 * spec.key_dim + spec.value_dim)
        self.i_bias = tensors["i_bias"].contiguous()
        self.f_bias = tensors["f_bias"].to(self.i_bias.dtype).contiguous()
        self.norm, self.w_o = tensors["norm"].to(self.i_bias.dtype).contiguous(), tensors["o"]

    def vectors(self, n: int):
        spec, ws = self.spec, self.rt.workspace
        return (ws.get("mstate.qk", (n, spec.num_heads, 2, spec.key_dim), torch.float32),
                ws.get("mstate.vals", (n, spec.num_heads, spec.value_dim + 1), torch.float32))

    def forward(self, x: torch.Tensor, ctx, call: int) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, H, dk, dv = x.shape[0], spec.num_heads, spec.key_dim, spec.value_dim
        packed = ws.get("mstate.packed", (n, self.width), rt.dtype)
        ops.gemm(x, self.w_packed, packed)
        gated = ws.get("mstate.gated", (n, H * dv), rt.dtype)
        y = ws.get("mixer.out", (n, spec.hidden_size), rt.dtype)
        plan = ctx.attention_plan
        if plan is not None and plan.decode_only and ops.state_step(
                False, packed, H, H, dk, dv, self.norm, spec.out_norm_eps, ctx.state(call), ctx.token_seq, ctx.cu_seqlens,
                ctx.state_slots, ctx.n_seqs, gated, i_bias=self.i_bias, f_bias=self.f_bias, cap=spec.gate_cap,
                max_state=ctx.state(call, "max"), denom_eps=spec.denom_eps):
            return ops.gemm(gated, self.w_o, y, defer_sum=True) or y
        gates = ws.get("mstate.gates", (n, H, 4), torch.float32)
        raw = ws.get("mstate.raw", (n, H, dv + 1), torch.float32)
        prepare = (packed, H, dk, dv, self.i_bias, self.f_bias, spec.gate_cap, ctx.state(call, "max"), ctx.token_seq, ctx.cu_seqlens,
                   ctx.state_slots, ctx.n_seqs)
        if (self.chunks(ops.state_chunks) is not None and step_paths(rt, ctx, "sum", H, dk, dv + 1) == (True, False)
                and ops.mlstm_chunks_serve(packed, dk, dv)):
            ops.mlstm_prepare(*prepare, None, None, gates)
            ops.mlstm_chunks(packed, gates, ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, H, dk, dv,
                             *step_chunk_scratch(rt, ctx, "sum", n, H, dk, dv + 1), raw)
        else:
            qk, vals = self.vectors(n)
            ops.mlstm_prepare(*prepare, qk, vals, gates)
            recurrence(rt, ctx, "sum", n, H, dk, dv + 1, raw, ops.state_scan, self.chunks(ops.state_chunks), qk, vals, gates, ctx.state(call),
                       ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, H, H, dk, dv + 1, False)
        ops.state_finish(raw, gates, packed, self.gate_offset, self.norm, H, dv, spec.out_norm_eps, ctx.token_seq, gated,
                         shared_weight=False, silu_gate=False, normaliser=True, denom_eps=spec.denom_eps)
        return ops.gemm(gated, self.w_o, y, defer_sum=True) or y


@dataclass(frozen=True)
class ChannelDeltaSpec(PartSpec):
    kind = "channel_delta"
    hidden_size: int = 0
    num_heads: int = 0
    num_kv_heads: int = 0
    key_dim: int = 0
    value_dim: int = 0
    conv_taps: int = 1                  # 1: no convolution (a single tap still scales each channel)
    decay_rank: int = 0                 # rows of W_a1
    gate_rank: int = 0                  # rows of W_g1
    unit_eps: float = 1e-6              # inside the root of a query's or key's length
    out_norm_eps: float = 1e-6          # of the per-head RMS of the output

    @property
    def conv_channels(self) -> int:
        return 2 * self.num_kv_heads * self.key_dim + self.num_heads * self.value_dim


@register_mixer(ChannelDeltaSpec.kind)
class ChannelDelta(ChunkedRecurrence):
    """Packed rows: [q | k | v | b, padded to a multiple of 8 | W_a1 h | W_g1 h, padded to a multiple of 32]. In steps with
    prompt portions the two second matrices are one product against the low-rank columns (block-diagonal, in float32
    rows [decays | gates]); in steps of single tokens the step's kernel makes them itself."""
    spec_class = ChannelDeltaSpec
    accepts_pending_norm = True         # the input is used by one packed product only
    accepts_fold = True                 # the output comes from one product

    @classmethod
    def tensors(cls, spec: ChannelDeltaSpec) -> Dict[str, TensorDecl]:
        hid, H = spec.hidden_size, spec.num_heads
        qk, dk, vd = spec.num_kv_heads * spec.key_dim, H * spec.key_dim, H * spec.value_dim
        return {"q": TensorDecl((qk, hid)), "k": TensorDecl((qk, hid)), "v": TensorDecl((vd, hid)), "b": TensorDecl((H, hid)),
                "q_conv": TensorDecl((qk, spec.conv_taps)), "k_conv": TensorDecl((qk, spec.conv_taps)),
                "v_conv": TensorDecl((vd, spec.conv_taps)),
                "A_log": TensorDecl((H,), init="zeros_normal"), "dt_bias": TensorDecl((dk,), init="zeros_normal"),
                "a1": TensorDecl((spec.decay_rank, hid)), "a2": TensorDecl((dk, spec.decay_rank)),
                "g1": TensorDecl((spec.gate_rank, hid)), "g2": TensorDecl((vd, spec.gate_rank)),
                "norm": TensorDecl((spec.value_dim,), init="ones_normal"), "o": TensorDecl((hid, vd))}

    @classmethod
    def state_shapes(cls, spec: ChannelDeltaSpec):
        shapes = {"state": ((spec.num_heads, spec.value_dim, spec.key_dim), torch.float32)}
        if spec.conv_taps > 1:
            shapes["conv"] = ((spec.conv_taps - 1, spec.conv_channels), None)      # the activation type
        return shapes

    def __init__(self, spec: ChannelDeltaSpec, tensors: Dict[str, torch.Tensor], rt: Runtime, position: Optional[object] = None):
        if min(spec.num_heads, spec.num_kv_heads, spec.key_dim, spec.value_dim, spec.conv_taps, spec.decay_rank, spec.gate_rank) < 1 \
                or spec.num_heads % spec.num_kv_heads:
            raise ValueError(f"channel-wise delta rule: bad sizes {spec}")
        self.spec, self.rt = spec, rt
        self.recurrence_sizes = ("channel", spec.num_heads, spec.key_dim, spec.value_dim)
        hid, H, dk, dv = spec.hidden_size, spec.num_heads, spec.key_dim, spec.value_dim
        ra, rg = spec.decay_rank, spec.gate_rank
        front = _pack(tensors, ("q", "k", "v", "b"), hid, "channel-wise delta rule")
        low = torch.cat([tensors["a1"], tensors["g1"]], dim=0)
        pad = (-low.shape[0]) % 32
        if pad:
            low = torch.cat([low, torch.zeros((pad, hid), dtype=low.dtype, device=low.device)], dim=0)
        self.b_offset, self.low_offset, self.low_width = spec.conv_channels, front.shape[0], low.shape[0]
        self.w_packed = torch.cat([front, low], dim=0).contiguous()
        self.width = self.w_packed.shape[0]
        second = torch.zeros((H * (dk + dv), self.low_width), dtype=low.dtype, device=low.device)
        second[:H * dk, :ra] = tensors["a2"]
        second[H * dk:, ra:ra + rg] = tensors["g2"]
        self.w_second = second.contiguous()
        self.conv_w = torch.cat([tensors["q_conv"], tensors["k_conv"], tensors["v_conv"]], dim=0).contiguous()
        dt = self.conv_w.dtype
        self.a_log, self.dt_bias = tensors["A_log"].to(dt).contiguous(), tensors["dt_bias"].to(dt).contiguous()
        self.a2t, self.g2t = tensors["a2"].to(dt).t().contiguous(), tensors["g2"].to(dt).t().contiguous()
        self.norm, self.w_o = tensors["norm"].to(dt).contiguous(), tensors["o"]

    def first_product(self):
        return self.w_packed.shape[0], self.w_packed.shape[1], False

    def vectors(self, n: int):
        spec, ws = self.spec, self.rt.workspace
        return (ws.get("mstate.qk", (n, spec.num_kv_heads, 2, spec.key_dim), torch.float32),
                ws.get("mstate.vals", (n, spec.num_heads, spec.value_dim), torch.float32),
                ws.get("mstate.beta", (n, spec.num_heads), torch.float32))

    def forward(self, x: torch.Tensor, ctx, call: int, fold=None) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, H, G, dk, dv = x.shape[0], spec.num_heads, spec.num_kv_heads, spec.key_dim, spec.value_dim
        packed = ws.get("mstate.packed", (n, self.width), rt.dtype)
        ops.gemm(x, self.w_packed, packed)
        gated = ws.get("mstate.gated", (n, H * dv), rt.dtype)
        y = ws.get("mixer.out", (n, spec.hidden_size), rt.dtype)
        conv_state = ctx.state(call, "conv") if spec.conv_taps > 1 else None
        plan = ctx.attention_plan
        if plan is not None and plan.decode_only and ops.channel_step(
                packed, H, G, dk, dv, spec.conv_taps, self.b_offset, self.low_offset, self.conv_w, self.a_log, self.dt_bias, self.a2t,
                self.g2t, self.norm, conv_state, ctx.state(call), spec.unit_eps, spec.out_norm_eps, ctx.token_seq, ctx.cu_seqlens,
                ctx.state_slots, ctx.n_seqs, gated):
            return ops.gemm(gated, self.w_o, y, defer_sum=True, fold=fold) or y
        z = ws.get("mstate.z", (n, H * (dk + dv)), torch.float32)
        ops.gemm(packed[:, self.low_offset:self.low_offset + self.low_width], self.w_second, z)
        raw = ws.get("mstate.raw", (n, H, dv), torch.float32)
        if (self.chunks(ops.channel_chunks) is not None and step_paths(rt, ctx, "channel", H, dk, dv) == (True, False)
                and ops.delta_chunks_conv_serve(packed, dk, dv, spec.conv_taps, self.conv_w, self.dt_bias, conv_state, z)):
            ops.delta_chunks_conv("channel", packed, self.b_offset, H, G, dk, dv, spec.conv_taps, self.conv_w, self.a_log, self.dt_bias, conv_state,
                                  spec.unit_eps, z, ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs,
                                  *step_chunk_scratch(rt, ctx, "channel", n, H, dk, dv), raw)
        else:
            qk, vals, beta = self.vectors(n)
            ops.channel_prepare(packed, H, G, dk, dv, spec.conv_taps, self.b_offset, self.conv_w, self.a_log, self.dt_bias, conv_state,
                                spec.unit_eps, ctx.token_seq, ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, qk, vals, beta, z)
            recurrence(rt, ctx, "channel", n, H, dk, dv, raw, ops.channel_scan, self.chunks(ops.channel_chunks), qk, vals, beta, z,
                       ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, H, G, dk, dv)
        ops.state_finish(raw, None, z, H * dk, self.norm, H, dv, spec.out_norm_eps, ctx.token_seq, gated, shared_weight=True,
                         silu_gate=False)
        return ops.gemm(gated, self.w_o, y, defer_sum=True, fold=fold) or y


@dataclass(frozen=True)
class ConstantDecaySpec(PartSpec):
    kind = "constant_decay"
    hidden_size: int = 0
    num_heads: int = 0
    key_dim: int = 0
    value_dim: int = 0
    decay: Tuple[float, ...] = ()       # one per head
    out_norm_eps: float = 1e-6          # of the RMS over all heads' outputs

    @property
    def inner(self) -> int:
        return self.num_heads * self.value_dim


@register_mixer(ConstantDecaySpec.kind)
class ConstantDecay(Mixer):
    spec_class = ConstantDecaySpec
    PACKED = ("q", "k", "v", "g")

    @classmethod
    def tensors(cls, spec: ConstantDecaySpec) -> Dict[str, TensorDecl]:
        hid, qk, vd = spec.hidden_size, spec.num_heads * spec.key_dim, spec.inner
        return {"q": TensorDecl((qk, hid)), "k": TensorDecl((qk, hid)), "v": TensorDecl((vd, hid)), "g": TensorDecl((vd, hid)),
                "norm": TensorDecl((vd,), init="ones_normal"), "o": TensorDecl((hid, vd))}

    @classmethod
    def state_shapes(cls, spec: ConstantDecaySpec):
        return {"state": ((spec.num_heads, spec.value_dim, spec.key_dim), torch.float32)}

    def __init__(self, spec: ConstantDecaySpec, tensors: Dict[str, torch.Tensor], rt: Runtime, position: Optional[object] = None):
        if min(spec.num_heads, spec.key_dim, spec.value_dim) < 1 or len(spec.decay) != spec.num_heads:
            raise ValueError(f"constant decay: bad sizes, or not one decay for each head: {spec}")
        self.spec, self.rt = spec, rt
        self.w_packed = _pack(tensors, self.PACKED, spec.hidden_size, "constant decay")
        self.width = self.w_packed.shape[0]
        self.decay = torch.tensor(spec.decay, dtype=torch.float32, device=rt.device)
        # prompts go chunk by chunk through matrix products where the decays' powers are powers of two's logarithm
        self.chunked = all(0.0 < d <= 1.0 for d in spec.decay)
        self.norm, self.w_o = tensors["norm"].contiguous(), tensors["o"]

    def recur(self, packed: torch.Tensor, base: int, ctx, call: int, beside: Optional[dict] = None):
        """From rows that hold this mixer's projections from column ``base`` on: (the rows that go into the output
        projection, a ``RowSums`` when they are still to be divided by their root mean square, whether ``beside`` ran).
        ``beside``: a query/key norm and cache write on the same rows, to run in the same launch where there is one."""
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, H, dk, dv = packed.shape[0], spec.num_heads, spec.key_dim, spec.value_dim
        gated = ws.get("mstate.gated", (n, H * dv), rt.dtype)
        plan = ctx.attention_plan
        if plan is not None and plan.decode_only:
            sums = ws.get("mstate.sums", (n, H), torch.float32)
            if ops.constant_step(packed, base, H, dk, dv, self.decay, self.norm, ctx.state(call), ctx.token_seq, ctx.state_slots, gated,
                                 sums, beside=beside):
                return gated, RowSums(sums, H * dv, spec.out_norm_eps), beside is not None
        raw = ws.get("mstate.raw", (n, H, dv), torch.float32)
        if self.chunked and plan is not None:
            chunks = plan.units(ops.constant_chunk_tokens())
            sums = ws.get("mstate.chunks", (chunks, H, dv, dk), torch.float32)
            ops.constant_chunks(packed, base, H, dk, dv, self.decay, ctx.state(call), ctx.token_seq, ctx.cu_seqlens, ctx.state_slots,
                                ctx.n_seqs, chunks, sums, raw)
        else:
            qk = ws.get("mstate.qk", (n, H, 2, dk), torch.float32)
            vals = ws.get("mstate.vals", (n, H, dv), torch.float32)
            gates = ws.get("mstate.gates", (n, H, 4), torch.float32)
            ops.constant_prepare(packed, base, H, dk, dv, self.decay, ctx.token_seq, qk, vals, gates)
            ops.state_scan(qk, vals, gates, ctx.state(call), ctx.cu_seqlens, ctx.state_slots, ctx.n_seqs, H, H, dk, dv, False, raw)
        ops.row_gate_finish(raw, packed, base + H * (2 * dk + dv), self.norm, spec.out_norm_eps, ctx.token_seq, gated)
        return gated, None, False

    def forward(self, x: torch.Tensor, ctx, call: int) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n = x.shape[0]
        packed = ws.get("mstate.packed", (n, self.width), rt.dtype)
        ops.gemm(x, self.w_packed, packed)
        gated, sums, _ = self.recur(packed, 0, ctx, call)
        if sums is not None:
            whole = ws.get("mstate.scaled", (n, spec.inner), rt.dtype)
            ops.scale_rows(gated, sums.sums, sums.sums.shape[1], sums.eps, whole)
            gated = whole
        y = ws.get("mixer.out", (n, spec.hidden_size), rt.dtype)
        return ops.gemm(gated, self.w_o, y, defer_sum=True) or y


@dataclass(frozen=True)
class GatedLinearSpec(PartSpec):
    kind = "gated_linear"
    hidden_size: int = 0
    num_heads: int = 0
    key_dim: int = 0
    value_dim: int = 0
    decay_rank: int = 0                 # rows of W_a1
    tau: float = 1.0                    # a channel's decay is sigmoid(z)^(1 / tau)
    out_norm_eps: float = 1e-6          # of the per-head RMS of the output
    out_scale: float = 1.0              # on the gated rows (it goes into the norm's weight)

    @property
    def inner(self) -> int:
        return self.num_heads * self.value_dim


@register_mixer(GatedLinearSpec.kind)
class GatedLinear(Mixer):
    """Packed rows: [q | k | v | g, padded to a multiple of 8 | W_a1 h, padded to a multiple of 32]. In steps with prompt
    portions W_a2 is one product with float32 rows; in steps of single tokens the step's kernel makes them itself."""
    spec_class = GatedLinearSpec
    accepts_pending_norm = True         # the input is used by one packed product only
    accepts_fold = True                 # the output comes from one product
    PACKED = ("q", "k", "v", "g")

    @classmethod
    def tensors(cls, spec: GatedLinearSpec) -> Dict[str, TensorDecl]:
        hid, qk, vd = spec.hidden_size, spec.num_heads * spec.key_dim, spec.inner
        return {"q": TensorDecl((qk, hid)), "k": TensorDecl((qk, hid)), "v": TensorDecl((vd, hid)), "g": TensorDecl((vd, hid)),
                "a1": TensorDecl((spec.decay_rank, hid)), "a2": TensorDecl((qk, spec.decay_rank)),
                "a2_bias": TensorDecl((qk,), init="zeros_normal"), "norm": TensorDecl((spec.value_dim,), init="ones_normal"),
                "o": TensorDecl((hid, vd))}

    @classmethod
    def state_shapes(cls, spec: GatedLinearSpec):
        return {"state": ((spec.num_heads, spec.value_dim, spec.key_dim), torch.float32)}

    def __init__(self, spec: GatedLinearSpec, tensors: Dict[str, torch.Tensor], rt: Runtime, position: Optional[object] = None):
        if min(spec.num_heads, spec.key_dim, spec.value_dim, spec.decay_rank) < 1 or not spec.tau > 0:
            raise ValueError(f"gated linear attention: bad sizes {spec}")
        self.spec, self.rt = spec, rt
        hid, qk = spec.hidden_size, spec.num_heads * spec.key_dim
        front = _pack(tensors, self.PACKED, hid, "gated linear attention")
        pad = (-spec.decay_rank) % 32
        low, a2 = tensors["a1"], tensors["a2"]
        self.a2t = a2.t().contiguous()
        if pad:
            low = torch.cat([low, torch.zeros((pad, hid), dtype=low.dtype, device=low.device)], dim=0)
            a2 = torch.cat([a2, torch.zeros((qk, pad), dtype=a2.dtype, device=a2.device)], dim=1)
        self.low_offset, self.low_width = front.shape[0], low.shape[0]
        self.w_packed = torch.cat([front, low], dim=0).contiguous()
        self.width = self.w_packed.shape[0]
        self.w_second = a2.contiguous()
        self.a2_bias = tensors["a2_bias"].to(torch.float32).contiguous()
        # float32: the constant on the output costs no rounding of its own
        self.norm = (tensors["norm"].to(torch.float32) * spec.out_scale).contiguous()
        self.w_o = tensors["o"]

    def first_product(self):
        return self.w_packed.shape[0], self.w_packed.shape[1], False

    def recur(self, packed: torch.Tensor, base: int, ctx, call: int, out: torch.Tensor, beside: Optional[dict] = None) -> bool:
        """From rows that hold this mixer's projections from column ``base`` on: the gated rows that go into the output
        projection, in ``out`` [n, heads * value_dim]. ``beside``: a convolution and cache write of a softmax mixer on the same
        rows (``Attention.conv_store_args``), to run in the same launch where there is one; returns whether it ran."""
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, H, dk, dv = packed.shape[0], spec.num_heads, spec.key_dim, spec.value_dim
        plan = ctx.attention_plan
        if plan is not None and plan.decode_only:
            ran = ops.gated_linear_step(packed, base, base + self.low_offset, H, dk, dv, self.a2t, self.a2_bias, spec.tau, self.norm,
                                        spec.out_norm_eps, ctx.state(call), ctx.token_seq, ctx.state_slots, out, beside=beside)
            if ran:
                return ran == 2
        z = ws.get("mstate.z", (n, H * dk), torch.float32)
        low = base + self.low_offset
        ops.gemm(packed[:, low:low + self.low_width], self.w_second, z)
        raw = ws.get("mstate.raw", (n, H, dv), torch.float32)
        chunks = plan.units(ops.gated_linear_chunk_tokens()) if plan is not None else n
        sums = ws.get("mstate.chunks", (chunks, H, dv, dk), torch.float32)
        decays = ws.get("mstate.decays", (chunks, H, dk), torch.float32)
        ops.gated_linear_chunks(packed, base, H, dk, dv, z, self.a2_bias, spec.tau, ctx.state(call), ctx.token_seq, ctx.cu_seqlens,
                                ctx.state_slots, ctx.n_seqs, chunks, sums, decays, raw)
        ops.state_finish(raw, None, packed, base + H * (2 * dk + dv), self.norm, H, dv, spec.out_norm_eps, ctx.token_seq, out,
                         shared_weight=True, silu_gate=True)
        return False

    def forward(self, x: torch.Tensor, ctx, call: int, fold=None) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n = x.shape[0]
        packed = ws.get("mstate.packed", (n, self.width), rt.dtype)
        ops.gemm(x, self.w_packed, packed)
        gated = ws.get("mstate.gated", (n, spec.inner), rt.dtype)
        self.recur(packed, 0, ctx, call, gated)
        y = ws.get("mixer.out", (n, spec.hidden_size), rt.dtype)
        return ops.gemm(gated, self.w_o, y, defer_sum=True, fold=fold) or y
