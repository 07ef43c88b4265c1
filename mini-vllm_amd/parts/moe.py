"""A mixture of gated feed-forward experts behind a softmax router.

Router logits z = W_router x in float32; scores s = softmax(z) over all router outputs. The last
``identity_experts`` outputs are identity experts (their output is x itself, they have no tensors), the
others are gated SiLU pairs down_e(silu(gate_e x) * (up_e x)). A token uses ``top`` experts: those with
the largest s + correction (the correction steers the choice only, never the weights), restricted to
the ``keep_groups`` of ``groups`` equal runs of neighbouring router outputs whose largest such number is
largest (outputs of other groups cannot be chosen whatever their number). The weights are the chosen
experts' scores divided by their sum (+ weight_sum_eps); the result is the weighted sum of the
chosen experts' outputs.

How it runs: in bfloat16, with widths that are multiples of 64 and where it takes less time (``wants_pairs``: many experts of
which few are chosen, or large steps), the chosen (token, expert) pairs are sorted by expert on the device, every expert's
pairs are cut into tiles of up to 128 rows, and two MFMA kernels compute gate/up with the weighted activation and the down
product for those tiles only; a last kernel sums a token's pairs in the order of choice and adds the identity experts'
share (csrc/moe_tile.hip). Otherwise gate and up matrices of all experts form one packed product and all down matrices one
second product; between them one kernel applies SiLU, the up factor and the router's weight (zero for experts that were not
chosen) before the single rounding, so the second product sums exactly the chosen experts.
That is exact and replays from graphs, but computes every expert: eight times the useful multiply-adds when a token uses an
eighth of the experts, and every expert's bytes in a decode step. Widths that are odd multiples of 32 may take the pairs
through plain MFMA kernels instead (``grouped``; operands straight from memory): only in steps of few rows against large
experts, as the spec's thresholds say, where bytes decide. Either way everything is decided on the device; nothing about
a step's routing reaches the host, so steps replay from graphs.

Options of the spec, each with the default that gives the above: ``scoring`` "sigmoid" scores every router
output by sigmoid(z) on its own; ``group_worth`` "top2" ranks a group by the sum of its two largest choices
instead of its largest; ``normalize`` False uses the chosen scores themselves as weights; ``activation``
"clamped" replaces the gated SiLU pair by g = min(gate, limit), u = clamp(up, -limit, limit),
g * sigmoid(gate_slope * g) * (u + 1).

``router`` "table": there is no router. A stored integer table [``table_rows``, ``top``] names the experts of every
token id (the step's ``ctx.token_ids``), each with the weight 1 / top; with all experts at once the activation kernel
looks the weights up itself, the chosen-pairs paths get the usual lists from ``moe_table_route``. ``shared_size`` > 0:
a shared expert (a gated pair like the others) runs for every token and is added: its rows ride in the two packed
products (and are one more expert of the tiled pairs), or, where steps may take the plain chosen-pairs kernels, it keeps two
products of its own.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Dict

import torch

from .base import FeedForward, PartSpec, Runtime, TensorDecl, register_feed_forward


@dataclass(frozen=True)
class RoutedExpertsSpec(PartSpec):
    kind = "routed_swiglu"
    hidden_size: int = 0
    expert_size: int = 0                 # width of one expert's gated pair
    num_experts: int = 0                 # experts with tensors
    identity_experts: int = 0            # router outputs behind them whose expert is the identity
    top: int = 1
    groups: int = 1
    keep_groups: int = 1
    correction: bool = False             # a stored number per router output added to the scores for the choice
    weight_sum_eps: float = 1e-20
    # bfloat16: the experts' products over the chosen (token, expert) pairs only. Widths that are multiples of 64 go in tiles
    # where that takes less time (``RoutedExperts.wants_pairs``); other multiples of 32, and steps that the tiles leave,
    # through plain kernels, with fewer than ``grouped_max_rows`` chosen rows an expert on average and experts of at
    # least ``grouped_min_weight`` elements a matrix (there a step is bound by the bytes of the experts it reads, and most
    # experts are not chosen)
    grouped: bool = True
    grouped_max_rows: float = 2.0
    grouped_min_weight: int = 4 * 1024 * 1024
    scoring: str = "softmax"             # or "sigmoid"
    group_worth: str = "max"             # or "top2": the sum of a group's two largest choices
    normalize: bool = True               # False: the weights are the chosen scores as they are
    activation: str = "swiglu"           # or "clamped" (with ``limit`` and ``gate_slope``)
    limit: float = 0.0
    gate_slope: float = 1.702
    # "table": no router product; a stored integer table [table_rows, top] names the experts of every token id, each
    # with the weight 1 / top (``groups``, ``correction``, ``scoring`` and ``normalize`` then mean nothing)
    router: str = "learned"
    table_rows: int = 0
    # > 0: a shared expert of that width (a gated pair like the others) runs for every token and is added
    shared_size: int = 0

    @property
    def router_outputs(self) -> int:
        return self.num_experts + self.identity_experts


@register_feed_forward(RoutedExpertsSpec.kind)
class RoutedExperts(FeedForward):
    spec_class = RoutedExpertsSpec

    @classmethod
    def tensors(cls, spec: RoutedExpertsSpec) -> Dict[str, TensorDecl]:
        if spec.router == "table":
            t = {"table": TensorDecl((spec.table_rows, spec.top), init=f"distinct_below:{spec.num_experts}", integer=True)}
        else:
            t = {"router": TensorDecl((spec.router_outputs, spec.hidden_size))}
        if spec.shared_size:
            t["shared.gate"] = TensorDecl((spec.shared_size, spec.hidden_size))
            t["shared.up"] = TensorDecl((spec.shared_size, spec.hidden_size))
            t["shared.down"] = TensorDecl((spec.hidden_size, spec.shared_size))
        if spec.correction:
            t["correction"] = TensorDecl((spec.router_outputs,), init="zeros_normal")
        for e in range(spec.num_experts):
            t[f"gate.{e}"] = TensorDecl((spec.expert_size, spec.hidden_size))
            t[f"up.{e}"] = TensorDecl((spec.expert_size, spec.hidden_size))
            t[f"down.{e}"] = TensorDecl((spec.hidden_size, spec.expert_size))
        return t

    def __init__(self, spec: RoutedExpertsSpec, tensors: Dict[str, torch.Tensor], rt: Runtime):
        E = spec.router_outputs
        if spec.num_experts < 0 or spec.identity_experts < 0 or E < 1 or spec.groups < 1 or E % spec.groups \
                or not (1 <= spec.keep_groups <= spec.groups) or not (1 <= spec.top <= E // spec.groups * spec.keep_groups):
            raise ValueError(f"routed experts: bad sizes {spec}")
        if spec.scoring not in ("softmax", "sigmoid") or spec.group_worth not in ("max", "top2") \
                or spec.activation not in ("swiglu", "clamped") or (spec.activation == "clamped" and not spec.limit > 0):
            raise ValueError(f"routed experts: unknown scoring, group worth or activation, or a clamped pair without a "
                             f"positive limit: {spec}")
        if spec.router not in ("learned", "table") or spec.shared_size < 0:
            raise ValueError(f"routed experts: the router is 'learned' or 'table' and a shared expert's width >= 0: {spec}")
        if spec.router == "table" and (spec.identity_experts or spec.correction or spec.table_rows < 1 or not spec.num_experts):
            raise ValueError(f"routed experts: a table names experts with tensors, for every token id: {spec}")
        if spec.shared_size and not spec.num_experts:
            raise ValueError("routed experts: a shared expert stands beside experts with tensors")
        self.spec, self.rt = spec, rt
        self.w_router = tensors.get("router")
        self.table = tensors.get("table")
        self.correction = tensors.get("correction")
        n_e = spec.num_experts
        if n_e:
            names = [f"{k}.{e}" for e in range(n_e) for k in ("gate", "up", "down")]
            if spec.shared_size:
                names += ["shared.gate", "shared.up", "shared.down"]
            dtypes = {tensors[name].dtype for name in names}
            if len(dtypes) != 1:
                raise ValueError(f"routed experts: the experts are stored in different dtypes {dtypes}; cannot pack them")
            # rows: every expert's gate block, then every expert's up block; the down matrices side by side. A shared
            # expert's gate and up rows come behind those and its down matrix behind the others' (one pair of products
            # serves all), unless steps may take the plain chosen-pairs kernels, which know no shared expert: then it keeps
            # matrices and products of its own
            always_tiled = self._tiled(dtypes.pop(), spec.shared_size) and self._always_pairs()
            self.shared_packed = bool(spec.shared_size) and (always_tiled or not self._grouped_possible())
            shared_rows = [tensors["shared.gate"], tensors["shared.up"]] if spec.shared_size else []
            self.w_gate_up = torch.cat([tensors[f"gate.{e}"] for e in range(n_e)] + [tensors[f"up.{e}"] for e in range(n_e)]
                                       + (shared_rows if self.shared_packed else []), dim=0).contiguous()
            self.w_down = torch.cat([tensors[f"down.{e}"] for e in range(n_e)]
                                    + ([tensors["shared.down"]] if self.shared_packed else []), dim=1).contiguous()
            if spec.shared_size and not self.shared_packed:
                self.w_shared_gate_up = torch.cat(shared_rows, dim=0).contiguous()
                self.w_shared_down = tensors["shared.down"]

    def _grouped_possible(self) -> bool:
        spec = self.spec
        return (spec.grouped and self.rt.ops.use_fast_kernels and self.rt.dtype == torch.bfloat16
                and spec.expert_size * spec.hidden_size >= spec.grouped_min_weight)

    def wants_grouped(self, n: int) -> bool:
        """Whether a step of n rows computes the chosen pairs only (where the kernels take the sizes)."""
        spec = self.spec
        return (spec.grouped and n * spec.top < spec.grouped_max_rows * spec.num_experts
                and spec.expert_size * spec.hidden_size >= spec.grouped_min_weight)

    def _tiled(self, stored: torch.dtype, shared_size: int) -> bool:
        """Whether the tiled products over the chosen pairs take these widths."""
        spec = self.spec
        return (spec.grouped and self.rt.ops.use_fast_kernels and self.rt.dtype == torch.bfloat16 and stored == torch.bfloat16
                and not (spec.hidden_size % 64 or spec.expert_size % 64 or shared_size % 64))

    def _always_pairs(self) -> bool:
        """Experts of which the chosen ones alone take less time whatever the number of rows (see ``wants_pairs``)."""
        E, expert = self.spec.num_experts, self.spec.expert_size * self.spec.hidden_size
        return E * expert >= 1024 * 1024 and E >= 3 * self.spec.top and (E >= 12 or expert >= 4 * 1024 * 1024)

    def wants_pairs(self, n: int) -> bool:
        """Whether a step of n rows goes through the tiled products over the chosen pairs (where the kernels take the sizes).
        They save the products and weights of the experts that are not chosen, and cost one launch more and rows of tiles that
        few pairs fill. Both sides on an MI355X (us a layer, pairs / all experts), width x expert, experts and choices:
        always, 1024 x 768, 32 of 4: 34 / 62 at one row, 66 / 80 at 128, 131 / 406 at 2,048; 16 of 4 33 / 40, 51 / 56, 115 / 210;
        12 of 4 32 / 37, 47 / 50, 109 / 176; 4096 x 3072, 8 of 2 66 / 233, 162 / 186, 593 / 1,108. In large steps only: 1024 x 768,
        8 of 4 53 / 48 at 128, 69 / 78 at 1,024; 4 of 2 49 / 32 and 55 / 51, 67 / 69 at 2,048; 16 of 8 67 / 56, 116 / 142. Large experts
        in steps that leave experts unchosen: 4096 x 3072, 8 of 4 95 / 252 at one row, 275 / 235 at 256; 4 of 2 68 / 229, 162 / 136.
        Small mixtures, bound by launches, never: 64 x 64, 8 of 2 19 / 16 and 35 / 27; 128 x 128, 16 of 4 22 / 18, 45 / 42."""
        spec, FS = self.spec, self.spec.shared_size if self.shared_packed else 0
        if not self._tiled(self.w_gate_up.dtype, FS):
            return False
        E, top, expert, shared = spec.num_experts, spec.top, spec.expert_size * spec.hidden_size, 1 if FS else 0
        return self._always_pairs() or (expert >= 4 * 1024 * 1024 and n * top < E) \
            or (E * expert >= 1024 * 1024 and E + shared >= 2 * (top + shared) and n * E >= self.LARGE_STEP)

    LARGE_STEP = 8192                    # (token, expert) pairs, chosen or not, from which a step is a large one

    def reserve(self, tokens: int) -> None:
        # a step of ``tokens`` may take the chosen pairs where a smaller one takes all experts
        for n in (tokens, min(tokens, (self.LARGE_STEP - 1) // max(1, self.spec.num_experts))):
            if n > 0 and self.spec.num_experts and not self.wants_pairs(n):
                self._all_experts_scratch(n)
                break
        if self.spec.shared_size and not self.shared_packed:
            self._shared_gate_up(tokens)            # (which numbers of rows go in one pass does not grow with them)

    def _shared_gate_up(self, n: int) -> torch.Tensor:
        return self.rt.workspace.get("moe.shared_gate_up", (n, 2 * self.spec.shared_size), self.rt.dtype)

    def _all_experts_scratch(self, n: int):
        spec, rt = self.spec, self.rt
        F, FS = spec.num_experts * spec.expert_size, spec.shared_size if self.shared_packed else 0
        return rt.workspace.get("moe.gate_up", (n, 2 * F + 2 * FS), rt.dtype), rt.workspace.get("moe.act", (n, F + FS), rt.dtype)

    def _pairs(self, x: torch.Tensor, dense, ids, weights, y) -> bool:
        """The chosen (token, expert) pairs only, a packed shared expert among them. False: the sizes are not served."""
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, n_e, F, FS = x.shape[0], spec.num_experts, spec.expert_size, spec.shared_size if self.shared_packed else 0
        pairs = n * (spec.top + (1 if FS else 0))
        return ops.lib.has("mv_moe_pairs") and ops.moe_pairs(
            x, self.w_gate_up, self.w_down, n_e, spec.identity_experts, F, FS, ids, weights, dense,
            ws.get("moe.ints", (ops.moe_pairs_ints(n, spec.top, n_e, FS),), torch.int32),
            ws.get("moe.pair_act", (pairs, max(F, FS)), rt.dtype), ws.get("moe.pair_out", (pairs, spec.hidden_size), torch.float32), y,
            limit=spec.limit if spec.activation == "clamped" else 0.0, slope=spec.gate_slope)

    def _grouped(self, x: torch.Tensor, ctx, dense, ids, weights, y) -> bool:
        """The chosen (token, expert) pairs only: sorted by expert on the device, tiles of 64 rows through MFMA.
        False: the sizes are not served."""
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, n_e, F = x.shape[0], spec.num_experts, spec.expert_size
        need = int(ops.lib.dll.mv_moe_grouped_ints(n, spec.top, n_e)) if ops.lib.has("mv_moe_grouped") else 0
        return bool(need) and ops.moe_grouped(
            x, self.w_gate_up, self.w_down, n_e, spec.identity_experts, F, ids, weights, dense,
            ws.get("moe.ints", (need,), torch.int32), ws.get("moe.pair_act", (n * spec.top, F), rt.dtype),
            ws.get("moe.pair_out", (n * spec.top, spec.hidden_size), torch.float32), y,
            limit=spec.limit if spec.activation == "clamped" else 0.0, slope=spec.gate_slope)

    def _add_shared(self, x: torch.Tensor, y: torch.Tensor) -> None:
        """y += the shared expert's output, as two products of its own."""
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        n, FS = x.shape[0], spec.shared_size
        if spec.activation != "swiglu":
            raise NotImplementedError("a shared expert with matrices of its own is a gated SiLU pair")
        act = ws.get("moe.shared_act", (n, FS), rt.dtype)
        if not ops.gemm_swiglu(x, self.w_shared_gate_up, act):
            gu = self._shared_gate_up(n)
            ops.gemm(x, self.w_shared_gate_up, gu)
            ops.swiglu(gu, act)
        ys = ws.get("moe.shared_out", (n, spec.hidden_size), rt.dtype)
        ops.gemm(act, self.w_shared_down, ys)
        ops.add_rows(y, ys)

    def forward(self, x: torch.Tensor, ctx) -> torch.Tensor:
        spec, rt, ops, ws = self.spec, self.rt, self.rt.ops, self.rt.workspace
        if not isinstance(x, torch.Tensor):
            x = x.materialize()
        n, E, n_e, F = x.shape[0], spec.router_outputs, spec.num_experts, spec.expert_size
        FS = spec.shared_size if n_e and self.shared_packed else 0
        apart = bool(spec.shared_size) and not FS
        dense = ws.get("moe.dense", (n, E), torch.float32)
        ids = ws.get("moe.ids", (n, spec.top), torch.int32)
        weights = ws.get("moe.weights", (n, spec.top), torch.float32)
        by_table = spec.router == "table"
        pairs = bool(n_e) and self.wants_pairs(n)
        grouped = bool(n_e) and not FS and ops.use_fast_kernels and self.wants_grouped(n)
        if by_table and (pairs or grouped):
            ops.moe_table_route(ctx.token_ids, self.table, n_e, dense, ids, weights)
        elif by_table:
            pass                  # all experts at once: the activation kernel looks the weights up itself
        else:
            logits = ws.get("moe.logits", (n, E), torch.float32)
            ops.gemm(x, self.w_router, logits)
            ops.moe_route(logits, self.correction, spec.groups, spec.keep_groups, spec.top, spec.weight_sum_eps, dense, ids, weights,
                          scoring=spec.scoring, group_worth=spec.group_worth, normalize=spec.normalize)
        y = ws.get("ffn.out", (n, spec.hidden_size), rt.dtype)
        # (sizes that are not served after all: the kernel below takes the dense weights or the table)
        if (pairs and self._pairs(x, dense, ids, weights, y)) or (grouped and self._grouped(x, ctx, dense, ids, weights, y)):
            if apart:
                self._add_shared(x, y)
            return y
        if n_e:
            gu, act = self._all_experts_scratch(n)
            ops.gemm(x, self.w_gate_up, gu)
            table = (ctx.token_ids, self.table) if by_table else None
            if spec.activation == "clamped":
                ops.moe_swiglu_scale(gu, None if by_table else dense, n_e, F, act, limit=spec.limit, slope=spec.gate_slope,
                                     shared=FS, table=table)
            else:
                ops.moe_swiglu_scale(gu, None if by_table else dense, n_e, F, act, shared=FS, table=table)
            ops.gemm(act, self.w_down, y)
            if apart:
                self._add_shared(x, y)
        if spec.identity_experts or not n_e:
            ops.moe_identity_add(y, x, dense, n_e, spec.identity_experts, overwrite=not n_e)
        return y
