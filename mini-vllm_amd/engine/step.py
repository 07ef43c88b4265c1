"""The step function's input and the context every part sees during a step.

A step is a batch of (request, its next tokens): portions of prompts beside single decoded
tokens, cut anywhere. Reference: the reference builds either a prefill input (whole uncached
prompts; minivllm/executor/executor.py:81-127) or a decode input (one token per request;
executor.py:130-153) and hands the layers a ``Context`` with cu_seqlens / slot_mapping /
cache_seqlens / block_table (minivllm/executor/context.py). Here one layout serves both and
any mix: flat token ids and positions, the sequence each token belongs to, per sequence the
range of its tokens and its context length, one block table per cache group; cache slots are
computed by the kernels from position and block table.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, List, Optional, Sequence

import torch

# token counts that steps with prompt portions are padded to when they are replayed from a graph:
# at most an eighth more than the step holds (from 9 tokens on 16, up to 8 tokens 8: there the products change hands, and a step
# is to add in the same order recorded and not; gemm_deep.hip knows these classes)
TOKEN_BUCKETS = ([8] + list(range(16, 129, 16)) + list(range(160, 257, 32)) + list(range(320, 513, 64))
                 + list(range(640, 1025, 128)) + list(range(1280, 2049, 256)) + list(range(2560, 4097, 512))
                 + list(range(5120, 8193, 1024)))


def class_rows(tokens: int) -> int:
    """The rows of a step of so many tokens when it is recorded (more than the largest class: the tokens)."""
    return next((b for b in TOKEN_BUCKETS if b >= tokens), tokens)


@dataclass
class SeqStep:
    """One request's share of a step.

    tokens        the next tokens of the request (>= 1)
    start         position of tokens[0] = number of the request's tokens already in the cache
    block_tables  per cache group, the request's page ids by page index (-1: given back)
    state_slot    row of the state tensors that belongs to the request
    want          indices into ``tokens`` whose logits are returned, in this order
    """
    tokens: Sequence[int]
    start: int
    block_tables: Sequence[Sequence[int]]
    state_slot: int = 0
    want: Sequence[int] = ()


@dataclass
class KVView:
    """Cache of one call as its mixer sees it: the page tensors its ``CacheNeed`` named
    (``[pages, *page shape]`` each), the block table of its group and the page size."""
    pages: Dict[str, torch.Tensor]
    block_table: torch.Tensor      # int32 [sequences, width] of the call's group
    page_size: int

    @property
    def k_pages(self) -> torch.Tensor:      # softmax attention: [pages, kv_heads, page_size, head_dim]
        return self.pages["k"]

    @property
    def v_pages(self) -> torch.Tensor:      # [pages, kv_heads, head_dim, page_size]
        return self.pages["v"]


def most_units(tokens: int, seqs: int, unit_tokens: int, least: int = 1) -> int:
    """The most runs of up to ``unit_tokens`` tokens that up to ``seqs`` sequences of at least ``least`` tokens each, ``tokens``
    in all, can have: each adds less than one to what its tokens fill."""
    return tokens // unit_tokens + min(seqs, tokens // least)


@dataclass
class AttentionPlan:
    """Host-side facts about the step that let the attention pick a kernel."""
    decode_only: bool              # every sequence brings exactly one token
    max_q_len: int
    max_context_len: int           # longest context the step (or the graph it is captured in) must serve
    n_seqs: int                    # rows of cu_seqlens - 1, padding sequences included
    q_lens: Sequence[int] = ()     # tokens per sequence, on the host
    cu_seqlens: Optional[torch.Tensor] = None   # int32 [n_seqs + 1] on the device
    workspace: Optional[object] = None          # where kernels take scratch memory from
    # decode steps: over how many workgroups a sequence's keys are dealt out; None lets the launch
    # rule choose (tests force counts)
    decode_splits: Optional[int] = None
    # prompt steps: (column tiles per wave, key groups per workgroup) of the MFMA kernel; None lets the
    # launch rule choose (tests force variants)
    prefill_variant: Optional[tuple] = None
    # steps recorded into a graph that serves any cut of up to (tokens, sequences): the kernels' grids
    # are then sized for the worst cut, not for ``q_lens`` (workgroups without work end at once)
    bound: Optional[tuple] = None
    # ... whose steps hold at least this many tokens
    bound_least: int = 1
    # ... and for which every part that chooses by the sequences' lengths and places (``Mixer.step_path``) chooses as for these
    path_lens: Sequence[int] = ()
    path_starts: Sequence[int] = ()
    # for measurement: keys in the cache of the step's sequences after the step (summed), and the
    # number of (query, visible key) pairs without windows
    kv_tokens: int = 0
    attention_pairs: int = 0
    # the position of each sequence's first token of the step and, for measurement, its number of tokens, on the
    # host (a recording for a size class clears ``q_lens``; these stay those of the step that was recorded)
    starts: Sequence[int] = ()
    step_q_lens: Sequence[int] = ()

    def cut(self) -> tuple:
        """Tokens and first positions of the sequences by which parts may choose: the step's own, or those that stand for a
        recording's; both empty where neither is known."""
        lens, starts = (self.q_lens, self.starts) if self.bound is None else (self.path_lens, self.path_starts)
        return (lens[:len(starts)], starts) if starts else ((), ())

    def units(self, unit_tokens: int, least: int = 1) -> int:
        """Runs of up to ``unit_tokens`` consecutive tokens of one sequence in the step, of the sequences that
        bring at least ``least``: counted from the host's lengths, or the most that any cut within ``bound`` can have."""
        if self.bound is not None:
            return most_units(*self.bound, unit_tokens, least)
        return sum(-(-ql // unit_tokens) for ql in self.q_lens if ql >= least)

    def has_long(self, tokens: int) -> bool:
        """Whether a sequence may bring at least so many tokens to the step."""
        return self.bound[0] >= tokens if self.bound is not None else any(q >= tokens for q in self.q_lens)

    def has_short(self, tokens: int) -> bool:
        """Whether a sequence may bring fewer."""
        if self.bound is not None:
            return self.bound[1] > 1 or self.bound_least < tokens
        return any(0 < q < tokens for q in self.q_lens)

    def busy_units(self, unit_tokens: int) -> int:
        """The units that hold tokens, for rules that weigh the work against the device: the count
        itself, or, of a bound, the units its tokens fill (the rest of ``units`` are spares that end
        at once)."""
        if self.bound is not None:
            return max(1, self.bound[0] // unit_tokens)
        return self.units(unit_tokens)


class StepContext:
    """Device tensors (int32) and host facts describing the step, handed to every part.

    token_ids [n]      positions [n]        token_seq [n] (sequence index, -1 = padding row)
    cu_seqlens [s+1]   context_lens [s]     state_slots [s]      logit_rows [m]
    """

    def __init__(self):
        self.n_tokens = 0
        self.n_seqs = 0
        self.n_logit_rows = 0
        self.token_ids: torch.Tensor = None
        self.positions: torch.Tensor = None
        self.token_seq: torch.Tensor = None
        self.cu_seqlens: torch.Tensor = None
        self.context_lens: torch.Tensor = None
        self.state_slots: torch.Tensor = None
        self.logit_rows: torch.Tensor = None
        self.block_tables: List[torch.Tensor] = []
        # host copies
        self.q_lens: List[int] = []
        self.starts: List[int] = []
        self.host_state_slots: List[int] = []
        self.attention_plan: Optional[AttentionPlan] = None
        # filled by the executor
        self._kv: Dict[int, "KVView"] = {}
        self._state: Dict[int, Dict[str, torch.Tensor]] = {}
        self.page_size = 0
        # rows that a position encoding had gathered for this step (PositionEncoding.step_gather), by part
        self.position_rows: Dict[object, torch.Tensor] = {}
        # what a part leaves for parts of later calls of the same step, by a key of their own choosing (the
        # values a layer projected, which later layers blend into theirs)
        self.carry: Dict[str, torch.Tensor] = {}

    def kv(self, call: int) -> KVView:
        try:
            return self._kv[call]
        except KeyError:
            raise KeyError(f"call {call} has no cache: its mixer declared no cache need") from None

    def state(self, call: int, name: str = "state") -> torch.Tensor:
        """``[slots, *shape]`` of the state ``name`` of a call ("state": the one a mixer's
        ``state_shape`` declares)."""
        try:
            return self._state[call][name]
        except KeyError:
            raise KeyError(f"call {call} has no state {name!r}: neither its mixer nor its block declared it") from None
