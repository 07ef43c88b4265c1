"""Which steps' walks over the keys are cut in two: room for their sums is there before the cache is sized, and the rule holds to its lines."""
import ctypes
import random
from types import SimpleNamespace

import pytest
import torch

from minivllm_amd.csrc import build
from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.kernels.library import KernelLibraryError
from minivllm_amd.kernels.ops import PROMPT_SPLIT_UNITS, Ops
from minivllm_amd.parts.base import Workspace

HEADS = [(16, 8), (32, 8), (64, 8), (4, 2), (24, 24), (6, 2)]


def rule():
    ops = SimpleNamespace(lib=SimpleNamespace(has=lambda name: True, dll=ctypes.CDLL(build.find_library("bf16") or build.build("bf16"))),
                          compute_units=256, use_fast_kernels=True, dtype=torch.bfloat16, _attn_counters=None)
    ops._prompt_counters = Ops._prompt_counters
    for name in ("_prefill_limit", "_prefill_room", "_counted_launch", "reserve_prompt_attention", "_prefill_variant"):
        setattr(ops, name, getattr(Ops, name).__get__(ops))
    return ops


def plan_of(lens, bound=None):
    return AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=max(lens), n_seqs=len(lens), q_lens=() if bound else list(lens), bound=bound,
                         workspace=Workspace(torch.device("meta")))


@pytest.mark.parametrize("H, Hkv", HEADS)
@pytest.mark.parametrize("D", [64, 128])
def test_any_steps_parts_fit_what_is_reserved(H, Hkv, D):
    ops, rng, cut = rule(), random.Random(H + D), 0
    for tokens, seqs in ((700, 8), (2048, 4), (8192, 288)):
        ws = Workspace(torch.device("meta"))
        Ops.reserve_prompt_attention(ops, ws, tokens, seqs, H, Hkv, D)
        ws.frozen = True                 # (a buffer that would have to grow raises)
        for _ in range(200):
            n = rng.choice([1, 1, 2, 3, min(5, seqs), seqs])
            total = rng.randint(n, tokens)
            ends = sorted(rng.sample(range(1, total), n - 1)) if n > 1 else []
            lens = [b - a for a, b in zip([0] + ends, ends + [total])]
            for plan in (plan_of(lens), plan_of(lens, bound=(total, rng.randint(n, seqs)))):
                nt, kw, units, busy, limit = ops._prefill_variant(plan, H // Hkv, Hkv)
                if limit:
                    cut += 1
                    assert kw == 1 and limit % 2 == 0 and units * Hkv <= PROMPT_SPLIT_UNITS
                    need = units * Hkv * ops.lib.dll.mv_attention_prefill_part_floats(nt, D)
                    ws.get("attn.prompt_partials", (need,), torch.float32)
    assert cut or H == 4                 # (two heads of two never fill the chip)


def test_the_lines():
    ops = rule()
    variant = lambda lens, H=16, keys=None, sums=False: ops._prefill_variant(plan_of(lens), H // 8, 8, keys, sums)
    assert variant([1408])[:2] == (1, 2) and variant([1408])[4] == 0
    assert variant([2048])[:2] == (1, 1) and variant([2048])[4] == 44
    assert variant([4096])[:2] == (2, 1) and variant([4096])[4] in (74, 76)
    assert variant([8192])[4] == 0                                        # enough units
    assert variant([2048], keys=1024)[4] == 0 and variant([2048], keys=2048)[4] == 44          # a window that no walk leaves
    assert variant([4096], sums=True)[:2] != (2, 1) or variant([4096], sums=True)[4] == 0      # sums of sigmoid weights: 16 columns a wave only
    assert ops._prefill_variant(plan_of([2048], bound=(2048, 1)), 2, 8)[4] == 44


@pytest.mark.parametrize("rows", [1408, 2048, 4096])
def test_a_plan_without_a_workspace_has_whole_walks(rows):
    """As every plan had before walks were cut; a forced cut has no room and is refused."""
    ops, plan, whole = rule(), plan_of([rows]), plan_of([rows])
    plan.workspace, ops_whole = None, rule()
    ops_whole._prefill_limit = lambda *args: 0
    nt, kw, units, busy, limit = ops._prefill_variant(plan, 2, 8)
    assert (nt, kw, units, busy, limit) == ops_whole._prefill_variant(whole, 2, 8)
    assert ops._prefill_room(plan.workspace, limit, nt, units, 8, 128) == (None, None, 0)
    with pytest.raises(KernelLibraryError):
        ops._prefill_room(None, 16, nt, units, 8, 128)


def test_two_workspaces_share_no_counters(monkeypatch):
    """Steps on two streams have a workspace each and may overlap, also on one ``Ops``: what a launch counts in is its workspace's, zero at first; a launch
    that fails leaves zeros behind, in its own."""
    ops, room = rule(), [Workspace(torch.device("cpu")) for _ in range(2)]
    taken = [ops._prefill_room(ws, 16, 1, 40, 8, 128) for ws in room]
    assert len({pointer for r in taken for pointer in r[:2]}) == 4 and ops._attn_counters is None
    counters = [ops._prompt_counters(ws, 320) for ws in room]
    assert [c.data_ptr() for c in counters] == [r[1] for r in taken] and not any(bool(c.any()) for c in counters)
    for c in counters:
        c[5] = 1
    room[0].frozen = True
    assert ops._prefill_room(room[0], 30, 1, 20, 8, 128)[1] == taken[0][1] and int(counters[0][5]) == 1      # (those of a launch on its way)

    def fails(entry, *args):
        raise KernelLibraryError(entry)
    ops.lib.call = fails
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    with pytest.raises(KernelLibraryError):
        ops._counted_launch(lambda: counters[0], "mv_attention_prefill")
    assert not bool(counters[0].any()) and int(counters[1][5]) == 1
