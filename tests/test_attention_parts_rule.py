"""Which steps' walks over the keys are cut in two: room for their sums is there before the cache is sized, and the rule holds to its lines."""
import ctypes
import random
from types import SimpleNamespace

import pytest
import torch

from minivllm_amd.csrc import build
from minivllm_amd.engine.step import AttentionPlan, class_rows
from minivllm_amd.kernels.library import KernelLibraryError
from minivllm_amd.kernels.ops import PROMPT_SPLIT_UNITS, Ops
from minivllm_amd.parts.base import Workspace

HEADS = [(16, 8), (32, 8), (64, 8), (4, 2), (24, 24), (6, 2)]


def rule():
    ops = SimpleNamespace(lib=SimpleNamespace(has=lambda name: True, dll=ctypes.CDLL(build.find_library("bf16") or build.build("bf16"))),
                          compute_units=256, use_fast_kernels=True, dtype=torch.bfloat16, _attn_counters=None)
    ops._prompt_counters = Ops._prompt_counters
    ops._keys_seen = Ops._keys_seen
    for name in ("_prompt_parts", "_cut_walks", "prompt_attention_path", "_prefill_room", "_counted_launch", "reserve_prompt_attention", "_prefill_variant"):
        setattr(ops, name, getattr(Ops, name).__get__(ops))
    return ops


def plan_of(lens, bound=None, starts=None):
    starts = [0] * len(lens) if starts is None else starts
    plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=max(map(sum, zip(lens, starts))), n_seqs=len(lens),
                         q_lens=() if bound else list(lens), starts=list(starts), bound=bound, workspace=Workspace(torch.device("meta")))
    if bound:
        plan.path_lens, plan.path_starts = tuple(lens), tuple(starts)
    return plan


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
            starts = [rng.choice([0, 0, rng.randint(0, 9000)]) for _ in lens]
            for plan in (plan_of(lens, starts=starts), plan_of(lens, (total, rng.randint(n, seqs)), starts)):
                nt, kw, units, busy, limit = ops._prefill_variant(plan, H // Hkv, Hkv)
                if limit:
                    cut += 1
                    assert kw == 1 and limit % 2 == 0 and units * Hkv <= PROMPT_SPLIT_UNITS
                    need = units * Hkv * ops.lib.dll.mv_attention_prefill_part_floats(nt, D)
                    ws.get("attn.prompt_partials", (need,), torch.float32)
    assert cut or H == 4                 # (two heads of two never fill the chip)


def test_the_lines():
    ops = rule()
    variant = lambda lens, H=16, keys=None, sums=False, **more: ops._prefill_variant(plan_of(lens, **more), H // 8, 8, keys, sums)
    assert variant([1408])[:2] == (1, 2) and variant([1408])[4] == 0
    assert variant([2048])[:2] == (1, 1) and variant([2048])[4] == 44
    assert variant([4096])[:2] == (2, 1) and variant([4096])[4] in (74, 76)
    assert variant([8192])[4] == 0                                        # enough units
    assert variant([2048], keys=1024)[4] == 0 and variant([2048], keys=2048)[4] == 44          # a window that no walk leaves
    assert variant([4096], sums=True)[:2] != (2, 1) or variant([4096], sums=True)[4] == 0      # sums of sigmoid weights: 16 columns a wave only
    assert ops._prefill_variant(plan_of([2048], bound=(2048, 1)), 2, 8)[4] == 44


WHOLE = {16: [[1024, 1024], [900, 1200], [1100, 700], [512] * 4, [256] * 8, [700] * 4, [1333] * 3, [1569, 805, 1625], [2000, 2000]],
         32: [[1024, 1024], [1177, 604], [1100, 700], [512] * 4, [256] * 8, [2000, 2000]], 64: [[1024, 1024], [1200], [512] * 4]}


@pytest.mark.parametrize("H", WHOLE)
def test_prompts_without_a_long_walk_of_their_own_stay_whole(H):
    """... in the launch that such a step has without the rule: no second half of a grid that ends at once, heavy units beside light ones, two key groups."""
    ops, uncut = rule(), rule()
    uncut._cut_walks = lambda *args: (0, 0)
    for lens in WHOLE[H]:
        for bound in (None, (class_rows(sum(lens)), 8)):
            plan = plan_of(lens, bound)
            assert ops._prefill_variant(plan, H // 8, 8) == uncut._prefill_variant(plan, H // 8, 8), lens


def test_the_walks_are_those_behind_the_contexts():
    """A portion's walks begin at position zero: the limit grows with the context, and walks that are about equally long stay whole where they make
    whole rounds. One long prompt beside others that are short is cut as it is alone."""
    ops = rule()
    variant = lambda lens, starts, H=16: ops._prefill_variant(plan_of(lens, starts=starts), H // 8, 8)
    for start in (1024, 2048, 4096, 8192):
        assert variant([2048], [start])[4] == 0 and variant([4096], [8192])[4] == 0
    limits = [variant([3000], [start])[4] for start in (0, 256, 1024, 2048, 4096)]
    assert limits == sorted(limits) and limits[0] < 50 and limits[-1] > 140
    assert all(variant([rows], [start])[4] > 0 for rows, start in ((1536, 1024), (1536, 8192), (1700, 2048), (4096, 2048), (5000, 8192)))
    assert variant([1900, 148], [0, 0])[4] > 0 and variant([3500, 100, 100], [0, 0, 0])[4] > 0
    assert variant([2000] + [1] * 40, [0] + list(range(1100, 1500, 10)))[4] == 0               # decoding requests have more walks than the prompt
    plan = plan_of([900, 1148])
    plan.starts = ()                                                      # (a plan that does not say where they start)
    assert ops._prefill_variant(plan, 2, 8)[4] == 0


@pytest.mark.parametrize("H, Hkv", HEADS)
def test_a_recordings_key_says_how_it_was_cut(H, Hkv):
    """Every step of a class that is cut alike runs the same launch: what the key holds is what the launch rule makes of any of its steps, and a class has
    few keys though its contexts differ."""
    ops, rng, keys = rule(), random.Random(H), {}
    for _ in range(3000):
        lens, starts = [rng.randint(600, 2048)], [rng.choice([0, rng.randint(1, 4000)])]
        if rng.random() < 0.3:
            lens, starts = lens + [rng.randint(1, 200)], starts + [rng.randint(0, 1000)]
        if sum(lens) > 2048:
            continue
        rows, seqs = class_rows(sum(lens)), len(lens)
        nt, limit = key = ops.prompt_attention_path(lens, starts, rows, H, Hkv, 128)
        got = ops._prefill_variant(plan_of(lens, (rows, seqs), starts), H // Hkv, Hkv)
        assert (got[0], got[4]) == key if limit else got[4] == 0
        cap = max(1024, 1 << (max(map(sum, zip(lens, starts))) - 1).bit_length())
        keys.setdefault((rows, seqs, cap), set()).add(key)
    assert max(map(len, keys.values())) <= 7 and sum(map(len, keys.values())) <= 3 * len(keys)
    assert ops.prompt_attention_path([2048], [0], 2048, H, Hkv, 96) is None


@pytest.mark.parametrize("rows", [1408, 2048, 4096])
def test_a_plan_without_a_workspace_has_whole_walks(rows):
    """As every plan had before walks were cut; a forced cut has no room and is refused."""
    ops, plan, whole = rule(), plan_of([rows]), plan_of([rows])
    plan.workspace, ops_whole = None, rule()
    ops_whole._cut_walks = lambda *args: (0, 0)
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
