"""A step whose requests and heads fill the chip scans: the chunks' work grows with both, the scan's time does not."""
from types import SimpleNamespace

import pytest

from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.parts.matrix_state import recurrence


def path(rule, heads, dk, lens, recorded):
    plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=4096, n_seqs=len(lens), q_lens=[] if recorded else lens)
    if recorded:
        plan.bound, plan.path_lens = (8192, 64), tuple(lens)
    ops = SimpleNamespace(delta_chunk_line=lambda: 128, delta_chunk_tokens=lambda: 32, delta_chunks_serve=lambda *a: True)
    rt, seen = SimpleNamespace(ops=ops, workspace=SimpleNamespace(get=lambda *a: None)), []
    recurrence(rt, SimpleNamespace(attention_plan=plan), rule, sum(lens), heads, dk, dk, None,
               lambda *a, below=0: seen.append("scan below" if below else "scan"), lambda *a: seen.append("chunks"))
    return seen


@pytest.mark.parametrize("recorded", [False, True])
@pytest.mark.parametrize("heads, dk, lens, want", [
    # both sides measured on an MI355X, at least 8 % apart
    (16, 64, [2048], ["chunks"]), (64, 64, [2048], ["chunks"]), (64, 64, [384], ["chunks"]), (16, 64, [512] * 4, ["chunks"]),
    (16, 64, [128] * 16, ["scan"]), (16, 64, [128] * 64, ["scan"]), (16, 64, [256] * 32, ["scan"]), (16, 64, [512] * 16, ["scan"]),
    (64, 64, [128] * 4, ["scan"]), (64, 64, [512] * 4, ["scan"]), (64, 64, [1024] * 8, ["scan"]),
    (16, 128, [128], ["scan"]), (16, 128, [2048], ["chunks"]), (16, 128, [256] * 16, ["scan"]),
    (16, 64, [800] + [1] * 64, ["chunks", "scan below"]), (16, 64, [230, 90, 176] + [1] * 17, ["scan"])])
@pytest.mark.parametrize("rule", ["delta", "gated", "channel"])
def test_the_path_that_is_faster(rule, heads, dk, lens, want, recorded):
    assert path(rule, heads, dk, lens, recorded) == want


def test_sums_take_chunks_further():
    assert path("sum", 64, 64, [2048], False) == ["chunks"] and path("sum", 16, 64, [1024] * 8, False) == ["chunks"]
    assert path("sum", 64, 64, [128] * 64, False) == ["scan"]
