"""Which of a recurrence's two paths a step takes: chunks for long requests, the scan for short ones, the scan alone where
a step brings both and the long ones are not long enough to pay for both."""
from types import SimpleNamespace

import pytest

from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.parts.matrix_state import CHUNKS_BESIDE_SHORT, CHUNKS_BESIDE_SHORT_CLASS, recurrence

LINE = 128


@pytest.mark.parametrize("q_lens, bound, least, want", [
    ([LINE - 1], None, 1, ["scan"]), ([LINE], None, 1, ["chunks"]), ([LINE, 2 * LINE], None, 1, ["chunks"]),
    ([1, CHUNKS_BESIDE_SHORT - 1], None, 1, ["scan"]), ([1, CHUNKS_BESIDE_SHORT], None, 1, ["chunks", "scan below"]),
    ((), (256, 1), 193, ["chunks"]), ((), (128, 1), 65, ["scan"]), ((), (CHUNKS_BESIDE_SHORT_CLASS - 1, 4), 1, ["scan"]),
    ((), (CHUNKS_BESIDE_SHORT_CLASS, 4), 1, ["chunks", "scan below"])])
def test_paths(q_lens, bound, least, want):
    plan = AttentionPlan(decode_only=False, max_q_len=max(q_lens or [bound[0] if bound else 1]), max_context_len=4096,
                         n_seqs=len(q_lens) or bound[1], q_lens=list(q_lens), cu_seqlens=None, workspace=None)
    plan.bound, plan.bound_least = bound, least
    ops = SimpleNamespace(delta_chunk_line=lambda: LINE, delta_chunk_tokens=lambda: 32, delta_chunks_serve=lambda *a: True)
    rt = SimpleNamespace(ops=ops, workspace=SimpleNamespace(get=lambda *a: None))
    seen = []
    recurrence(rt, SimpleNamespace(attention_plan=plan), "delta", 8, 2, 64, 64, None,
               lambda *a, below=0: seen.append("scan below" if below else "scan"), lambda *a: seen.append("chunks"))
    assert seen == want
