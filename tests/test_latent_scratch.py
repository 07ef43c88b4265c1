"""What a latent attention takes as scratch is there before the cache is sized, whichever way the largest step goes."""
from types import SimpleNamespace
from unittest.mock import MagicMock

import pytest
import torch

from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.kernels.ops import Ops
from minivllm_amd.parts.base import Workspace
from minivllm_amd.parts.latent_attention import LatentAttention, LatentAttentionSpec

POSITIONS = 512


def layer():
    spec = LatentAttentionSpec(hidden_size=64, num_heads=2, plain_dim=128, rot_dim=64, value_dim=128, q_rank=32, kv_rank=128)
    ops = MagicMock(compute_units=256)
    ops.latent_heads_serve.return_value = True
    ops.gemm.return_value = None
    ops.latent_heads = lambda *a: Ops.latent_heads(ops, *a)
    ops.latent_heads_most = lambda *a: Ops.latent_heads_most(ops, *a)
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device("cpu")), max_positions=POSITIONS)
    return LatentAttention(spec, {name: torch.zeros(decl.shape, dtype=torch.bfloat16) for name, decl in LatentAttention.tensors(spec).items()}, rt,
                           SimpleNamespace(rotary=lambda: (torch.zeros(POSITIONS, 64), False)))


def step(part, lens, starts):
    """Runs the part over a step; whether it made the heads' own keys."""
    plan = AttentionPlan(decode_only=max(lens) == 1, max_q_len=max(lens), max_context_len=POSITIONS, n_seqs=len(lens), q_lens=lens, starts=starts)
    part.rt.ops.reset_mock()
    part.rt.ops.gemm.return_value = None
    part.forward(torch.zeros(sum(lens), 64, dtype=torch.bfloat16), MagicMock(attention_plan=plan), 0)
    return part.rt.ops.latent_expand.called


@pytest.mark.parametrize("largest, own", [(([300], [0]), True), (([30] * 10, [0] * 10), True), (([66] + [1] * 234, [0] + [500] * 234), False)])
def test_scratch_stands_at_the_start(largest, own):
    part = layer()
    part.reserve(300, 256)
    assert step(part, *largest) is own
    part.rt.workspace.frozen = True                  # (a buffer that would have to grow raises)
    ways = {step(part, *cut) for cut in [([64], [0]), ([1] * 60, [500] * 60), ([200], [300]), ([66] + [1] * 60, [0] + [500] * 60), ([4] * 60, [508] * 60)]}
    assert ways == {True, False}
