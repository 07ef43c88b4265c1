"""What the recurrences over chunks take as scratch is there before the cache is sized, however later steps are cut."""
import random
from types import SimpleNamespace
from unittest.mock import MagicMock

import pytest
import torch

from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.parts import MIXERS, Workspace
from minivllm_amd.parts.delta_rule import DeltaRuleSpec
from minivllm_amd.parts.matrix_state import ChannelDeltaSpec, GatedDeltaSpec, MLSTMSpec

SIZES = dict(hidden_size=64, num_heads=2, key_dim=64, value_dim=64)
SPECS = [DeltaRuleSpec(hidden_size=64, num_heads=2, head_dim=64, decay_rank=64), GatedDeltaSpec(num_kv_heads=1, conv_taps=4, **SIZES), MLSTMSpec(**SIZES),
         ChannelDeltaSpec(num_kv_heads=1, conv_taps=4, decay_rank=16, gate_rank=16, **SIZES)]


@pytest.mark.parametrize("spec", SPECS, ids=lambda spec: spec.kind)
def test_vectors_of_short_requests_have_room_before_any_come(spec):
    """An engine of so few requests that its dry step's all go in chunks, straight from the packed rows: a short request beside long ones, or alone, and
    requests so many that all are scanned, want their rows' vectors in memory."""
    ops = MagicMock(compute_units=256)
    ops.delta_chunk_line.return_value, ops.delta_chunk_tokens.return_value, ops.gemm.return_value = 128, 32, None
    for straight in ("delta_chunks_rows", "delta_chunks_conv", "mlstm_chunks"):
        getattr(ops, straight + "_serve").return_value = True
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device("meta")), max_positions=1024)
    cls = MIXERS.get(spec.kind)
    part = cls(spec, {name: torch.zeros(decl.shape, dtype=torch.bfloat16, device="meta") for name, decl in cls.tensors(spec).items()}, rt)

    def step(lens):
        plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=max(lens), n_seqs=len(lens), q_lens=lens)
        ops.reset_mock()
        part.forward(torch.zeros(sum(lens), 64, dtype=torch.bfloat16, device="meta"), MagicMock(attention_plan=plan), 0)
        return any(getattr(ops, straight).called for straight in ("delta_chunks_rows", "delta_chunks_conv", "mlstm_chunks"))

    part.reserve(1024, 4)
    assert step([512, 512]), "the dry step wants no vectors"
    rt.workspace.frozen = True                  # (a buffer that would have to grow raises)
    assert not any(step(lens) for lens in ([1000, 24], [700, 100, 100, 124], [100], [127] * 8))


def test_no_cut_has_more_units():
    from minivllm_amd.engine.step import most_units
    rng = random.Random(1)
    for _ in range(300):
        least, seqs = rng.choice([1, 128]), rng.randint(1, 40)
        lens = [rng.randint(1, rng.choice([3, 150, 1000])) for _ in range(seqs)]
        plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=4096, n_seqs=seqs, q_lens=lens)
        assert plan.units(32, least) <= most_units(sum(lens), seqs, 32, least)
    lens = [129] * 7
    plan = AttentionPlan(decode_only=False, max_q_len=129, max_context_len=4096, n_seqs=7, q_lens=lens)
    assert plan.units(32, 128) == 35 == most_units(7 * 129, 40, 32, 128)
    plan.q_lens = [1] * 500 + [160]
    assert plan.units(32, 128) == 5, "requests that do not go in chunks count"


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("requests, rank", [(64, 8), (4, 64)])
def test_scratch_stands_at_the_start(graphs, requests, rank):
    """An engine that sizes its cache from the memory that is left: first long prompts of every kind of cut allocate no scratch. With four requests its
    dry step's all go in chunks, and with a rank of 64 straight from the packed rows."""
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.engine.step import SeqStep
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    mlp = {"kind": "dense", "ff": 128}
    arch, cfg = config_from_dict({"architecture": "Bolapel", "vocab": 256, "width": 128, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                  "logit_softcap": 20.0,
                                  "layers": [{"type": "general_delta", "mixer": {"heads": 2, "dim": 64, "rank": rank}, "mlp": mlp}]})
    source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device("cuda:0"), std=0.05)
    ex = Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=1024, max_num_batched_tokens=1024, max_num_batched_seqs=requests,
                               kv_cache_block_size=16, gpu_memory_utilization=0.05, use_cuda_graph=graphs), model=(arch, cfg, source))
    areas = lambda: [ws.bytes() for ws in (ex.rt.workspace, ex._graph_workspace) if ws is not None]
    at_start = areas()
    assert len(at_start) == 1 + graphs
    for lens in ([1024], [129] * 7, [700] + [1] * 60, [128], [383, 385, 200, 50], [900, 24], [1]):
        if len(lens) > requests:
            continue
        ex.step([SeqStep(tokens=[i % 256 for i in range(q)], start=0, block_tables=[[]] * len(ex.groups), state_slot=s, want=[q - 1])
                 for s, q in enumerate(lens)])
        torch.cuda.synchronize()
        assert areas() == at_start, lens
