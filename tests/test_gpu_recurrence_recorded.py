"""Recorded steps with prompt portions take the recurrences' paths that the same step takes eagerly, whatever else was recorded
for their size class."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def executor(graphs):
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    mlp = {"kind": "dense", "ff": 128}
    arch, cfg = config_from_dict({"architecture": "Bolapel", "vocab": 256, "width": 128, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                  "logit_softcap": 20.0,
                                  "layers": [{"type": "general_delta", "mixer": {"heads": 2, "dim": 64, "rank": 8}, "mlp": mlp}] * 2})
    source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device("cuda:0"), std=0.08)
    return Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=1024, max_num_batched_tokens=1024, max_num_batched_seqs=16,
                                 kv_cache_block_size=16, kv_cache_num_blocks=16, use_cuda_graph=graphs), model=(arch, cfg, source))


def test_paths_of_recorded_steps():
    """Pairs of steps of one size class that differ in their longest or shortest request, each several times, in turn: what
    ran, the logits and the states left behind against eager steps (bfloat16 products differ in order: 2e-2)."""
    from minivllm_amd.engine.step import SeqStep
    recorded, eager = executor(True), executor(False)
    g = torch.Generator().manual_seed(2)
    text = [torch.randint(0, 256, (700,), generator=g).tolist() for _ in range(9)]
    steps = [([440, 440], {"mv_delta_chunks"}), ([600] + [1] * 8, {"mv_delta_chunks", "mv_delta_scan"}), ([250, 250], {"mv_delta_chunks"}),
             ([380, 120], {"mv_delta_scan"}), ([400, 110], {"mv_delta_chunks", "mv_delta_scan"}), ([127, 3], {"mv_delta_scan"}),
             ([130], {"mv_delta_chunks"})]
    for turn in range(3):
        for lens, want in steps:
            known = set(recorded.graph_ledger)
            made = [SeqStep(tokens=text[s][:q], start=0, block_tables=[[]] * len(recorded.groups), state_slot=s, want=[q - 1])
                    for s, q in enumerate(lens)]
            got, plain = recorded.step(made).clone(), eager.step(made).clone()
            torch.cuda.synchronize()
            new = [k for k in recorded.graph_ledger if k not in known]
            assert len(new) == (1 if turn == 0 else 0), lens
            if new:
                ran = {e[0] for e in recorded.graph_ledger[new[0]]}
                assert ran & {"mv_delta_chunks", "mv_delta_scan"} == want, lens
            assert float((got - plain).abs().max() / plain.abs().max()) <= 2e-2, lens
            for call in recorded.state_tensors:
                a, b = (ex.state_tensors[call]["state"][:len(lens)] for ex in (recorded, eager))
                assert float((a - b).abs().max() / b.abs().max()) <= 2e-2, lens
