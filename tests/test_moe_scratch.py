"""What a mixture takes as scratch where a step computes all experts is there before the cache is sized, also where the largest
step computes the chosen pairs only."""
import pytest
import torch

from test_moe_paths import experts


@pytest.mark.parametrize("hid, F, E, top, most, want", [
    (1024, 768, 8, 4, 16384, 1023), (1024, 768, 8, 4, 1024, 1023), (1024, 768, 8, 4, 700, 700), (4096, 3072, 4, 2, 8192, 2047),
    (1024, 768, 32, 4, 16384, None), (64, 64, 8, 2, 16384, 16384)])
def test_the_largest_step_that_computes_all_experts(hid, F, E, top, most, want):
    part, seen = experts(hid, F, E, top), []
    part._all_experts_scratch = seen.append
    part.reserve(most)
    assert seen == ([] if want is None else [want])
    assert want is None or want == max(n for n in range(1, most + 1) if not part.wants_pairs(n))


@pytest.mark.gpu
@pytest.mark.parametrize("graphs", [True, False])
def test_scratch_stands_at_the_start(graphs):
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.engine.step import SeqStep
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    latent = {"heads": 2, "dim": 16, "rot_dim": 16, "vdim": 16, "q_rank": 64, "kv_rank": 64, "scale": 0.1, "rot": {"dims": 16, "base": 1e4}}
    moe = {"kind": "moe", "expert": {"ff": 256}, "router": {"experts": 8, "identity": 0, "top": 4, "groups": {"count": 1, "keep": 1}}}
    arch, cfg = config_from_dict({"architecture": "Dutilix", "vocab": 256, "width": 512, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                  "logit_scale": 1.0, "layers": [{"type": "latent_attention", "mixer": latent, "mlp": moe}]})
    source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device("cuda:0"), std=0.05)
    ex = Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=2048, max_num_batched_tokens=2048, max_num_batched_seqs=64,
                               kv_cache_block_size=16, gpu_memory_utilization=0.05, use_cuda_graph=graphs), model=(arch, cfg, source))
    areas = lambda: [ws.bytes() for ws in (ex.rt.workspace, ex._graph_workspace) if ws is not None]
    at_start = areas()
    assert len(at_start) == 1 + graphs
    for q in (1000, 1023, 1024, 2048, 300):
        ex.step([SeqStep(tokens=[i % 256 for i in range(q)], start=0, block_tables=[list(range(-(-q // 16)))], state_slot=0, want=[q - 1])])
        torch.cuda.synchronize()
        assert areas() == at_start, q
