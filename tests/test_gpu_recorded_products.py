"""A step recorded for its size class against the same step run eagerly, at the sizes that the kernels are made for: the rows
behind the step's own are padding, and what is added up for the others keeps its order."""
import math

import pytest
import torch

from helpers import rel_err
from minivllm_amd.engine.executor import TOKEN_BUCKETS
from test_gpu_kernels import ops_for

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("N,K", [(4096, 1024), (1024, 2048), (1024, 3072), (2048, 512), (64, 1024)])
@pytest.mark.parametrize("gated", [False, True])
def test_products_of_a_class(N, K, gated):
    ops = ops_for(BF)
    g = torch.Generator().manual_seed(N + K)
    a = torch.randn(64, K, generator=g).to(BF).cuda()
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(BF).cuda()
    width = N // 2 if gated else N
    run = ops.gemm_swiglu if gated else ops.gemm
    for rows in range(2, 65):
        padded = next(b for b in TOKEN_BUCKETS if b >= rows)
        own, recorded = torch.empty(rows, width, dtype=BF, device="cuda"), torch.empty(padded, width, dtype=BF, device="cuda")
        run(a[:rows], w, own)
        run(a[:padded], w, recorded)
        assert torch.equal(own, recorded[:rows]), (rows, padded)


def steps_of(shape, use_graph, portions, seed):
    """The logits of one request's last row at every portion of its prompt."""
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.config.shapes import named_shape
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.engine.step import SeqStep
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    raw = dict(named_shape(shape), torch_dtype="bfloat16")
    raw.update({"layers": raw["layers"][:4], "vocab": 512} if "layers" in raw else {"num_hidden_layers": 3, "vocab_size": 512})
    arch, cfg = config_from_dict(raw)
    source = DeviceRandomSource(expected_tensors(arch, cfg), 1, BF, torch.device("cuda:0"), std=0.64 / cfg.hidden_size ** 0.5)
    ex = Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=512, max_num_batched_tokens=256, max_num_batched_seqs=4,
                               kv_cache_block_size=16, kv_cache_num_blocks=64, use_cuda_graph=use_graph), model=(arch, cfg, source))
    manager = ex.new_cache_manager()
    tokens = torch.randint(0, 512, (sum(portions),), generator=torch.Generator().manual_seed(seed)).tolist()
    manager.admit(0)
    manager.reserve(0, len(tokens))
    at, out = 0, []
    for n in portions:
        out.append(ex.step([SeqStep(tokens=tokens[at:at + n], start=at, want=[n - 1], state_slot=manager.sequence(0).state_slot,
                                    block_tables=[list(manager.block_table(0, g)) for g in range(len(manager.groups))])]).clone().cpu())
        at += n
    assert bool(ex._mixed_graphs) == use_graph
    return out


@pytest.mark.parametrize("shape", ["0.6b", "dutilix-0.6b", "furanex-0.6b"])
def test_steps_of_a_class(shape):
    portions = [20, 2, 3, 5, 8, 7, 12, 16, 4, 30, 6]
    recorded, eager = (steps_of(shape, use_graph, portions, seed=5) for use_graph in (True, False))
    errors = [rel_err(a.numpy(), b.numpy()) for a, b in zip(recorded, eager)]
    print(shape, " ".join(f"{e:.1e}" for e in errors))
    assert max(errors) == 0.0
