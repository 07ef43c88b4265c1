"""Recorded steps with prompt portions take the latent attention's kernel that the same step takes eagerly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def executor(graphs):
    from minivllm_amd.config import EngineConfig
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.models import config_from_dict, expected_tensors
    from minivllm_amd.weights.device_random import DeviceRandomSource
    latent = {"heads": 2, "dim": 16, "rot_dim": 64, "vdim": 16, "q_rank": 64, "kv_rank": 128, "scale": 0.1, "rot": {"dims": 64, "base": 1e4}}
    arch, cfg = config_from_dict({"architecture": "Dutilix", "vocab": 256, "width": 128, "norm": {"eps": 1e-5}, "torch_dtype": "bfloat16",
                                  "logit_scale": 1.0, "layers": [{"type": "latent_attention", "mixer": latent,
                                                                  "mlp": {"kind": "dense", "ff": 128}}] * 2})
    source = DeviceRandomSource(expected_tensors(arch, cfg), 1, torch.bfloat16, torch.device("cuda:0"), std=0.08)
    return Executor(EngineConfig(model="", dtype="bfloat16", max_model_len=1024, max_num_batched_tokens=1024, max_num_batched_seqs=16,
                                 kv_cache_block_size=16, kv_cache_num_blocks=256, use_cuda_graph=graphs), model=(arch, cfg, source))


def test_kernels_of_recorded_steps():
    """Steps of one size class that differ in where their tokens stand or how they are dealt out, each several times, in turn: what
    ran, and the logits against eager steps (bfloat16, sums in another order: 2e-2)."""
    from minivllm_amd.engine.step import SeqStep
    recorded, eager = executor(True), executor(False)
    g = torch.Generator().manual_seed(2)
    text = [torch.randint(0, 256, (700,), generator=g).tolist() for _ in range(8)]
    tables = [list(range(44 * s, 44 * s + 44)) for s in range(4)]
    for s in range(4):                                   # contexts for the steps that begin behind position 0
        for ex in (recorded, eager):
            ex.step([SeqStep(tokens=text[s][:600], start=0, block_tables=[tables[s]], state_slot=s, want=[])])
    shared, apart = "mv_attention_latent_prompt", "mv_attention_latent_mfma"
    steps = [([(20, 0)], apart), ([(20, 400)], shared), ([(20, 40)], apart), ([(12, 600), (1, 599)], shared),
             ([(6, 600), (7, 599)], apart), ([(12, 0), (1, 20)], apart)]
    for turn in range(3):
        for cut, want in steps:
            known = set(recorded.graph_ledger)
            made = [SeqStep(tokens=text[s][start:start + q], start=start, block_tables=[tables[s]], state_slot=s, want=[q - 1])
                    for s, (q, start) in enumerate(cut)]
            got, plain = recorded.step(made).clone(), eager.step(made).clone()
            torch.cuda.synchronize()
            for key in set(recorded.graph_ledger) - known:
                assert turn == 0
                ran = {e[0] for e in recorded.graph_ledger[key]}
                assert want in ran and not ran & ({shared, apart} - {want}), cut
            eager.ops.ledger = []
            eager.step(made)
            ran, eager.ops.ledger = {e[0] for e in eager.ops.ledger}, None
            assert want in ran and not ran & ({shared, apart} - {want}), cut
            assert float((got - plain).abs().max() / plain.abs().max()) <= 2e-2, cut
    # (the third step has the choice of the first, and its recording)
    assert len(recorded.graph_ledger) == 5


def test_sizes_without_a_choice_are_recorded_once():
    """Latents that the sharing kernel does not take, and the float32 engine, have no choice to make."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    assert all(ops.latent_shares_serve(*sizes) for sizes in ((64, 0), (128, 0), (192, 0), (256, 0), (128, 64), (256, 64)))
    assert not any(ops.latent_shares_serve(*sizes) for sizes in ((64, 32), (128, 32), (192, 64), (16, 4), (512, 64)))
    assert not get_ops(torch.float32).latent_shares_serve(256, 64)
