"""Between a gated pair's two products lies a buffer that steps of one pass do not need: it is there before the cache is sized, also
where the largest step goes in one pass and a smaller one does not."""
from types import SimpleNamespace

import pytest
import torch

from minivllm_amd.parts.base import Workspace
from minivllm_amd.parts.mlp import ClampedGLU, ClampedGLUSpec, SwiGLU, SwiGLUSpec
from minivllm_amd.parts.moe import RoutedExperts, RoutedExpertsSpec


def part_of(cls, spec, one_pass):
    ops = SimpleNamespace(use_fast_kernels=True, gemm_swiglu=lambda x, w, out, *a, **k: one_pass(x.shape[0]), gemm=lambda *a, **k: None,
                          swiglu=lambda *a, **k: None, add_rows=lambda *a: None)
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device("cpu")))
    return cls(spec, {name: torch.zeros(decl.shape, dtype=torch.bfloat16) for name, decl in cls.tensors(spec).items()}, rt)


@pytest.mark.parametrize("cls, spec", [
    (SwiGLU, SwiGLUSpec(hidden_size=64, intermediate_size=128)),
    (ClampedGLU, ClampedGLUSpec(hidden_size=64, intermediate_size=128, limit=7.0)),
    # (experts whose chosen pairs may go through the plain kernels: the shared one keeps matrices of its own)
    (RoutedExperts, RoutedExpertsSpec(hidden_size=64, expert_size=96, num_experts=4, top=2, shared_size=32, grouped_min_weight=1))])
@pytest.mark.parametrize("one_pass", [lambda n: n > 128, lambda n: n < 100 or n > 128, lambda n: n != 77, lambda n: n > 1])
def test_no_smaller_step_needs_more(cls, spec, one_pass):
    part, most = part_of(cls, spec, one_pass), 300
    ws = part.rt.workspace
    if cls is RoutedExperts:
        assert not part.shared_packed
        run = lambda n: part._add_shared(torch.zeros(n, 64), torch.zeros(n, 64))
    else:
        run = lambda n: part.forward(torch.zeros(n, 64), None)
    part.reserve(most)
    run(most)
    ws.frozen = True                     # (a buffer that would have to grow raises)
    for n in range(1, most + 1):
        run(n)


def test_the_rule_for_one_pass_is_not_monotone():
    """What makes the buffer necessary: more rows go in one pass where fewer do not."""
    import ctypes
    from minivllm_amd.csrc import build
    shape = ctypes.CDLL(build.find_library("bf16") or build.build("bf16")).mv_gemm_pair_shape
    assert shape(1024, 256, 128, 256) and not shape(128, 256, 128, 256)
    assert shape(2048, 12288, 2048, 256) and not shape(1792, 12288, 2048, 256)


def test_the_librarys_workspace_is_there_before_the_dry_run():
    """The dry run's own products may all be the engine's; a smaller step's need not be."""
    from unittest.mock import MagicMock, patch
    from minivllm_amd.engine.executor import Executor
    from minivllm_amd.kernels.ops import Ops
    engine = MagicMock(page_size=16, num_state_slots=4, groups=[None],
                       config=SimpleNamespace(max_num_batched_seqs=4, max_model_len=64, use_cuda_graph=False))
    ops = SimpleNamespace(_lt_work=None, use_library_gemm=True,
                          lib=SimpleNamespace(has=lambda name: True, dll=SimpleNamespace(mv_gemm_lt_workspace=lambda: 1 << 20)))
    engine.ops.reserve_library = lambda device: Ops.reserve_library(ops, torch.device("cpu"))
    engine.step = lambda seqs: seen.append(ops._lt_work)
    seen = []
    with patch("torch.cuda.synchronize"), patch("torch.cuda.empty_cache"), patch("torch.cuda.is_current_stream_capturing", return_value=False):
        Executor._warmup(engine, 64)
        assert len(seen) == 1 and seen[0].numel() == 1 << 20
        Ops.reserve_library(ops, torch.device("cpu"))
        assert ops._lt_work is seen[0]
        ops.use_library_gemm, ops._lt_work = False, None             # (the float32 engine has no such product)
        Ops.reserve_library(ops, torch.device("cpu"))
        assert ops._lt_work is None


def test_scratch_of_folded_norms_is_there_before_the_dry_run():
    """The largest step folds no norm, smaller ones do."""
    from minivllm_amd.parts import NORMS, RMSNormSpec
    from minivllm_amd.parts.block import PreNormBlock
    most = 1024
    ops = SimpleNamespace(most_fold_rows=lambda width: most, can_fold_norm=lambda n, size, consumer: n <= most)
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device("cpu")))
    norm = NORMS.get("rmsnorm")(RMSNormSpec(size=128), {"weight": torch.ones(128)}, rt)
    block = PreNormBlock(None, {"mixer": norm, "ffn": norm}, None, SimpleNamespace())
    block.reserve(4096)
    rt.workspace.frozen = True
    for n in (1, 97, 512, most):
        assert norm.fold(SimpleNamespace(resid=torch.zeros(n, 128)), None, (64, 128, False)) is not None
    assert norm.fold(SimpleNamespace(resid=torch.zeros(most + 1, 128)), None, (64, 128, False)) is None
