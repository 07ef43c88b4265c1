"""Which steps of a mixture compute the chosen pairs only: those where that was measured to take less time."""
from types import SimpleNamespace

import pytest
import torch


def experts(hid, F, E, top, shared=0, **options):
    from minivllm_amd.parts.moe import RoutedExperts, RoutedExpertsSpec
    spec = RoutedExpertsSpec(hidden_size=hid, expert_size=F, num_experts=E, top=top, shared_size=shared, **options)
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=SimpleNamespace(use_fast_kernels=True))
    return RoutedExperts(spec, {name: torch.empty(decl.shape, dtype=torch.bfloat16, device="meta")
                                for name, decl in RoutedExperts.tensors(spec).items()}, rt)


@pytest.mark.parametrize("hid, F, E, top, pairs, all_experts", [
    # both sides measured on an MI355X, more than 4 % apart
    (1024, 768, 32, 4, [1, 8, 128, 2048], []), (1024, 768, 16, 4, [1, 64, 8192], []), (1024, 768, 64, 2, [1, 16, 8192], []),
    (4096, 3072, 8, 2, [1, 64, 512, 8192], []), (1024, 768, 8, 4, [1024, 2048], [1, 2, 128, 256]), (1024, 768, 4, 2, [4415], [1, 8, 64, 128, 512, 1024]),
    (1024, 3072, 2, 1, [4415], [1, 64, 128, 512, 1024]), (1024, 3072, 2, 2, [], [1, 64, 1024, 8192]), (4096, 3072, 8, 4, [1, 512 * 2], [256]),
    (4096, 3072, 4, 2, [1, 2048], [64, 256]), (64, 64, 8, 2, [], [1, 64, 1024, 8192]), (128, 128, 16, 4, [], [1, 128, 512, 8192]),
    (1024, 768, 16, 8, [1024, 2048], [64, 128])])
def test_the_path_that_is_faster(hid, F, E, top, pairs, all_experts):
    part = experts(hid, F, E, top)
    for n in pairs:
        assert part.wants_pairs(n), n
    for n in all_experts:
        assert not part.wants_pairs(n), n


def test_widths_that_the_tiles_do_not_take():
    assert not experts(96, 768, 32, 4).wants_pairs(64) and not experts(1024, 800, 32, 4).wants_pairs(64)
    assert not experts(1024, 768, 32, 4, grouped=False).wants_pairs(64)
