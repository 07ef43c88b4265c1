"""Steps with prompt portions: when the latent attention's workgroups share key rows among a request's tokens."""
from types import SimpleNamespace

import pytest

from minivllm_amd.engine.step import AttentionPlan
from minivllm_amd.kernels.ops import Ops


@pytest.mark.parametrize("heads, prompts, decoding, want", [
    # (tokens, first position) of prompts, (requests, position) of decoded tokens: both sides measured, at least 8 % apart
    (16, [(20, 0)], (0, 0), False), (16, [(48, 0)], (0, 0), False), (16, [(160, 0)], (0, 0), True), (16, [(8, 200)], (0, 0), True),
    (16, [(9, 0)] * 100, (0, 0), False), (64, [(60, 0)] * 5, (0, 0), True), (64, [(9, 0)] * 100, (0, 0), False), (64, [(128, 0)] * 16, (0, 0), True),
    (16, [(16, 0)], (8, 1900), True), (16, [(16, 0)], (300, 40), False), (16, [(16, 0)], (300, 1000), True), (64, [(16, 0)], (100, 1000), True),
    (64, [(16, 0)], (200, 300), False), (64, [(16, 0)], (300, 1000), False), (64, [(9, 500)] * 100, (0, 0), True),
    (16, [(7, 500)], (8, 1900), False)])
@pytest.mark.parametrize("window", [-1, 1 << 20])
def test_the_kernel_that_is_faster(heads, prompts, decoding, want, window):
    lens, starts = [1] * decoding[0] + [q for q, _ in prompts], [decoding[1] - 1] * decoding[0] + [s for _, s in prompts]
    assert Ops.latent_shares(SimpleNamespace(compute_units=256), heads, window, lens, starts) is want


def test_keys_in_front_of_a_window_do_not_count():
    shares = lambda window: Ops.latent_shares(SimpleNamespace(compute_units=256), 16, window, [20], [2000])
    assert shares(-1) and shares(500) and not shares(30)


def test_the_cut_that_choices_follow():
    plan = AttentionPlan(decode_only=False, max_q_len=9, max_context_len=30, n_seqs=3, q_lens=[9, 1, 0], starts=[0, 29])
    assert plan.cut() == ([9, 1], [0, 29])
    plan.bound, plan.q_lens = (16, 4), ()
    assert plan.cut() == ((), ())                       # a recording that has to serve any cut
    plan.path_lens, plan.path_starts = (9, 1), (0, 29)
    assert plan.cut() == ((9, 1), (0, 29))
    assert Ops.latent_shares(SimpleNamespace(compute_units=256), 16, -1, *AttentionPlan(False, 9, 30, 1, q_lens=[9]).cut())


@pytest.mark.parametrize("heads, prompts, decoding, own", [
    # up to 64 tokens stay where sums leave the latent's space in float32
    (16, [(20, 0)], (0, 0), False), (16, [(16, 2000)], (0, 0), False), (16, [(16, 0)], (8, 1000), False), (16, [(65, 0)], (0, 0), True),
    (16, [(56, 0)], (8, 300), False), (64, [(64, 1000)], (0, 0), False), (64, [(65, 1000)], (0, 0), True),
    # both sides measured, at least 8 % apart: (tokens, first position) of prompts, (requests, position) of decoded tokens
    (16, [(2048, 0)], (0, 0), True), (16, [(64, 0)], (17, 700), False), (16, [(300, 0)], (16, 1900), False), (16, [(16, 0)], (64, 1000), False), (16, [(9, 500)] * 40, (0, 0), False),
    (64, [(100, 0)], (0, 0), True), (64, [(16, 0)], (16, 1000), False), (64, [(300, 0)], (16, 1000), False)])
def test_when_the_heads_have_keys_of_their_own(heads, prompts, decoding, own):
    lens, starts = [1] * decoding[0] + [q for q, _ in prompts], [decoding[1] - 1] * decoding[0] + [s for _, s in prompts]
    room = Ops.latent_heads(SimpleNamespace(compute_units=256), heads, lens, starts)
    assert (room > 0) is own
    assert room == 0 or room * 32 >= sum(lens) + sum(starts)


def test_room_for_own_keys_is_bounded():
    """Steps of similar sizes have one room; no step has more than what is reserved for the engine's sizes."""
    ops = SimpleNamespace(compute_units=256)
    rooms = {Ops.latent_heads(ops, 16, [n], [0]) for n in range(1800, 2049)}
    assert rooms == {64}
    assert Ops.latent_heads(ops, 16, [], []) == 0 and Ops.latent_heads(ops, 16, [1, 1], [900, 20]) == 0
    most = Ops.latent_heads_most(ops, 16, 512, 4, 1024)
    for lens, starts in (([512], [0]), ([128] * 4, [896] * 4), ([2] * 4, [1022] * 4), ([2], [0]), ([100, 100, 100], [924, 100, 0])):
        assert Ops.latent_heads(ops, 16, lens, starts) <= most
    assert Ops.latent_heads(ops, 64, [64], [40000]) == 0 and Ops.latent_heads_most(ops, 64, 8192, 256, 40960) == 512


def test_layers_of_one_spec_that_store_their_maps_differently_choose_for_themselves():
    """A layer whose maps are stored in 32 bits stays in the latent's space, its neighbour of the same spec does not: a recording's key
    holds both choices, whichever layer comes last."""
    import torch
    from minivllm_amd.models.causal_lm import CausalLM
    from minivllm_amd.parts.latent_attention import LatentAttention, LatentAttentionSpec
    spec = LatentAttentionSpec(hidden_size=256, num_heads=2, plain_dim=128, rot_dim=64, value_dim=128, kv_rank=128)
    ops = SimpleNamespace(compute_units=256, latent_heads_serve=lambda *sizes: True, latent_shares_serve=lambda *sizes: True)
    ops.latent_heads, ops.latent_shares = lambda *a: Ops.latent_heads(ops, *a), lambda *a: Ops.latent_shares(ops, *a)
    rt = SimpleNamespace(dtype=torch.bfloat16, ops=ops)

    def layer(*wide):
        return LatentAttention(spec, {name: torch.zeros(decl.shape, dtype=torch.float32 if name in wide else torch.bfloat16)
                                      for name, decl in LatentAttention.tensors(spec).items()}, rt,
                               SimpleNamespace(rotary=lambda: (torch.zeros(1, 64), False)))
    both = [layer(), layer("uk")]
    lens, starts = [100], [0]
    own, latent = (m.step_path(lens, starts) for m in both)
    assert own != latent
    for mixers in (both, both[::-1], both + [layer(), layer("uv"), None]):
        assert set(CausalLM.step_paths(SimpleNamespace(_choosers=None, mixers=mixers), lens, starts)) == {own, latent}
    assert len(CausalLM.step_paths(SimpleNamespace(_choosers=None, mixers=[layer(), layer(), layer()]), lens, starts)) == 1


def test_maps_without_a_rotary_part_stay_in_the_latents_space():
    import torch
    from minivllm_amd.parts.latent_attention import LatentAttention, LatentAttentionSpec
    ops = SimpleNamespace(latent_heads_serve=lambda *sizes: True)
    for rot_dim in (0, 64):
        spec = LatentAttentionSpec(hidden_size=256, num_heads=2, plain_dim=128, rot_dim=rot_dim, value_dim=128, kv_rank=128)
        part = LatentAttention(spec, {name: torch.zeros(decl.shape, dtype=torch.bfloat16) for name, decl in LatentAttention.tensors(spec).items()},
                               SimpleNamespace(dtype=torch.bfloat16, ops=ops), SimpleNamespace(rotary=lambda: (torch.zeros(1, 64), False)))
        assert (part.heads_operands is not None) is (rot_dim > 0)


def mixed_load(rng, steps, positions):
    """Steps of one to three prompt portions beside up to fifteen requests that decode."""
    for _ in range(steps):
        lens, starts = [1] * rng.randint(0, 15), []
        starts += [rng.randint(20, positions - 1) for _ in lens]
        for _ in range(rng.randint(1, 3)):
            lens.append(rng.randint(20, 500))
            starts.append(rng.choice([0, rng.randint(0, positions - 500)]))
        yield lens, starts


def size_class(lens, starts):
    """Tokens, sequences and context that a recording of such a step is made for."""
    from minivllm_amd.engine.executor import GRAPH_BUCKETS, TOKEN_BUCKETS
    cap = max(1024, 1 << (max(map(sum, zip(lens, starts))) - 1).bit_length())
    return next(b for b in TOKEN_BUCKETS if b >= sum(lens)), next(b for b in GRAPH_BUCKETS if b >= len(lens)), cap


def test_a_growing_context_needs_no_recording_of_its_own():
    """Of a size class there is one recording for each of the three ways, whatever the keys that its steps' contexts hold."""
    import random
    import torch
    from minivllm_amd.parts.latent_attention import LatentAttention
    ops = SimpleNamespace(compute_units=256, latent_shares_serve=lambda *sizes: True)
    ops.latent_heads, ops.latent_shares = lambda *a: Ops.latent_heads(ops, *a), lambda *a: Ops.latent_shares(ops, *a)
    part = SimpleNamespace(rt=SimpleNamespace(ops=ops), heads_operands=(), spec=SimpleNamespace(num_heads=16, window=None, kv_rank=256, rot_dim=64))
    keys = {}
    for lens, starts in mixed_load(random.Random(1), 1500, 1900):
        keys.setdefault(size_class(lens, starts), set()).add(LatentAttention.step_path(part, lens, starts))
    assert len(keys) > 50 and max(map(len, keys.values())) <= 3
    assert sum(map(len, keys.values())) <= 1.5 * len(keys)


@pytest.mark.parametrize("heads, units", [(1, 256), (3, 64), (16, 256), (16, 304), (20, 128), (64, 256), (128, 256)])
def test_the_room_reserved_holds_every_step(heads, units):
    import random
    rng, ops, own = random.Random(heads), SimpleNamespace(compute_units=units), 0
    cuts = list(mixed_load(rng, 400, 1900)) + list(mixed_load(rng, 200, 4000))
    for _ in range(600):                                 # portions of any length at any place, none of them decoded tokens
        n = int(2 ** rng.uniform(0, 5))
        cuts.append(([int(2 ** rng.uniform(1, 9)) for _ in range(n)], [rng.choice([0, rng.randint(0, 3000)]) for _ in range(n)]))
    for lens, starts in cuts:
        room = Ops.latent_heads(ops, heads, lens, starts)
        own += room > 0
        assert room <= Ops.latent_heads_most(ops, heads, sum(lens), len(lens), max(map(sum, zip(lens, starts))))
        if sum(lens) <= 2048:
            of_class = Ops.latent_heads_most(ops, heads, *size_class(lens, starts))
            assert room <= of_class <= Ops.latent_heads_most(ops, heads, 2048, 64, 4096)           # (what an engine of such steps reserves)
    assert own > 100


def test_no_room_is_reserved_that_no_step_can_take():
    ops = SimpleNamespace(compute_units=256)
    assert Ops.latent_heads_most(ops, 16, 64, 256, 4096) == 0
    # 256 requests of 4,096 positions have 32,768 blocks; beside 512 tokens the latent's space is ahead from 1,000 on
    assert 800 <= Ops.latent_heads_most(ops, 16, 512, 256, 4096) <= 1250
