"""In float32 a request's rows and state have the same bits whatever else is in the step and however its tokens are cut."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def part(kind, H=2, dk=64, hid=64):
    from minivllm_amd.kernels.ops import get_ops
    from minivllm_amd.parts.base import MIXERS, Runtime, Workspace
    cls = MIXERS.get(kind)
    sizes = {"delta_rule": dict(num_heads=H, head_dim=dk, decay_rank=8)}.get(
        kind, dict(num_heads=H, key_dim=dk, value_dim=dk))
    if kind in ("gated_delta", "channel_delta"):
        sizes.update(num_kv_heads=1, conv_taps=3)
    if kind == "channel_delta":
        sizes.update(decay_rank=8, gate_rank=8)
    spec = cls.spec_class(hidden_size=hid, **sizes)
    g = torch.Generator(device=DEV).manual_seed(4)
    tensors = {}
    for name, decl in cls.tensors(spec).items():
        t = torch.randn(decl.shape, generator=g, device=DEV) * (decl.shape[-1] ** -0.5 if len(decl.shape) == 2 else 0.3)
        tensors[name] = t + 1 if decl.init == "ones_normal" else t
    rt = Runtime(device=torch.device(DEV), dtype=torch.float32, ops=get_ops(torch.float32), workspace=Workspace(torch.device(DEV)),
                 max_positions=4096)
    return cls(spec, tensors, rt), cls.state_shapes(spec)


def step(mixer, state, x, lens, slots):
    from minivllm_amd.engine.step import AttentionPlan, StepContext
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ends = [0]
    for q in lens:
        ends.append(ends[-1] + q)
    ctx = StepContext()
    ctx.token_seq, ctx.cu_seqlens, ctx.state_slots = i32([s for s, q in enumerate(lens) for _ in range(q)]), i32(ends), i32(slots)
    ctx.n_tokens, ctx.n_seqs, ctx._state = ends[-1], len(lens), {0: state}
    ctx.attention_plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=4096, n_seqs=len(lens), q_lens=list(lens),
                                       cu_seqlens=ctx.cu_seqlens)
    y = mixer.forward(x, ctx, 0)
    y = y if isinstance(y, torch.Tensor) else y.materialize()
    torch.cuda.synchronize()
    return y.clone()


@pytest.mark.parametrize("kind", ["delta_rule", "gated_delta", "mlstm", "channel_delta"])
def test_neighbours_and_cuts_do_not_show(kind):
    mixer, shapes = part(kind)
    g = torch.Generator(device=DEV).manual_seed(7)
    x = torch.randn(700, 64, generator=g, device=DEV)
    other = torch.randn(900, 64, generator=g, device=DEV)
    results = []
    for before, portions in (([], [700]), ([1], [700]), ([600], [700]), ([1, 390, 5], [300, 250, 150]), ([], [127] * 5 + [65])):
        state = {name: torch.zeros((4,) + tuple(dims), dtype=dt or torch.float32, device=DEV) for name, (dims, dt) in shapes.items()}
        rows, at = [], 0
        for q in portions:
            mine = torch.cat([other[:sum(before)], x[at:at + q]])
            rows.append(step(mixer, state, mine, before + [q], list(range(1, 1 + len(before))) + [0])[sum(before):])
            at += q
        results.append((torch.cat(rows), {name: t[0].clone() for name, t in state.items()}))
    rows, kept = results[0]
    for other_rows, other_kept in results[1:]:
        assert torch.equal(other_rows, rows)
        for name in kept:
            assert torch.equal(other_kept[name], kept[name]), name
