"""Finishing heads of 64 channels, four channels a lane, against the kernel that has a channel a lane: the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def rows(gen, n, width, dtype):
    return torch.randn(n, width, generator=gen, device=DEV).to(dtype)


# one head, a workgroup's sixteen less one, exactly and more, and several
@pytest.mark.parametrize("n, H", [(1, 1), (5, 3), (1, 16), (17, 1), (67, 5)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("weight_dtype", [torch.float32, torch.bfloat16])
def test_same_bits_as_a_channel_a_lane(n, H, dtype, weight_dtype):
    from minivllm_amd.kernels.ops import Ops
    ops = Ops(dtype)
    gen = torch.Generator(device=DEV).manual_seed(n + H)
    inner = 64 * H
    # (a pitch that stores of four do not fit goes to the other kernel)
    outs = [torch.full((n, inner + extra), 7.0, dtype=dtype, device=DEV) for extra in (4, 1)]
    raw, packed, weight = rows(gen, n, inner, torch.float32), rows(gen, n, 4 * inner + 4, dtype), rows(gen, 1, inner, weight_dtype)[0]
    raw[0, :64] = 0.0                                       # a head that says nothing
    for out in outs:
        ops.delta_finish(raw, packed, weight, H, 64, 1e-5, out[:, :inner])
    assert torch.equal(outs[0][:, :inner], outs[1][:, :inner])
    o = raw.view(n, H, 64).double()
    want = (o / (o.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()).view(n, inner) * weight.double() * torch.sigmoid(packed[:, 3 * inner:4 * inner].double())
    # a dozen float32 operations, or the rounding to eight bits
    assert bool(((outs[0][:, :inner].double() - want).abs() <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -19) * want.abs()).all())
    token_seq = torch.tensor([-1 if t % 4 == 2 else 0 for t in range(n)], dtype=torch.int32, device=DEV)
    for normaliser in (False, True):
        raw, gates = rows(gen, n, H * (64 + normaliser), torch.float32).view(n, H, -1), rows(gen, n, 4 * H, torch.float32).view(n, H, 4).abs()
        for gate_dtype in {torch.float32, dtype}:
            packed = rows(gen, n, 8 + inner, gate_dtype)
            for shared, silu in ((True, True), (False, False)):
                w = weight[:64].contiguous() if shared else weight
                for out in outs:
                    ops.state_finish(raw, gates, packed, 4, w, H, 64, 1e-5, token_seq, out[:, :inner], shared_weight=shared, silu_gate=silu,
                                     normaliser=normaliser, denom_eps=1e-6)
                assert torch.equal(outs[0][:, :inner], outs[1][:, :inner])
                assert not outs[0][:, :inner][token_seq < 0].any() and bool((outs[0][:, inner:] == 7.0).all())
