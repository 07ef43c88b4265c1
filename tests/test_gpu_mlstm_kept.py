"""The running maximum that an mLSTM keeps for the next step is the one its last row's factors were made from."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("lens", [[128 + 3 * s for s in range(60)], [1024, 1025, 2047, 2048, 2100, 64, 127, 1]])
def test_kept_maximum(lens):
    """The state carries exp(-m) of a request's last row, and the next step scales it by what is kept: gates[2] = exp(-m) of the
    kept m to the rounding of one exponential (2 units of 2^-23, on top of the stored result's half)."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    H, d, n, S = 8, 64, sum(lens), len(lens)
    g = torch.Generator(device=DEV).manual_seed(n)
    packed = torch.randn(n, 4 * H * d + 2 * H, generator=g, device=DEV)
    packed[:, 4 * H * d:4 * H * d + H] *= 4
    packed = packed.bfloat16()
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    ends = [0]
    for q in lens:
        ends.append(ends[-1] + q)
    kept = torch.randn(S, H, generator=g, device=DEV)
    gates = torch.empty(n, H, 4, device=DEV)
    bias = torch.randn(2, H, generator=g, device=DEV).bfloat16()
    ops.mlstm_prepare(packed, H, d, d, bias[0].contiguous(), (bias[1] + 2).contiguous(), 15.0, kept, i32([s for s, q in enumerate(lens) for _ in range(q)]),
                      i32(ends), i32(list(range(S))), S, torch.empty(n, H, 2, d, device=DEV), torch.empty(n, H, d + 1, device=DEV), gates)
    torch.cuda.synchronize()
    last = gates[torch.tensor(ends[1:], device=DEV) - 1, :, 2].double()
    assert float((last / torch.exp(-kept.double()) - 1).abs().max()) <= 3e-7
