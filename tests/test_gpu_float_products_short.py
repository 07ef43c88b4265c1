"""The exact product of many rows and a short K, whose tiles one wave makes alone: the same bits as tiles of eight waves."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("adtype, wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("K", [1, 8, 15, 17, 36, 64, 100, 128, 130, 512, 513])
@pytest.mark.parametrize("M, N", [(500, 1030), (2100, 1100)])
def test_one_wave_a_tile(adtype, wdtype, K, M, N):
    """One block of k and part of one, fewer blocks than partial sums and as many, several rounds of them, and K on both sides of
    the lines between the forms; rows and columns that fill their last tiles in part; operands that four elements can and
    cannot be loaded from at once. Every 97th row is also taken alone. 3e-6 of the largest, as the float sums elsewhere."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(adtype)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    a = torch.randn(M, K + 3, generator=g, device=DEV).to(adtype)[:, :K]
    w = (torch.randn(N, K, generator=g, device=DEV) / math.sqrt(K)).to(wdtype)
    b = torch.randn(N, generator=g, device=DEV).to(wdtype)
    out = torch.full((M + 1, N), float("nan"), dtype=torch.float32, device=DEV)
    ops.gemm(a, w, out[:M], b, exact=True)
    want = a.double() @ w.double().T + b.double()
    assert float((out[:M].double() - want).abs().max() / want.abs().max()) <= 3e-6
    assert bool(torch.isnan(out[M]).all())
    dense = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops.gemm(a.contiguous(), w, dense, b, exact=True)
    assert torch.equal(dense, out[:M])
    one = torch.empty(1, N, dtype=torch.float32, device=DEV)
    for m in range(0, M, 97):
        ops.gemm(a[m:m + 1], w, one, b, exact=True)
        assert torch.equal(one[0], out[m]), m
