"""The exact product on the float matrix unit at the edges of its tiles and of its blocks of k."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("adtype, wdtype", [(torch.float32, torch.float32), (torch.float32, torch.bfloat16), (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("K", [3, 16, 131, 1024])
@pytest.mark.parametrize("M, N", [(1, 15), (16, 16500), (17, 65), (33, 4160), (65, 16384), (300, 6200)])
def test_every_tile_gives_a_row_the_same_bits(adtype, wdtype, K, M, N):
    """Each choice of tile (one row block against narrow and wide weights, 32 rows, 64, and rounds that leave 32 x 64), K below
    a block of 16, whole blocks and a remainder, rows in a wider buffer that no four elements can be loaded from at once.
    A sum of K products of numbers of variance 1 / K, added in partial sums: 3e-6 of the largest, as the float sums elsewhere."""
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
    ops.gemm(a[M - 1:M], w, one, b, exact=True)
    assert torch.equal(one, out[M - 1:M])
