"""The float products' LDS ring where a workgroup walks several tiles of several chunks: its stream of loads goes on into the
next tile while the sums of the last one are added up, and an odd number of chunks changes the register buffers over."""
import math

import pytest
import torch

from helpers import rel_err
from test_gpu_kernels import ops_for

pytestmark = pytest.mark.gpu
XCDS = 8


def tiles_of(shape, M, N, units):
    """Tiles that the XCDs get, and the workgroups that walk an XCD's."""
    tiles = -(-M // (16 * (shape // 10))) * -(-N // (16 * (shape % 10)))
    shares = [tiles * (x + 1) // XCDS - tiles * x // XCDS for x in range(XCDS)]
    return shares, min(-(-tiles // XCDS), units // XCDS)


# two chunks and odd numbers of them, XCDs with unequal shares, workgroups with unequal numbers of tiles, ragged edges
@pytest.mark.parametrize("shape, M, N, K", [(22, 97, 5030, 384), (22, 33, 17000, 256), (22, 40, 9001, 640), (22, 24, 20000, 384),
                                            (24, 70, 9100, 384), (24, 500, 4111, 256), (24, 129, 17003, 640), (24, 224, 6144, 1024),
                                            (44, 600, 3000, 384), (44, 300, 6100, 384), (44, 300, 6100, 256), (44, 700, 2503, 640)])
def test_a_workgroup_walks_several_tiles(shape, M, N, K):
    """The bits are those of the product that takes rows at any address: the same rows shifted by one element. Against 64
    bits 3e-6 of the largest, as elsewhere."""
    ops = ops_for(torch.float32)
    if ops.compute_units != 256:
        pytest.skip("the sizes are made for 256 compute units")
    assert ops.lib.dll.mv_gemm_ref_ring_shape(M, N, K) == shape
    shares, groups = tiles_of(shape, M, N, ops.compute_units)
    assert groups == 32 and min(shares) > groups and K // 128 >= 2
    g = torch.Generator().manual_seed(M + N + K)
    a = torch.randn(M, K, generator=g).cuda()
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).cuda()
    b = torch.randn(N, generator=g).cuda()
    out = torch.full((M, N + 3), float("nan"), device="cuda")
    ops.gemm(a, w, out[:, :N], b, exact=True)
    odd = torch.empty(M * (K + 4) + 1, device="cuda")[1:].view(M, K + 4)[:, :K]
    odd.copy_(a)
    plain = torch.empty(M, N, device="cuda")
    ops.gemm(odd, w, plain, b, exact=True)
    assert torch.equal(out[:, :N], plain)
    assert bool(torch.isnan(out[:, N:]).all())
    want = a.double() @ w.double().T + b.double()
    assert rel_err(plain.cpu().numpy(), want.cpu().numpy()) <= 3e-6
