"""Float outputs of bfloat16 products (scores that choices are made by): a row's bits do not depend on how many rows an entry
point is given, up to where its callers hand over to another one."""
import math

import pytest
import torch

from test_gpu_kernels import ops_for

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def operands(M, N, K):
    g = torch.Generator().manual_seed(N + K)
    return torch.randn(M, K, generator=g).to(BF).cuda(), (torch.randn(N, K, generator=g) / math.sqrt(K)).to(BF).cuda()


# (weights of 16 MB and more are read by another kernel up to 16 rows)
@pytest.mark.parametrize("N,K", [(64, 1024), (2048, 1024), (1024, 3072), (6144, 1024)])
def test_of_few_rows(N, K):
    ops = ops_for(BF)
    a, w = operands(64, N, K)
    whole = None
    for M in (64, 33, 17, 16, 9, 8, 1):
        out = torch.full((M, N), float("nan"), device="cuda")
        ops.lib.call("mv_gemm_skinny", a.data_ptr(), K, w.data_ptr(), K, 0, out.data_ptr(), N, 0, M, N, K, 0, ops._stream())
        whole = out if whole is None else whole
        assert torch.equal(out, whole[:M]), M


@pytest.mark.parametrize("N,K", [(4096, 1024), (4096, 512)])
def test_of_many_rows(N, K):
    ops = ops_for(BF)
    a, w = operands(512, N, K)
    whole = None
    for M in (512, 300, 129, 128, 65, 40):
        assert int(ops.lib.dll.mv_gemm_tile_splits(M, N, K, 0, 0)) == 1
        out = torch.full((M, N), float("nan"), device="cuda")
        ops.lib.call("mv_gemm_tile", a.data_ptr(), K, w.data_ptr(), 0, out.data_ptr(), N, 0, M, N, K, 0, 0, 0, 0, 0.0, 1.0, 0, ops._stream())
        whole = out if whole is None else whole
        assert torch.equal(out, whole[:M]), M
