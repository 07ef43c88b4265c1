"""The product of many values of k a step (gemm_deep.hip), every tile and form of it, against 64 bits."""
import math

import pytest
import torch

from helpers import rel_err
from test_gpu_kernels import OP_TOL, ops_for

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


def operands(M, N, K, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(M, K + 8, generator=g).to(BF).cuda()[:, :K]          # rows with a stride of their own
    w = (torch.randn(N, K, generator=g) / math.sqrt(K)).to(BF).cuda()
    b = torch.randn(N, generator=g).to(BF).cuda()
    return a, w, b


def exact(a, w, b):
    return a.double().cpu() @ w.double().cpu().T + (0.0 if b is None else b.double().cpu())


# one chunk, fewer and more than a ring holds; rows and columns at the edges of the tiles, one column beyond them, odd widths
SIZES = [(1, 16, 256), (16, 48, 512), (17, 33, 768), (5, 35, 1792), (32, 64, 1024), (33, 65, 2304), (64, 130, 3072), (100, 200, 512)]


@pytest.mark.parametrize("shape", [11, 12, 22, 24])
@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("with_bias, floats, scaled", [(False, False, False), (True, True, False), (True, False, True)])
def test_products(shape, M, N, K, with_bias, floats, scaled):
    """bfloat16 operands, float sums: the output's rounding, or 3e-6 of the largest for float outputs."""
    ops = ops_for(BF)
    a, w, b = operands(M, N, K, M + N + K + shape)
    b = b if with_bias else None
    out = torch.full((M, N + 3), float("nan"), dtype=torch.float32 if floats else BF, device="cuda")
    P = 300 if M < 17 else 5
    partial = (torch.rand(M, P, generator=torch.Generator().manual_seed(3)) + 0.5).cuda() * K / P
    ops.lib.call("mv_gemm_deep", a.data_ptr(), a.stride(0), w.data_ptr(), 0 if b is None else b.data_ptr(), out.data_ptr(), N + 3,
                 0 if floats else 1, M, N, K, 0, partial.data_ptr() if scaled else 0, P, 1e-6, 0.0, 1.0, 0, shape, ops._stream())
    want = exact(a, w, None)
    if scaled:
        want = want / torch.sqrt(partial.double().cpu().sum(1, keepdim=True) / K + 1e-6)
    if b is not None:
        want = want + b.double().cpu()
    assert rel_err(out[:, :N].float().cpu().numpy(), want.numpy()) <= (3e-6 if floats else OP_TOL[BF])
    assert bool(torch.isnan(out[:, N:].float()).all())


@pytest.mark.parametrize("shape", [12, 22, 24])
@pytest.mark.parametrize("M,I,K", [(1, 16, 256), (16, 40, 1024), (17, 33, 768), (33, 66, 2304), (64, 130, 512)])
@pytest.mark.parametrize("limit, scaled", [(0.0, False), (7.0, True)])
def test_gated_pairs(shape, M, I, K, limit, scaled):
    ops = ops_for(BF)
    a, w, b = operands(M, 2 * I, K, M + I + K)
    out = torch.full((M, I + 1), float("nan"), dtype=BF, device="cuda")
    P = 7
    partial = (torch.rand(M, P, generator=torch.Generator().manual_seed(3)) + 0.5).cuda() * K / P
    ops.lib.call("mv_gemm_deep", a.data_ptr(), a.stride(0), w.data_ptr(), b.data_ptr(), out.data_ptr(), I + 1, 1, M, 2 * I, K, 1,
                 partial.data_ptr() if scaled else 0, P, 1e-6, limit, 1.702 if limit else 1.0, 0, shape, ops._stream())
    want = exact(a, w, None)
    if scaled:
        want = want / torch.sqrt(partial.double().cpu().sum(1, keepdim=True) / K + 1e-6)
    want = want + b.double().cpu()
    g, u = want[:, :I], want[:, I:]
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        want = g * torch.sigmoid(1.702 * g) * (u + 1)
    else:
        want = g * torch.sigmoid(g) * u
    assert rel_err(out[:, :I].float().cpu().numpy(), want.numpy()) <= OP_TOL[BF]
    assert bool(torch.isnan(out[:, I:].float()).all())


@pytest.mark.parametrize("shape", [11, 12, 22, 24])
@pytest.mark.parametrize("M,N,K", [(1, 16, 256), (16, 36, 1024), (17, 64, 768), (33, 132, 2304), (96, 100, 512)])
@pytest.mark.parametrize("with_bias, unit_offset", [(False, 0), (True, 1)])
def test_in_front_of_a_norm(shape, M, N, K, with_bias, unit_offset):
    """The residual takes the product's rounded row: a unit in the last place of bfloat16 where the sums differ; the
    weighted rows and the sums of squares are the new residual's to float rounding."""
    ops = ops_for(BF)
    a, w, b = operands(M, N, K, M + N + K)
    g = torch.Generator().manual_seed(8)
    start = torch.randn(M, N, generator=g)
    resid, nw = start.cuda(), torch.randn(N, generator=g).to(BF).cuda()
    weighted = torch.full((M, N), float("nan"), dtype=BF, device="cuda")
    P = (N + 15) // 16
    partial = torch.full((M, P), float("nan"), device="cuda")
    ops.lib.call("mv_gemm_deep_fold", a.data_ptr(), a.stride(0), w.data_ptr(), b.data_ptr() if with_bias else 0, resid.data_ptr(), N,
                 nw.data_ptr(), 1, unit_offset, weighted.data_ptr(), N, partial.data_ptr(), P, M, N, K, shape, ops._stream())
    x = resid.double().cpu()
    assert rel_err(x.numpy(), (start.double() + exact(a, w, b if with_bias else None)).numpy()) <= OP_TOL[BF]
    assert rel_err(weighted.float().cpu().numpy(), (x * (nw.double().cpu() + unit_offset)).numpy()) <= OP_TOL[BF]
    columns = torch.nn.functional.pad(x, (0, 16 * P - N)).view(M, P, 16)
    assert rel_err(partial.cpu().numpy(), columns.pow(2).sum(-1).numpy()) <= 1e-6


def test_which_sizes_come_here():
    ops = ops_for(BF)
    shape = ops.lib.dll.mv_gemm_deep_shape
    if ops.compute_units != 256:
        pytest.skip("the rule counts compute units")
    assert [shape(*s) for s in [(9, 4096, 1024, 0), (16, 6144, 4096, 0), (1, 4096, 12288, 0), (9, 6144, 1024, 1), (64, 4096, 1024, 0),
                                (128, 4096, 1024, 0), (64, 6144, 1024, 1), (64, 1024, 3072, 0), (256, 1024, 3072, 0), (512, 1024, 3072, 0)]] == \
        [11, 12, 11, 12, 22, 24, 24, 11, 22, 24]
    assert [shape(*s) for s in [(8, 4096, 1024, 0), (16, 4096, 256, 0), (16, 4096, 1000, 0), (17, 4096, 4096, 0), (8, 24576, 4096, 1),
                                (129, 4096, 1024, 0), (513, 1024, 1024, 0), (0, 1024, 1024, 0), (16, 1023, 1024, 0)]] == [0] * 9


# (weights of 8 Mi elements, where the kernel in front changes its form, and on both sides of it)
@pytest.mark.parametrize("N,K", [(4096, 1024), (1024, 2048), (1024, 3072), (2048, 4096), (2032, 4096), (8192, 1024), (4096, 4096), (4096, 12288)])
def test_sums_are_as_exact_as_those_of_the_kernel_in_front(N, K):
    """Float sums of N(0, 1) operands against 64 bits, 2-norms over 16 rows of four draws, which are good to a percent."""
    ops = ops_for(BF)
    errors = {"mv_gemm_skinny": 0.0, "mv_gemm_deep": 0.0}
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        a = torch.randn(16, K, generator=g, device="cuda").to(BF)
        w = (torch.randn(N, K, generator=g, device="cuda") / math.sqrt(K)).to(BF)
        want = a.double() @ w.double().T
        for entry in errors:
            out = torch.empty(16, N, device="cuda")
            if entry == "mv_gemm_skinny":
                ops.lib.call(entry, a.data_ptr(), K, w.data_ptr(), K, 0, out.data_ptr(), N, 0, 16, N, K, 0, ops._stream())
            else:
                ops.lib.call(entry, a.data_ptr(), K, w.data_ptr(), 0, out.data_ptr(), N, 0, 16, N, K, 0, 0, 0, 0.0, 0.0, 1.0, 0, 0, ops._stream())
            errors[entry] += float(((out.double() - want).norm() / want.norm()) ** 2)
    print(K, {entry: math.sqrt(e / 4) for entry, e in errors.items()})
    assert math.sqrt(errors["mv_gemm_deep"]) <= 1.02 * math.sqrt(errors["mv_gemm_skinny"])
