"""The decode attention's grid: a workgroup's number gives its sequence and its head by a reciprocal, for any number of heads."""
import pytest
import torch

from helpers import rel_err
from test_gpu_kernels import OP_TOL, make_plan, ops_for

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.mark.parametrize("heads, kv_heads", [(2, 1), (2, 2), (6, 3), (5, 5), (7, 7), (24, 12)])
@pytest.mark.parametrize("n", [1, 9, 700])
def test_every_sequence_and_head_is_its_own(heads, kv_heads, n):
    """Contexts of 1 to 40 tokens, each on pages of its own, against the general kernel: both round an output once."""
    ops = ops_for(BF)
    D, ps, width = 64, 16, 3
    g = torch.Generator().manual_seed(kv_heads)
    lens = torch.randint(1, 41, (n,), generator=g)
    k = torch.randn(n * width, kv_heads, ps, D, generator=g).to(BF).cuda()
    v = torch.randn(n * width, kv_heads, D, ps, generator=g).to(BF).cuda()
    q = torch.randn(n, heads * D, generator=g).to(BF).cuda()
    table = torch.randperm(n * width, generator=g).to(torch.int32).view(n, width).cuda()
    positions, seq = (lens - 1).to(torch.int32).cuda(), torch.arange(n, dtype=torch.int32, device="cuda")
    out = {}
    for name, plan in (("mv_attention_decode", make_plan([1] * n, lens.tolist())), ("mv_attention_ref", None)):
        out[name] = torch.full((n, heads * D), float("nan"), dtype=BF, device="cuda")
        ledger, ops.ledger = ops.ledger, []
        try:
            ops.attention(q, out[name], k, v, table, ps, positions, seq, heads, kv_heads, D, D ** -0.5, None, plan=plan)
            assert [line[0] for line in ops.ledger] == [name]
        finally:
            ops.ledger = ledger
    got, want = (out[name].float().cpu() for name in ("mv_attention_decode", "mv_attention_ref"))
    assert rel_err(got.numpy(), want.numpy()) <= 2 * OP_TOL[BF]
