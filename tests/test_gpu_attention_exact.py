"""The float attention on the matrix unit (attention_exact.hip) on keys that are no numbers, against 64 bits."""
import pytest
import torch

from helpers import rel_err
from test_gpu_kernels import make_plan, ops_for, reference_attention

pytestmark = pytest.mark.gpu
NAN, INF = float("nan"), float("inf")


@pytest.mark.parametrize("tokens, decode", [(150, False), (17, True), (40, True), (161, True)])
@pytest.mark.parametrize("broken", [(16, 17), (16, 32), (0, 16), (0, 150), (3, 4), (144, 160)])
@pytest.mark.parametrize("value", [NAN, INF, -INF])
def test_keys_that_are_no_numbers(tokens, decode, broken, value):
    """One key, a whole block of 16 (all that a wave sees of a short context), all of a prompt: a row that sees a key that is
    no number is none itself, minus infinity as a score has no weight, and the other rows are what they were: 5e-6, softmax
    over N(0, 1) scores and sums of up to 161 floats."""
    ops = ops_for(torch.float32)
    H, Hkv, D, ps = 4, 2, 64, 16
    g = torch.Generator().manual_seed(tokens)
    pages = -(-tokens // ps)
    k = torch.randn(pages * ps, Hkv, D, generator=g)
    v = torch.randn(pages * ps, Hkv, D, generator=g)
    k[broken[0]:min(broken[1], tokens)] = value
    n = 1 if decode else tokens
    q = torch.randn(n, H, D, generator=g).abs()                     # (so that an infinite key's scores have one sign)
    positions = torch.arange(tokens - n, tokens, dtype=torch.int32)
    seq = torch.zeros(n, dtype=torch.int32)
    out = torch.full((n, H * D), 7.0, device="cuda")
    ledger, ops.ledger = ops.ledger, []
    try:
        ops.attention(q.view(n, H * D).cuda(), out, k.view(pages, ps, Hkv, D).transpose(1, 2).contiguous().cuda(),
                      v.view(pages, ps, Hkv, D).permute(0, 2, 3, 1).contiguous().cuda(),
                      torch.arange(pages, dtype=torch.int32, device="cuda")[None], ps, positions.cuda(), seq.cuda(), H, Hkv, D,
                      D ** -0.5, None, plan=make_plan([n], [tokens]))
        assert [line[0] for line in ops.ledger] == ["mv_attention_exact"]
    finally:
        ops.ledger = ledger
    got = out.view(n, H, D).cpu()
    want = reference_attention(q.double(), [k.double()], [v.double()], positions, seq, H, Hkv, D ** -0.5, None)
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    good = ~torch.isnan(want)
    if bool(good.any()):
        assert rel_err(got[good].numpy(), want[good].numpy()) <= 5e-6
