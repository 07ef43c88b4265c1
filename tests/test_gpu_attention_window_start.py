"""The general attention loads four neighbouring values at once wherever a window starts: the same bits as one at a time."""
import math

import pytest
import torch

from test_gpu_kernels import OP_TOL, dev, fill_pages, make_plan, ops_for, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D", [64, 20])
@pytest.mark.parametrize("window, first", [(w, 0) for w in (0, 1, 2, 3, 4, 5, 126, 127, 128, 129, 258)] + [(9, 3), (130, 5)])
def test_windows_that_start_anywhere(D, window, first):
    """Windows that start at every distance from a multiple of four and end inside and behind a tile of 128 keys, kept first
    positions in front: pages of 16 slots (four values a load) against pages of 6 (no four slots of which are neighbours
    in memory for sure), and both against float64."""
    ops, H, Hkv = ops_for(torch.float32), 2, 1
    g = torch.Generator().manual_seed(D + window)
    ctx_lens, q_lens = [41, 300], [41, 70]
    k = [torch.randn(c, Hkv, D, generator=g).double() for c in ctx_lens]
    v = [torch.randn(c, Hkv, D, generator=g).double() for c in ctx_lens]
    positions = torch.tensor([p for c, q in zip(ctx_lens, q_lens) for p in range(c - q, c)], dtype=torch.int32)
    token_seq = torch.tensor([s for s, q in enumerate(q_lens) for _ in range(q)], dtype=torch.int32)
    n, scale = len(positions), 1.0 / math.sqrt(D)
    q = torch.randn(n, H, D, generator=g)
    outs = []
    for ps in (16, 6):
        per = [-(-c // ps) for c in ctx_lens]
        tables = [list(range(per[0])), list(range(per[0], sum(per)))]
        kp, vp = fill_pages(k, v, tables, ps, Hkv, D, sum(per), torch.float32)
        bt = torch.full((2, max(per)), -1, dtype=torch.int32)
        for s, t in enumerate(tables):
            bt[s, :len(t)] = torch.tensor(t, dtype=torch.int32)
        out = torch.full((n, H * D), float("nan"), device="cuda")
        ops.attention(dev(q.view(n, H * D)), out, kp, vp, dev(bt), ps, dev(positions), dev(token_seq), H, Hkv, D, scale, window,
                      plan=make_plan(q_lens, ctx_lens), **({"keep_first": first} if first else {}))
        outs.append(out.cpu())
    assert torch.equal(outs[0], outs[1])
    want = torch.zeros(n, H, D, dtype=torch.float64)
    for i in range(n):
        s, p = int(token_seq[i]), int(positions[i])
        keys = [j for j in range(p + 1) if j >= p - window or j < first]
        for h in range(H):
            want[i, h] = torch.softmax(k[s][keys, 0] @ q[i, h].double() * scale, dim=0) @ v[s][keys, 0]
    assert rel_err(outs[0].view(n, H, D).numpy(), want.numpy()) <= OP_TOL[torch.float32]
