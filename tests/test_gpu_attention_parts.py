"""The MFMA prompt attention with walks over the keys cut in two, a workgroup each, against attention in 64 bits."""
import math

import numpy as np
import pytest
import torch

from test_gpu_kernels import OP_TOL, dev, fill_pages, make_plan, ops_for, rel_err

pytestmark = pytest.mark.gpu


# limits of one pair of blocks (every walk of ten blocks and more in halves), between the walks' lengths, at and beside a walk's length
# less the eight blocks that a second part has at least
@pytest.mark.parametrize("nt, limit", [(1, 2), (1, 16), (1, 26), (1, 28), (2, 2), (2, 16), (2, 30)])
@pytest.mark.parametrize("H, Hkv, D, ps, window, first", [(4, 2, 128, 16, None, 0), (16, 8, 128, 32, 400, 0), (6, 2, 64, 16, None, 0), (8, 2, 64, 16, 350, 40)])
def test_walks_in_two_parts(nt, limit, H, Hkv, D, ps, window, first):
    """Walks of 1, 9, 10, 35 and 36 blocks, portions behind a context, single tokens beside them (the narrow form with 16 columns a wave), a window with pages given
    back, slots behind a context that hold NaN. Launches follow each other on one set of counters and have the same bits."""
    ops, dtype = ops_for(torch.bfloat16), torch.bfloat16
    g = torch.Generator().manual_seed(83 + D)
    ctx_lens, q_lens = [19, 288, 289, 1120, 1131, 700], [19, 40, 1, 130, 70, 1]
    k_all = [torch.randn(c, Hkv, D, generator=g).to(dtype).double() for c in ctx_lens]
    v_all = [torch.randn(c, Hkv, D, generator=g).to(dtype).double() for c in ctx_lens]
    pages_per = [-(-c // ps) for c in ctx_lens]
    perm = torch.randperm(sum(pages_per) + 3, generator=g).tolist()
    tables, cur = [], 0
    for n_p in pages_per:
        tables.append(perm[cur:cur + n_p])
        cur += n_p
    if window is not None:
        for s, (c, ql) in enumerate(zip(ctx_lens, q_lens)):
            for i in range(-(-first // ps), max(0, (c - ql) - window) // ps):
                tables[s][i] = -1
    kp, vp = fill_pages(k_all, v_all, tables, ps, Hkv, D, len(perm), dtype)
    bt = torch.full((len(tables), max(pages_per)), -1, dtype=torch.int32)
    for s, t in enumerate(tables):
        bt[s, :len(t)] = torch.tensor(t, dtype=torch.int32)
    positions = torch.tensor([p for c, ql in zip(ctx_lens, q_lens) for p in range(c - ql, c)], dtype=torch.int32)
    token_seq = torch.tensor([s for s, ql in enumerate(q_lens) for _ in range(ql)], dtype=torch.int32)
    n, ends, scale = len(positions), np.cumsum(q_lens) - 1, 1.0 / math.sqrt(D)
    q = torch.randn(n, H, D, generator=g)
    for s, row in enumerate(ends):                 # every request's last query singles out its first visible key, the first part's
        far = 0 if window is None or first else max(0, ctx_lens[s] - 1 - window)
        q[row] = 6.0 * k_all[s][far].float().repeat_interleave(H // Hkv, dim=0) / math.sqrt(D)
    q = q.to(dtype)
    outs = []
    plan = make_plan(q_lens, ctx_lens)
    plan.prefill_variant = (nt, 1, limit)
    args = dev(q.view(n, H * D)), kp, vp, dev(bt), dev(positions), dev(token_seq)
    for _ in range(3):
        out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
        ops.attention(args[0], out, args[1], args[2], args[3], ps, args[4], args[5], H, Hkv, D, scale, window, plan=plan,
                      **({"keep_first": first} if first else {}))
        outs.append(out)
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    assert not bool(ops._prompt_counters(plan.workspace).any())
    want = torch.zeros(n, H, D, dtype=torch.float64)
    for i in range(n):
        s, p = int(token_seq[i]), int(positions[i])
        lo = 0 if window is None else max(0, p - window)
        keys = list(range(min(first, lo))) + list(range(lo, p + 1))
        for kvh in range(Hkv):
            h = slice(kvh * H // Hkv, (kvh + 1) * H // Hkv)
            want[i, h] = torch.softmax(q[i, h].double() @ k_all[s][keys, kvh].T * scale, dim=-1) @ v_all[s][keys, kvh]
    assert rel_err(outs[0].float().cpu().view(n, H, D).numpy(), want.numpy()) <= 2 * OP_TOL[dtype]


@pytest.mark.parametrize("chunk, gated", [(0, False), (600, True)])
def test_sums_of_sigmoid_weights_in_two_parts(chunk, gated):
    """Without a normalisation the two parts just add: against the whole walks, half a step of bfloat16 (2^-9) a result for each rounding of the two."""
    ops, dtype, H, Hkv, D, ps, n = ops_for(torch.bfloat16), torch.bfloat16, 4, 2, 128, 16, 1500
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    q, kp, vp = rand(n, H * D), rand(-(-n // ps), Hkv, ps, D), rand(-(-n // ps), Hkv, D, ps)
    gate = rand(n, H) if gated else None
    pos, seq = torch.arange(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    bt = torch.arange(-(-n // ps), dtype=torch.int32, device="cuda").view(1, -1)
    bias = torch.full((H,), -math.log(n), device="cuda")
    outs = []
    for variant in ((1, 1), (1, 1, 4), (1, 1, 20)):
        plan = make_plan([n], [n])
        plan.prefill_variant = variant
        out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
        ops.attention_sigmoid(q, out, kp, vp, bt, ps, pos, seq, H, Hkv, D, D, D ** -0.5, chunk or None, None, bias, gate, plan=plan)
        outs.append(out.double())
    for out in outs[1:]:
        assert float((out - outs[0]).norm() / outs[0].norm()) <= 2 * 2.0 ** -9


@pytest.mark.parametrize("rows", [[2048], [1700], [4000], [900, 1200]])
def test_the_rule_cuts_long_walks(rows):
    """What the launch rule chooses for whole prompts gives what whole walks give, to the roundings of bfloat16 weights and results: 2^-9 each."""
    ops, dtype, H, Hkv, D, ps = ops_for(torch.bfloat16), torch.bfloat16, 16, 8, 128, 16
    n, pages = sum(rows), [-(-r // ps) for r in rows]
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    q, kp, vp = rand(n, H * D), rand(sum(pages), Hkv, ps, D), rand(sum(pages), Hkv, D, ps)
    bt = torch.zeros(len(rows), max(pages), dtype=torch.int32)
    for s, p in enumerate(pages):
        bt[s, :p] = torch.arange(p) + sum(pages[:s])
    pos = torch.cat([torch.arange(r) for r in rows]).int().cuda()
    seq = torch.cat([torch.full((r,), s) for s, r in enumerate(rows)]).int().cuda()
    outs = []
    for variant in ((1, 1), None):
        plan = make_plan(rows, rows)
        plan.prefill_variant = variant
        out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
        ops.attention(q, out, kp, vp, bt.cuda(), ps, pos, seq, H, Hkv, D, D ** -0.5, None, plan=plan)
        outs.append(out.double())
    assert ops._prefill_variant(plan, 2, Hkv)[4] > 0
    assert float((outs[1] - outs[0]).norm() / outs[0].norm()) <= 2 * 2.0 ** -9
