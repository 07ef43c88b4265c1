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


@pytest.mark.parametrize("rows, starts", [([2048], [0]), ([1700], [0]), ([4000], [0]), ([1500, 300], [0, 0]), ([1536], [1000]), ([1700], [4096]), ([3000], [700])])
def test_the_rule_cuts_long_walks(rows, starts):
    """What the launch rule chooses gives what whole walks give, to the roundings of bfloat16 weights and results: 2^-9 each."""
    ops, dtype, H, Hkv, D, ps = ops_for(torch.bfloat16), torch.bfloat16, 16, 8, 128, 16
    ctx = [r + s for r, s in zip(rows, starts)]
    n, pages = sum(rows), [-(-c // ps) for c in ctx]
    g = torch.Generator(device="cuda").manual_seed(7)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    q, kp, vp = rand(n, H * D), rand(sum(pages), Hkv, ps, D), rand(sum(pages), Hkv, D, ps)
    bt = torch.zeros(len(rows), max(pages), dtype=torch.int32)
    for s, p in enumerate(pages):
        bt[s, :p] = torch.arange(p) + sum(pages[:s])
    pos = torch.cat([torch.arange(s, s + r) for r, s in zip(rows, starts)]).int().cuda()
    seq = torch.cat([torch.full((r,), s) for s, r in enumerate(rows)]).int().cuda()
    outs = []
    for variant in ((1, 1), None):
        plan = make_plan(rows, ctx)
        plan.starts, plan.prefill_variant = starts, variant
        out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
        ops.attention(q, out, kp, vp, bt.cuda(), ps, pos, seq, H, Hkv, D, D ** -0.5, None, plan=plan)
        outs.append(out.double())
    limit = ops._prefill_variant(plan, 2, Hkv)[4]
    assert limit > 0 and max(-(-c // 32) for c in ctx) >= limit + 8
    assert float((outs[1] - outs[0]).norm() / outs[0].norm()) <= 2 * 2.0 ** -9


@pytest.mark.parametrize("nt", [1, 2])
@pytest.mark.parametrize("form", [{"softcap": 20.0}, {"slopes": True}, {"sink": True}, {"softcap": 10.0, "slopes": True, "sink": True}])
def test_scored_walks_in_two_parts(nt, form):
    """Capped scores, a distance bias and a sink, which the two parts' maxima and sums count in once: as the whole walks, to the roundings of bfloat16."""
    ops, dtype, H, Hkv, D, ps, n = ops_for(torch.bfloat16), torch.bfloat16, 4, 2, 64, 16, 900
    g = torch.Generator(device="cuda").manual_seed(11)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    q, kp, vp = rand(n, H * D), rand(-(-n // ps), Hkv, ps, D), rand(-(-n // ps), Hkv, D, ps)
    pos, seq = torch.arange(n, dtype=torch.int32, device="cuda"), torch.zeros(n, dtype=torch.int32, device="cuda")
    bt = torch.arange(-(-n // ps), dtype=torch.int32, device="cuda").view(1, -1)
    if "slopes" in form:
        form = dict(form, slopes=torch.tensor([2.0 ** -(h + 3) for h in range(H)], device="cuda"))
    outs = []
    for variant in ((nt, 1), (nt, 1, 2), (nt, 1, 12)):
        plan = make_plan([n], [n])
        plan.prefill_variant = variant
        out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
        ops.attention(q, out, kp, vp, bt, ps, pos, seq, H, Hkv, D, D ** -0.5, None, plan=plan, **form)
        outs.append(out.double())
    for out in outs[1:]:
        assert float((out - outs[0]).norm() / outs[0].norm()) <= 2 * 2.0 ** -9


def test_a_recording_cuts_the_walks_of_any_step_of_its_class():
    """Recorded for a class with more units than its steps have, replayed with eager work between for other cuts of it, one long prompt or several short ones,
    behind contexts and not: the eager whole walks' results to the roundings of bfloat16, the same bits again, and counters at zero after every replay."""
    from minivllm_amd.engine.step import class_rows
    ops, dtype, H, Hkv, D, ps, rows, seqs = ops_for(torch.bfloat16), torch.bfloat16, 16, 8, 128, 16, 2048, 4
    steps = [([2048], [0]), ([1900], [0]), ([1793], [100]), ([1800, 100, 1], [0, 0, 900]), ([500, 600, 700], [0, 300, 0]), ([2000], [0])]
    g = torch.Generator(device="cuda").manual_seed(13)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").to(dtype)
    pages = 4 * 128
    q, kp, vp = rand(rows, H * D), rand(pages, Hkv, ps, D), rand(pages, Hkv, D, ps)
    bt = torch.arange(pages, dtype=torch.int32, device="cuda").view(seqs, -1)

    def tensors(lens, starts):
        pad = [0] * (rows - sum(lens))
        pos = torch.tensor([p for r, s in zip(lens, starts) for p in range(s, s + r)] + pad, dtype=torch.int32)
        seq = torch.tensor([i for i, r in enumerate(lens) for _ in range(r)] + [-1] * len(pad), dtype=torch.int32)
        ends = np.cumsum([0] + lens).tolist()
        return pos, seq, torch.tensor(ends + [ends[-1]] * (seqs - len(lens)), dtype=torch.int32)
    pos, seq, cu = (t.cuda() for t in tensors(*steps[0]))
    plan = make_plan([2048], [2048])
    plan.bound, plan.bound_least, plan.q_lens, plan.path_lens, plan.path_starts = (rows, seqs), 1793, (), tuple(steps[0][0]), tuple(steps[0][1])
    plan.n_seqs, plan.cu_seqlens = seqs, cu
    assert class_rows(1793) == rows and ops._prefill_variant(plan, H // Hkv, Hkv)[4] == 44
    out = torch.zeros(rows, H * D, dtype=dtype, device="cuda")
    run = lambda: ops.attention(q, out, kp, vp, bt, ps, pos, seq, H, Hkv, D, D ** -0.5, None, plan=plan)
    run()
    torch.cuda.synchronize()
    plan.workspace.frozen = True
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    counters = ops._prompt_counters(plan.workspace)
    seen = {}
    for lens, starts in steps + steps[::-1]:
        for t, new in zip((pos, seq, cu), tensors(lens, starts)):
            t.copy_(new)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert not bool(counters.any())
        n = sum(lens)
        whole = make_plan(lens, [r + s for r, s in zip(lens, starts)])
        whole.prefill_variant = (1, 1)
        ref = torch.empty(n, H * D, dtype=dtype, device="cuda")
        ops.attention(q[:n], ref, kp, vp, bt[:len(lens)].contiguous(), ps, pos[:n], seq[:n], H, Hkv, D, D ** -0.5, None, plan=whole)
        assert float((out[:n].double() - ref.double()).norm() / ref.double().norm()) <= 2 * 2.0 ** -9
        assert torch.equal(seen.setdefault(str((lens, starts)), out[:n].clone()), out[:n])
