"""The MFMA prompt attention's narrow units (at most 16 columns: decoding requests in a step with prompts, a prompt's last
tokens), each wave on blocks of its own, against attention in 64 bits."""
import math

import numpy as np
import pytest
import torch

from test_gpu_kernels import OP_TOL, dev, fill_pages, make_plan, ops_for, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt, kw", [(1, 1), (1, 2), (2, 2)])
@pytest.mark.parametrize("H, Hkv, D, ps", [(4, 2, 128, 16), (16, 1, 64, 32), (3, 1, 128, 64), (10, 2, 64, 16)])
@pytest.mark.parametrize("window, first", [(None, 0), (90, 0), (70, 40)])
def test_narrow_units(nt, kw, H, Hkv, D, ps, window, first):
    """Contexts of one key, of a block and a key to each side, of one round of the waves (four or eight blocks) and a block to
    each side, of many rounds; under a window with pages given back, with kept first positions; units of one token, of as
    many as a tile holds and of one more (the wide form). Slots behind a context hold NaN."""
    ops, dtype = ops_for(torch.bfloat16), torch.bfloat16
    g = torch.Generator().manual_seed(71 + D)
    group = H // Hkv
    tile = 16 // group
    ctx_lens = [1, 31, 32, 33, 96, 127, 129, 256, 257, 500, 1200, tile, 300, 301, 64 + tile + 1]
    q_lens = [1] * 11 + [tile, tile, tile + 1, tile + 1]
    q_lens[3] = 2
    k_all = [torch.randn(c, Hkv, D, generator=g).to(dtype).double() for c in ctx_lens]
    v_all = [torch.randn(c, Hkv, D, generator=g).to(dtype).double() for c in ctx_lens]
    pages_per = [-(-c // ps) for c in ctx_lens]
    num_pages = sum(pages_per) + 3
    perm = torch.randperm(num_pages, generator=g).tolist()
    tables, cur = [], 0
    for n_p in pages_per:
        tables.append(perm[cur:cur + n_p])
        cur += n_p
    if window is not None:
        for s, (c, ql) in enumerate(zip(ctx_lens, q_lens)):
            for i in range(-(-first // ps), max(0, (c - ql) - window) // ps):
                tables[s][i] = -1
    kp, vp = fill_pages(k_all, v_all, tables, ps, Hkv, D, num_pages, dtype)
    bt = torch.full((len(tables), max(pages_per)), -1, dtype=torch.int32)
    for s, t in enumerate(tables):
        bt[s, :len(t)] = torch.tensor(t, dtype=torch.int32)
    positions = torch.tensor([p for c, ql in zip(ctx_lens, q_lens) for p in range(c - ql, c)], dtype=torch.int32)
    token_seq = torch.tensor([s for s, ql in enumerate(q_lens) for _ in range(ql)], dtype=torch.int32)
    n, ends, scale = len(positions), np.cumsum(q_lens) - 1, 1.0 / math.sqrt(D)
    q = torch.randn(n, H, D, generator=g)
    for s, row in enumerate(ends):                 # every request's last query singles out its first visible key
        far = 0 if window is None or first else max(0, ctx_lens[s] - 1 - window)
        q[row] = 6.0 * k_all[s][far].float().repeat_interleave(group, dim=0) / math.sqrt(D)
    q = q.to(dtype)
    out = torch.full((n, H * D), float("nan"), dtype=dtype, device="cuda")
    plan = make_plan(q_lens, ctx_lens)
    plan.prefill_variant = (nt, kw)
    ops.attention(dev(q.view(n, H * D)), out, kp, vp, dev(bt), ps, dev(positions), dev(token_seq), H, Hkv, D, scale, window, plan=plan,
                  **({"keep_first": first} if first else {}))
    want = torch.zeros(n, H, D, dtype=torch.float64)
    for i in range(n):
        s, p = int(token_seq[i]), int(positions[i])
        keys = [j for j in range(p + 1) if window is None or j >= p - window or j < first]
        for h in range(H):
            w = torch.softmax((k_all[s][keys, h // group] @ q[i, h].double()) * scale, dim=0)
            want[i, h] = w @ v_all[s][keys, h // group]
    assert rel_err(out.float().cpu().view(n, H, D).numpy(), want.numpy()) <= 2 * OP_TOL[dtype]
