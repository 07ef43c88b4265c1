"""Attention over a cached latent for steps with prompt portions: the kernel whose workgroups share key rows among a request's
neighbouring tokens, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


@pytest.mark.parametrize("R, DR", [(256, 64), (128, 64), (256, 0), (192, 0), (128, 0), (64, 0)])
@pytest.mark.parametrize("page, H", [(16, 16), (8, 3), (64, 37)])
@pytest.mark.parametrize("window, sinks", [(None, False), (0, False), (5, True), (40, False), (100, True)])
def test_tokens_that_share_key_rows(R, DR, page, H, window, sinks):
    """Five requests in one step: whole runs of tokens, remainders and single tokens, at positions on and off the blocks and
    pages, beside two padding rows and a padding request. What no query may see is NaN: slots behind a request's last token,
    pages in front of every window, pages of nobody. Weights and values are bfloat16: 1.2e-2 of the largest, as for the other
    kernels."""
    from minivllm_amd.engine.step import AttentionPlan
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    unit = int(ops.lib.dll.mv_attention_latent_prompt_tokens())
    lens, starts = [1, unit, 3 * unit + 5, 70, 2], [63, 96, 27, 0, 200]
    g = torch.Generator(device=DEV).manual_seed(R + H + page)
    D, n = R + DR, sum(lens)
    width = max(s + q for s, q in zip(starts, lens)) // page + 1
    count = sum((s + q - 1) // page + 1 for s, q in zip(starts, lens)) + 3
    perm = torch.randperm(count, generator=g, device=DEV).tolist()
    pages = torch.full((count, page, D), float("nan"), dtype=torch.bfloat16, device=DEV)
    table = torch.full((len(lens) + 1, width), -1, dtype=torch.int32)
    keys, at = [], 0
    for s, (q, start) in enumerate(zip(lens, starts)):
        rows = torch.randn(start + q, D, generator=g, device=DEV).bfloat16()
        keys.append(rows)
        low = 0 if window is None else max(0, start - window) // page
        for p in range((start + q - 1) // page + 1):
            if p >= low:
                table[s, p] = perm[at]
                part = rows[p * page:(p + 1) * page]
                pages[perm[at], :len(part)] = part
            at += 1
    q = torch.randn(n + 2, H, D, generator=g, device=DEV)
    pos = [start + t for m, start in zip(lens, starts) for t in range(m)] + [0, 0]
    seq = [s for s, m in enumerate(lens) for _ in range(m)] + [-1, -1]
    ends = [0]
    for m in lens:
        ends.append(ends[-1] + m)
    plan = AttentionPlan(decode_only=False, max_q_len=max(lens), max_context_len=202, n_seqs=len(lens) + 1, q_lens=lens + [0],
                         cu_seqlens=i32(ends + [ends[-1]]))
    sink = torch.linspace(-2.0, 3.0, H, device=DEV) if sinks else None
    out = torch.full((n + 2, H, R), float("nan"), device=DEV)
    ops.ledger = []
    scale = 0.7 / D ** 0.5
    ops.attention_latent(q, out, pages, table.to(DEV), page, i32(pos), i32(seq), H, R, DR, scale, plan=plan, window=window, sink=sink,
                         pages_t=pages[:, :, :R].transpose(1, 2).contiguous())
    torch.cuda.synchronize()
    ran, ops.ledger = [e[0] for e in ops.ledger], None
    assert ran == ["mv_attention_latent_prompt"]
    for t in range(n):
        k = keys[seq[t]][:pos[t] + 1].double()
        if window is not None:
            k = k[max(0, pos[t] - window):]
        s = q[t].double() @ k.T * scale
        top = s.max(-1, keepdim=True).values
        if sinks:
            top = torch.maximum(top, sink.double()[:, None])
        e = torch.exp(s - top)
        den = e.sum(-1, keepdim=True) + (torch.exp(sink.double()[:, None] - top) if sinks else 0.0)
        want = (e / den) @ k[:, :R]
        off = float((out[t].double() - want).abs().max() / want.abs().max())
        assert off <= 1.2e-2, f"row {t} at position {pos[t]} of request {seq[t]}: {off}"
    assert bool((out[n:] == 0).all()), "padding rows are zeros"
