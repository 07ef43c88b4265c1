"""The recurrences with a matrix state as products over chunks of tokens, against the same recurrence token by token in
float64, and beside the scans that take the shorter requests of the step."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
RULES = ("delta", "channel", "gated", "sum")


def ops_for(dtype):
    from minivllm_amd.kernels.ops import get_ops
    return get_ops(dtype)


def i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def unit(x):
    return x / x.pow(2).sum(-1, keepdim=True).sqrt()


def make(rule, n, H, G, dk, dv, seed, forgetting, dtype):
    """Operands of the scan of that rule, and (w, a, b, x, r, v) per head in float64: p = a^T S; S <- w S + b p^T + x v^T; o = S^T r.
    ``forgetting``: how much of the decays' range is used: 0 every decay one, 3 down to exact zeros."""
    g = torch.Generator().manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g)
    wide = dk if rule in ("delta", "channel") else 1
    w = torch.exp(-forgetting * torch.rand(n, H, wide, generator=g) ** 4)
    if forgetting >= 3:
        w[torch.rand(n, H, wide, generator=g) < 0.02] = 0.0
        w[torch.rand(n, H, wide, generator=g) < 0.02] = 1e-30
    if rule == "delta":
        r, k, v = rand(n, H, dk), rand(n, H, dk), rand(n, H, dv)
        u, rate = unit(k), torch.rand(n, H, dk, generator=g)
        rows = torch.cat([r.flatten(1), k.flatten(1), v.flatten(1)], 1).to(dtype)
        v = rows[:, 2 * H * dk:].float().view(n, H, dv)
        ops_in = [rows.to(DEV), torch.stack([w, rate * u, u, k, r], 2).contiguous().to(DEV)]
        plain = (w, u, -rate * u, k, r, v)
    else:
        q, k, v, strength = rand(n, G, dk) * dk ** -0.5, unit(rand(n, G, dk)), rand(n, H, dv), torch.rand(n, H, generator=g)
        qh, kh = (t.repeat_interleave(H // G, 1) for t in (q, k))
        first = [torch.stack([q, k], 2).contiguous().to(DEV), v.to(DEV)]
        if rule == "channel":
            z = torch.cat([w.flatten(1), rand(n, 8)], 1).contiguous()
            ops_in = first + [strength.to(DEV), z.to(DEV)]
        else:
            ops_in = first + [torch.cat([w, strength[..., None], rand(n, H, 2)], 2).contiguous().to(DEV)]
        if rule == "sum":
            plain = (w, torch.zeros_like(kh), torch.zeros_like(kh), kh, qh, strength[..., None] * v)
        else:
            plain = (w, w * kh, -strength[..., None] * kh, strength[..., None] * kh, qh, v)
    return ops_in, [t.double() for t in plain]


def walk(plain, S):
    """Token by token: S [H, dk, dv] float64."""
    w, a, b, x, r, v = plain
    out = torch.empty_like(v)
    S = S.clone()
    for t in range(v.shape[0]):
        p = torch.einsum("hk,hkv->hv", a[t], S)
        S = w[t][:, :, None] * S + b[t][:, :, None] * p[:, None] + x[t][:, :, None] * v[t][:, None]
        out[t] = torch.einsum("hk,hkv->hv", r[t], S)
    return out, S


def run(ops, rule, ops_in, state, lens, slots, pad_seqs, H, G, dk, dv, raw, units):
    ends = [0]
    for q in lens:
        ends.append(ends[-1] + q)
    cu = i32(ends + [ends[-1]] * pad_seqs)
    where = (cu, i32(list(slots) + [0] * pad_seqs), len(lens) + pad_seqs)
    scratch = (torch.empty((units, H) + ((dk, dk) if rule != "sum" else ()), dtype=torch.float32, device=DEV),
               torch.empty((units, H, dv, dk), dtype=torch.float32, device=DEV),
               torch.empty((raw.shape[0], H, dk), dtype=torch.float32, device=DEV))
    line = ops.delta_chunk_line()
    if rule == "delta":
        args = (*ops_in, state, *where, H, dk)
        ops.delta_chunks(*args, *scratch, raw)
        ops.delta_scan(*args, raw, below=line)
    elif rule == "channel":
        args = (*ops_in, state, *where, H, G, dk, dv)
        ops.channel_chunks(*args, *scratch, raw)
        ops.channel_scan(*args, raw, below=line)
    else:
        args = (*ops_in, state, *where, H, G, dk, dv, rule == "gated")
        ops.state_chunks(*args, *scratch, raw)
        ops.state_scan(*args, raw, below=line)
    torch.cuda.synchronize()


def close(got, want, tol, what):
    off = float((got.double().cpu() - want).abs().max()) / max(1e-30, float(want.abs().max()))
    assert off <= tol, f"{what}: {off}"


@pytest.mark.parametrize("rule", RULES)
@pytest.mark.parametrize("H, G, dk, dv", [(3, 3, 64, 64), (4, 2, 64, 65), (2, 1, 64, 80), (2, 2, 64, 1), (2, 1, 128, 128), (2, 2, 128, 33),
                                          (1, 1, 128, 144)])
@pytest.mark.parametrize("forgetting", [0.0, 0.5, 3.0])
def test_chunks_and_scan_of_one_step(rule, H, G, dk, dv, forgetting):
    """Requests on both sides of the line (127 and 128 tokens), whole chunks and remainders of one token, on slots out of
    order with states that are not zero; two padding rows and a padding request. Float sums of up to a few hundred
    products of numbers of size one: 2e-5 of the largest, as for the scans. With decays of one and weights of random
    keys the state grows with the token count, which the largest value takes in."""
    if rule == "delta" and (dv != dk or G != H):
        pytest.skip("square heads with keys of their own")
    dtype = torch.bfloat16 if dk == 64 else torch.float32
    ops = ops_for(dtype)
    assert ops.delta_chunks_serve(rule, dk, dv)
    line = ops.delta_chunk_line()
    lens, slots = [line + 1, 1, line - 1, 2 * line + 17, line], [2, 5, 0, 4, 1]
    n = sum(lens)
    ops_in, plain = make(rule, n + 2, H, G, dk, dv, dk + dv + H, forgetting, dtype)
    S0 = 0.3 * torch.randn(7, H, dk, dv, generator=torch.Generator().manual_seed(9))
    state = S0.transpose(2, 3).contiguous().to(DEV)
    raw = torch.full((n + 2, H * dv) if rule == "delta" else (n + 2, H, dv), float("nan"), dtype=torch.float32, device=DEV)
    C = ops.delta_chunk_tokens()
    run(ops, rule, ops_in, state, lens, slots, 1, H, G, dk, dv, raw, sum(-(-q // C) for q in lens) + 3)
    base = 0
    for q, slot in zip(lens, slots):
        want, S = walk([t[base:base + q] for t in plain], S0[slot].double())
        close(raw[base:base + q].view(q, H, dv), want, 2e-5, f"outputs of {q} tokens")
        close(state[slot].transpose(1, 2), S, 2e-5, f"state after {q} tokens")
        base += q
    for slot in (3, 6):
        assert torch.equal(state[slot].cpu(), S0[slot].transpose(1, 2)), "a slot nobody holds was touched"
    assert bool(torch.isnan(raw[n:]).all()), "a padding row was written"


@pytest.mark.parametrize("rule", RULES)
def test_many_requests_and_the_scan_alone_agree(rule):
    """300 requests of which every eleventh is long (the search for a chunk's request goes round more than once): the
    rows of the scan over everything."""
    H, G, dk, dv = (1, 1, 64, 64)
    ops = ops_for(torch.bfloat16)
    line = ops.delta_chunk_line()
    lens = [line + s % 40 if s % 11 == 0 else s % 3 for s in range(300)]
    n = sum(lens)
    ops_in, _ = make(rule, n, H, G, dk, dv, 5, 0.5, torch.bfloat16)
    rows, states = [], []
    for chunked in (True, False):
        state = torch.zeros(300, H, dv, dk, dtype=torch.float32, device=DEV)
        raw = torch.zeros((n, H * dv) if rule == "delta" else (n, H, dv), dtype=torch.float32, device=DEV)
        if chunked:
            run(ops, rule, ops_in, state, lens, range(300), 0, H, G, dk, dv, raw, sum(-(-q // 32) for q in lens))
        else:
            ends = [0]
            for q in lens:
                ends.append(ends[-1] + q)
            where = (i32(ends), i32(list(range(300))), 300)
            if rule == "delta":
                ops.delta_scan(*ops_in, state, *where, H, dk, raw)
            elif rule == "channel":
                ops.channel_scan(*ops_in, state, *where, H, G, dk, dv, raw)
            else:
                ops.state_scan(*ops_in, state, *where, H, G, dk, dv, rule == "gated", raw)
            torch.cuda.synchronize()
        rows.append(raw)
        states.append(state)
    close(rows[0], rows[1].double().cpu(), 2e-5, "rows")
    close(states[0], states[1].double().cpu(), 2e-5, "states")
