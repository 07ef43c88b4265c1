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


# the general rule's vectors made in the chunks' kernel: a rank of one to four blocks, requests that end inside a run and inside a chunk, of the least
# number of tokens, with a request that brings none between them
@pytest.mark.parametrize("H, rank, weights", [(2, 16, torch.bfloat16), (3, 64, torch.float32), (1, 48, torch.bfloat16)])
@pytest.mark.parametrize("lens", [[128], [193, 0, 160], [145, 271]])
def test_chunks_straight_from_the_rows(H, rank, weights, lens):
    """Against the recurrence in float64 from the same rows: errors of float32 sums, 2^-24 a term, over what a chunk adds up."""
    dtype, D, rate, eps, pad = torch.bfloat16, 64, 0.6, 1e-6, 8
    ops, n = ops_for(dtype), sum(lens)
    inner = H * D
    g = torch.Generator().manual_seed(rank + n)
    rows = torch.randn(n, 5 * inner + rank + pad, generator=g).to(dtype)
    rows[:, 5 * inner + rank:] = float("nan")
    w2t, w0, ab = ((torch.randn(*s, generator=g) * f).to(weights) for s, f in (((rank, inner), rank ** -0.5), ((inner,), 1.0), ((inner,), 1.0)))
    f = rows.double()
    r, k, v, _, a = (f[:, j * inner:(j + 1) * inner].view(n, H, D) for j in range(5))
    w = torch.exp(-rate * torch.sigmoid(torch.tanh(f[:, 5 * inner:5 * inner + rank]) @ w2t.double() + w0.double())).view(n, H, D)
    u = k / (k.pow(2).sum(-1, keepdim=True) + eps).sqrt()
    plain = w, u, -torch.sigmoid(a + ab.double().view(H, D)) * u, k, r, v
    slots = list(range(len(lens)))[::-1]
    state = torch.randn(len(lens), H, D, D, generator=g)
    packed, cu = rows.to(DEV), i32([0] + torch.tensor(lens).cumsum(0).tolist())
    units = sum(-(-x // ops.delta_chunk_tokens()) for x in lens) + 2
    scratch = [torch.empty(units, H, D, D, device=DEV), torch.empty(units, H, D, D, device=DEV), torch.empty(n, H, D, device=DEV)]
    raw, dstate = torch.empty(n, inner, device=DEV), state.to(DEV)
    weights_dev = [t.to(DEV) for t in (w2t, w0, ab)]
    assert ops.delta_chunks_rows_serve(packed, D, rank, weights_dev[2])
    ops.delta_chunks_rows(packed, H, D, rank, *weights_dev, rate, eps, dstate, cu, i32(slots), len(lens), *scratch, raw)
    # ... and as close as the vectors laid out in memory are
    coef, raw2, dstate2 = torch.empty(n, H, 5, D, device=DEV), torch.empty(n, inner, device=DEV), state.to(DEV)
    ops.delta_prepare(packed, H, D, rank, *weights_dev, rate, eps, coef)
    ops.delta_chunks(packed, coef, dstate2, cu, i32(slots), len(lens), H, D, *scratch, raw2)
    first = 0
    for s, count in enumerate(lens):
        if count:
            want, S = walk([t[first:first + count] for t in plain], state[slots[s]].double().transpose(1, 2))
            for got, got2, ref in ((raw[first:first + count].view(count, H, D), raw2[first:first + count].view(count, H, D), want),
                                   (dstate[slots[s]].transpose(1, 2), dstate2[slots[s]].transpose(1, 2), S)):
                err, err2 = (float((x.double().cpu() - ref).norm() / ref.norm()) for x in (got, got2))
                assert err <= 5e-6 and err <= 1.5 * err2 + 2.0 ** -24, (err, err2)
        else:
            assert torch.equal(dstate[slots[s]].cpu(), state[slots[s]])
        first += count


# the convolution's rules' vectors made in the chunks' kernel: every number of taps, groups of one and two heads, requests that start behind kept inputs,
# end inside a run and inside a chunk, bring the least number of tokens or none
@pytest.mark.parametrize("rule", ["gated", "channel"])
@pytest.mark.parametrize("H, G, taps, weights", [(2, 1, 4, torch.bfloat16), (3, 3, 3, torch.float32), (4, 2, 2, torch.bfloat16)])
@pytest.mark.parametrize("lens", [[128], [193, 0, 160], [145, 271]])
def test_chunks_straight_from_convolved_rows(rule, H, G, taps, weights, lens):
    """Against the recurrence in float64 from the same rows: errors of float32 sums, 2^-24 a term over the 64 channels of a length and the tokens of a
    request, and no larger than those of the vectors laid out in memory and the chunks behind them, which add up the same terms in another
    order. The kept inputs are the same bits."""
    dtype, D, eps = torch.bfloat16, 64, 1e-6
    ops, n, channel = ops_for(dtype), sum(lens), rule == "channel"
    C = 2 * G * D + H * D
    gate_off = C + H * D
    g = torch.Generator().manual_seed(17 * taps + n)
    rand = lambda *s: torch.randn(*s, generator=g)
    packed = rand(n, (gate_off + 2 * H + 7) // 8 * 8 + 8).to(dtype).to(DEV)
    conv_w, a_log = (rand(C, taps) / taps ** 0.5).to(weights).to(DEV), (rand(H) - 1).to(weights).to(DEV)
    dt_bias = rand(H * D if channel else H).to(weights).to(DEV)
    kept, state = rand(len(lens) + 1, taps - 1, C).to(dtype).to(DEV), rand(len(lens) + 1, H, D, D).to(DEV)
    z = rand(n, 2 * H * D).to(DEV) if channel else None
    ends = torch.tensor([0] + lens).cumsum(0).tolist()
    cu, slots, count = i32(ends), i32(list(range(len(lens), 0, -1))), len(lens)
    token_seq = i32([s for s, q in enumerate(lens) for _ in range(q)])
    units = sum(-(-x // ops.delta_chunk_tokens()) for x in lens) + 2
    scratch = [torch.empty(units, H, D, D, device=DEV), torch.empty(units, H, D, D, device=DEV), torch.empty(n, H, D, device=DEV)]
    results = []
    for straight in (True, False):
        k2, s2, raw, z2 = kept.clone(), state.clone(), torch.empty(n, H, D, device=DEV), z.clone() if channel else None
        if straight:
            assert ops.delta_chunks_conv_serve(packed, D, D, taps, conv_w, dt_bias, k2, z2)
            ops.delta_chunks_conv(rule, packed, gate_off, H, G, D, D, taps, conv_w, a_log, dt_bias, k2, eps, z2, s2, cu, slots, count, *scratch, raw)
            assert z2 is None or torch.equal(z2, z)
        else:
            qk, vals = torch.empty(n, G, 2, D, device=DEV), torch.empty(n, H, D, device=DEV)
            if channel:
                beta = torch.empty(n, H, device=DEV)
                ops.channel_prepare(packed, H, G, D, D, taps, gate_off, conv_w, a_log, dt_bias, k2, eps, token_seq, cu, slots, count, qk, vals, beta, z2)
                ops.channel_chunks(qk, vals, beta, z2, s2, cu, slots, count, H, G, D, D, *scratch, raw)
            else:
                gates = torch.empty(n, H, 4, device=DEV)
                ops.gated_delta_prepare(packed, H, G, D, D, taps, conv_w, a_log, dt_bias, k2, eps, token_seq, cu, slots, count, qk, vals, gates)
                ops.state_chunks(qk, vals, gates, s2, cu, slots, count, H, G, D, D, True, *scratch, raw)
        results.append((raw, s2, k2))
    for got, want in zip(results[0][:2], results[1][:2]):
        assert bool(torch.isfinite(want).all())
        assert float((got.double() - want.double()).norm() / want.double().norm()) <= 16 * 2.0 ** -24 * 64 ** 0.5
    assert torch.equal(results[0][2], results[1][2])
    f, taps_w, rate, bias = packed.double().cpu(), conv_w.double().cpu(), -torch.exp(a_log.double().cpu()), dt_bias.double().cpu()
    for s, count in enumerate(lens):
        first, slot = ends[s], len(lens) - s
        if not count:
            assert torch.equal(results[0][1][slot], state[slot])
            continue
        rows = f[first:first + count]
        inputs = torch.cat([kept[slot].double().cpu(), rows[:, :C]])
        x = torch.nn.functional.silu(sum(inputs[j:j + count] * taps_w[:, j] for j in range(taps)))
        lengths = lambda t: t / (t.pow(2).sum(-1, keepdim=True) + eps).sqrt()
        q, k = (lengths(x[:, j * G * D:(j + 1) * G * D].view(count, G, D)).repeat_interleave(H // G, 1) for j in range(2))
        v, beta = x[:, 2 * G * D:].view(count, H, D), torch.sigmoid(rows[:, gate_off:gate_off + H])[..., None]
        if channel:
            before = z[first:first + count, :H * D].double().cpu() + bias
            w = torch.exp(rate[:, None] * torch.nn.functional.softplus(before).view(count, H, D))
        else:
            w = torch.exp(rate * torch.nn.functional.softplus(rows[:, gate_off + H:gate_off + 2 * H] + bias))[..., None]
        want, S = walk((w, w * k, -beta * k, beta * k, q * D ** -0.5, v), state[slot].double().cpu().transpose(1, 2))
        for straight, laid_out, ref in ((results[0][0][first:first + count], results[1][0][first:first + count], want),
                                        (results[0][1][slot].transpose(1, 2), results[1][1][slot].transpose(1, 2), S)):
            err, err2 = (float((t.double().cpu() - ref).norm() / ref.norm()) for t in (straight, laid_out))
            assert err <= 5e-6 and err <= 1.5 * err2 + 2.0 ** -24, (err, err2)


@pytest.mark.parametrize("H", [1, 3])
@pytest.mark.parametrize("lens", [[128], [193, 0, 160], [145, 271]])
def test_mlstm_chunks_straight_from_the_rows(H, lens):
    """The bits of the vectors laid out in memory and the chunks behind them: heads of 64 x 64, requests that end inside a run and inside a chunk."""
    ops, n, D = ops_for(torch.bfloat16), sum(lens), 64
    g = torch.Generator().manual_seed(H + n)
    packed = torch.randn(n, (4 * H * D + 2 * H + 7) // 8 * 8 + 8, generator=g).bfloat16().to(DEV)
    bias = [torch.randn(H, generator=g).bfloat16().to(DEV) for _ in range(2)]
    cu, slots, count = i32(torch.tensor([0] + lens).cumsum(0).tolist()), i32(list(range(len(lens), 0, -1))), len(lens)
    token_seq = i32([s for s, q in enumerate(lens) for _ in range(q)])
    state = torch.randn(len(lens) + 1, H, D + 1, D, generator=g).to(DEV)
    units = sum(-(-x // ops.delta_chunk_tokens()) for x in lens) + 2
    scratch = [torch.empty(units, H, device=DEV), torch.empty(units, H, D + 1, D, device=DEV), torch.empty(n, H, D, device=DEV)]
    results = []
    for straight in (True, False):
        s2, raw, gates, most = state.clone(), torch.empty(n, H, D + 1, device=DEV), torch.empty(n, H, 4, device=DEV), torch.zeros(len(lens) + 1, H, device=DEV)
        qk, vals = (None, None) if straight else (torch.empty(n, H, 2, D, device=DEV), torch.empty(n, H, D + 1, device=DEV))
        ops.mlstm_prepare(packed, H, D, D, *bias, 15.0, most, token_seq, cu, slots, count, qk, vals, gates)
        if straight:
            assert ops.mlstm_chunks_serve(packed, D, D)
            ops.mlstm_chunks(packed, gates, s2, cu, slots, count, H, D, D, *scratch, raw)
        else:
            ops.state_chunks(qk, vals, gates, s2, cu, slots, count, H, H, D, D + 1, False, *scratch, raw)
        results.append((raw, s2, gates, most))
    assert bool(torch.isfinite(results[1][0]).all())
    for got, want in zip(*results):
        assert torch.equal(got, want)
