"""The kernels that prepare a recurrence's vectors eight rows a wave, and the mLSTM gates' maxima as a prefix: the vectors
of a long step against the same rows in short steps (which go one row a workgroup) bit for bit, the gates against 64 bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def i32(values):
    return torch.tensor(list(values), dtype=torch.int32, device=DEV)


def ops_for(dtype):
    from minivllm_amd.kernels.ops import Ops
    return Ops(dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rule", ["scalar", "channel"])
@pytest.mark.parametrize("taps", [2, 3, 4])
@pytest.mark.parametrize("H, G, DK, DV", [(16, 8, 64, 64), (6, 6, 40, 24), (9, 3, 65, 130), (8, 4, 128, 72), (4, 4, 256, 256)])
def test_eight_rows_a_wave(dtype, rule, taps, H, G, DK, DV):
    """Requests that begin and end inside runs of eight rows, one with kept inputs, padding rows behind; the
    short steps cut the requests at rows that are no multiple of eight."""
    ops, cut = ops_for(dtype), 21
    lens = [1, 2, 900, 13, 800, 5]                           # (rows x heads enough for the long form at every size above)
    pad = 3
    n, C = sum(lens) + pad, 2 * G * DK + H * DV
    g = torch.Generator().manual_seed(DK + taps)
    ld = C + H * DV + 2 * H
    packed = torch.randn(n, ld, generator=g).to(dtype).to(DEV)
    cw = torch.randn(C, taps, generator=g).bfloat16().to(DEV)
    al, db = torch.randn(H, generator=g).bfloat16().to(DEV), torch.randn(H * (DK if rule == "channel" else 1), generator=g).bfloat16().to(DEV)
    hist0 = torch.randn(len(lens), taps - 1, C, generator=g).to(dtype).to(DEV)
    z0 = torch.randn(n, H * DK, generator=g).to(DEV)

    def step(rows, q_lens, slots, hist, z):
        m = rows.shape[0]
        seq = [s for s, k in enumerate(q_lens) for _ in range(k)]
        seq = i32(seq + [-1] * (m - len(seq)))
        cu, sl = i32(np.concatenate([[0], np.cumsum(q_lens)])), i32(slots)
        outs = [torch.full(s, 7.0, device=DEV) for s in ((m, G, 2, DK), (m, H, DV), (m, H) if rule == "channel" else (m, H, 4))]
        if rule == "channel":
            ops.channel_prepare(rows, H, G, DK, DV, taps, C, cw, al, db, hist, 1e-6, seq, cu, sl, len(q_lens), *outs, z)
            outs.append(z)
        else:
            ops.gated_delta_prepare(rows, H, G, DK, DV, taps, cw, al, db, hist, 1e-6, seq, cu, sl, len(q_lens), *outs)
        return outs

    hist, z = hist0.clone(), z0.clone()
    got = step(packed, lens, range(len(lens)), hist, z)
    assert all(bool((t[n - pad:] == 7.0).all()) for t in got[:3]), "a padding row was written"
    base = 0
    kept = hist0.clone()
    for s, k in enumerate(lens):
        for a in range(base, base + k, cut):
            b = min(a + cut, base + k)
            want = step(packed[a:b].contiguous(), [b - a], [s], kept, z0[a:b].clone())
            for name, x, y in zip(("queries and keys", "values", "gates", "decays"), got, want):
                assert torch.equal(x[a:b], y), (name, s, a)
        base += k
    assert torch.equal(hist, kept), "kept inputs"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("length", [127, 128, 1023, 1024, 1025, 2100])
def test_gate_maxima_as_a_prefix(dtype, length):
    """Maxima, and the factors made from them. A maximum is at most ~3 caps from 0 and so is every partial sum on the way to
    the one that wins; 12 steps of the prefix round each by 2^-24 of that, the gates' own functions by a few units each."""
    ops, H, dk, dv, cap = ops_for(dtype), 3, 8, 12, 15.0
    g = torch.Generator().manual_seed(length)
    lens, n = [5, length, 200], length + 205
    g0 = 2 * H * dk + 2 * H * dv
    packed = torch.randn(n, g0 + 2 * H, generator=g)
    packed[:, g0:] *= torch.tensor([1.0, 6.0, 20.0]).repeat(2)       # maxima that move often, and gates that are cut off
    packed = packed.to(dtype)
    ib, fb = torch.randn(H, generator=g).bfloat16(), (2 + torch.randn(H, generator=g)).bfloat16()
    kept = torch.randn(3, H, generator=g)
    maxima = kept.clone().to(DEV)
    qk, vals, gates = [torch.empty(s, device=DEV) for s in ((n, H, 2, dk), (n, H, dv + 1), (n, H, 4))]
    seq = i32([s for s, k in enumerate(lens) for _ in range(k)])
    ops.mlstm_prepare(packed.to(DEV), H, dk, dv, ib.to(DEV), fb.to(DEV), cap, maxima, seq, i32([0, 5, 5 + length, n]), i32([1, 2, 0]), 3,
                      qk, vals, gates)
    p = packed.double()
    li = cap * torch.tanh((p[:, g0:g0 + H] + ib.double()) / cap)
    lf = torch.nn.functional.logsigmoid(cap * torch.tanh((p[:, g0 + H:g0 + 2 * H] + fb.double()) / cap))
    want = torch.empty(n, H, 3, dtype=torch.float64)
    base = 0
    tol = (12 * 3 * cap + 16 * cap) * 2.0 ** -24
    for k, slot in zip(lens, [1, 2, 0]):
        m = kept[slot].double()
        for t in range(base, base + k):
            new = torch.maximum(lf[t] + m, li[t])
            want[t] = torch.stack([torch.exp(lf[t] + m - new), torch.exp(li[t] - new), torch.exp(-new)], dim=-1)
            m = new
        base += k
        assert float((maxima[slot].double().cpu() - m).abs().max()) <= tol
    err = ((gates[..., :3].double().cpu() - want).abs() / want.abs().clamp_min(1e-30))
    assert float(err[..., 2].max()) <= tol and float((gates[..., :2].double().cpu() - want[..., :2]).abs().max()) <= 2 * tol
