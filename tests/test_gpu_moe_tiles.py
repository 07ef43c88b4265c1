"""Every shape of tile that a mixture's products choose from, against the mixture in float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("limit", [0.0, 1.5])
@pytest.mark.parametrize("n, hid, F, FS, E, top, tiles", [
    # (rows of a tile, columns of a tile of the first product, of the second)
    (20, 64, 64, 0, 8, 1, (32, 64, 64)), (20, 832, 64, 0, 48, 2, (32, 64, 128)), (100, 320, 64, 0, 200, 1, (32, 64, 256)),
    (20, 64, 448, 0, 96, 2, (32, 256, 64)), (1500, 64, 64, 64, 24, 2, (64, 128, 128)), (1100, 320, 64, 64, 96, 2, (64, 128, 256)),
    (1100, 64, 192, 64, 96, 2, (64, 256, 128)), (300, 64, 64, 64, 150, 2, (96, 128, 128)), (300, 576, 64, 64, 150, 2, (96, 128, 256)),
    (300, 64, 192, 64, 150, 2, (96, 256, 128)), (1100, 320, 448, 64, 24, 2, (128, 128, 128)), (1500, 832, 192, 64, 48, 2, (128, 128, 256)),
    (1500, 320, 448, 64, 48, 2, (128, 256, 128)), (1500, 576, 448, 64, 24, 2, (160, 128, 128)), (1000, 1024, 768, 768, 32, 4, (160, 256, 256)),
    # as many pairs as the threads that sort them keep, and more
    (2048, 64, 64, 64, 24, 4, (96, 128, 128)), (2100, 64, 64, 64, 24, 4, (96, 128, 128))])
def test_tiles(n, hid, F, FS, E, top, tiles, limit):
    """Full and partial tiles, an expert that most tokens chose, empty ones, tokens without an expert. bfloat16 operands summed in float,
    activations rounded once to bfloat16 (2^-9 of each of F terms of random sign): 1e-2 of the largest output, and each row's share of it."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    shape = ops.lib.dll.mv_moe_pairs_shape(n, top, E, hid, F, FS, 256)
    assert (shape & 1023, shape >> 10 & 1023, shape >> 20) == tiles
    g = torch.Generator(device=DEV).manual_seed(n + hid + E)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x = rand(n, hid).bfloat16()
    gate_up, down = (rand(2 * E * F + 2 * FS, hid) / hid ** 0.5).bfloat16(), (rand(hid, E * F + FS) / F ** 0.5).bfloat16()
    ids = torch.rand(n, E, generator=g, device=DEV).argsort(1)[:, :top].int().contiguous()
    ids[: n // 3, 0] = 2
    ids[ids == E - 1] = E - 2
    ids[-1] = -1
    weights = torch.rand(n, top, generator=g, device=DEV)
    pairs = n * (top + (1 if FS else 0))
    act = torch.full((pairs, max(F, FS)), float("nan"), dtype=torch.bfloat16, device=DEV)
    out, y = torch.full((pairs, hid), float("nan"), device=DEV), torch.full((n + 1, hid), 3.0, dtype=torch.bfloat16, device=DEV)
    ints = torch.full((ops.moe_pairs_ints(n, top, E, FS),), -7, dtype=torch.int32, device=DEV)
    assert ops.moe_pairs(x, gate_up, down, E, 0, F, FS, ids, weights, None, ints, act, out, y[:n], limit=limit, slope=1.702)
    xd, want = x.double(), torch.zeros(n, hid, dtype=torch.float64, device=DEV)

    def expert(rows, gate, up, back):
        p, u = rows @ gate.double().T, rows @ up.double().T
        if limit > 0:
            p, u = p.clamp(max=limit), u.clamp(-limit, limit)
            return (p * torch.sigmoid(1.702 * p) * (u + 1)) @ back.double().T
        return (p * torch.sigmoid(p) * u) @ back.double().T
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            block = slice(e * F, (e + 1) * F)
            want.index_add_(0, t, weights[t, k].double()[:, None] * expert(xd[t], gate_up[block], gate_up[E * F:][block], down[:, block]))
    if FS:
        want += expert(xd, gate_up[2 * E * F:2 * E * F + FS], gate_up[2 * E * F + FS:], down[:, E * F:])
    error = (y[:n].double() - want).abs().amax(1)
    assert float(error.max() / want.abs().max()) <= 1e-2
    assert bool((error <= 0.05 * want.abs().amax(1) + 1e-3 * want.abs().max()).all()), "a row is another's"
    assert bool((y[n] == 3.0).all())


def test_activations_at_the_ends():
    """What the activation makes of infinite, huge and no numbers (one expert, one token, products that are the inputs)."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    gates = [float("inf"), float("-inf"), float("nan"), 3e38, -3e38, 90.0, -90.0, -1e4, 0.0, -0.0, 20.0, -20.0]
    n, hid, F = len(gates), 64, 64
    x = torch.zeros(n, hid, device=DEV)
    x[:, 0], x[:, 1] = torch.tensor([v if abs(v) < 1e30 else (1.0 if v != v else v) for v in gates], device=DEV), 2.0
    x[2, 0] = float("nan")
    x[:, 0].clamp_(-3e38, 3e38)
    gate_up = torch.zeros(2 * F, hid, dtype=torch.bfloat16, device=DEV)
    gate_up[:F, 0], gate_up[F:, 1] = 1.0, 1.0
    down = torch.zeros(hid, F, dtype=torch.bfloat16, device=DEV)
    down[:, 0] = 1.0
    ids, weights = torch.zeros(n, 1, dtype=torch.int32, device=DEV), torch.ones(n, 1, device=DEV)
    act, out = torch.zeros(n, F, dtype=torch.bfloat16, device=DEV), torch.zeros(n, hid, device=DEV)
    y = torch.zeros(n, hid, dtype=torch.bfloat16, device=DEV)
    ints = torch.zeros(ops.moe_pairs_ints(n, 1, 1, 0), dtype=torch.int32, device=DEV)
    assert ops.moe_pairs(x.bfloat16(), gate_up, down, 1, 0, F, 0, ids, weights, None, ints, act, out, y)
    v = x.bfloat16()[:, 0].float()
    want = (torch.nn.functional.silu(v) * 2).bfloat16().float()
    got = act[:, 0].float()
    assert torch.equal(got.isnan(), want.isnan())
    ok = ~want.isnan()
    assert torch.allclose(got[ok], want[ok], rtol=2.0 ** -8, atol=1e-30)
