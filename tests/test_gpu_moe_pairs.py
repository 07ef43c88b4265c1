"""A mixture's tiled products over the chosen (token, expert) pairs, against the mixture in float64 from the same lists."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.mark.parametrize("n", [1, 6, 33, 130, 700])
@pytest.mark.parametrize("hid, F, FS, E, identity, top, limit", [(64, 64, 0, 5, 2, 3, 0.0), (192, 128, 64, 12, 0, 2, 0.0),
                                                                 (128, 64, 192, 3, 0, 3, 0.0), (320, 192, 0, 40, 0, 4, 1.5),
                                                                 (128, 576, 128, 1, 1, 1, 0.0), (64, 64, 0, 1000, 0, 2, 0.0)])
def test_pairs_against_the_mixture(n, hid, F, FS, E, identity, top, limit):
    """Few and many rows an expert (each height of a tile, full and partial), an expert that nobody chose and one that most
    chose, experts without tensors among the choices, pairs without an expert, a shared expert narrower and wider than
    the others, widths that are no multiple of a tile. bfloat16 operands summed in float, activations rounded once to bfloat16
    (2^-9 of each of F terms of random sign): 1e-2 of the largest output."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(n + hid + E)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x = rand(n, hid).bfloat16()
    gate_up = (rand(2 * E * F + 2 * FS, hid) / hid ** 0.5).bfloat16()
    down = (rand(hid, E * F + FS) / F ** 0.5).bfloat16()
    ids = torch.stack([torch.randperm(E + identity, generator=g, device=DEV)[:top] for _ in range(n)]).int()
    if E > 2:
        ids[: n // 2 + 1, 0] = 1                             # a crowded expert (a token may name it twice)
        ids[ids == E - 1] = E - 2                            # an empty one
    if n > 4:
        ids[3, top - 1] = -1
    weights = torch.rand(n, top, generator=g, device=DEV)
    dense = torch.zeros(n, E + identity, device=DEV)
    for k in range(top):
        ok = ids[:, k] >= 0
        dense[ok.nonzero().flatten(), ids[ok, k].long()] += weights[ok, k]
    pairs = n * (top + (1 if FS else 0))
    ints = torch.full((ops.moe_pairs_ints(n, top, E, FS),), -7, dtype=torch.int32, device=DEV)
    act = torch.full((pairs, max(F, FS)), float("nan"), dtype=torch.bfloat16, device=DEV)
    out = torch.full((pairs, hid), float("nan"), device=DEV)
    y = torch.full((n + 1, hid), 3.0, dtype=torch.bfloat16, device=DEV)
    assert ops.moe_pairs(x, gate_up, down, E, identity, F, FS, ids, weights, dense, ints, act, out, y[:n], limit=limit, slope=1.702)
    torch.cuda.synchronize()
    xd, gu, dn = x.double(), gate_up.double(), down.double()

    def expert(rows, e):
        if e == E:
            a, b, d = gu[2 * E * F:2 * E * F + FS], gu[2 * E * F + FS:], dn[:, E * F:]
        else:
            a, b, d = gu[e * F:(e + 1) * F], gu[(E + e) * F:(E + e + 1) * F], dn[:, e * F:(e + 1) * F]
        p, u = rows @ a.T, rows @ b.T
        if limit > 0:
            p, u = p.clamp(max=limit), u.clamp(-limit, limit)
            return (p * torch.sigmoid(1.702 * p) * (u + 1)) @ d.T
        return (p * torch.sigmoid(p) * u) @ d.T
    want = torch.zeros(n, hid, dtype=torch.float64, device=DEV)
    for e in range(E):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            want.index_add_(0, t, weights[t, k].double()[:, None] * expert(xd[t], e))
    want += dense[:, E:].double().sum(1, keepdim=True) * xd
    if FS:
        want += expert(xd, E)
    assert float((y[:n].double() - want).abs().max() / want.abs().max()) <= 1e-2
    assert bool((y[n] == 3.0).all())
    again = torch.empty_like(y)
    assert ops.moe_pairs(x, gate_up, down, E, identity, F, FS, ids, weights, dense, ints, act, out, again[:n], limit=limit, slope=1.702)
    assert torch.equal(again[:n], y[:n]), "the order of an expert's pairs shows"


def test_widths_that_are_not_served_are_left_alone():
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    z = lambda *s, dt=torch.bfloat16: torch.zeros(*s, dtype=dt, device=DEV)
    for hid, F in ((96, 64), (64, 32)):
        assert not ops.moe_pairs(z(2, hid), z(2 * F, hid), z(hid, F), 1, 0, F, 0, z(2, 1, dt=torch.int32), z(2, 1, dt=torch.float32), None,
                                 z(ops.moe_pairs_ints(2, 1, 1, 0), dt=torch.int32), z(2, F), z(2, hid, dt=torch.float32), z(2, hid))
