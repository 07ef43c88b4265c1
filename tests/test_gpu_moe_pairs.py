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


@pytest.mark.parametrize("n", [3, 200])
@pytest.mark.parametrize("hid, F, FS, E, identity, top, router, activation", [
    (256, 256, 0, 16, 2, 4, "learned", "swiglu"), (256, 256, 192, 20, 0, 3, "table", "swiglu"), (256, 320, 64, 16, 0, 2, "learned", "clamped"),
    (2048, 2048, 1024, 12, 0, 2, "table", "swiglu"), (2048, 2048, 1024, 12, 0, 2, "learned", "clamped")])
def test_the_part_takes_its_shared_expert_along(n, hid, F, FS, E, identity, top, router, activation):
    """The feed-forward part at widths the tiles take: the routing and one call for the pairs, a shared expert among them also
    where the experts are large enough for the plain pairs' kernels. Against float64, choices from the part's own logits."""
    from types import SimpleNamespace
    from minivllm_amd.kernels.ops import get_ops
    from minivllm_amd.parts.base import Runtime, Workspace
    from minivllm_amd.parts.moe import RoutedExperts, RoutedExpertsSpec
    ops = get_ops(torch.bfloat16)
    spec = RoutedExpertsSpec(hidden_size=hid, expert_size=F, num_experts=E, identity_experts=identity, top=top, router=router, table_rows=50,
                             shared_size=FS, activation=activation, limit=1.5 if activation == "clamped" else 0.0)
    g = torch.Generator(device=DEV).manual_seed(n + hid)
    w = {}
    for name, decl in RoutedExperts.tensors(spec).items():
        if decl.integer:
            w[name] = torch.rand(decl.shape[0], E, generator=g, device=DEV).argsort(1)[:, :top].to(torch.int32).contiguous()
        else:
            w[name] = (torch.randn(decl.shape, generator=g, device=DEV) / decl.shape[1] ** 0.5).bfloat16()
    rt = Runtime(device=torch.device(DEV), dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device(DEV)), max_positions=64)
    part = RoutedExperts(spec, w, rt)
    assert part.shared_packed == bool(FS)
    x = torch.randn(n, hid, generator=g, device=DEV).bfloat16()
    ctx = SimpleNamespace(token_ids=torch.randint(0, 50, (n,), generator=g, device=DEV, dtype=torch.int32))
    ops.ledger = []
    y = part.forward(x, ctx)
    torch.cuda.synchronize()
    ran, ops.ledger = [e[0] for e in ops.ledger], None
    assert ran[-1] == "mv_moe_pairs" and len(ran) == (3 if router == "learned" else 2), ran
    ids, weights = (rt.workspace.get(name, (n, top), dt) for name, dt in (("moe.ids", torch.int32), ("moe.weights", torch.float32)))

    def pair(rows, gate, up, down):
        p, u = rows @ gate.double().T, rows @ up.double().T
        if activation == "clamped":
            p, u = p.clamp(max=1.5), u.clamp(-1.5, 1.5)
            return (p * torch.sigmoid(1.702 * p) * (u + 1)) @ down.double().T
        return (p * torch.sigmoid(p) * u) @ down.double().T
    xd = x.double()
    want = pair(xd, w["shared.gate"], w["shared.up"], w["shared.down"]) if FS else torch.zeros_like(xd)
    for e in range(E + identity):
        t, k = (ids == e).nonzero(as_tuple=True)
        if t.numel():
            rows = pair(xd[t], w[f"gate.{e}"], w[f"up.{e}"], w[f"down.{e}"]) if e < E else xd[t]
            want.index_add_(0, t, weights[t, k].double()[:, None] * rows)
    assert float((y.double() - want).abs().max() / want.abs().max()) <= 1e-2
