"""The residual add and the norm between two products of a prompt's rows, taken apart into both, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def make(M, N, K, N2, gated, bias, offset, norm_dtype, seed=3):
    from minivllm_amd.kernels.ops import get_ops
    from minivllm_amd.parts import NORMS, HiddenStream, RMSNormSpec, Runtime, Workspace
    ops = get_ops(torch.bfloat16)
    rt = Runtime(device=torch.device(DEV), dtype=torch.bfloat16, ops=ops, workspace=Workspace(torch.device(DEV)), max_positions=16)
    g = torch.Generator(device=DEV).manual_seed(seed)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    spec = RMSNormSpec(size=N, eps=1e-5, unit_offset=offset)
    norm = NORMS.get(spec.kind)(spec, {"weight": ((0 if offset else 1) + 0.1 * rand(N)).to(norm_dtype)}, rt)
    rows2 = 2 * N2 if gated else N2
    t = dict(resid=3 * rand(M, N), a=rand(M, K + 8).bfloat16()[:, :K], w1=(rand(N, K) / K ** 0.5).bfloat16(), w2=(rand(rows2, N) / N ** 0.5).bfloat16(),
             b1=rand(N).bfloat16() if bias else None, b2=rand(rows2).bfloat16() if bias else None)
    return ops, norm, t, lambda resid: HiddenStream(resid.clone(), torch.empty_like(resid))


def run(ops, norm, t, stream, gated, N2):
    M, N = stream.resid.shape
    fold = norm.fold(stream, None, (t["w2"].shape[0], N, gated))
    assert fold is not None
    ops.ledger = []
    y = torch.full((M, N), 7.0, dtype=torch.bfloat16, device=DEV)
    rows = ops.gemm(t["a"][:M], t["w1"], y, t["b1"], defer_sum=True, fold=fold)
    assert rows.is_weighted_rows and bool((y == 7.0).all())
    out = torch.full((M + 1, N2), 7.0, dtype=torch.bfloat16, device=DEV)
    if gated: assert ops.gemm_swiglu(rows, t["w2"], out[:M], t["b2"])
    else: ops.gemm(rows, t["w2"], out[:M], t["b2"])
    ran, ops.ledger = [e[0] for e in ops.ledger], None
    assert ran == ["mv_gemm_into_norm", "mv_gemm_behind_norm"] and bool((out[M] == 7.0).all())
    return out[:M]


# the deep product in front (up to 512 rows of the first size) and the tiles of 64 x 64, their last rows and last round; the same choices behind
@pytest.mark.parametrize("M, N, K, N2, gated", [(129, 1024, 2048, 4096, False), (512, 1024, 3072, 3072, True), (513, 1024, 2048, 4096, False), (1000, 1024, 3072, 3072, True),
                                                (1024, 1024, 512, 592, False), (300, 384, 64, 200, True), (257, 2048, 320, 1000, False), (1023, 128, 128, 104, True)])
@pytest.mark.parametrize("bias, offset, norm_dtype", [(False, False, torch.bfloat16), (True, True, torch.float32)])
def test_folded_into_the_products_around_it(M, N, K, N2, gated, bias, offset, norm_dtype):
    """The sum is rounded where a delta of its own is (bfloat16, half a step of 2^-8 of it; a sum near the middle may fall the other way). Weighted rows and
    results are rounded to bfloat16 once each, 2^-9 of the result's size and of the terms that make it up, root mean square."""
    ops, norm, t, stream_of = make(M, N, K, N2, gated, bias, offset, norm_dtype)
    stream = stream_of(t["resid"])
    out = run(ops, norm, t, stream, gated, N2)
    delta = t["a"].double() @ t["w1"].double().T + (t["b1"].double() if bias else 0)
    x = t["resid"].double() + delta
    assert bool(((stream.resid.double() - x).abs() <= 2.0 ** -8 * delta.abs() + 1e-5).all())
    x = stream.resid.double()
    w = norm.weight.double() + (1 if offset else 0)
    z = (x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w) @ t["w2"].double().T + (t["b2"].double() if bias else 0)
    want = torch.nn.functional.silu(z[:, :N2]) * z[:, N2:] if gated else z
    assert float((out.double() - want).norm() / want.norm()) <= 2.0 ** -7.5
    rows = norm.fold(stream_of(t["resid"]), None, (t["w2"].shape[0], N, gated))
    weighted = ops.gemm(t["a"], t["w1"], torch.empty(M, N, dtype=torch.bfloat16, device=DEV), t["b1"], fold=rows)
    h = weighted.materialize().double()                       # for whoever wants the rows themselves
    normed = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * w
    assert float((h - normed).norm() / normed.norm()) <= 2.0 ** -8


@pytest.mark.parametrize("M, padded, N, K, N2, gated", [(130, 144, 1024, 2048, 4096, False), (208, 224, 1024, 512, 592, False), (481, 512, 1024, 3072, 3072, True),
                                                        (560, 576, 1024, 2048, 3104, False), (961, 1024, 1024, 3072, 3072, True)])
def test_a_steps_rows_have_the_bits_of_its_class(M, padded, N, K, N2, gated):
    """A recorded step is padded to its class: other tiles, the same bits."""
    ops, norm, t, stream_of = make(padded, N, K, N2, gated, True, False, torch.bfloat16)
    few, all_rows = stream_of(t["resid"][:M]), stream_of(t["resid"])
    a, b = run(ops, norm, t, few, gated, N2), run(ops, norm, t, all_rows, gated, N2)
    assert torch.equal(a, b[:M]) and torch.equal(few.resid, all_rows.resid[:M])
