"""The gated pair of a prompt's rows: every shape of tile and its edges, against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def pair(x, w, bias, limit, slope):
    p = x.double() @ w.double().T + (0 if bias is None else bias.double())
    g, u = p[:, :p.shape[1] // 2], p[:, p.shape[1] // 2:]
    if limit > 0:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
        return g * torch.sigmoid(slope * g) * (u + 1)
    return g * torch.sigmoid(slope * g) * u


@pytest.mark.parametrize("bm", [64, 128, 192, 256])
@pytest.mark.parametrize("bn", [64, 128, 192])
@pytest.mark.parametrize("M, I, K, bias, limit", [(1, 8, 64, False, 0.0), (255, 100, 128, True, 0.0), (257, 97, 192, True, 1.5), (300, 192, 640, False, 0.0),
                                                  (577, 333, 320, True, 1.5)])
def test_tiles(bm, bn, M, I, K, bias, limit):
    """Rows, columns and chunks of K that end inside, at and behind a tile and the ring's stages; columns at odd places, pitches of the
    rows. Sums are float: what remains is the rounding of the result to bfloat16, 2^-9 of it (2^-8 with the sums' own error where
    gate and up nearly cancel)."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(M + I)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x = rand(M, K + 8).bfloat16()[:, :K]
    w = (rand(2 * I, K) / K ** 0.5 * 2).bfloat16()
    b = rand(2 * I).bfloat16() if bias else None
    out = torch.full((M + 1, I + 3), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.lib.call("mv_gemm_pair", x.data_ptr(), x.stride(0), w.data_ptr(), 0 if b is None else b.data_ptr(), out.data_ptr(), out.stride(0), M, 2 * I, K,
                 limit, 1.702 if limit else 1.0, bm << 16 | bn, torch.cuda.current_stream().cuda_stream)
    want = pair(x, w, b, limit, 1.702 if limit else 1.0)
    error = (out[:M, :I].double() - want).abs()
    assert bool((error <= 2.0 ** -8 * want.abs() + 1e-4).all())
    assert bool((out[M] == 7.0).all()) and bool((out[:, I:] == 7.0).all())


@pytest.mark.parametrize("M, I, K", [(129, 3072, 1024), (512, 3072, 1024), (2048, 768, 512)])
def test_prompts_take_it(M, I, K):
    """Through the engine's entry point, which leaves these sizes to it, with and without the pitch that stores of four need."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(2 * I, K, device=DEV) / K ** 0.5).bfloat16()
    for pitch in (I, I + 1):
        out = torch.zeros(M, pitch, dtype=torch.bfloat16, device=DEV)[:, :I]
        ops.ledger = []
        assert ops.gemm_swiglu(x, w, out)
        ran, ops.ledger = [e[0] for e in ops.ledger], None
        assert ran == ["mv_gemm_tile" if M <= 1536 else "mv_gemm_pair"]      # (the same kernel inside the tiled product's entry point)
        want = pair(x, w, None, 0.0, 1.0)
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.parametrize("bm", [64, 128, 192, 256])
@pytest.mark.parametrize("bn", [64, 96, 128, 192])
@pytest.mark.parametrize("M, N, K, bias", [(1, 8, 64, False), (255, 101, 128, True), (257, 193, 192, True), (300, 384, 640, False), (577, 333, 320, True)])
def test_plain_tiles(bm, bn, M, N, K, bias):
    """As above without the activation: the result is rounded by half a step of its eight bits, 2^-8 of it at most; sums of up to 640
    terms of a tenth in float32 are off by 1e-5 at most."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(M + N)
    rand = lambda *s: torch.randn(*s, generator=g, device=DEV)
    x, w = rand(M, K + 8).bfloat16()[:, :K], (rand(N, K) / K ** 0.5).bfloat16()
    b = rand(N).bfloat16() if bias else None
    out = torch.full((M + 1, N + 3), 7.0, dtype=torch.bfloat16, device=DEV)
    ops.lib.call("mv_gemm_round", x.data_ptr(), x.stride(0), w.data_ptr(), 0 if b is None else b.data_ptr(), out.data_ptr(), out.stride(0), M, N, K,
                 bm << 16 | bn, torch.cuda.current_stream().cuda_stream)
    want = x.double() @ w.double().T + (0 if b is None else b.double())
    assert bool(((out[:M, :N].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-5).all())
    assert bool((out[M] == 7.0).all()) and bool((out[:, N:] == 7.0).all())


@pytest.mark.parametrize("M, N, K", [(600, 5184, 1024), (1000, 592, 1024), (2048, 3104, 1024), (700, 1024, 1024)])
def test_plain_products_of_prompts_take_it(M, N, K):
    """Through the engine's entry point, rows with and without a pitch that loads of eight need."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    w, b = (torch.randn(N, K, device=DEV) / K ** 0.5).bfloat16(), torch.randn(N, device=DEV).bfloat16()
    for pitch in (K, K + 8, K + 4):
        x = torch.randn(M, pitch, device=DEV).bfloat16()[:, :K]
        out = torch.zeros(M, N, dtype=torch.bfloat16, device=DEV)
        ops.ledger = []
        ops.gemm(x, w, out, bias=b)
        ran, ops.ledger = [e[0] for e in ops.ledger], None
        assert (ran == ["mv_gemm_round"]) == (pitch % 8 == 0)
        want = x.double() @ w.double().T + b.double()
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4).all())


@pytest.mark.parametrize("M", [129, 150, 160, 256])
def test_short_prompts_stay_with_the_deep_product(M):
    """Pairs of few weight rows that both kernels serve: the bits of the one that the tiled product had them in."""
    from minivllm_amd.kernels.ops import get_ops
    ops, N, K = get_ops(torch.bfloat16), 2048, 1024
    assert ops.lib.dll.mv_gemm_deep_shape(M, N, K, 1) and ops.lib.dll.mv_gemm_pair_shape(M, N, K, 256) and ops.wants_tile(M, N, K, gated=True)
    x, w = torch.randn(M, K, device=DEV).bfloat16(), (torch.randn(N, K, device=DEV) / K ** 0.5).bfloat16()
    got, deep = (torch.zeros(M, N // 2, dtype=torch.bfloat16, device=DEV) for _ in range(2))
    assert ops.gemm_swiglu(x, w, got)
    ops.lib.call("mv_gemm_deep", x.data_ptr(), K, w.data_ptr(), 0, deep.data_ptr(), N // 2, 1, M, N, K, 1, 0, 0, 0.0, 0.0, 1.0, 0, 0,
                 torch.cuda.current_stream().cuda_stream)
    assert torch.equal(got, deep)


@pytest.mark.parametrize("lo, hi, limit", [(-60, -40, 0.0), (-40, -8, 0.0), (-8, 8, 0.0), (-8, 8, 7.0)])
def test_the_activation_is_float32_up_to_the_rounding(lo, hi, limit):
    """Gates and ups that are exact: what the activation is off shows where a result is not the 16-bit number nearest to the exact one.
    At 2^-24 x 5 off (a limit's slope * g is rounded in front of the exponential, 2^-24 x 12) 1.5e-4 (3.7e-4) of the results lie
    close enough to the middle of two, which are at least 2^-8 apart, if all are off that far the wrong way."""
    from minivllm_amd.kernels.ops import get_ops
    ops = get_ops(torch.bfloat16)
    gen, M, I, K = torch.Generator(device=DEV).manual_seed(7), 512, 2048, 64
    rand = lambda n, a, b: (torch.rand(n, generator=gen, device=DEV) * (b - a) + a).bfloat16()
    x, w = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV), torch.zeros(2 * I, K, dtype=torch.bfloat16, device=DEV)
    x[:, 0], x[:, 1], w[:I, 0], w[I:, 1] = rand(M, 0.95, 1.0), rand(M, 1.0, 2.0), rand(I, lo, hi), rand(I, 0.5, 3.0)
    out = torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
    ops.lib.call("mv_gemm_pair", x.data_ptr(), K, w.data_ptr(), 0, out.data_ptr(), I, M, 2 * I, K, limit, 1.702 if limit else 1.0, 128 << 16 | 128,
                 torch.cuda.current_stream().cuda_stream)
    want = pair(x, w, None, limit, 1.702 if limit else 1.0)
    assert float((out != want.float().bfloat16()).double().mean()) <= (3.7e-4 if limit else 1.5e-4)
