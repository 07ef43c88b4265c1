"""Products of a little more rows than fill the compute units a whole number of times go to the library in two calls:
the rows on both sides of the seam, against 64 bits."""
import pytest
import torch

from test_gpu_kernels import OP_TOL, dev, ops_for, rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("front, behind, N, calls", [(4096, 0, 4096, 1), (4096, 1, 4096, 2), (4096, 1024, 4096, 2), (4096, 1025, 4096, 1),
                                                    (2048, 7, 8192, 2), (4096, 9, 6144, 1), (8192, 300, 4096, 2)])
@pytest.mark.parametrize("form", ["plain", "bias", "rows apart", "float32"])
def test_rows_behind_whole_rounds(front, behind, N, calls, form):
    ops, dtype, M, K = ops_for(torch.bfloat16), torch.bfloat16, front + behind, 256
    if ops.compute_units != 256:
        pytest.skip("the sizes are those of 256 compute units")
    g = torch.Generator().manual_seed(M + N)
    a, w = torch.randn(M, K, generator=g).to(dtype), (torch.randn(N, K, generator=g) / 16).to(dtype)
    bias = torch.randn(N, generator=g).to(dtype) if form == "bias" else None
    wide = torch.full((M, N + 64), float("nan"), dtype=torch.float32 if form == "float32" else dtype, device="cuda")
    out = wide[:, :N] if form == "rows apart" else torch.empty(M, N, dtype=wide.dtype, device="cuda")
    ledger, ops.ledger = ops.ledger, []
    try:
        ops.gemm(dev(a), dev(w), out, None if bias is None else dev(bias))
        seen = [line[0] for line in ops.ledger]
    finally:
        ops.ledger = ledger
    assert seen == ["mv_gemm_lt"] * calls, seen
    rows = sorted({0, 1, front - 1, min(front, M - 1), M - 1} | set(range(0, M, 97)))
    want = a[rows].double() @ w.double().T + (0.0 if bias is None else bias.double())
    assert rel_err(out[rows].float().cpu().numpy(), want.numpy()) <= (3e-6 if form == "float32" else OP_TOL[dtype])
    if form == "rows apart":
        assert bool(torch.isnan(wide[:, N:]).all())
