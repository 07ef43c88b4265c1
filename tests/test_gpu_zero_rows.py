"""The launch that clears the states of starting requests: exactly the named rows of every tensor."""
import pytest
import torch

pytestmark = pytest.mark.gpu

# rows below, at and above what a workgroup clears, of odd sizes, and sizes no 16-byte store fits
SHAPES = [((4096,), torch.float32), ((4100,), torch.float32), ((3,), torch.bfloat16), ((1,), torch.float32),
          ((16, 64, 65), torch.float32), ((8191,), torch.bfloat16), ((64,), torch.bfloat16)]


@pytest.mark.parametrize("rows", [[0], [4, 1], [2, 2], list(range(69, -1, -1)), []])
def test_only_the_named_rows_are_cleared(rows):
    from minivllm_amd.kernels.ops import Ops, StateRows
    ops = Ops(torch.bfloat16)
    count = 70
    tensors = [torch.randn((count,) + dims, device="cuda").to(dt) for dims, dt in SHAPES]
    tensors.insert(3, torch.empty((count, 0), device="cuda"))
    want = [t.clone() for t in tensors]
    for w in want:
        w[rows] = 0
    ops.zero_rows(StateRows(tensors), rows)
    for t, w in zip(tensors, want):
        assert torch.equal(t, w)


def test_rows_outside_and_tensors_that_do_not_fit_are_refused():
    from minivllm_amd.kernels.ops import KernelLibraryError, Ops, StateRows
    ops = Ops(torch.bfloat16)
    t = torch.randn(4, 32, device="cuda")
    for bad in ([4], [-1], [0, 7]):
        with pytest.raises(KernelLibraryError, match="zero_rows"):
            ops.zero_rows(StateRows([t]), bad)
    with pytest.raises(KernelLibraryError, match="zero_rows"):
        StateRows([t, torch.randn(5, 32, device="cuda")])
    with pytest.raises(KernelLibraryError, match="zero_rows"):
        StateRows([t[:, :16]])
    ops.zero_rows(StateRows([]), [])
