"""The router whose waves take a row each (up to 64 experts) against the one that goes through LDS, which the same rows reach
behind enough experts that nothing can choose: scores of minus infinity and zero weight."""
import pytest
import torch

from test_gpu_kernels import ops_for

pytestmark = pytest.mark.gpu
INF = float("inf")


def route(z, correction, groups, keep, top, **options):
    ops = ops_for(torch.float32)
    n, E = z.shape
    dense = torch.full((n, E), 7.0, device="cuda")
    ids, weights = torch.full((n, top), -7, dtype=torch.int32, device="cuda"), torch.full((n, top), 7.0, device="cuda")
    ops.moe_route(z.cuda(), None if correction is None else correction.cuda(), groups, keep, top, 1e-20, dense, ids, weights, **options)
    return dense.cpu(), ids.cpu(), weights.cpu()


# one expert, one group, groups of one, of two and of half the experts; rows that end with a workgroup's four and that don't
@pytest.mark.parametrize("E, groups, keep, top, n", [(1, 1, 1, 1, 5), (2, 2, 1, 1, 4), (8, 8, 3, 2, 7), (16, 8, 3, 6, 64), (32, 4, 2, 4, 129),
                                                     (33, 1, 1, 5, 6), (60, 3, 3, 8, 9), (64, 2, 1, 32, 3), (64, 1, 1, 64, 2), (64, 64, 64, 64, 1)])
@pytest.mark.parametrize("scoring, worth, normalize", [("softmax", "max", True), ("sigmoid", "top2", True), ("sigmoid", "max", False)])
@pytest.mark.parametrize("ties", [False, True])
def test_against_the_kernel_for_more_experts(E, groups, keep, top, n, scoring, worth, normalize, ties):
    """The same choices in the same order and the same bits of the weights; with ``ties`` the logits are one of three values
    (two of them zero with either sign), so that nearly every choice is one among equals, and half of the corrections say that
    an expert is not to be chosen, so that some rows have too few."""
    g = torch.Generator().manual_seed(E * top + groups)
    z = torch.randint(0, 3, (n, E), generator=g).float() - 1 if ties else 2 * torch.randn(n, E, generator=g)
    correction = None
    if ties:
        z[z == 0] = -0.0
        z[:, ::3][z[:, ::3] == 0] = 0.0
        correction = torch.where(torch.rand(E, generator=g) < 0.5, -INF, 0.0)
    options = dict(scoring=scoring, group_worth=worth, normalize=normalize)
    dense, ids, weights = route(z, correction, groups, keep, top, **options)
    per = E // groups
    more = max(1, -(-(65 - E) // per))
    wide = torch.cat([z, torch.full((n, more * per), -INF)], 1)
    wide_correction = torch.cat([torch.zeros(E) if correction is None else correction, torch.full((more * per,), -INF)])
    if keep == groups:                                      # all groups stay, also those behind
        want = route(wide, wide_correction, groups + more, groups + more, top, **options)
    else:
        want = route(wide, wide_correction, groups + more, keep, top, **options)
    assert torch.equal(ids, want[1]) and torch.equal(weights, want[2]) and torch.equal(dense, want[0][:, :E])
    chosen = ids >= 0
    assert bool((weights[~chosen] == 0).all()) and bool((want[0][:, E:] == 0).all())


@pytest.mark.parametrize("value", [float("nan"), -float("nan")])
@pytest.mark.parametrize("where", ["logits", "correction"])
def test_a_score_that_is_no_number_is_not_lost(value, where):
    """It comes first, as in a sort, and the row's weights say so; every other row keeps its choice."""
    g = torch.Generator().manual_seed(1)
    z, correction = torch.randn(6, 32, generator=g), torch.zeros(32)
    plain = route(z, correction, 1, 1, 4, scoring="sigmoid")
    z2, c2 = z.clone(), correction.clone()
    if where == "logits":
        z2[2, 17] = value
    else:
        c2[17] = value
    dense, ids, weights = route(z2, c2, 1, 1, 4, scoring="sigmoid")
    rows = [2] if where == "logits" else range(6)
    for r in range(6):
        if r in rows:
            assert ids[r, 0] == 17
            others = [e for e in plain[1][r].tolist() if e != 17]
            assert ids[r, 1:].tolist() == others[:3]
            assert where == "correction" or bool(torch.isnan(weights[r]).all())
        else:
            assert torch.equal(ids[r], plain[1][r]) and torch.equal(weights[r], plain[2][r])
    # all of a row: every choice is still an expert, each once
    z2[3] = value
    ids = route(z2, correction, 1, 1, 4, scoring="softmax")[1]
    assert len(set(ids[3].tolist())) == 4 and bool(((ids >= 0) & (ids < 32)).all())
