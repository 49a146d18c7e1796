"""Populations from the size on at which their matrix comes from the orders of the objectives, and those orders from shares placed in
LDS (``objective_shares_kernel``, ``objective_order_stream_kernel``), against the pairwise matrix.  Reference:
src/evox/operators/selection/non_dominate.py:6-26, :172-254."""

import pytest
import torch

from evox_amd import runtime
from evox_amd.operators.selection import nd_environmental_selection, non_dominate_rank_until

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _population(kind, n, m):
    g = torch.Generator("cpu").manual_seed(n + m)
    f = torch.rand(n, m, generator=g)
    if kind == "levels":  # every share of an order holds one value or two, values reach over many shares
        f = (f * 3).floor() / 3
    elif kind == "plane":
        f = f / f.sum(dim=1, keepdim=True)
    elif kind == "decades":  # values over many binades, of both signs, and both zeros
        f = torch.pow(10.0, 70.0 * f - 38.0) * torch.where(torch.rand(n, m, generator=g) < 0.5, -1.0, 1.0)
        f[::97] *= 0.0
    return f


@pytest.mark.parametrize("kind", ["uniform", "levels", "plane", "decades"])
@pytest.mark.parametrize("n,m", [(40960, 3), (32769, 4), (33333, 5), (32769, 7), (70001, 8), (33000, 16)])
def test_selection_equals_that_from_the_pairwise_matrix(kind, n, m):
    f = _population(kind, n, m).to(DEV)
    x = torch.arange(n, dtype=torch.int32, device=DEV)[:, None]
    topk = n // 3
    got = nd_environmental_selection(x, f, topk)
    ranks = non_dominate_rank_until(f, topk)
    assert runtime.last_status()["error"] == 0
    with runtime.options(prefix_min_rows=0):
        want = nd_environmental_selection(x, f, topk)
        want_ranks = non_dominate_rank_until(f, topk)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    # (the same quotients, added in another order: m units in the last place of float32, with room)
    torch.testing.assert_close(got[3], want[3], rtol=1e-5, atol=0.0, equal_nan=True)
    kept = torch.sort(want_ranks).values[topk - 1]
    assert torch.equal(ranks[want_ranks <= kept], want_ranks[want_ranks <= kept]) and bool((ranks[want_ranks > kept] > kept).all())
    runtime.release_workspaces()


@pytest.mark.parametrize("n,m,levels,share", [(60000, 4, 4, 1.0), (60000, 4, 16, 1.0), (40961, 3, 60, 1.0), (33001, 5, 5, 0.5), (33001, 7, 1, 0.3)])
def test_samples_of_few_levels(n, m, levels, share):
    # (levels in the middle of the sample, alone or among rows of other values; sixty do not crowd; a level within the span of the others' bucket)
    g = torch.Generator("cpu").manual_seed(n + levels)
    f = torch.rand(n, m, generator=g)
    steps = ((f * levels).floor() + 0.5) / levels
    f = torch.where(torch.rand(n, m, generator=g) < share, steps, f).to(DEV)
    x = torch.arange(n, dtype=torch.int32, device=DEV)[:, None]
    got = nd_environmental_selection(x, f, n // 2)
    assert runtime.last_status()["error"] == 0
    with runtime.options(prefix_min_rows=0):
        want = nd_environmental_selection(x, f, n // 2)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and torch.equal(got[2], want[2])
    # (the same quotients, added in another order: m units in the last place of float32, with room)
    torch.testing.assert_close(got[3], want[3], rtol=1e-5, atol=0.0, equal_nan=True)
    runtime.release_workspaces()
