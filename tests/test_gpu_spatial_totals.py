"""Selections of large populations that keep less than front 0 holds: from the third call of a shape on the dominators are
counted in spatial order, without a matrix.  Against the same selection with the matrix: objectives on either side of the
tile sizes, populations on either side of the rule, equal rows, equal keys, values on a grid, all rows alike, a NaN, and a
population whose front 0 falls short after others whose did not."""

import pytest
import torch

from evox_amd import runtime
from evox_amd.operators.selection import nd_environmental_selection

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _population(kind, n, m, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    d = torch.randn(n, m, generator=g).abs()
    if kind == "shell":  # most rows on the first front, the others behind it
        f = d / d.norm(dim=1, keepdim=True) * (1.0 - 0.05 * torch.log1p(-torch.rand(n, 1, generator=g)))
    elif kind == "grid":  # a plane of integers: equal rows and many equal values, and rows one step behind
        f = torch.randint(0, 60, (n, m), generator=g).float()
        f[:, -1] = 60.0 * m - f[:, :-1].sum(dim=1)
        f[::5] += 1.0
        f[1] = f[0]
    elif kind == "alike":
        f = torch.full((n, m), 0.5)
        f[7] = 0.75
    else:  # "uniform": front 0 holds a small part
        f = torch.rand(n, m, generator=g)
    return f.to(DEV)


def _same(a, b):
    return torch.equal(torch.nan_to_num(a.float(), nan=-7.0), torch.nan_to_num(b.float(), nan=-7.0))


@pytest.mark.parametrize("n,m", [(57343, 5), (57344, 5), (90113, 3), (90200, 4), (60001, 8), (58000, 9), (60000, 10), (57345, 15), (57344, 16)])
def test_totals_in_spatial_order(n, m):
    runtime.release_workspaces()
    x = torch.arange(n, dtype=torch.int32, device=DEV)[:, None]
    k = n // 4
    kinds = ["shell", "shell", "shell", "grid", "grid", "grid", "alike", "uniform", "shell", "shell", "shell", "nan"]
    for call, kind in enumerate(kinds):
        f = _population("shell" if kind == "nan" else kind, n, m, 10 * n + m + call)
        if kind == "nan":
            f[5, 1] = float("nan")
        got = nd_environmental_selection(x, f, k)
        assert runtime.last_status()["error"] == 0
        with runtime.options(prefix_count_first=0):
            want = nd_environmental_selection(x, f, k)
        assert all(_same(a, b) for a, b in zip(got, want)), (call, kind)
    runtime.release_workspaces()
