"""Last fronts ordered by sorted runs of 512 keys: sizes around the ends of the runs and of the groups of runs that a lane
searches together, ties across runs, zeros of either sign, NaN; against the plain-C checker and the radix path.  A
selection of up to three objectives takes this path from the second call of a shape on, so every call is made three
times."""

import numpy as np
import pytest
import torch

from evox_amd import runtime
from evox_amd.operators.selection import crowding_distance, nd_environmental_selection, nd_environmental_selection_two_part
from oracle import c_oracle
from tests.cases import as_np

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _front(n, m, kind):
    """n rows, none of which dominates another: every row's objectives add up to the same integer."""
    g = torch.Generator("cpu").manual_seed(n * 31 + m)
    if m == 2:
        a = torch.randperm(4 * n, generator=g)[:n].float() if kind != "ties" else torch.randint(0, n // 3, (n,), generator=g).float()
        f = torch.stack([a - 7.0, 7.0 - a], dim=1)
    else:
        top = 300 if kind == "ties" else 100000
        f = torch.randint(0, top, (n, m), generator=g).float()
        f[:, -1] = top * m - f[:, :-1].sum(dim=1)
    if kind == "odd":
        f[:: n // 7, 0] = float("nan")  # (dominates nothing and is dominated by nothing)
        at = torch.arange(5) * (n // 5) + 1
        f[at + 1] = f[at]
        f[at, 0] = 0.0
        f[at + 1, 0] = -0.0
    return f


def _same(a, b):
    return torch.equal(torch.nan_to_num(a.float(), nan=-7.0), torch.nan_to_num(b.float(), nan=-7.0))


SIZES = [(1025, 6), (1536, 5), (1537, 9), (2049, 3), (4097, 2), (4608, 4), (6144, 3), (6145, 5), (8192, 3), (8193, 3), (20481, 3),
         (24577, 4), (32767, 2), (32768, 6)]


@pytest.mark.parametrize("kind", ["plain", "ties", "odd"])
@pytest.mark.parametrize("n,m", SIZES)
def test_front_of_one_selection(n, m, kind):
    f = _front(n, m, kind)
    x = torch.arange(n, dtype=torch.int32)[:, None]
    k = n // 2 + 1
    order, rank, dist, _ = c_oracle.select(as_np(f), k)
    xd, fd = x.to(DEV), f.to(DEV)
    h = n // 3
    with runtime.options(mid_argsort=0):
        old = nd_environmental_selection(xd, fd, k)
    for call in range(3):
        if call == 2:
            got = nd_environmental_selection_two_part(xd[:h], fd[:h], xd[h:], fd[h:], k)
        else:
            got = nd_environmental_selection(xd, fd, k)
        assert runtime.last_status()["error"] == 0
        assert np.array_equal(as_np(got[0])[:, 0].astype(np.int64), order), (n, m, kind, call)
        assert all(_same(a, b) for a, b in zip(got, old)), (n, m, kind, call)
        gd, wd = as_np(got[3]), dist[order]
        fin = np.isfinite(wd)
        assert np.array_equal(np.isnan(gd), np.isnan(wd)) and np.array_equal(np.isfinite(gd), fin)
        np.testing.assert_allclose(gd[fin], wd[fin], rtol=1e-5)
    runtime.release_workspaces()


@pytest.mark.parametrize("n,m,kept", [(1030, 5, 0), (1030, 5, 1), (5000, 3, 1537), (9000, 12, 9000), (32768, 2, 16385)])
def test_distances_of_a_mask(n, m, kept):
    g = torch.Generator("cpu").manual_seed(n)
    costs = torch.randint(-50, 50, (n, m), generator=g).float() * 0.5
    mask = torch.zeros(n, dtype=torch.bool)
    mask[torch.randperm(n, generator=g)[:kept]] = True
    want = c_oracle.crowding(as_np(costs), as_np(mask)) if kept else np.full(n, -np.inf, np.float32)
    got = as_np(crowding_distance(costs.to(DEV), mask.to(DEV)))
    assert np.array_equal(np.isinf(got), np.isinf(want)) and np.array_equal(np.isnan(got), np.isnan(want))
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-5)
    runtime.release_workspaces()


@pytest.mark.parametrize("b,n,m", [(20, 1500, 4), (3, 6145, 3), (40, 2100, 5)])
def test_fronts_of_many_populations(b, n, m):
    """Populations of one shape in the same launches: as each on its own."""
    f = torch.stack([_front(n, m, "ties" if i % 2 else "plain")[torch.randperm(n, generator=torch.Generator("cpu").manual_seed(i))] for i in range(b)]).to(DEV)
    x = torch.arange(n, dtype=torch.int32, device=DEV)[None, :, None].expand(b, n, 1).contiguous()
    for _ in range(2):
        got = nd_environmental_selection(x, f, n // 2)
    for i in range(0, b, 7):
        with runtime.options(mid_argsort=0):
            one = nd_environmental_selection(x[i], f[i], n // 2)
        assert all(_same(a[i], c) for a, c in zip(got, one)), i
    runtime.release_workspaces()
