"""The steps of the first-front mask (sampled champions, grid, pairs, leaves in spatial order) at the sizes where one takes
over from another, against the C checker: masks are whole numbers and must be equal."""

import numpy as np
import pytest
import torch

from oracle import c_oracle

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


def population(kind, n, m, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    f = torch.rand(n, m, generator=g)
    if kind == "uniform":
        return f
    d = torch.randn(n, m, generator=g).abs()
    if kind == "one front":
        return d / d.sum(dim=1, keepdim=True)
    f = d / d.norm(dim=1, keepdim=True) * (1.0 - 0.1 * torch.log1p(-torch.rand(n, 1, generator=g)))
    if kind == "ties":  # equal rows and equal values in every objective
        f = torch.round(f * 32) / 32
    if kind == "special":  # penalties, infinities, signed zeros, NaN
        f[: n // 3] = 1e9
        f[::101, 0] = -0.0
        f[1::103, m - 1] = 0.0
        f[2::107, 0] = INF
        f[3::109, m - 1] = -INF
        f[4::113, m // 2] = NAN
    return f


@pytest.mark.parametrize("kind", ["uniform", "shell", "one front", "ties", "special"])
@pytest.mark.parametrize("n,m", [(1, 3), (63, 2), (64, 1), (65, 16), (100, 3), (513, 9), (1025, 3), (1024, 16), (512, 16), (1536, 8),
                                 (1537, 8), (2457, 5), (2458, 5), (4096, 3), (4097, 3), (4097, 16), (16384, 3), (16385, 2), (16385, 3), (21000, 4), (65536, 3),
                                 (65537, 2), (65537, 3), (65537, 4), (70001, 7), (131072, 3), (131073, 3)])
def test_mask_at_the_edges_of_the_steps(n, m, kind):
    from evox_amd.operators.selection import non_dominated_mask

    f = population(kind, n, m, n + m)
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    assert np.array_equal(got, c_oracle.first_front(f.numpy()))


@pytest.mark.parametrize("finite", [True, False])
@pytest.mark.parametrize("n,m", [(65601, 5), (65601, 6), (65601, 9), (65700, 12), (65601, 16)])
def test_leaves_of_more_objectives(n, m, finite):
    """Rows on one front, more of them than are compared pair by pair."""
    from evox_amd.operators.selection import non_dominated_mask

    f = population("one front", n if finite else n + n // 4, m, n + m)
    if not finite:
        f[2::1007, 0] = INF
        f[4::1013, m // 2] = NAN
        f[3::40001, m - 1] = -INF
        f[7] = INF
    want = c_oracle.first_front(f.numpy())
    assert 65536 < want.sum()
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    assert np.array_equal(got, want)


@pytest.mark.parametrize("n,m", [(5, 3), (100, 2), (130, 9), (1024, 3), (4096, 2), (4100, 3)])
def test_masks_of_several_small_populations(n, m):
    from evox_amd.operators.selection import non_dominated_mask

    f = torch.stack([population(kind, n, m, n + b) for b, kind in enumerate(("uniform", "one front", "special", "ties"))])
    wide = torch.full((4, n, m + 2), -1.0)
    wide[:, :, 1 : m + 1] = f
    for view in (f.to("cuda"), wide.to("cuda")[:, :, 1 : m + 1], f.transpose(1, 2).contiguous().to("cuda").transpose(1, 2)):
        got = non_dominated_mask(view).cpu().numpy()
        for b in range(4):
            assert np.array_equal(got[b], c_oracle.first_front(f[b].numpy())), b


@pytest.mark.parametrize("n,m", [(4097, 3), (5000, 16), (20000, 7), (70001, 2), (66000, 8), (300001, 3)])
@pytest.mark.parametrize("good", [1, 17])
def test_few_rows_that_dominate_the_rest(n, m, good):
    """At places that no sample by position holds; among the others infinities and sums that overflow."""
    from evox_amd.operators.selection import non_dominated_mask

    g = torch.Generator("cpu").manual_seed(n + m)
    f = torch.rand(n, m, generator=g) + 1.0
    f[::1009, 0] = INF
    f[5::1013] = 3e38
    f[7::1019, m - 1] = -3e38
    at = torch.randint(n // 3, n, (good,), generator=g)
    f[at] = 0.9 * torch.rand(good, m, generator=g)
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    assert np.array_equal(got, c_oracle.first_front(f.numpy()))


def test_masks_of_several_large_populations():
    from evox_amd.operators.selection import non_dominated_mask

    f = torch.stack([population(kind, 66000, 3, 5) for kind in ("uniform", "one front", "special")])
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    for b in range(3):
        assert np.array_equal(got[b], c_oracle.first_front(f[b].numpy())), b


@pytest.mark.parametrize("n,m", [(120001, 2), (120001, 3), (90001, 4), (70003, 5)])
def test_rows_that_a_leaf_asks_one_by_one(n, m):
    """Three rows in four are slightly worse copies of a row of the front, by steps from below a leaf's extent to well above
    it: after a leaf's nearest neighbours a few of its rows are open, some of which only a distant row dominates."""
    from evox_amd.operators.selection import non_dominated_mask

    g = torch.Generator("cpu").manual_seed(n + m)
    f = population("one front", n, m, n - m)
    copies = n * 3 // 4
    step = 10.0 ** (-5.5 + 4.0 * torch.rand(copies, 1, generator=g))
    f[:copies] = f[torch.randint(copies, n, (copies,), generator=g)] + step * torch.rand(copies, m, generator=g)
    f = f[torch.randperm(n, generator=g)]
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    assert np.array_equal(got, c_oracle.first_front(f.numpy()))


@pytest.mark.parametrize("n,m", [(1000, 3), (3000, 5), (20000, 3), (66000, 8), (70001, 2), (70001, 3)])
def test_masks_in_a_graph(n, m):
    """One capture, replayed on other populations with eager calls in between: nothing is left over from a replay."""
    from evox_amd import runtime
    from evox_amd.operators.selection import non_dominated_mask

    static = population("shell", n, m, n).to("cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        non_dominated_mask(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = non_dominated_mask(static)
    for seed, kind in enumerate(("shell", "one front", "uniform", "special", "one front")):
        f = population(kind, n, m, n + seed).to("cuda")
        static.copy_(f)
        graph.replay()
        eager = non_dominated_mask(f)
        torch.cuda.synchronize()
        assert torch.equal(out, eager), kind
    del graph
    runtime.release_workspaces()  # (those of the capture's stream among them)
