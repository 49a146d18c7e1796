"""Populations of up to 1024 rows and three to eight objectives: one launch up to 256 rows (``few_whole_kernel``), the matrix by
the whole device and the rest by one workgroup above (``few_dominance_kernel``, ``few_finish_kernel``), against the CPU
restatement.  Reference: src/evox/operators/selection/non_dominate.py:172-254."""

import numpy as np
import pytest
import torch

from evox_amd import runtime
from evox_amd.operators.selection import nd_environmental_selection, nd_environmental_selection_two_part, non_dominate_rank, non_dominate_rank_until
from oracle import eager_restatement as er
from tests.cases import as_np

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


def _population(kind, n, m, seed):
    g = torch.Generator("cpu").manual_seed(seed)
    f = torch.rand(n, m, generator=g)
    if kind == "plane":  # one front
        f = f / f.sum(dim=1, keepdim=True)
    elif kind == "grid":  # ties, copies
        f = (f * 4).floor() / 4
    elif kind == "decades":
        f = torch.pow(10.0, 60.0 * f - 30.0)
    elif kind == "special":  # NaN, infinities, signed zeros, in rows and in copies of rows
        f = (f * 5).floor() / 5
        for i, v in enumerate((float("nan"), float("inf"), -float("inf"), -0.0, 0.0)):
            f[i:: 11, i % m] = v
    elif kind == "chain":
        f = torch.randperm(n, generator=g).float()[:, None].repeat(1, m)
    return f, torch.arange(n, dtype=torch.float32)[:, None].repeat(1, 3)


def _same(got, want, what):
    assert torch.equal(got[0].cpu(), want[0]), what
    assert np.array_equal(as_np(got[1]), as_np(want[1]), equal_nan=True), what
    assert torch.equal(got[2].cpu(), want[2]), what
    g, w = as_np(got[3]), as_np(want[3])
    fin = np.isfinite(w)
    assert np.array_equal(np.isfinite(g), fin) and np.array_equal(g[~fin], w[~fin], equal_nan=True), what
    # (a sum of m quotients in another order: m units in the last place of float32, with room)
    np.testing.assert_allclose(g[fin], w[fin], rtol=1e-5, err_msg=str(what))


@pytest.mark.parametrize("kind", ["uniform", "plane", "grid", "decades", "special", "chain"])
@pytest.mark.parametrize("n,m", [(1, 3), (64, 5), (65, 3), (200, 8), (256, 4), (257, 3), (385, 6), (1000, 7), (1023, 3), (1024, 8)])
def test_selections_and_ranks(kind, n, m):
    f, x = _population(kind, n, m, 13 * n + m)
    fd, xd = f.to(DEV), x.to(DEV)
    ranks = er.ranks_by_peeling(f)
    assert np.array_equal(as_np(non_dominate_rank(fd)), as_np(ranks))
    for topk in sorted({1, max(1, n // 2), n}):
        _same(nd_environmental_selection(xd, fd, topk), er.environmental_selection(x, f, topk), (kind, n, m, topk))
    cut = max(1, n // 2)
    until = as_np(non_dominate_rank_until(fd, cut))
    worst = int(torch.sort(ranks).values[cut - 1])
    kept = as_np(ranks) <= worst
    assert np.array_equal(until[kept], as_np(ranks)[kept]) and (until[~kept] > worst).all()


@pytest.mark.parametrize("n_a,n_b,m", [(100, 100, 3), (1, 255, 5), (300, 211, 3), (512, 512, 4), (0, 700, 3)])
def test_two_parts_and_strides(n_a, n_b, m):
    n = n_a + n_b
    f, x = _population("uniform", n, m, n + m)
    want = er.environmental_selection(x, f, max(1, n // 2))
    fd, xd = f.to(DEV), x.to(DEV)
    _same(nd_environmental_selection_two_part(xd[:n_a].clone(), fd[:n_a].clone(), xd[n_a:].clone(), fd[n_a:].clone(), max(1, n // 2)), want, "clones")
    padded = torch.zeros(n, m + 3, device=DEV)
    padded[:, 1:m + 1] = fd
    columns = fd.t().contiguous().t()  # column-major
    _same(nd_environmental_selection(xd, padded[:, 1:m + 1], max(1, n // 2)), want, "padded")
    _same(nd_environmental_selection(xd, columns, max(1, n // 2)), want, "columns")
    if n_a:
        # parts of different strides
        _same(nd_environmental_selection_two_part(xd[:n_a], columns[:n_a], xd[n_a:].clone(), padded[n_a:, 1:m + 1], max(1, n // 2)), want, "strides differ")


@pytest.mark.parametrize("b,n,m", [(2, 200, 3), (5, 600, 3), (33, 520, 5), (3, 1024, 4)])
def test_several_populations(b, n, m):
    fs, xs = zip(*(_population("uniform" if i % 2 else "plane", n, m, 100 * i + n) for i in range(b)))
    got = nd_environmental_selection(torch.stack(xs).to(DEV), torch.stack(fs).to(DEV), n // 2)
    for i in range(b):
        _same([t[i] for t in got], er.environmental_selection(xs[i], fs[i], n // 2), (b, i))
    assert runtime.last_status()["error"] == 0


@pytest.mark.parametrize("m", [3, 8])
@pytest.mark.parametrize("n", [65, 200, 256, 257, 512, 700, 1000, 1024])
@pytest.mark.parametrize("levels", [1, 2, 4, 16, 30])
def test_last_fronts_of_few_levels(n, m, levels):
    """Candidates that crowd a bucket of the placement: of one value, of several (levels, with copies at both ends and between)."""
    g = torch.Generator("cpu").manual_seed(n + m + levels)
    f = torch.randint(0, levels, (n, m), generator=g).float()
    f[:, 0] = torch.where(torch.rand(n, generator=g) < 0.1, f[:, 0] * 1e-12 * torch.rand(n, generator=g), f[:, 0])  # (close ones beside)
    x = torch.arange(n * 2.0).reshape(n, 2)
    for data in (f, -f, torch.cat([f[: n // 2] * 1e30, f[n // 2:] * 1e-30])):
        for k in (1, n // 2, n):
            _same(nd_environmental_selection(x.to(DEV), data.to(DEV), k), er.environmental_selection(x, data, k), (levels, n, m, k))
            batch = nd_environmental_selection(x.expand(32, n, 2).to(DEV), data.expand(32, n, m).to(DEV), k)  # (without pairs above 256 rows)
            _same([t[7] for t in batch], er.environmental_selection(x, data, k), (levels, n, m, k, "batch"))


def test_host_threads_on_one_stream():
    """Threads whose calls take several launches each on the workspace of the default stream: every result is its own population's."""
    import threading

    populations = [_population("uniform", n, m, n)[0] for n, m in ((300, 3), (700, 5), (1000, 3), (2500, 3))]
    want = [as_np(er.ranks_by_peeling(f)) for f in populations]
    on_device = [f.to(DEV) for f in populations]
    results, errors = [], []

    def work(first):
        try:
            mine = []
            for rep in range(100):
                i = (first + rep) % len(on_device)
                mine.append((i, non_dominate_rank(on_device[i])))
            results.append(mine)
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(first,)) for first in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for mine in results:
        for i, rank in mine:
            assert np.array_equal(as_np(rank), want[i]), i


@pytest.mark.parametrize("n,m", [(300, 3), (1000, 8), (2500, 3)])
def test_a_captured_call_keeps_its_workspace(n, m):
    """Captured on a stream whose buffer a larger call then replaces: replays neither read nor write what the allocator has
    given away since."""
    f = torch.rand(n, m, generator=torch.Generator("cpu").manual_seed(n))
    static = f.to(DEV)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        non_dominate_rank(static)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = non_dominate_rank(static)
    with torch.cuda.stream(side):
        non_dominate_rank(torch.rand(9000, m, device=DEV))
        taken = [torch.full((1 << shift,), 7, dtype=torch.uint8, device=DEV) for shift in range(9, 25) for _ in range(3)]
    torch.cuda.synchronize()
    for seed in range(4):
        f = torch.rand(n, m, generator=torch.Generator("cpu").manual_seed(seed))
        static.copy_(f)
        graph.replay()
        eager = non_dominate_rank(f.to(DEV))
        torch.cuda.synchronize()
        assert torch.equal(out, eager) and np.array_equal(as_np(eager), as_np(er.ranks_by_peeling(f))), seed
    assert all(bool((t == 7).all()) for t in taken)
    del graph
    runtime.release_workspaces()
