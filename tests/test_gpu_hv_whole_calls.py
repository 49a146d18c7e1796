"""The hypervolume functions as whole calls in the library, at the edges of their kernels: steps of points, workgroups of 64
samples, shares and tiles of samples, objectives held in registers, the number of samples from which fewer waves share the
points, strided inputs, values that are not finite -- against the restatement on the CPU, which shares no kernel with them,
and against the same functions around the operators."""

import pytest
import torch

from evox_amd import hype, ops
from evox_amd.metrics import hv
from oracle import eager_restatement as er

pytestmark = pytest.mark.gpu
DEV = "cuda"

SIZES = [
    (1, 1, 1), (2, 3, 63), (7, 3, 64), (8, 2, 65), (9, 4, 127), (64, 5, 128), (65, 6, 129), (255, 7, 1000), (257, 8, 1025),
    (300, 9, 4097), (1000, 16, 2000), (2000, 3, 10000), (5003, 3, 20001), (130, 3, 65536), (1001, 3, 65537), (20000, 2, 300),
]


def _both(monkeypatch, call):
    out = []
    for whole in (True, False):
        with monkeypatch.context() as patch:
            if not whole:
                patch.setattr(ops, "hv_whole_call_fits", lambda *a: False)
            torch.manual_seed(5)
            with torch.device(DEV):
                out.append(call())
    return out


def _close(got, want, rtol):
    assert got.shape == want.shape and got.dtype == want.dtype and got.device == want.device
    assert torch.allclose(got, want, rtol=rtol, atol=0.0, equal_nan=True), (got, want)


def _against_the_restatement(objs, ref, n_sample, seed):
    u = torch.rand(n_sample, objs.size(1), generator=torch.Generator().manual_seed(seed))
    n, m = objs.shape
    pop = max(1, n // 2)
    assert ops.hv_whole_call_fits(objs.to(DEV), ref.to(DEV), n_sample)
    # the counts are equal; the quotient and the product of m sides are rounded m + 1 times on either side
    got = ops.hv_estimate(objs.to(DEV), ref.to(DEV), u.to(DEV)).cpu()
    _close(got, er.hv_estimate(objs, ref, u), rtol=2 * (m + 1) * 2.0**-24)
    # weights, none of them negative, are products of up to n rounded quotients, and n_sample of them are added up
    got = ops.hype_contributions(objs.to(DEV), ref.to(DEV), pop, u.to(DEV)).cpu()
    _close(got, er.hv_contributions(objs, ref, pop, u), rtol=(n_sample + 2 * n + 2 * m + 8) * 2.0**-24)


@pytest.mark.parametrize("n", [1, 7, 8, 9, 15, 16, 17, 31, 32, 33, 255, 257])
@pytest.mark.parametrize("m", range(1, 17))
def test_whole_calls_against_the_restatement(n, m):
    g = torch.Generator().manual_seed(100 * n + m)
    objs = torch.randn(n, m, generator=g).abs()
    objs = objs / objs.sum(dim=1, keepdim=True)
    _against_the_restatement(objs, objs.max(dim=0).values * 1.1 + 0.05, 641, n + m)


@pytest.mark.parametrize("m", [1, 3, 8, 9, 16])
@pytest.mark.parametrize("value", [float("inf"), -float("inf"), float("nan")])
def test_values_that_are_not_finite_against_the_restatement(m, value):
    """A point of infinite cost leaves everything else finite; the others make the box and with it every result infinite or NaN."""
    objs = torch.rand(300, m, generator=torch.Generator().manual_seed(m))
    objs[17, m // 2] = value
    objs[290, m - 1] = value
    _against_the_restatement(objs, torch.full((m,), 1.2), 1500, m)


@pytest.mark.parametrize("m", [1, 4, 8, 13, 17])
def test_samples_that_are_not_finite(m):
    """The operators, whose samples may be anything, against the tests written out: differences for the contributions, in
    which infinity minus itself is no cover, comparisons for the metric."""
    g = torch.Generator().manual_seed(m)
    fit, samples = torch.rand(400, m, generator=g), 0.4 + torch.rand(700, m, generator=g)
    for t in (fit, samples):
        t[::7, 0] = float("inf")
        t[3::11, m // 2] = -float("inf")
        t[5::13, m - 1] = float("nan")
    covers = torch.stack([(fit - s <= 0).all(dim=1) for s in samples])
    assert not torch.equal(covers, torch.stack([(fit <= s).all(dim=1) for s in samples]))
    alpha = torch.rand(400, generator=g)
    want = covers.double().t() @ alpha[(covers.sum(dim=1) - 1).clamp(min=0)].double()
    got = ops.hv_contributions(fit.to(DEV), samples.to(DEV), alpha.to(DEV), 1.0).cpu().double()
    assert torch.allclose(got, want, rtol=702 * 2.0**-24, atol=0.0)
    exceeded = torch.stack([(s < fit).all(dim=1).any() for s in samples]).sum()
    assert int(ops.hv_covered_count(fit.to(DEV), samples.to(DEV))) == int(exceeded)


@pytest.mark.parametrize("n, m, n_sample", SIZES)
def test_whole_calls_match_the_operators(monkeypatch, n, m, n_sample):
    g = torch.Generator().manual_seed(n + m)
    wide = torch.rand(n, 2 * m, generator=g).to(DEV)
    for objs in (wide[:, :m].contiguous(), wide[:, ::2], wide[:, :m].t().contiguous().t()):
        ref = (objs.max(dim=0).values * 1.1)
        assert ops.hv_whole_call_fits(objs, ref, n_sample)
        # the counts are equal; the quotient and the product of m sides are rounded m + 1 times on either side
        _close(*_both(monkeypatch, lambda: hv(objs, ref, n_sample)), rtol=2 * (m + 1) * 2.0**-24)
        # the sums have one order; a weight is a product of up to n rounded quotients on the operators' side
        _close(*_both(monkeypatch, lambda: hype.cal_hv(objs, ref, max(1, n // 2), n_sample)), rtol=(2 * n + 2 * m + 8) * 2.0**-24)


def test_values_that_are_not_finite(monkeypatch):
    base = torch.rand(200, 3, generator=torch.Generator().manual_seed(3)).to(DEV)
    ref = torch.full((3,), 1.2, device=DEV)
    for value in (float("nan"), float("inf"), -float("inf")):
        objs = base.clone()
        objs[17, 1] = value
        _close(*_both(monkeypatch, lambda: hv(objs, ref, 3000)), rtol=1e-6)
        _close(*_both(monkeypatch, lambda: hype.cal_hv(objs, ref, 100, 3000)), rtol=4e-5)


def test_calls_that_keep_to_the_operators():
    objs, ref = torch.rand(20, 3, device=DEV), torch.ones(3, device=DEV)
    assert ops.hv_whole_call_fits(objs, ref, 100)
    assert not ops.hv_whole_call_fits(objs.double(), ref, 100)
    assert not ops.hv_whole_call_fits(objs.clone().requires_grad_(), ref, 100)
    assert not ops.hv_whole_call_fits(objs, ref[:1], 100)
    assert not ops.hv_whole_call_fits(objs[:0], ref, 100)
    assert not ops.hv_whole_call_fits(torch.rand(20, 17, device=DEV), torch.ones(17, device=DEV), 100)
    seen = []
    torch.vmap(lambda f: seen.append(ops.hv_whole_call_fits(f, ref, 100)) or f)(objs.view(2, 10, 3))
    with torch.autograd.forward_ad.dual_level():
        seen.append(ops.hv_whole_call_fits(objs, ref, 100))
    assert seen == [False, False]
    # a gradient still reaches the points (through the volume of the box)
    leaf = objs.clone().requires_grad_()
    torch.manual_seed(2)
    with torch.device(DEV):
        hv(leaf, ref, 1000).backward()
    assert float(leaf.grad.abs().sum()) > 0.0


@pytest.mark.parametrize("n, m, n_sample", [(100003, 3, 64), (70000, 3, 1), (65537, 8, 130), (40001, 17, 65), (30011, 5, 1000),
                                            (300000, 1, 100), (20000, 16, 63), (20001, 8, 2000)])
def test_points_shared_by_several_workgroups(n, m, n_sample):
    """Few samples against many points, where several workgroups have the same samples, against counts made on the CPU.
    Some samples are covered by no point, some only by points of the last steps."""
    g = torch.Generator().manual_seed(n + m)
    fit = torch.randn(n, m, generator=g).abs()
    fit = fit / fit.norm(dim=1, keepdim=True) + 0.3
    fit[-5:] *= 0.9
    samples = 0.25 + 1.1 * torch.rand(n_sample, m, generator=g)
    samples[::3] = fit[torch.randint(n - 16, n, (len(samples[::3]),), generator=g)]
    covers = torch.stack([(fit <= s).all(dim=1) for s in samples])
    count = covers.sum(dim=1)
    alpha = torch.rand(n, generator=g)
    weight = alpha[(count - 1).clamp(min=0)].double()
    got = ops.hv_contributions(fit.to(DEV), samples.to(DEV), alpha.to(DEV), 1.0).cpu().double()
    want = covers.double().t() @ weight
    assert torch.allclose(got, want, rtol=(n_sample + 2) * 2.0**-24, atol=0.0)
    # the metric: points above the samples
    points, below = fit.to(DEV), samples.to(DEV)
    exceeded = torch.stack([(s < fit).all(dim=1).any() for s in samples]).sum()
    for _ in range(2):
        assert int(ops.hv_covered_count(points, below)) == int(exceeded)


@pytest.mark.parametrize("n, m, n_sample", [(500, 3, 5000), (30011, 3, 300), (20001, 8, 130)])
def test_hypervolume_in_a_graph(n, m, n_sample):
    """One capture, replayed on other points with eager calls in between; the counts of workgroups that share samples start
    from zero in every replay."""
    g = torch.Generator().manual_seed(n)

    def draw():
        return torch.rand(n, m, generator=g).to(DEV), torch.rand(n_sample, m, generator=g).to(DEV)

    objs, u = draw()
    ref, alpha = torch.full((m,), 1.2, device=DEV), torch.rand(n, generator=g).to(DEV)

    def calls(objs, u):
        return (ops.hv_estimate(objs, ref, u), ops.hype_contributions(objs, ref, n // 2, u), ops.hv_covered_count(objs, u),
                ops.hv_contributions(objs, u, alpha, 1.0))

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        calls(objs, u)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = calls(objs, u)
    for _ in range(4):
        new = draw()
        objs.copy_(new[0])
        u.copy_(new[1])
        graph.replay()
        eager = calls(*new)
        torch.cuda.synchronize()
        for got, want in zip(out, eager):
            assert torch.equal(got, want)
