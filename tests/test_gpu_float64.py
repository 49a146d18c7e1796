"""float64 fitness with torch's default dtype set to float64 (the reference computes the crowding distance in the
default dtype, src/evox/operators/selection/non_dominate.py:224): crowding distances and the selection against the
CPU restatement run in float64 on the same inputs.  The distances come from the same IEEE operations on the same
operands (a difference, a quotient), so they are compared exactly per objective sum up to the order of the M terms
(rtol 1e-12); ranks, the selected order and the positions of the infinities and NaN exactly."""

import numpy as np
import pytest
import torch

from evox_amd.operators.selection import crowding_distance, nd_environmental_selection, non_dominate_rank
from oracle import eager_restatement as er
from tests.cases import as_np, edge_cases

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
EDGE = edge_cases()


@pytest.fixture
def float64_default():
    torch.set_default_dtype(torch.float64)
    yield
    torch.set_default_dtype(torch.float32)


def _close(got, want, what):
    got, want = as_np(got), as_np(want)
    assert got.dtype == np.float64 and got.shape == want.shape, what
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    inf = np.isinf(want)
    assert np.array_equal(np.isinf(got), inf) and np.array_equal(got[inf], want[inf]), what
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-12, atol=0, err_msg=what)


def _populations():
    g = torch.Generator("cpu").manual_seed(64)
    out = [(name, f.double(), ks) for name, f, ks in EDGE]
    # values that differ only below float32's resolution, with ties, duplicates, a NaN and signed zeros
    fine = 1.0 + torch.randint(0, 400, (3000, 3), generator=g).double() * 1e-13
    fine[17, 1] = float("nan")
    fine[30] = fine[31]
    fine[40, 0], fine[41, 0] = 0.0, -0.0
    out.append(("below_float32_resolution", fine, [1, 700, 1500, 3000]))
    out.append(("uniform_5000x4", torch.rand(5000, 4, generator=g, dtype=torch.float64), [2500]))
    out.append(("uniform_9000x2", torch.rand(9000, 2, generator=g, dtype=torch.float64), [4500]))
    return out


POPS = _populations()


@pytest.mark.parametrize("name,f,ks", POPS, ids=[p[0] for p in POPS])
def test_float64_crowding_and_selection(float64_default, name, f, ks):
    fd = f.to(DEV)
    n = f.size(0)
    rank = er.ranks_by_peeling(f)
    assert np.array_equal(as_np(non_dominate_rank(fd)), as_np(rank))
    _close(crowding_distance(fd, None), er.crowding(f, None), (name, "no mask"))
    for r in sorted(set(as_np(rank).tolist()))[:3]:
        mask = rank == r
        _close(crowding_distance(fd, mask.to(DEV)), er.crowding(f, mask), (name, "front", r))
    x = torch.arange(n, dtype=torch.int64)[:, None]
    for k in ks:
        want = er.environmental_selection(x, f, k)
        got = nd_environmental_selection(x.to(DEV), fd, k)
        assert got[1].dtype == torch.float64 and got[2].dtype == torch.int32 and got[3].dtype == torch.float64
        assert torch.equal(got[0].cpu(), want[0]), (name, k)
        assert np.array_equal(as_np(got[1]), as_np(want[1]), equal_nan=True)
        assert torch.equal(got[2].cpu(), want[2])
        _close(got[3], want[3], (name, k))


def test_float64_batched_and_errors(float64_default):
    g = torch.Generator("cpu").manual_seed(65)
    f = torch.rand(3, 600, 3, generator=g, dtype=torch.float64)
    x = torch.arange(600, dtype=torch.int64)[None, :, None].repeat(3, 1, 1)
    got = nd_environmental_selection(x.to(DEV), f.to(DEV), 250)
    dist = crowding_distance(f.to(DEV), None)
    for b in range(3):
        want = er.environmental_selection(x[b], f[b], 250)
        assert torch.equal(got[0][b].cpu(), want[0]) and torch.equal(got[2][b].cpu(), want[2])
        _close(got[3][b], want[3], b)
        _close(dist[b], er.crowding(f[b], None), b)
    with pytest.raises(RuntimeError):
        nd_environmental_selection(x[0].to(DEV), f[0].to(DEV), 601)
    with pytest.raises(IndexError):
        nd_environmental_selection(x[0].to(DEV), f[0].to(DEV), 0)
    with pytest.raises(RuntimeError):  # float32 costs under a float64 default: the reference's scatter refuses them
        crowding_distance(f[0].float().to(DEV), None)


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.uint8])
def test_integer_fitness_crowding_and_selection(dtype):
    """Integer fitness (the reference accepts it: exact integer differences, divided in the default float dtype,
    non_dominate.py:218-225), 64-bit values beyond float32's 2**24 included."""
    g = torch.Generator("cpu").manual_seed(66)
    if dtype == torch.int64:
        f = (2**40 + torch.randint(0, 3000, (2500, 3), generator=g)).to(dtype)
    elif dtype == torch.int32:
        f = torch.randint(-50, 50, (2500, 2), generator=g, dtype=dtype)
    else:
        f = torch.randint(0, 256, (1500, 4), generator=g).to(dtype)
    fd = f.to(DEV)
    rank = er.ranks_by_peeling(f)
    for mask in (None, rank == 0, rank == 2):
        want = er.crowding(f, mask)
        got = crowding_distance(fd, None if mask is None else mask.to(DEV))
        assert got.dtype == torch.float32
        gw, ww = as_np(got), as_np(want)
        assert np.array_equal(np.isnan(gw), np.isnan(ww)) and np.array_equal(np.isinf(gw), np.isinf(ww))
        fin = np.isfinite(ww)
        np.testing.assert_allclose(gw[fin], ww[fin], rtol=1e-5)
    x = torch.arange(f.size(0), dtype=torch.int64)[:, None]
    for k in (1, 700, f.size(0)):
        want = er.environmental_selection(x, f, k)
        got = nd_environmental_selection(x.to(DEV), fd, k)
        assert got[1].dtype == dtype and torch.equal(got[1].cpu(), want[1])
        assert torch.equal(got[2].cpu(), want[2])
        gw, ww = as_np(got[3]), as_np(want[3])
        assert np.array_equal(np.isnan(gw), np.isnan(ww)) and np.array_equal(np.isinf(gw), np.isinf(ww))
        # the selected rows: equal but for distances that tie within float32 rounding at the cut
        if not torch.equal(got[0].cpu(), want[0]):
            assert sorted(as_np(got[0])[:, 0].tolist()) == sorted(as_np(want[0])[:, 0].tolist()) or np.allclose(
                np.sort(gw[np.isfinite(gw)]), np.sort(ww[np.isfinite(ww)]), rtol=1e-5)


def test_float64_long_sorts_and_vmap(float64_default):
    """Orders of more than 32 768 positions come from the radix sort, shorter ones from the kernels that sort in
    LDS; mapped populations go through the same operators."""
    g = torch.Generator("cpu").manual_seed(67)
    f = torch.rand(40000, 2, generator=g, dtype=torch.float64)
    f[:5000, 0] = f[5000:10000, 0]  # ties
    mask = torch.rand(40000, generator=g) < 0.4
    _close(crowding_distance(f.to(DEV), mask.to(DEV)), er.crowding(f, mask), "40000 rows")
    _close(crowding_distance(f.to(DEV), None), er.crowding(f, None), "40000 rows, no mask")
    fb = torch.rand(4, 300, 3, generator=g, dtype=torch.float64)
    mb = torch.rand(4, 300, generator=g) < 0.5
    mapped = torch.vmap(crowding_distance)(fb.to(DEV), mb.to(DEV))
    xb = torch.arange(300, dtype=torch.int64)[None, :, None].repeat(4, 1, 1)
    sel = torch.vmap(lambda x, f: nd_environmental_selection(x, f, 120))(xb.to(DEV), fb.to(DEV))
    for b in range(4):
        _close(mapped[b], er.crowding(fb[b], mb[b]), ("vmap", b))
        want = er.environmental_selection(xb[b], fb[b], 120)
        assert torch.equal(sel[0][b].cpu(), want[0]) and torch.equal(sel[2][b].cpu(), want[2])
        _close(sel[3][b], want[3], ("vmap selection", b))


def test_float64_selection_either_side_of_the_direct_limit(float64_default):
    """Up to 24 576 rows the last front's distances and order come from kernels that look for every candidate's
    neighbours among the candidates (whatever the size of the front: here one front of all rows, ties included);
    above, from sorts of all rows.  The larger populations hold values that float32 represents exactly, so that the C
    checker (float32) gives their ranks and, to float32's rounding, their distances."""
    from oracle import c_oracle

    g = torch.Generator("cpu").manual_seed(68)
    a = (torch.rand(6000, generator=g, dtype=torch.float64) * 900).round() / 900  # one front with duplicates
    f = torch.stack([a, 1.0 - a], dim=1)
    x = torch.arange(6000, dtype=torch.int64)[:, None]
    for k in (1, 3000, 6000):
        want = er.environmental_selection(x, f, k)
        got = nd_environmental_selection(x.to(DEV), f.to(DEV), k)
        assert torch.equal(got[2].cpu(), want[2]), k
        _close(got[3], want[3], ("one front", k))
        if not torch.equal(got[0].cpu(), want[0]):  # (equal distances at the cut may change places only among themselves)
            gw, ww = as_np(got[3]), as_np(want[3])
            assert np.array_equal(np.sort(gw[np.isfinite(gw)]), np.sort(ww[np.isfinite(ww)])), k
    # a front beyond what those kernels are meant for: the first selection of the shape goes through them all the same,
    # the next ones through the sorts (the library remembers what the last selection of a shape found)
    a = torch.rand(12000, generator=g, dtype=torch.float64)
    f = torch.stack([a, 1.0 - a], dim=1)
    x = torch.arange(12000, dtype=torch.int64)[:, None]
    want = er.environmental_selection(x, f, 7000)
    for call in range(3):
        got = nd_environmental_selection(x.to(DEV), f.to(DEV), 7000)
        assert torch.equal(got[0].cpu(), want[0]) and torch.equal(got[2].cpu(), want[2]), call
        _close(got[3], want[3], ("one front of 12000", call))
    for n, m in ((24576, 2), (30000, 3)):
        f32 = torch.rand(n, m, generator=g)
        k = n // 2
        order, rank, dist, _ = c_oracle.select(f32.numpy(), k)
        order, rank, dist = as_np(order)[:k], as_np(rank), as_np(dist)
        got = nd_environmental_selection(torch.arange(n, dtype=torch.int64, device=DEV)[:, None], f32.double().to(DEV), k)
        assert got[3].dtype == torch.float64
        rows = as_np(got[0])[:, 0]
        assert np.array_equal(as_np(got[2]), rank[rows]) and np.array_equal(np.sort(rank[rows]), np.sort(rank[order])), (n, m)
        worst = rank[order].max()
        assert np.array_equal(np.sort(rows[rank[rows] < worst]), np.sort(order[rank[order] < worst])), (n, m)
        gd, wd = as_np(got[3]), dist[rows]
        fin = np.isfinite(wd)
        assert np.array_equal(np.isfinite(gd), fin), (n, m)
        np.testing.assert_allclose(gd[fin], wd[fin], rtol=1e-4, err_msg=str((n, m)))  # (the checker's sums are float32)
        cut = rank[rows] == worst  # taken from the cut front by descending distance
        assert (gd[cut][:-1] >= gd[cut][1:]).all(), (n, m)


@pytest.mark.parametrize("dtype", [torch.float64, torch.int64])
def test_dense_rank_image(dtype):
    """The float32 image that the ranking takes in place of 8-byte fitness: per objective, the number of distinct
    values below a row's value (one kernel behind a sort of every objective), against numpy."""
    from evox_amd import ops

    g = torch.Generator("cpu").manual_seed(69)
    for shape in ((1, 1), (5, 2), (4097, 3), (3, 50000, 2), (2, 2, 700, 4)):
        if dtype == torch.float64:
            f = (torch.rand(*shape, generator=g, dtype=torch.float64) * 50).round() / 50
            flat = f.view(-1)
            if flat.numel() > 40:
                flat[3], flat[11] = 0.0, -0.0
                flat[5], flat[20] = float("nan"), float("nan")
                flat[7], flat[9] = float("inf"), -float("inf")
                flat[13] = 1.0 + 2.0**-40  # not a float32 value
        else:
            f = torch.randint(-(2**40), 2**40, shape, generator=g, dtype=torch.int64)
            f.view(-1)[::3] //= 2**38  # ties
        got = as_np(ops._order_preserving_f32(f.to(DEV), "fitness"))
        assert got.dtype == np.float32 and got.shape == tuple(shape)
        cols = f.numpy().reshape(-1, shape[-2], shape[-1])
        for b in range(cols.shape[0]):
            for k in range(shape[-1]):
                col = cols[b][:, k]
                want = np.full(col.shape, np.nan, dtype=np.float32)
                ok = ~np.isnan(col) if dtype == torch.float64 else np.ones(col.shape, bool)
                values = np.unique(col[ok] + 0.0 if dtype == torch.float64 else col[ok])  # (-0.0 + 0.0 == 0.0)
                want[ok] = np.searchsorted(values, col[ok]).astype(np.float32)
                assert np.array_equal(got.reshape(cols.shape)[b][:, k], want, equal_nan=True), (shape, b, k)


@pytest.mark.parametrize("shape", [(1023, 1), (1024, 2), (1025, 3), (4096, 1), (20001, 3), (300000, 2), (300, 1500, 1), (100, 3000, 2), (7, 5001, 3)])
def test_dense_rank_parts(shape):
    """The same image where a sorted row is one part, one part per workgroup of values and a remainder, parts of several
    passes, and where rows outnumber the compute units: runs of equal values across the ends of parts, NaN at the end."""
    from evox_amd import ops

    g = torch.Generator("cpu").manual_seed(71)
    f = torch.rand(*shape, generator=g, dtype=torch.float64)
    f.view(-1)[::2] = (f.view(-1)[::2] * 9).round() / 9 - 0.5  # long runs, among them -0.0
    f.view(-1)[5::701] = float("nan")
    got = ops._order_preserving_f32(f.to(DEV), "fitness").cpu()
    cols = f.reshape(-1, *shape[-2:])
    for b in range(cols.size(0)):
        for k in range(shape[-1]):
            col = cols[b, :, k]
            ok = ~torch.isnan(col)
            want = torch.full(col.shape, float("nan"))
            want[ok] = torch.unique(col[ok] + 0.0, return_inverse=True)[1].float()
            assert torch.equal(got.reshape(cols.shape)[b, :, k].nan_to_num(-1.0), want.nan_to_num(-1.0)), (shape, b, k)


def test_batches_of_8_byte_fitness_share_their_launches(float64_default):
    """Several populations of float64 or int64 fitness in one call: the same as one population at a time."""
    g = torch.Generator("cpu").manual_seed(70)
    f64 = (torch.rand(5, 3000, 3, generator=g, dtype=torch.float64) * 300).round() / 300
    f64[1, 7, 2] = float("nan")
    f64[2, :, 1] = 1.0 - f64[2, :, 0]
    f64[3] = f64[3, :1]  # every row the same
    i64 = torch.randint(-(2**40), 2**40, (3, 9000, 2), generator=g, dtype=torch.int64)
    for f, k in ((f64, 1200), (f64, 3000), (i64, 4000)):
        batch, n = f.shape[:2]
        x = torch.rand(batch, n, 3, generator=g, dtype=torch.float64)
        fd, xd = f.to(DEV), x.to(DEV)
        got = nd_environmental_selection(xd, fd, k)
        for b in range(batch):
            alone = nd_environmental_selection(xd[b], fd[b], k)
            for part, (a, c) in enumerate(zip(got, alone)):
                assert a[b].dtype == c.dtype and np.array_equal(as_np(a[b]), as_np(c), equal_nan=True), (f.dtype, k, b, part)
    # no decision columns, populations along another dimension
    none = nd_environmental_selection(torch.empty(5, 3000, 0, device=DEV), f64.to(DEV), 1200)
    want = nd_environmental_selection(torch.zeros(5, 3000, 1, device=DEV), f64.to(DEV), 1200)
    assert none[0].shape == (5, 1200, 0) and torch.equal(none[2], want[2]) and np.array_equal(as_np(none[3]), as_np(want[3]), equal_nan=True)
    mapped = torch.vmap(lambda a, c: nd_environmental_selection(a, c, 1200), in_dims=(1, 1))(
        torch.zeros(3000, 5, 1, device=DEV), f64.permute(1, 0, 2).contiguous().to(DEV))
    assert torch.equal(mapped[2], want[2]) and np.array_equal(as_np(mapped[1]), as_np(want[1]), equal_nan=True)
