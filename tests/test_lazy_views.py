"""Views whose memory holds other bytes than their values -- the imaginary part of a conjugated tensor has a negative bit, a
conjugated one a conjugate bit -- give what their resolved copies give: calls that go past the dispatcher must not read the
memory as it is."""

import pytest
import torch

from evox_amd import ops
from evox_amd.hype import cal_hv
from evox_amd.metrics import hv
from evox_amd.operators import selection
from evox_amd.operators.selection import non_dominate


def _negative_view(t):
    view = torch.complex(torch.zeros_like(t), -t).conj().imag
    assert type(view) is torch.Tensor and view.is_neg() and torch.equal(view, t)
    return view


def test_lazy_views_keep_to_the_operator():
    f = torch.rand(5, 3)
    assert non_dominate._plain(ops.nd_rank, f) is not ops.nd_rank
    assert non_dominate._plain(ops.nd_rank, _negative_view(f)) is ops.nd_rank
    x = torch.complex(f, f)
    assert non_dominate._plain(ops.nd_select, x, f) is not ops.nd_select
    assert non_dominate._plain(ops.nd_select, x.conj(), f) is ops.nd_select


def test_the_choice_can_be_traced():
    @torch.compile(fullgraph=True, backend="eager")
    def kept(f):
        return f + 1.0 if non_dominate._plain(ops.nd_rank, f) is ops.nd_rank else f

    assert torch.equal(kept(torch.zeros(3)), torch.ones(3))


CALLS = {
    "rank": lambda f: selection.non_dominate_rank(f),
    "rank until": lambda f: selection.non_dominate_rank_until(f, f.size(0) // 2),
    "first front": lambda f: selection.non_dominated_mask(f),
    "crowding": lambda f: selection.crowding_distance(f, None),
    "select": lambda f: selection.nd_environmental_selection(f, f, f.size(0) // 2),
    "two part": lambda f: selection.nd_environmental_selection_two_part(f, f, f, f, f.size(0) // 2),
    "conjugated rows": lambda f: selection.nd_environmental_selection(
        torch.complex(f, f).conj() if f.is_neg() else torch.complex(f, -f), f, f.size(0) // 2),
    "tournament": lambda f: selection.tournament_selection_multifit(64, [f[:, 0], f[:, 1]]),
    "hypervolume": lambda f: hv(f, torch.full((f.size(1),), 1.5, device=f.device), 5000),
    "hypervolume, reference": lambda f: hv(f.detach().clone(), f[0] + 1.0 if not f.is_neg() else _negative_view(f[0] + 1.0), 5000),
    "contributions": lambda f: cal_hv(f, torch.full((f.size(1),), 1.5, device=f.device), f.size(0) // 2, 5000),
}


@pytest.mark.gpu
@pytest.mark.parametrize("call", CALLS)
@pytest.mark.parametrize("n", [150, 3000])
def test_lazy_views_give_what_their_copies_give(call, n):
    f = torch.rand(n, 3, generator=torch.Generator().manual_seed(n)).cuda()
    out = []
    for fitness in (_negative_view(f), f):
        torch.manual_seed(11)
        got = CALLS[call](fitness)
        out.append(got if isinstance(got, tuple) else (got,))
    # the operators' statements round a volume m + 1 times in an order of their own, and a weight up to n times
    rtol = {"hypervolume": 8 * 2.0**-24, "hypervolume, reference": 8 * 2.0**-24, "contributions": (2 * n + 14) * 2.0**-24}.get(call, 0.0)
    for got, want in zip(*out):
        assert got.dtype == want.dtype and torch.allclose(got, want, rtol=rtol, atol=0.0)
