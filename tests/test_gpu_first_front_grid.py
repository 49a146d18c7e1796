"""The first front of more rows than one pass of the grid's workgroups holds (four rows to each of 1024 threads, on every
compute unit), where a workgroup drops what its own rows dominate and the grid's cells lie apart in memory, against the C
checker: masks are whole numbers and must be equal."""

import numpy as np
import pytest
import torch

from oracle import c_oracle

pytestmark = pytest.mark.gpu

INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("n", [200001, 600007, 1050001])
@pytest.mark.parametrize("m", [2, 3])
def test_rows_dropped_by_their_own_workgroup(n, m):
    from evox_amd.operators.selection import non_dominated_mask

    g = torch.Generator("cpu").manual_seed(n + m)
    d = torch.randn(n, m, generator=g).abs()
    f = d / d.norm(dim=1, keepdim=True) * (1.0 - 0.1 * torch.log1p(-torch.rand(n, 1, generator=g)))
    f[::3] = torch.round(f[::3] * 64) / 64  # ties, equal rows and zeros among them
    f[1::1009, 0] = INF
    f[2::1013, m - 1] = -0.0
    f[3::50021, m - 1] = -INF
    f[4::1019, m // 2] = NAN
    got = non_dominated_mask(f.to("cuda")).cpu().numpy()
    assert np.array_equal(got, c_oracle.first_front(f.numpy()))
