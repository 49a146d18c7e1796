"""The argsort that holds all keys in LDS (8193 to 32 768 positions) where some or all keys are the largest there is --
the rank of the rows behind a cut -- against numpy's stable order."""

import numpy as np
import pytest
import torch

from evox_amd.utils import lexsort

pytestmark = pytest.mark.gpu
TOP = 2**31 - 1


@pytest.mark.parametrize("n", [8193, 24576, 24577, 32768])
@pytest.mark.parametrize("keys", ["ranks", "next to the largest", "wide", "all the largest", "one other", "low words"])
def test_largest_key(n, keys):
    rng = np.random.default_rng(n)
    if keys == "ranks":
        key = np.where(rng.random(n) < 0.5, TOP, rng.integers(0, 30, n)).astype(np.int32)
    elif keys == "next to the largest":
        key = rng.integers(TOP - 2, TOP + 1, n).astype(np.int32)
    elif keys == "wide":
        key = np.where(rng.random(n) < 0.3, TOP, rng.integers(-(2**31), TOP, n)).astype(np.int32)
    elif keys == "all the largest":
        key = np.full(n, TOP, np.int32)
    elif keys == "one other":
        key = np.full(n, TOP, np.int32)
        key[n // 2] = -(2**31)
    else:  # 64-bit keys, sorted by their low and then by their high words
        key = np.where(rng.random(n) < 0.5, -1, rng.integers(-5, 2**33, n)).astype(np.int64)
    got = lexsort([torch.from_numpy(key).cuda()]).cpu().numpy()
    assert np.array_equal(got, np.argsort(key, kind="stable"))
