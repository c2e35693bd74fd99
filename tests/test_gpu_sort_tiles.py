"""The key sort at the edges of its tiles and of the sizes where the tile changes: the order is numpy's
stable argsort of the keys, so equal keys keep their input order."""

import numpy as np
import pytest
import torch

from pytreegrav_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 255, 256, 257, 65535, 65536, 65537, 65536 + 511, 262144, 262145, 262144 + 1023,
                               1048576, 1048577, 1048576 + 2047])
def test_order_is_the_stable_sort(n):
    # a lattice of 256 cells a side with several particles on a place: runs of equal keys
    rng = np.random.default_rng(n)
    q = rng.integers(0, 256, (n, 3))
    q[0], q[-1] = 0, 256
    x = q / 256.0
    key = np.zeros(n, dtype=np.uint64)
    cell = np.minimum(q.astype(np.uint64) << np.uint64(13), np.uint64((1 << 21) - 1))
    for b in range(21):
        for k in range(3):
            key |= ((cell[:, k] >> np.uint64(b)) & np.uint64(1)) << np.uint64(3 * b + k)
    got = engine.morton_order(torch.from_numpy(x).to(engine.device())).cpu().numpy()
    assert np.array_equal(got, np.argsort(key, kind="stable"))
