"""Ray-traced columns along the axes of a lattice, where particles and whole nodes lie exactly on the rays, against
the oracle: products of one factor and sums of zeros, so that both see the same r^2 - z^2 there.  Within 1e-12 of
the largest column (r / h stays below 60: 2^-53 r^2 / h^2 < 4e-13, 20 particles a ray)."""

import numpy as np
import pytest
import torch

import oracle
from pytreegrav_amd import ConstructTree, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,scale", [(16, 1.0), (20, 1.0), (17, 0.3)])
@pytest.mark.parametrize("path", ["bundles", "own", "per target"])
def test_axis_rays_of_a_lattice(k, scale, path):
    g = (np.arange(k) + 0.5) / k * scale
    x = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    t = x[np.random.default_rng(0).choice(len(x), 300)]
    h = np.full(len(x), 0.6 / k * scale)
    rays = np.concatenate([np.eye(3), -np.eye(3)])
    tree = ConstructTree(x, np.ones(len(x)), h).dev
    if path == "per target":
        got = engine.column_rays(tree, t, np.tile(rays, (len(t), 1, 1)), per_target=True)
    else:
        ctr = torch.zeros(1, dtype=torch.int64, device=engine.device()) if path == "own" else None
        got = engine.column_rays(tree, t, rays, counters=ctr)
    want = oracle.column_rays(oracle.build_tree(x, np.ones(len(x)), h), t, rays)
    assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * np.abs(want).max()
