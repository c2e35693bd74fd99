"""The bundle walk of ray-traced columns (ptg_column_bundles) and its target orders (ptg_ray_orders)
against the oracle, within 1e-12 of the largest column: the chord's b^2 = r^2 - z^2 carries 2^-53 r^2,
and r / h stays below 100 here."""

import numpy as np
import pytest
import torch

import oracle
from pytreegrav_amd import ConstructTree, engine

pytestmark = pytest.mark.gpu


def _rays(k):
    u = np.random.default_rng(k).normal(size=(k, 3))
    u[0] = [0.0, 0.0, -1.0]
    return u / np.linalg.norm(u, axis=1, keepdims=True)


def _check(x, m, h, targets, rays):
    t = ConstructTree(x, m, h)
    got = engine.column_rays(t.dev, targets, rays)
    assert torch.equal(got, engine.column_rays(t.dev, targets, rays))
    want = oracle.column_rays(oracle.build_tree(x, m, h), targets, rays)
    assert np.abs(got.cpu().numpy() - want).max() <= 1e-12 * max(np.abs(want).max(), 1e-300)


# bundles of 64 targets and their remainders; radii of one size, and over two decades with zeros (wide
# rectangles against small reaches: quarters, then single targets)
@pytest.mark.parametrize("nt,nr", [(1, 1), (63, 2), (64, 1), (65, 3), (129, 2), (1500, 5)])
@pytest.mark.parametrize("radii", ["equal", "spread"])
def test_bundles_match_oracle(nt, nr, radii):
    rng = np.random.default_rng(nt)
    x = rng.normal(size=(4000, 3))
    h = np.full(len(x), 0.2) if radii == "equal" else 10.0 ** rng.uniform(-1.0, 0.7, len(x))
    if radii == "spread":
        h[::7] = 0.0
    targets = np.concatenate([x, rng.normal(size=(500, 3)) * 3.0])[rng.permutation(4500)[:nt]]
    _check(x, rng.uniform(0.0, 1.0, len(x)), h, targets, _rays(nr))


def test_deep_and_massless_trees():
    # 2000 coincident points: a chain of buckets hundreds of levels deep, past the LDS stack
    rng = np.random.default_rng(3)
    x = np.concatenate([rng.normal(size=(500, 3)), np.full((2000, 3), 0.25)])
    m = np.ones(len(x))
    m[::3] = 0.0
    _check(x, m, np.full(len(x), 0.3), x[:200] + 0.1, _rays(2))


def test_non_finite_targets_leave_their_neighbours_alone():
    rng = np.random.default_rng(5)
    x = rng.normal(size=(2000, 3))
    t = ConstructTree(x, np.ones(2000), np.full(2000, 0.3))
    targets = rng.normal(size=(40, 3))
    want = engine.column_rays(t.dev, targets, _rays(2))
    bad = targets.copy()
    bad[0], bad[17], bad[39] = np.nan, np.inf, -np.inf
    got = engine.column_rays(t.dev, bad, _rays(2))
    keep = np.ones(40, bool)
    keep[[0, 17, 39]] = False
    assert torch.allclose(got[keep], want[keep], rtol=1e-12, atol=0.0) and not bool(got[~keep].any())


@pytest.mark.parametrize("nt,nr", [(1, 1), (1000, 3), (2049, 1), (300, 70)])
def test_ray_orders_sort_every_ray_by_its_own_plane(nt, nr):
    rng = np.random.default_rng(nt + nr)
    tp = torch.from_numpy(rng.normal(size=(nt, 3))).cuda()
    rays = _rays(nr)
    order = engine._ray_orders(tp, torch.from_numpy(rays).cuda()).cpu().numpy()
    assert np.array_equal(np.sort(order, 1), np.tile(np.arange(nt), (nr, 1)))
    if nt >= 1000:  # neighbours in the order are neighbours across the ray: far nearer than at random
        x = tp.cpu().numpy()[order[0]]
        a = x - np.outer(x @ rays[0], rays[0])
        assert np.median(np.linalg.norm(np.diff(a, axis=0), axis=1)) < 0.2
