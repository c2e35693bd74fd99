"""The FP64 walk's slices, deferred traversals and squared opening test against the oracle: equal
interaction and visit counters, fields within 1e-10 of the largest value (sums of up to 1e5 terms in
another order, 1e5 * 2^-53 ~ 1e-11), and the same bits on a second run."""

import numpy as np
import pytest

import oracle
from pytreegrav_amd.sampling import plummer_truncated

pytestmark = pytest.mark.gpu


def _lattice(k):
    g = (np.arange(k) + 0.5) / k
    return np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)


def _check(x, m, h, t, ht, gs, theta, quad, mask):
    import torch

    from pytreegrav_amd import ConstructTree, engine

    tree = ConstructTree(x, m, h, quadrupole=quad)
    perm = torch.arange(len(t), dtype=torch.int64, device=engine.device())
    outs = []
    for _ in range(2):
        ctr = torch.zeros(4, dtype=torch.int64, device=engine.device())
        outs.append(engine.walk(tree.dev, t, ht, perm, mask, quadrupole=quad, group_size=gs, theta=theta,
                                precision="float64", counters=ctr))
    assert torch.equal(outs[0], outs[1])
    ot = oracle.build_tree(x, m, h, quadrupole=quad)
    ref, rctr = oracle.fields_grouped(ot, t, ht, potential=bool(mask & 1), accel=bool(mask & 2), tidal=bool(mask & 4),
                                      quadrupole=quad, group_size=gs, theta=theta, return_counters=True)
    assert int(ctr[0]) == rctr["interactions"] and int(ctr[1]) == rctr["visits"]
    got = {k: v.cpu().numpy() for k, v in engine.unpack_fields(outs[0], mask).items()}
    for k in ref:
        assert np.abs(got[k] - ref[k]).max() <= 1e-10 * np.abs(ref[k]).max(), k


# scattered targets: every group's box spans the sphere and opens most of its 7e4 elements, past the
# budgets of all rounds; group sizes at the edges of the slices and of the targets per lane
@pytest.mark.parametrize("gs,quad,mask", [(1, False, 2), (2, False, 3), (5, True, 7), (8, False, 2), (8, True, 4),
                                          (9, False, 4), (32, False, 3), (33, True, 2), (64, False, 1), (65, False, 7),
                                          (256, True, 7)])
def test_groups_wider_than_the_cells(gs, quad, mask):
    x, m = plummer_truncated(50_000, seed=17)
    h = np.full(len(x), 0.02)
    pick = np.random.default_rng(gs).choice(len(x), 3 * gs + gs // 2 + 1, replace=False)
    t = x[pick] * 1.5
    t[: gs] = x[pick[: gs]]  # the first group sits on particles: self terms, softened pairs
    _check(x, m, h, t, np.full(len(t), 0.03), gs, 0.7, quad, mask)


# lattice sources and targets meet the opening radius exactly (r_min = size / theta); scales where
# squares of distances leave the range of ordinary sizes
@pytest.mark.parametrize("theta,scale", [(1.0, 1.0), (0.5, 1.0), (1.0, 2.0 ** 250), (0.5, 2.0 ** -250)])
def test_opening_test_at_ties(theta, scale):
    x = _lattice(16) * scale
    t = np.concatenate([_lattice(8), _lattice(8) + 1.0, _lattice(8) * 4.0]) * scale
    _check(x, np.full(len(x), 1.0), np.zeros(len(x)), t, np.zeros(len(t)), 8, theta, False, 2)


@pytest.mark.parametrize("n", [4_097, 200_000])
def test_self_gravity_sizes(n):
    x, m = plummer_truncated(n, seed=n)
    h = np.full(n, 0.01)
    t = oracle.build_tree(x, m, h)
    xs = np.ascontiguousarray(x[t.TreewalkIndices])
    _check(x, m, h, xs, h, 8, 0.7, False, 3)
