"""Angle-binned columns through a tree whose every level leaves its most on the traversal stack: 30 levels of seven
filled octants each around the corner that the next level refines, all opened from there (about 448 entries a
level).  Against the oracle, within 1e-11 of the largest bin (some ten thousand terms)."""

import numpy as np
import pytest

import oracle
from pytreegrav_amd import ConstructTree, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("levels", [18, 30])
def test_spilled_traversals(levels):
    g = (np.arange(4) + 0.5) / 4
    cube = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    octants = [(i, j, k) for i in (0, 1) for j in (0, 1) for k in (0, 1) if (i, j, k) != (1, 1, 1)]
    # level l fills the octants of [-2^-l, 0]^3 but the last, which is level l + 1's cube
    x = np.concatenate([((cube + o) / 2 - 1) * 2.0 ** -l for l in range(levels) for o in octants])
    x = np.concatenate([x, (cube - 1) * 2.0 ** -levels])
    m, h = np.ones(len(x)), np.full(len(x), 2.0 ** -levels)
    t = -np.random.default_rng(1).uniform(0, 1, (5, 3)) * 2.0 ** -levels
    got = engine.column_binned(ConstructTree(x, m, h).dev, t, group_size=5, theta=0.1).cpu().numpy()
    want = oracle.column_binned(oracle.build_tree(x, m, h), t, group_size=5, theta=0.1)
    assert np.abs(got - want).max() <= 1e-11 * np.abs(want).max()
