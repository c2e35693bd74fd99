"""The FP64 walk and the angle-binned columns at the ends of the number range: separations whose squares
overflow or nearly do, infinite and nan targets among ordinary ones, nan, infinite and zero softenings.  Each
value is the oracle's (IEEE square roots and divisions): to 1e-11 of itself (sums of some hundred terms), the
same infinities and the same nans.  (The first target of a group is an ordinary one: the oracle's box starts there.)"""

import numpy as np
import pytest
import torch

import oracle
from pytreegrav_amd import ConstructTree, engine

pytestmark = pytest.mark.gpu


def _same(got, want):
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    f = np.isfinite(want)
    tiny = 1e-300  # sums of terms below the ordinary numbers carry no digits
    assert (np.abs(got[f] - want[f]) <= 1e-11 * np.abs(want[f]) + tiny).all()


def _sources(scale):
    rng = np.random.default_rng(8)
    n = 700
    return rng.uniform(0.5, 1.5, (n, 3)) * scale, rng.uniform(0.5, 1.5, n), rng.uniform(0.0, 0.2, n) * scale


def _targets(x, h, gs):
    # a group of ordinary targets, then one ordinary target and the odd ones of a kind per group
    s = np.abs(x).max()
    odd = [[1e150, 0.0, 0.0], [2e150, 3e150, 1e150], [1.2e154, 0.0, 0.0], [-1.5e154, 1e154, 0.0], [1e200, 1e200, -1e200],
           [np.nan, 0.0, 0.0], [s, np.nan, s], [s, s, np.nan], [np.inf, 0.0, 0.0], [s, -np.inf, np.inf],
           [np.nan, np.inf, 0.0]]
    soft = [np.nan, np.inf, 0.0, 1e-170]
    t, th = [x[i] for i in range(gs)], [h[i] for i in range(gs)]
    for k, o in enumerate(odd):
        row = [x[40 + k] + 0.3 * s] + [o] * (gs - 1)
        t += row
        th += [h[40 + k]] * len(row)
    for k, hk in enumerate(soft):
        row = [x[60 + gs * k + i] + 0.01 * s * (i % 3) for i in range(gs)]
        t += row
        th += [h[60 + gs * k]] + [hk] * (gs - 1)
    return np.array(t), np.array(th)


@pytest.mark.parametrize("scale", [1.0, 1e149, 1e-40])
@pytest.mark.parametrize("gs,quad,mask", [(2, False, 3), (8, False, 7), (8, True, 3), (65, False, 2)])
def test_walk(scale, gs, quad, mask):
    x, m, h = _sources(scale)
    t, th = _targets(x, h, gs)
    tree = ConstructTree(x, m, h, quadrupole=quad)
    perm = torch.arange(len(t), dtype=torch.int64, device=engine.device())
    out = engine.walk(tree.dev, t, th, perm, mask, quadrupole=quad, group_size=gs, theta=0.7, precision="float64")
    ref = oracle.fields_grouped(oracle.build_tree(x, m, h, quadrupole=quad), t, th, potential=bool(mask & 1),
                                accel=bool(mask & 2), tidal=bool(mask & 4), quadrupole=quad, group_size=gs, theta=0.7)
    for k, v in engine.unpack_fields(out, mask).items():
        got, want = v.cpu().numpy().reshape(len(t), -1), ref[k].reshape(len(t), -1)
        # accelerations and tidal tensors cancel: to the largest term of their group's ordinary targets
        if k == "potential":
            _same(got, want)
        else:
            assert np.array_equal(np.isnan(got), np.isnan(want))
            assert np.array_equal(np.isinf(got), np.isinf(want))
            f = np.isfinite(want)
            assert (np.abs(got - want)[f] <= 1e-10 * np.abs(want[f]).max()).all()


@pytest.mark.parametrize("scale", [1.0, 1e149, 1e-40])
@pytest.mark.parametrize("gs", [2, 8])
def test_binned_columns(scale, gs):
    x, m, h = _sources(scale)
    h[::5] = 0.0
    t, _ = _targets(x, h, gs)
    with np.errstate(all="ignore"):
        tree = ConstructTree(x, m, h)
        got = engine.column_binned(tree.dev, t, group_size=gs, theta=0.7).cpu().numpy()
        want = oracle.column_binned(oracle.build_tree(x, m, h), t, group_size=gs, theta=0.7)
    _same(got, want)
