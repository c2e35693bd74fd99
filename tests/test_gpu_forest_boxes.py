"""Per-system bounding cubes reduced in parts (as many blocks a system as fit, down to one), and the
finiteness check of the key pass: the cubes are the exact minima and maxima, and a non-finite input of any
system is refused."""

import numpy as np
import pytest

from pytreegrav_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsys", [2, 3, 511, 1024, 1025, 1500])
def test_cubes(nsys):
    rng = np.random.default_rng(nsys)
    ns = rng.integers(2, 40, nsys)
    ns[nsys // 2] = 70_001
    off = np.concatenate([[0], np.cumsum(ns)])
    x = rng.standard_normal((off[-1], 3)) * np.repeat(10.0 ** rng.uniform(-3, 3, nsys), ns)[:, None]
    f = engine.DeviceTree(x, np.ones(len(x)), np.zeros(len(x)), offsets=off)
    cubes = f.cubes.cpu().numpy()
    lo, hi = np.minimum.reduceat(x, off[:-1]), np.maximum.reduceat(x, off[:-1])
    assert np.array_equal(cubes[:, :3], 0.5 * (hi + lo))
    assert np.array_equal(cubes[:, 3], (hi - lo).max(1))


@pytest.mark.parametrize("offsets", [[0, 3000], [0, 1000, 1002, 3000]])
@pytest.mark.parametrize("what,value", [("x", np.nan), ("x", np.inf), ("m", -np.inf), ("h", np.nan)])
def test_non_finite_inputs_are_refused(offsets, what, value):
    rng = np.random.default_rng(1)
    v = {"x": rng.standard_normal((3000, 3)), "m": np.ones(3000), "h": np.full(3000, 0.1)}
    v[what][2999] = value
    with pytest.raises(Exception, match="non-finite"):
        engine.DeviceTree(v["x"], v["m"], v["h"], offsets=np.array(offsets))
