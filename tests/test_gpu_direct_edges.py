"""The direct sum at the edges of its split: more than 131072 targets (64 to a block, one slice a wave), and
subnormal softenings, whose reciprocal is infinite.  Against the oracle with test_gpu_direct_split.py's bounds."""

import numpy as np
import pytest

import oracle
from pytreegrav_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [131072, 131073, 131136])
@pytest.mark.parametrize("mask", [2, 7])
def test_many_targets(nt, mask):
    rng = np.random.default_rng(nt)
    ns = 65
    xs, xt = rng.normal(size=(ns, 3)), rng.normal(size=(nt, 3))
    xt[-ns:] = xs
    ms, hs, ht = rng.random(ns) + 0.1, rng.random(ns) * 0.3, rng.random(nt) * 0.2
    ref = oracle.fields_target_bruteforce(xt, ht, xs, ms, hs, potential=bool(mask & 1), accel=True, tidal=bool(mask & 4))
    for prec, tol in (("float64", 1e-13), ("float32", 1e-4)):
        got = engine.unpack_fields(engine.direct(xt, ht, xs, ms, hs, mask, precision=prec).cpu(), mask)
        for k in ref:
            assert np.abs(got[k].numpy() - ref[k]).max() <= tol * np.abs(ref[k]).max(), k


@pytest.mark.parametrize("n", [2, 17, 1000, 2000])
@pytest.mark.parametrize("prec,h,tol", [("float64", 5e-310, 1e-13), ("float32", 1e-40, 1e-4 * np.sqrt(2))])
def test_subnormal_softenings(n, prec, h, tol):
    rng = np.random.default_rng(n)
    x, m = rng.normal(size=(n, 3)), rng.random(n) + 0.1
    ref = oracle.fields_self_bruteforce(x, m, np.zeros(n), potential=True, accel=True, tidal=True)
    out = engine.direct(x, np.full(n, h), x, m, np.full(n, h), 7, self_mode=True, precision=prec)
    got = engine.unpack_fields(out.cpu(), 7)
    for k in ref:
        assert np.abs(got[k].numpy() - ref[k]).max() <= tol * np.abs(ref[k]).max(), k
