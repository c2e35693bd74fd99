"""The direct sum's split over waves and lane slices: every count of targets and sources around the
sizes where the split changes, pairs off the plain path (coincident, softened, at extreme distances),
against the oracle (FP64 1e-13 and FP32 10 * 1e-5 sqrt(N / 1000) of the largest value, the bounds of
test_gpu_direct.py)."""

import numpy as np
import pytest

import oracle
from pytreegrav_amd import engine

pytestmark = pytest.mark.gpu


def _compare(got, ref, tol):
    for k in ref:
        s = np.abs(ref[k]).max()
        assert np.abs(got[k].numpy() - ref[k]).max() <= tol * (s if s > 0 else 1.0), k


@pytest.mark.parametrize("nt,ns", [(1, 1), (3, 15), (4, 17), (5, 1023), (1024, 64), (1025, 65), (16, 4096), (17, 0),
                                   (2049, 33)])
@pytest.mark.parametrize("mask", [2, 7])
def test_targets_and_sources(nt, ns, mask):
    rng = np.random.default_rng(nt * 7 + ns)
    xs, xt = rng.normal(size=(ns, 3)), rng.normal(size=(nt, 3))
    k = min(nt, ns) // 2
    xt[:k] = xs[:k]  # coincident pairs
    ms, hs, ht = rng.random(ns) + 0.1, rng.random(ns) * 0.3, rng.random(nt) * 0.2
    ref = oracle.fields_target_bruteforce(xt, ht, xs, ms, hs, potential=bool(mask & 1), accel=True, tidal=bool(mask & 4),
                                          G=1.5)
    for prec, tol in (("float64", 1e-13), ("float32", 1e-4 * np.sqrt(max(ns, 1000) / 1000))):
        out = engine.direct(xt, ht, xs, ms, hs, mask, G=1.5, self_mode=False, precision=prec)
        _compare(engine.unpack_fields(out.cpu(), mask), ref, tol)


@pytest.mark.parametrize("n", [2, 1024, 1025])
def test_self_mode_with_coincident_particles(n):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, 3))
    x[n // 2:] = x[: n - n // 2]  # every position twice: the softened potential stays, the force does not
    m, h = rng.random(n) + 0.1, np.full(n, 0.1)
    ref = oracle.fields_self_bruteforce(x, m, h, potential=True, accel=True, tidal=True)
    for prec, tol in (("float64", 1e-13), ("float32", 1e-4 * np.sqrt(max(n, 1000) / 1000))):
        out = engine.direct(x, h, x, m, h, 7, self_mode=True, precision=prec)
        _compare(engine.unpack_fields(out.cpu(), 7), ref, tol)


def test_extreme_distances():
    # squares past the largest and below the smallest ordinary number of either type
    x = np.array([[0.0, 0, 0], [1e-160, 0, 0], [1.0, 0, 0], [0, 1e160, 0]])
    m, h = np.ones(4), np.zeros(4)
    ref = oracle.fields_self_bruteforce(x, m, h, potential=True)["potential"]
    got = engine.direct(x, h, x, m, h, 1, self_mode=True).cpu().numpy()[:, 0]
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    ok = np.isfinite(ref)
    assert np.allclose(got[ok], ref[ok], rtol=1e-13, atol=0.0)
    x32 = np.array([[0.0, 0, 0], [1.0, 0, 0], [0, 1e25, 0], [2.0 ** -70, 0, 0]])
    got = engine.direct(x32, h, x32, m, np.full(4, 0.5), 2, self_mode=True, precision="float32").cpu().numpy()
    ref = oracle.fields_self_bruteforce(x32, m, np.full(4, 0.5), accel=True)["accel"]
    assert np.allclose(got, ref, rtol=1e-5, atol=1e-12)
