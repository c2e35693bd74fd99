"""Cut traversals of the FP32 walk: targets of which the last few groups spread over the whole domain, so
that each opens most of the tree and is finished in shares (systems of 1024 groups, 2048 with tidal
tensors).  The fields follow the FP64 walk of the same groups to the reference's FP32 tolerances (RMS 1e-5,
worst 1e-2 where an opening decision flips), the visit counts to 1e-3, and a second run gives the same bits."""

import numpy as np
import pytest
import torch

from pytreegrav_amd import ConstructTree, engine
from pytreegrav_amd.sampling import plummer_truncated

pytestmark = pytest.mark.gpu


def _setup(n, nt, quad, wide=300):
    # nt - wide targets in a small ball far from the mass, then `wide` drawn from all of it
    x, m = plummer_truncated(n, seed=23)
    h = np.full(n, 0.02)
    t = ConstructTree(x, m, h, quadrupole=quad)
    rng = np.random.default_rng(nt)
    far = np.array([400.0, 0.0, 0.0]) + rng.standard_normal((nt - wide, 3))
    tx = np.concatenate([far, x[rng.choice(n, wide, replace=False)] * 1.1])
    return t.dev, tx, np.full(nt, 0.03), torch.arange(nt, dtype=torch.int64, device=engine.device())


@pytest.mark.parametrize("nt,gs,quad,mask", [(65535, 64, False, 2), (65537, 64, False, 3), (65600, 64, True, 3),
                                             (131072, 128, False, 2), (262150, 256, True, 3),
                                             (20 * 2048 + 7, 20, False, 4), (131100, 64, True, 7)])
def test_wide_groups_follow_the_fp64_walk(nt, gs, quad, mask):
    t, tx, th, perm = _setup(60_000, nt, quad)
    kw = dict(quadrupole=quad, group_size=gs, theta=0.7, grouping="fixed")
    outs = []
    for _ in range(2):
        ctr = torch.zeros(4, dtype=torch.int64, device=engine.device())
        outs.append(engine.walk(t, tx, th, perm, mask, precision="float32", counters=ctr, **kw))
    assert torch.equal(outs[0], outs[1])
    c64 = torch.zeros(4, dtype=torch.int64, device=engine.device())
    ref = engine.walk(t, tx, th, perm, mask, precision="float64", counters=c64, **kw)
    assert abs(int(ctr[1]) / int(c64[1]) - 1) < 1e-3
    for k, v in engine.unpack_fields(outs[0], mask).items():
        if k == "tidal":  # the reference states no FP32 bar for it: the rounding of the coordinates rules it
            continue
        r = engine.unpack_fields(ref, mask)[k]
        rms = r.square().mean().sqrt()
        assert (v - r).square().mean().sqrt() <= 1e-5 * rms, k
        assert (v - r).abs().max() <= 1e-2 * torch.maximum(rms, r.abs().max()), k


@pytest.mark.parametrize("rel", [0.0, 3.0])
def test_group_expansion_in_shares(rel):
    # the folded far field of each share is evaluated for its group: the same truncation as uncut, so the
    # unfolded walk is met to the expansion's tolerance (1e-3 of the RMS field per element, far less in sum)
    t, tx, th, perm = _setup(60_000, 65_900, False)
    kw = dict(group_size=64, theta=0.7, grouping="cells", precision="float32")
    plain = engine.walk(t, tx, th, perm, 3, **kw)
    scale = float(plain[:, 1:].square().sum(1).mean().sqrt())
    a = engine.walk(t, tx, th, perm, 3, expansion=1e-3 * scale, expansion_rel=rel, **kw)
    assert torch.equal(a, engine.walk(t, tx, th, perm, 3, expansion=1e-3 * scale, expansion_rel=rel, **kw))
    assert float((a - plain)[:, 1:].square().sum(1).mean().sqrt()) <= 1e-2 * scale


def test_deferral_under_graph_replay():
    t, tx, th, perm = _setup(60_000, 65_700, False)
    xd, hd = engine.to_dev(tx, (-1, 3)), engine.to_dev(th, (65_700,))
    kw = dict(group_size=64, theta=0.7, grouping="fixed", precision="float32", _check=False, _ws_slot=7)
    want = engine.walk(t, xd, hd, perm, 3, **kw)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        engine.walk(t, xd, hd, perm, 3, **kw)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        out = engine.walk(t, xd, hd, perm, 3, **kw)
    for _ in range(3):
        out.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
