"""Every field of cut FP32 traversals against the same groups uncut: groups spread over the whole domain, in a call
of enough groups to be cut (1024, 2048 with tidal tensors) and alone.  Both sum the same n terms in FP32, each in an
order of its own: they differ by at most 2 n 2^-24 times the sum of the terms' sizes.  Tensors are symmetric bit for
bit, and the control block shows that the groups were cut, and their shares again."""

import numpy as np
import pytest
import torch

from pytreegrav_amd import ConstructTree, engine
from pytreegrav_amd.sampling import plummer_truncated

pytestmark = pytest.mark.gpu

NGROUP, NTASK = 288, 289  # words of the walk's control block


@pytest.mark.parametrize("gs,groups,quad,mask", [(64, 1030, False, 3), (128, 1030, True, 2), (20, 2050, False, 4),
                                                 (64, 2050, True, 7), (256, 2050, False, 6), (33, 2050, True, 5)])
def test_cut_equals_uncut(gs, groups, quad, mask):
    n, wide = 60_000, 6
    x, m = plummer_truncated(n, seed=23)
    h = np.full(n, 0.02)
    tree = ConstructTree(x, m, h, quadrupole=quad).dev
    rng = np.random.default_rng(gs)
    tw = x[rng.choice(n, wide * gs, replace=False)] * 1.1
    far = np.array([400.0, 0.0, 0.0]) + rng.standard_normal(((groups - wide) * gs, 3))

    def walk(t):
        ctr = torch.zeros(4, dtype=torch.int64, device=engine.device())
        perm = torch.arange(len(t), dtype=torch.int64, device=engine.device())
        out = engine.walk(tree, t, np.full(len(t), 0.03), perm, mask, quadrupole=quad, group_size=gs, theta=0.7,
                          grouping="fixed", precision="float32", counters=ctr)
        key = (torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream, 0)
        return engine.unpack_fields(out, mask), ctr, engine._walk_ws[key][:8192].view(torch.int32).cpu()

    cut, _, c = walk(np.concatenate([far, tw]))
    # cut as groups into at most 16 shares each, and some of those again
    assert int(c[NGROUP]) == wide and int(c[NTASK]) > 16 * wide
    alone, ctr, c = walk(tw)
    assert int(c[NGROUP]) == 0
    terms = 2 * int(ctr[0]) // len(tw)  # of one target, with a factor for groups that list more than others
    r = torch.cdist(engine.to_dev(tw, (-1, 3)), engine.to_dev(x, (-1, 3))).clamp_min(0.03)
    md = engine.to_dev(m, (n,))
    # sizes of the terms, spline and quadrupoles included: |phi| <= 2.8 m / r, |a| <= 12 m / r^2, |T| <= 90 m / r^3
    size = {"potential": 2.8 * (md / r).sum(1), "accel": 12 * (md / r ** 2).sum(1), "tidal": 90 * (md / r ** 3).sum(1)}
    for k, v in cut.items():
        got, want = v[-len(tw):], alone[k]
        d = (got - want).abs().reshape(len(tw), -1).amax(1)
        assert bool((d <= 2 * terms * 2.0 ** -24 * size[k]).all()), k
        assert float(d.max()) <= 1e-3 * float(want.abs().max()), k  # and far closer than a misplaced component
        if k == "tidal":
            assert torch.equal(got, got.transpose(1, 2))
