"""Cut traversals when the tables of groups and tasks are full: every target's group spreads over the whole
domain, in groups of the largest rows, so that few of them fit at a time.  A group's fields are the same bits
as in calls with few such groups, where all fit, and the counters add up; so too with walks on two streams."""

import numpy as np
import pytest
import torch

from pytreegrav_amd import ConstructTree, engine
from pytreegrav_amd.sampling import plummer_truncated

pytestmark = pytest.mark.gpu

NGROUP, BACK, BATCH = 288, 1120, 1123  # words of the walk's control block


def _control():
    return engine._walk_ws[(torch.cuda.current_device(), torch.cuda.current_stream().cuda_stream, 0)][:8192].view(torch.int32).cpu()


def _tree(n, quad):
    x, m = plummer_truncated(n, seed=5)
    return ConstructTree(x, m, np.full(n, 0.02), quadrupole=quad).dev, x


def _wide(x, groups, gs):
    # each group's targets are drawn from the whole domain
    pick = np.random.default_rng(gs).choice(len(x), groups * gs)
    return x[pick] * 1.1


def _walk(t, tx, gs, mask, precision, quad):
    ctr = torch.zeros(4, dtype=torch.int64, device=engine.device())
    perm = torch.arange(len(tx), dtype=torch.int64, device=engine.device())
    out = engine.walk(t, tx, np.full(len(tx), 0.03), perm, mask, quadrupole=quad, group_size=gs, theta=0.7,
                      grouping="fixed", precision=precision, counters=ctr)
    return out, ctr


@pytest.mark.parametrize("gs,quad,mask,groups,part", [(256, True, 7, 420, 42), (256, False, 4, 700, 70)])
def test_fp64(gs, quad, mask, groups, part):
    t, x = _tree(30_000, quad)
    tx = _wide(x, groups, gs)
    full, ctr = _walk(t, tx, gs, mask, "float64", quad)
    c = _control()
    assert int(c[BATCH]) > 0 and int(c[BACK]) == 0  # groups were put back, and all were walked
    again, ctr2 = _walk(t, tx, gs, mask, "float64", quad)
    assert torch.equal(full, again) and torch.equal(ctr, ctr2)
    total = torch.zeros_like(ctr)
    for g in range(0, groups, part):
        few, k = _walk(t, tx[g * gs:(g + part) * gs], gs, mask, "float64", quad)
        c = _control()
        assert int(c[BATCH]) == 0 and int(c[NGROUP]) == part  # all cut, all fit
        assert torch.equal(few, full[g * gs:(g + part) * gs])
        total += k
    assert torch.equal(total, ctr)


@pytest.mark.parametrize("quad,mask,groups,part", [(False, 3, 1100, 100), (True, 6, 2100, 30)])
def test_fp32(quad, mask, groups, part):
    # cuts of a system depend on its number of groups: the calls with few wide groups are filled up with
    # groups far away, each of the same targets
    gs = 256
    t, x = _tree(60_000, quad)
    tx = _wide(x, groups, gs)
    far = np.tile(np.array([400.0, 0.0, 0.0]) + np.random.default_rng(1).standard_normal((gs, 3)), (groups, 1))
    full, ctr = _walk(t, tx, gs, mask, "float32", quad)
    c = _control()
    assert int(c[BATCH]) > 0 and int(c[BACK]) == 0
    again, ctr2 = _walk(t, tx, gs, mask, "float32", quad)
    assert torch.equal(full, again) and torch.equal(ctr, ctr2)
    _, ctr_far = _walk(t, far, gs, mask, "float32", quad)
    total = torch.zeros_like(ctr)
    for g in range(0, groups, part):
        n = min(part, groups - g)
        few, k = _walk(t, np.concatenate([tx[g * gs:(g + n) * gs], far[n * gs:]]), gs, mask, "float32", quad)
        c = _control()
        assert int(c[BATCH]) == 0 and int(c[NGROUP]) == n
        assert torch.equal(few[:n * gs], full[g * gs:(g + n) * gs])
        total += k - (groups - n) * torch.div(ctr_far, groups, rounding_mode="floor")
    assert torch.equal(total, ctr)


def test_binned_columns():
    t, x = _tree(30_000, False)
    gs, groups, part = 64, 2_000, 250
    tx = _wide(x, groups, gs)

    def columns(targets):
        ctr = torch.zeros(2, dtype=torch.int64, device=engine.device())
        return engine.column_binned(t, targets, group_size=gs, theta=0.5, counters=ctr), ctr

    full, ctr = columns(tx)
    again, ctr2 = columns(tx)
    assert torch.equal(full, again) and torch.equal(ctr, ctr2)
    total = torch.zeros_like(ctr)
    for g in range(0, groups, part):
        few, k = columns(tx[g * gs:(g + part) * gs])
        assert torch.equal(few, full[g * gs:(g + part) * gs])
        total += k
    assert torch.equal(total, ctr)


def test_two_streams():
    t, x = _tree(30_000, False)
    tx = _wide(x, 500, 256)
    want = _walk(t, tx, 256, 7, "float64", False)[0]
    want32 = _walk(t, np.tile(tx, (3, 1)), 256, 7, "float32", False)[0]
    t3 = engine.to_dev(np.tile(tx, (3, 1)), (-1, 3))
    t1 = engine.to_dev(tx, (-1, 3))
    h = torch.full((len(t3),), 0.03, dtype=torch.float64, device=engine.device())
    perm = torch.arange(len(t3), dtype=torch.int64, device=engine.device())
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    outs = []
    for s, (p, prec) in zip(streams, ((t1, "float64"), (t3, "float32"))):
        with torch.cuda.stream(s):
            outs.append(engine.walk(t, p, h[:len(p)], perm[:len(p)], 7, group_size=256, theta=0.7, grouping="fixed",
                                    precision=prec, _check=False))
    for s in streams:
        with torch.cuda.stream(s):
            engine.check_walk()
    torch.cuda.synchronize()
    assert torch.equal(outs[0], want) and torch.equal(outs[1], want32)
