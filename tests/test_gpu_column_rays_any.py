"""Ray-traced columns of shared rays where bundles cannot give them: rays that are not of unit length, and trees
all of whose nodes are opened, past the bundles' stack.  The same bits as the targets' own walks (which
test_gpu_column.py compares with the oracle)."""

import numpy as np
import pytest
import torch

from pytreegrav_amd import ConstructTree, _lib, engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [40, 300])
def test_rays_of_other_lengths(nt):
    rng = np.random.default_rng(2)
    x, h = rng.normal(size=(3000, 3)), rng.uniform(0.05, 0.3, 3000)
    u = rng.normal(size=(6, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    u[0] *= 2.0
    u[1] *= 0.5
    u[2] = u[2].astype(np.float32)  # of unit length to 1e-7
    u[3] = 0.0
    t = rng.normal(size=(nt, 3))
    tree = ConstructTree(x, np.ones(3000), h).dev
    own = engine.column_rays(tree, t, u, counters=torch.zeros(1, dtype=torch.int64, device=engine.device()))
    assert torch.equal(engine.column_rays(tree, t, u), own)
    for i in range(4):
        assert torch.equal(engine.column_rays(tree, t, u[i:i + 1]), own[:, i:i + 1])


def test_every_node_opened():
    # radii of the whole domain: the children of 64 elements a step pass the bundles' 1024 entries
    rng = np.random.default_rng(4)
    n = 300_000
    tree = ConstructTree(rng.uniform(size=(n, 3)), np.ones(n), np.full(n, 2.0)).dev
    t, rays = rng.uniform(size=(70, 3)), np.array([[0.0, 0.0, 1.0], [0.6, 0.0, 0.8]])
    out = torch.empty((70, 2), dtype=torch.float64, device=engine.device())
    err = torch.zeros(1, dtype=torch.int32, device=engine.device())
    td, rd = engine.to_dev(t, (-1, 3)), engine.to_dev(rays)
    engine.check(_lib.load().ptg_column_bundles(_lib.ctypes.byref(tree.pack(_lib.PTG_F64, False)["wt"]), _lib.ptr(td), 70,
                                                _lib.ptr(rd), 2, None, _lib.ptr(out), _lib.ptr(err), engine.stream()),
                 "ptg_column_bundles")
    assert int(err) == 2
    own = engine.column_rays(tree, t, rays, counters=torch.zeros(1, dtype=torch.int64, device=engine.device()))
    assert torch.equal(engine.column_rays(tree, t, rays), own)
