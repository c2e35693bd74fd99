"""Workspaces sized for n particles serve fewer: the sizes do not fall as n grows (the key sort's tiles get longer
at some numbers of keys).  Sizes only, no GPU."""

import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.skipif(not os.path.exists(os.path.join(ROOT, "pytreegrav_amd", "libptg_hip.so")),
                                reason="libptg_hip.so not built")

SIZES = sorted({max(1, (1 << k) + d) for k in (0, 4, 8, 12, 15, 16, 17, 18, 19, 20, 21, 22, 24)
                for d in (-300, -1, 0, 1, 2, 300)})


@pytest.mark.parametrize("name,args", [("ptg_build_workspace_bytes", (1,)), ("ptg_build_workspace_bytes", (128,)),
                                       ("ptg_groups_workspace_bytes", (1,)), ("ptg_groups_workspace_bytes", (128,)),
                                       ("ptg_ray_orders_workspace_bytes", (1,)), ("ptg_ray_orders_workspace_bytes", (3,))])
def test_sizes_grow_with_n(name, args):
    from pytreegrav_amd import _lib

    f = getattr(_lib.load(), name)
    got = [f(n, *args) for n in SIZES]
    assert got == sorted(got), [n for n, a, b in zip(SIZES[1:], got, got[1:]) if b < a]
