"""hx_plan_walk_info: what the walks of a plan keep."""
import ctypes

import pytest

from test_walk4_program import _tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,T,cherries,dropped", [("balanced", 64, 32, 32), ("balanced", 2, 1, 0),
                                                      ("caterpillar", 9, 1, 1), ("balanced", 3, 1, 1)])
def test_dropped_cherries(gpu, shape, T, cherries, dropped):
    """The FP32 walks leave every cherry but the root out of memory."""
    from torchtree_amd import _lib
    from torchtree_amd.likelihood import Plan

    plan = Plan(T, _tree(shape, T), 0)
    out = [ctypes.c_int(-1) for _ in range(5)]
    _lib.check(_lib.load().hx_plan_walk_info(plan.handle, *map(ctypes.byref, out)))
    assert [o.value for o in out[2:]] == [cherries, dropped, dropped]
