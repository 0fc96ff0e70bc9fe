"""kgmt_get_frontier's size query and its two outputs, each alone and together,
before a plan, between steps and after plans that end early."""
import ctypes as C

import numpy as np
import pytest

from kgmt_amd import _lib
from kgmt_amd import workloads as W
from kgmt_amd.planner import KGMT, _ptr

pytestmark = pytest.mark.gpu


def _read(g, flags, counts, cap):
    n = C.c_uint32(0xFFFFFFFF)
    f, r = np.full(cap, 99, np.uint8), np.full(cap, 99, np.uint32)
    rc = _lib.lib().kgmt_get_frontier(g._h, _ptr(f) if flags else None, _ptr(r) if counts else None, cap, C.byref(n))
    return rc, n.value, f, r


@pytest.mark.parametrize("name", ["di6d", "dubins5d", "quad12d", "unicycle2d"])
def test_frontier_outputs(name):
    q = W.make_query(name, 4, capacity=20000, max_iter=8)
    g = KGMT(q.cfg)
    assert _read(g, False, False, 0)[:2] == (0, 0)

    def check(size):
        f, r = g.frontier()
        assert len(f) == size == len(r)
        rc, n, a, b = _read(g, True, False, size)
        assert (rc, n) == (0, size) and np.array_equal(a, f) and (b == 99).all()
        rc, n, a, b = _read(g, False, True, size)
        assert (rc, n) == (0, size) and np.array_equal(b, r) and (a == 99).all()
        assert _read(g, True, True, size - 1)[0] != 0

    g.plan_begin(q.start, q.goal, q.obstacles, len(q.obstacles))
    check(1)
    while not g.plan_step():
        check(g.h_treeSize_)
    check(g.h_treeSize_)
    last = g.frontier()
    res = g.plan(q.start, q.goal, q.obstacles, len(q.obstacles))
    check(res.tree_size)
    assert all(np.array_equal(x, y) for x, y in zip(last, g.frontier()))
