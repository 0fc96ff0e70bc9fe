"""A launch shape set while a step-by-step plan is in progress: the plan keeps
the shape that its scene and tiles were made for, the next one takes the new."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd._lib import KgmtError
from kgmt_amd.planner import KGMT
from tests.test_gpu_plan import _same_plan

pytestmark = pytest.mark.gpu

SHAPES = [dict(propagate_block=512, lanes_per_child=1), dict(propagate_block=256, lanes_per_child=4),
          dict(propagate_block=256, lanes_per_child=2), dict(propagate_block=128, lanes_per_child=1)]


def _finish(g, after=None):
    done = False
    while not done:
        done = g.plan_step()
        if after is not None:
            g.set_launch(**after)
    return g


@pytest.mark.parametrize("name,boxes", [("quad12d", 0), ("quad12d", 50), ("quad12d", 1500), ("dubins5d", 100)])
@pytest.mark.parametrize("first,then", [(1, 0), (2, 0), (2, 3), (0, 1), (0, 3), (3, 2)])
def test_shape_set_between_steps(name, boxes, first, then, orc):
    print(f"{name} boxes={boxes} {SHAPES[first]} then {SHAPES[then]}", flush=True)
    q = W.make_query(name, 3, capacity=3000, max_iter=4)
    obs = W.random_boxes(np.random.default_rng(boxes), boxes, 0.02, 0.05, [(q.start[:3], 0.06)]) if boxes else \
        np.zeros((0, 6), np.float32)
    ref = orc.plan(q.cfg, q.start, q.goal, obs)
    g = KGMT(q.cfg)
    g.set_launch(**SHAPES[first])
    g.plan_begin(q.start, q.goal, obs, len(obs))
    g.set_launch(**SHAPES[then])
    _finish(g, SHAPES[then])
    _same_tree(g, ref)
    # the next plans run in the shape set last
    _same_plan(g, g.plan(q.start, q.goal, obs, len(obs)), ref)
    g.plan_begin(q.start, q.goal, obs, len(obs))
    _same_tree(_finish(g), ref)


def test_refused_calls_leave_a_plan_in_progress(orc):
    q = W.make_query("quad12d", 3, capacity=3000, max_iter=4)
    ref = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
    g = KGMT(q.cfg)
    g.set_launch(**SHAPES[1])
    g.plan_begin(q.start, q.goal, q.obstacles, len(q.obstacles))
    g.set_launch(**SHAPES[0])
    many = np.tile(q.obstacles, (40, 1))
    with pytest.raises(KgmtError):
        g.plan(q.start, q.goal, many, len(many))
    _same_tree(_finish(g), ref)


def _same_tree(g, ref):
    s, p, c = g.tree()
    assert np.array_equal(p, ref["parents"])
    assert np.array_equal(s.view(np.uint32), ref["samples"].view(np.uint32))
    assert np.array_equal(c.view(np.uint32), ref["costs"].view(np.uint32))
