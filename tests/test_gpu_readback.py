"""Paths and trees read back after a plan: paths of one wave's 64 rows and
longer, single and in a batch, and trees of one to many nodes, against the
oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.abi import KGMT_MAX_SAMPLE
from kgmt_amd.planner import KGMT, BatchKGMT

pytestmark = pytest.mark.gpu

EMPTY = np.zeros((0, 6), np.float32)


def _straight(steps, seed):
    """A node flies straight to the goal, one edge of one step an iteration."""
    q = W.make_query("di6d", seed, capacity=8000, max_iter=300)
    start = np.zeros_like(q.start)
    start[:4] = (0.1, 0.1, 0.1, 1.0)
    goal = start.copy()
    goal[0] = 0.9
    zero = [0.0] * 4
    return q.cfg.replace(dt=0.8 / steps, steps_min=1, steps_max=1, children_per_entry=1, root_repeat=1, repeat_sparse=1,
                         ctrl_min=zero, ctrl_max=zero, goal_thresh=0.02, epsilon=0.0, r1_len=20), start, goal


def _padded(samples):
    return np.stack([np.pad(x, (0, KGMT_MAX_SAMPLE - len(x))) for x in samples])


@pytest.mark.parametrize("steps,rows", [(5, 7), (30, 37), (52, 62), (53, 64), (54, 65), (90, 107)])
def test_path_of_any_length_matches_oracle(steps, rows, orc):
    cfgs, starts, goals = zip(*[_straight(steps, seed) for seed in (1, 2, 3)])
    refs = [orc.plan(c, x0, xg, EMPTY) for c, x0, xg in zip(cfgs, starts, goals)]
    assert refs[0]["stats"]["path_rows"] == rows
    print(steps, [r["stats"]["path_rows"] for r in refs], flush=True)
    b = BatchKGMT(cfgs)
    zero = np.zeros(len(cfgs), np.uint32)
    for graph in (False, True):
        results, _ = b.plan(_padded(starts), _padded(goals), EMPTY, zero, zero, use_graph=graph)
        for i, ref in enumerate(refs):
            assert results[i].path_rows == ref["stats"]["path_rows"], i
            assert np.array_equal(b.path(i).view(np.uint32), ref["path"].view(np.uint32)), i
            assert np.float32(results[i].path_cost) == np.float32(ref["stats"]["path_cost"])
            assert np.float32(results[i].path_length) == np.float32(ref["stats"]["path_length"])
    g = KGMT(cfgs[0])
    g.plan(starts[0], goals[0], EMPTY, 0)
    assert np.array_equal(g.path().view(np.uint32), refs[0]["path"].view(np.uint32))


@pytest.mark.parametrize("name,cap", [("unicycle2d", 300), ("dubins5d", 257), ("quad12d", 1000), ("di6d", 9000)])
def test_tree_rows_match_oracle(name, cap, orc):
    q = W.make_query(name, 4, capacity=cap, max_iter=4)
    ref = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
    g = KGMT(q.cfg)
    g.plan_begin(q.start, q.goal, q.obstacles, len(q.obstacles))
    s, p, c = g.tree()  # the root
    assert s.shape[0] == 1 and p[0] == -1
    while not g.plan_step():
        g.tree()  # leaves the plan in progress as it is
    s, p, c = g.tree()
    assert np.array_equal(s.view(np.uint32), ref["samples"].view(np.uint32))
    assert np.array_equal(p, ref["parents"]) and np.array_equal(c.view(np.uint32), ref["costs"].view(np.uint32))
