"""Quadcopter plans at the sizes where a tile's work changes hands: few and
many children, edges of one step and of hundreds, box counts around the words
of the box masks, unusual boxes, every workgroup size; node by node against
the oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.planner import KGMT, BatchKGMT
from tests.test_gpu_plan import _odd_boxes, _same_plan

pytestmark = pytest.mark.gpu

CASES = [
    (0, dict(capacity=3000, max_iter=6), {}),
    (1, dict(capacity=700, max_iter=5, root_repeat=1), {}),
    (63, dict(capacity=5000, max_iter=5, children_per_entry=1, root_repeat=100), {}),
    (64, dict(capacity=5000, max_iter=6, steps_min=1, steps_max=1), {}),
    (65, dict(capacity=5000, max_iter=5, children_per_entry=33), dict(propagate_block=128)),
    (128, dict(capacity=5000, max_iter=5), dict(propagate_block=512)),
    (129, dict(capacity=4000, max_iter=4, dt=0.002, steps_min=100, steps_max=300), {}),
    (300, dict(capacity=6000, max_iter=5, children_per_entry=1000, root_repeat=2), dict(propagate_block=128)),
    (1300, dict(capacity=3000, max_iter=4), dict(propagate_block=512, propagate_grid=3)),
    (200, dict(capacity=4000, max_iter=5), dict(lanes_per_child=2, propagate_block=256)),
    (200, dict(capacity=4000, max_iter=5), dict(lanes_per_child=4, propagate_block=256)),
    (90, dict(capacity=6000, max_iter=6), dict(propagate_grid=2)),
]


@pytest.mark.parametrize("boxes,kw,launch", CASES)
def test_quadcopter_tiles_match_oracle(boxes, kw, launch, orc):
    print(f"quadcopter boxes={boxes} {kw} {launch}", flush=True)
    q = W.make_query("quad12d", 3, **kw)
    rng = np.random.default_rng(boxes)
    obs = W.random_boxes(rng, boxes, 0.02, 0.08, [(q.start[:3], 0.06)]) if boxes else np.zeros((0, 6), np.float32)
    ref = orc.plan(q.cfg, q.start, q.goal, obs)
    g = KGMT(q.cfg)
    g.set_launch(**launch)
    for _ in range(2):
        res = g.plan(q.start, q.goal, obs, len(obs))
        _same_plan(g, res, ref)


def test_unusual_boxes_match_oracle(orc):
    q = W.make_query("quad12d", 7, capacity=8000, max_iter=6)
    obs = _odd_boxes(3, np.random.default_rng(21))
    ref = orc.plan(q.cfg, q.start, q.goal, obs)
    g = KGMT(q.cfg)
    _same_plan(g, g.plan(q.start, q.goal, obs, len(obs)), ref)
    assert ref["stats"]["tree_size"] > 50


def test_large_workspace_matches_oracle(orc):
    """The reference's own configuration: a workspace of 100 units."""
    cfg = W.config("reference_quad", capacity=6000, max_iter=6, seed=5)
    rng = np.random.default_rng(8)
    start, goal = np.zeros(17, np.float32), np.zeros(17, np.float32)
    start[:3], goal[:3] = (10, 8, 5), (80, 95, 90)
    obs = W.random_boxes(rng, 150, 2.0, 9.0, [(start[:3], 6.0)], ws=(0.0, 100.0))
    ref = orc.plan(cfg, start, goal, obs)
    g = KGMT(cfg)
    _same_plan(g, g.plan(start, goal, obs, len(obs)), ref)


def test_mixed_tiles_in_one_workgroup_match_oracle(orc):
    """Few workgroups take the tiles of every model in turn."""
    qs = []
    for k, name in enumerate(["quad12d", "di6d", "quad12d", "dubins5d", "di6d", "quad12d"]):
        q = W.make_query(name, 20 + k, capacity=3000 + 500 * k, max_iter=5)
        qs.append(q)
    b = BatchKGMT([x.cfg for x in qs])
    b.set_launch(propagate_grid=3, chunk_grid=5)
    for graph in (False, True):
        results, _ = b.plan(*W.pack_batch(qs)[1:], use_graph=graph)
        for i, x in enumerate(qs):
            ref = orc.plan(x.cfg, x.start, x.goal, x.obstacles)
            st, r = ref["stats"], results[i]
            assert (r.iterations, r.tree_size, r.expanded) == (st["iterations"], st["tree_size"], st["expanded"]), i
            s, p, c = b.tree(i)
            assert np.array_equal(p, ref["parents"]), i
            assert np.array_equal(s.view(np.uint32), ref["samples"].view(np.uint32)), i
