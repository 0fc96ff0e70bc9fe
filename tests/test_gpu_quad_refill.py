"""Quadcopter tiles of two children per lane, whose children start in the order
of their steps: a batch large enough that a few thousand children reach them,
with every range of steps, workgroup size and odd counts; against the oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.planner import BatchKGMT

pytestmark = pytest.mark.gpu

LARGE = [
    dict(capacity=9000, max_iter=4),
    dict(capacity=8191, max_iter=5, steps_min=1, steps_max=1),
    dict(capacity=5003, max_iter=5, steps_min=1, steps_max=3, children_per_entry=7),
    dict(capacity=7000, max_iter=4, dt=0.002, steps_min=3, steps_max=299),
    dict(capacity=4100, max_iter=6, root_repeat=100, children_per_entry=1000),
]


@pytest.mark.parametrize("launch", [{}, dict(propagate_block=128), dict(propagate_block=512),
                                    dict(propagate_grid=2), dict(lanes_per_child=2, propagate_block=256)])
def test_two_children_per_lane_match_oracle(launch, orc):
    print(f"quadcopter batch {launch}", flush=True)
    qs = [W.make_query("quad12d", k, **(LARGE[k // 13] if k % 13 == 0 else dict(capacity=40, max_iter=2)))
          for k in range(13 * len(LARGE))]
    b = BatchKGMT([q.cfg for q in qs])
    b.set_launch(**launch)
    results, _ = b.plan(*W.pack_batch(qs)[1:])
    for k in range(0, len(qs), 13):
        q = qs[k]
        ref = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
        st, r = ref["stats"], results[k]
        assert (r.iterations, r.tree_size, r.expanded) == (st["iterations"], st["tree_size"], st["expanded"]), k
        s, p, c = b.tree(k)
        assert np.array_equal(p, ref["parents"]), k
        assert np.array_equal(s.view(np.uint32), ref["samples"].view(np.uint32)), k
