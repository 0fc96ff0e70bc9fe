"""Plans over region grids of every storage class of the region counters: one
region to 8100, and one bit of subregions per region to 250 words; node by
node against the oracle, alone and in one batch."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.planner import KGMT, BatchKGMT
from tests.test_gpu_plan import _same_plan

pytestmark = pytest.mark.gpu

# model, r1_len, r2_len
GRIDS = [
    ("di6d", 1, 1), ("di6d", 1, 20), ("di6d", 2, 3), ("di6d", 2, 4), ("di6d", 3, 5), ("di6d", 5, 6), ("di6d", 20, 1),
    ("unicycle2d", 1, 90), ("unicycle2d", 3, 8), ("unicycle2d", 4, 9), ("unicycle2d", 5, 5), ("unicycle2d", 32, 3),
    ("unicycle2d", 33, 11), ("unicycle2d", 64, 2), ("unicycle2d", 90, 1), ("dubins5d", 17, 2), ("quad12d", 7, 1),
]


def _query(name, r1, r2):
    cap = 2500 if name == "quad12d" else 6000
    return W.make_query(name, r1 + r2, capacity=cap, max_iter=6, r1_len=r1, r2_len=r2)


@pytest.mark.parametrize("name,r1,r2", GRIDS)
def test_region_grid_matches_oracle(name, r1, r2, orc):
    print(f"{name} r1={r1} r2={r2}", flush=True)
    q = _query(name, r1, r2)
    ref = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
    g = KGMT(q.cfg)
    for graph in (False, True, True):
        g.set_graph(graph)
        _same_plan(g, g.plan(q.start, q.goal, q.obstacles, len(q.obstacles)), ref)


@pytest.mark.parametrize("planar", [False, True])
def test_region_grids_in_one_batch_match_oracle(planar, orc):
    qs = [_query(*x) for x in GRIDS if (x[0] == "unicycle2d") == planar]
    b = BatchKGMT([q.cfg for q in qs])
    results, _ = b.plan(*W.pack_batch(qs)[1:])
    for i, q in enumerate(qs):
        ref = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
        st, r = ref["stats"], results[i]
        assert (r.iterations, r.tree_size, r.expanded) == (st["iterations"], st["tree_size"], st["expanded"]), i
        s, p, c = b.tree(i)
        assert np.array_equal(p, ref["parents"]), i
        assert np.array_equal(s.view(np.uint32), ref["samples"].view(np.uint32)), i
