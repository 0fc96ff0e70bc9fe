"""Batches around the sizes where the work lists change hands (one query, up to
256, more), with queries that end in different iterations, every workgroup size
and grids smaller than the work; query by query against the oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.planner import BatchKGMT

pytestmark = pytest.mark.gpu


def _queries(n):
    names = ["di6d", "dubins5d", "quad12d"]
    return [W.make_query(names[k % 3], k % 7, capacity=300 + 61 * (k % 29), max_iter=1 + k % 5, children_per_entry=4)
            for k in range(n)]


@pytest.fixture(scope="module")
def wanted(orc):
    refs = {}

    def get(k, q):
        key = (k % 3, k % 7, k % 29, k % 5)
        if key not in refs:
            refs[key] = orc.plan(q.cfg, q.start, q.goal, q.obstacles)
        return refs[key]

    return get


@pytest.mark.parametrize("n,launch", [
    (1, {}), (2, {}), (63, {}), (64, dict(propagate_block=128)), (65, dict(propagate_block=512)),
    (129, dict(propagate_grid=3, chunk_grid=2)), (255, {}), (256, {}), (257, {}), (300, dict(chunk_grid=5)),
])
def test_batch_of_any_size_matches_oracle(n, launch, wanted):
    print(f"{n} queries {launch}", flush=True)
    qs = _queries(n)
    b = BatchKGMT([q.cfg for q in qs])
    b.set_launch(**launch)
    for graph in (False, True):
        results, _ = b.plan(*W.pack_batch(qs)[1:], use_graph=graph)
        for k, q in enumerate(qs):
            st, r = wanted(k, q)["stats"], results[k]
            assert (r.iterations, r.tree_size, r.expanded) == (st["iterations"], st["tree_size"], st["expanded"]), k
            assert (r.goal_index if r.success else -1) == st["goal_index"], k
        for k in range(0, n, 1 + n // 20):
            s, p, c = b.tree(k)
            assert np.array_equal(p, wanted(k, qs[k])["parents"]), k
            assert np.array_equal(s.view(np.uint32), wanted(k, qs[k])["samples"].view(np.uint32)), k
