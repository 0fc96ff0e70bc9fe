"""kgmt_propagate_collide at counts around one and two turns of its lanes (1024
workgroups of 256 for the quadcopter, 2048 for the other models); bit for bit
against the oracle."""
import numpy as np
import pytest

from tests.test_gpu_edges import CASES, _boxes, _run, _same, parent_states

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case,turn", [("quad12d", 1024 * 256), ("di_ref", 2048 * 256), ("unicycle", 2048 * 256)])
@pytest.mark.parametrize("turns,more", [(1, -1), (1, 0), (1, 1), (2, 0), (2, 1)])
def test_turns_of_the_lanes(case, turn, turns, more, orc):
    n = turns * turn + more
    print(f"{case} edges n={n}", flush=True)
    cfg = CASES[case]().replace(steps_min=1, steps_max=2)
    rng = np.random.default_rng(n)
    X = parent_states(cfg, 900, seed=4)
    pidx = rng.integers(0, 900, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, n)
    obs = _boxes(cfg, 5, rng)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), orc.propagate_children(cfg, pidx, X, ctrl, steps, obs))
