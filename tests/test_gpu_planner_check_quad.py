"""The quadcopter's children through the planner's own tiles on caller buffers:
counts around a tile of as many children as lanes (256) and of twice as many,
box counts around the words of the box masks and the largest scene, parents out
of range; bit for bit against the oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.abi import KGMT_CHECK_ONE_PASS
from tests.test_gpu_planner_check import assert_bit_exact, run_planner_check
from tests.test_gpu_parity import CASES, parent_states

pytestmark = pytest.mark.gpu


def _boxes(cfg, boxes, seed):
    span = cfg.ws_max - cfg.ws_min
    if not boxes:
        return np.zeros((0, 6), np.float32)
    return W.random_boxes(np.random.default_rng(seed), boxes, 0.01 * span, 0.05 * span, ws=(cfg.ws_min, cfg.ws_max))


@pytest.mark.parametrize("n", [1, 63, 255, 256, 257, 511, 512, 513, 767, 768, 769, 1280, 3001])
@pytest.mark.parametrize("boxes", [0, 1, 64, 65, 129])
def test_tile_edges(n, boxes, orc):
    print(f"quadcopter planner check n={n} boxes={boxes}", flush=True)
    cfg = CASES["quad12d"]()
    X = parent_states(cfg, 40)
    pidx = np.random.default_rng(n).integers(0, 40, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, n)
    _, chk = assert_bit_exact(cfg, pidx, X, ctrl, steps, _boxes(cfg, boxes, n), orc)
    assert (chk == KGMT_CHECK_ONE_PASS).all()


@pytest.mark.parametrize("boxes", [333, 1500])
def test_large_scenes(boxes, orc):
    cfg = CASES["quad12d"]()
    n = 20000
    X = parent_states(cfg, 700)
    pidx = np.random.default_rng(boxes).integers(0, 700, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 2, 0, n)
    want, _ = assert_bit_exact(cfg, pidx, X, ctrl, steps, _boxes(cfg, boxes, 1), orc)
    assert 0 < want[1].sum() < n


def test_parents_out_of_range(orc):
    cfg = CASES["quad12d"]()
    n, npar = 2000, 50
    X = parent_states(cfg, npar)
    rng = np.random.default_rng(3)
    good = rng.integers(0, npar, n).astype(np.int32)
    bad = rng.random(n) < 0.2
    pidx = np.where(bad, rng.choice([-1, npar, 2**31 - 1, -2**31], n), good).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 2, 0, n)
    obs = _boxes(cfg, 40, 2)
    want = orc.propagate_children(cfg, good, X, ctrl, steps, obs)
    child, valid, r1, r2, _, _ = run_planner_check(cfg, pidx, X, ctrl, steps, obs)
    assert not child[:, bad].any() and not valid[bad].any() and (r1[bad] == -1).all() and (r2[bad] == -1).all()
    assert np.array_equal(child[:, ~bad].view(np.uint32), want[0][:, ~bad].view(np.uint32))
    assert np.array_equal(valid[~bad], want[1][~bad]) and np.array_equal(r1[~bad], want[2][~bad])
    assert np.array_equal(r2[~bad], want[3][~bad])
