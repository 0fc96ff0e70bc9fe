"""Quadcopter steps over a sweep of speeds, rates and angles under a drag and a
damping that make the roots and the quotients the state's largest terms: where
the step's short forms do not round as the plain operations do, the state's
bits show it. Against the oracle, one step an edge."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from tests.test_gpu_edges import _run, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", range(4))
def test_steps_over_a_sweep_match_oracle(seed, orc):
    n = 250000
    print(f"quadcopter short forms, seed {seed}: {n} steps", flush=True)
    rng = np.random.default_rng(seed)
    cfg = W.config("quad12d", dt=0.25, steps_min=1, steps_max=1, quad_nu=1.0, quad_mu=1.0, quad_ix=1.0, quad_iy=1.0,
                   quad_iz=1.0, v_min=-1e30, v_max=1e30, ws_min=-1e6, ws_max=1e6)
    X = np.zeros((12, n), np.float32)
    k = np.arange(n)
    # angles in even strides, speeds and rates over six binades each
    X[3] = (k * 0.61803398875 % 1.0 - 0.5) * 6.0
    X[4] = (k * 0.41421356237 % 1.0 - 0.5) * 3.1
    X[5] = (k * 0.73205080757 % 1.0 - 0.5) * 6.0
    X[6:] = rng.choice([-1.0, 1.0], (6, n)) * np.exp2(rng.uniform(-4.0, 2.0, (6, n)))
    ctrl = np.zeros((4, n), np.float32)
    ctrl[0] = rng.uniform(0.0, 19.0, n)
    ctrl[1:] = rng.uniform(-1.0, 1.0, (3, n))
    pidx, steps = np.arange(n, dtype=np.int32), np.ones(n, np.int32)
    obs = np.zeros((0, 6), np.float32)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), orc.propagate_children(cfg, pidx, X, ctrl, steps, obs))


@pytest.mark.parametrize("group", [64, 4096])
def test_largest_cosines_below_one(group, orc):
    """A pitch whose cosine is the float below 1 and its neighbours, by exact
    powers of two: the quotient of the one divisor whose reciprocal's
    refinement can stop at a tie. Few edges (a quad of lanes each) and many."""
    th = np.unique(np.float32(np.linspace(1e-5, 9e-4, 4096)))
    n = len(th) // group * group
    rng = np.random.default_rng(group)
    cfg = W.config("quad12d", dt=0.25, steps_min=1, steps_max=1, quad_nu=0.0, quad_mu=0.0, v_min=-1e30, v_max=1e30,
                   ws_min=-1e6, ws_max=1e6)
    X = np.zeros((12, n), np.float32)
    X[4] = th[:n]
    X[6:9] = 1.0
    X[9:11] = 0.5
    X[11] = np.ldexp(1.0, rng.integers(-20, 4, n)) * rng.choice([-1.0, 1.0], n)  # the yaw rate's quotient by cos theta
    ctrl = np.zeros((4, n), np.float32)
    steps, obs = np.ones(group, np.int32), np.zeros((0, 6), np.float32)
    for k in range(0, n, group):
        pidx = np.arange(k, k + group, dtype=np.int32)
        c = np.ascontiguousarray(ctrl[:, k:k + group])
        _same(_run(cfg, pidx, X, c, steps, obs), orc.propagate_children(cfg, pidx, X, c, steps, obs))
