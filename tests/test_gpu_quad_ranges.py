"""Quadcopter edges from states at the ends of the ranges where the step's
quotients and roots take the short form: rates, speeds and angles of zero, just
below, at and above the bound, cosines near zero, huge and non-finite ones; one
wave of one such state, and all of them mixed; bit for bit against the oracle."""
import numpy as np
import pytest

from kgmt_amd import workloads as W
from tests.test_gpu_edges import _run, _same

pytestmark = pytest.mark.gpu

# of an angle, a velocity or a rate; the bound is 2^-40 for an operand, so
# 2^-20 for a component under a root
VALUES = [0.0, -0.0, 1e-38, 2.0**-40, 2.0**-40 * (1 + 2.0**-23), 2.0**-41, 2.0**-20, -(2.0**-21), 1e-3, 1.5, np.pi / 2,
          -1.5707964, 1.5707963, 3.1415927, 100.0, 12868.0, 1e5, 2.0**61, -1e19, 3e38, np.inf, np.nan]


def _states(seed):
    """One parent per value and component of angles, velocity and rates."""
    rng = np.random.default_rng(seed)
    base = rng.uniform(-0.6, 0.6, (12, 9 * len(VALUES))).astype(np.float32)
    base[:3] = 0.5
    for k, v in enumerate(VALUES):
        for c in range(9):
            base[3 + c, 9 * k + c] = v
    return base


@pytest.mark.parametrize("per", [1, 4, 64, 200])
@pytest.mark.parametrize("rest", [False, True])
def test_quadcopter_ranges_match_oracle(per, rest, orc):
    print(f"quadcopter ranges: {per} children a state, at rest {rest}", flush=True)
    cfg = W.config("quad12d", steps_min=3, steps_max=12)
    X = _states(per)
    if rest:
        X[6:] = np.where(np.isin(np.abs(X[6:]), np.abs(np.float32(VALUES))), X[6:], 0.0)
    npar = X.shape[1]
    pidx = np.repeat(np.arange(npar, dtype=np.int32), per)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, len(pidx))
    obs = W.random_boxes(np.random.default_rng(2), 40, 0.02, 0.1)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), orc.propagate_children(cfg, pidx, X, ctrl, steps, obs))
