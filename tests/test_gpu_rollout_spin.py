"""Rollouts that turn fast: a stage's angles advance by less and by more than
0.1 rad, the bound between turned and recomputed sines, alone and side by side
in one wave; against the oracle's FP64 cost and adjoint."""
import numpy as np
import pytest
import torch

from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W

pytestmark = pytest.mark.gpu

# the bounds of the parity tests of this entry
RTOL = 1e-4
TURNS = [0.0, 0.05, 0.0999, 0.1, 0.1001, 0.199, 0.2001, 0.5, 1.0, 2.0]  # of a whole step


@pytest.mark.parametrize("n", [len(TURNS), 1100, 2200])
@pytest.mark.parametrize("mixed", [False, True])
def test_fast_turns_match_fp64(n, mixed, orc):
    print(f"turns: n={n} mixed={mixed}", flush=True)
    rng = np.random.default_rng(n)
    cfg = W.config("quad12d", dt=0.02)
    ap = W.refine_params(cfg, "hover")
    T = 12
    x0 = np.zeros((12, n), np.float32)
    x0[:3] = rng.uniform(0.3, 0.7, (3, n))
    x0[3:6] = rng.uniform(-0.4, 0.4, (3, n))
    x0[6:9] = rng.uniform(-0.3, 0.3, (3, n))
    turn = np.array(TURNS)[np.arange(n) % len(TURNS) if mixed else np.arange(n) * len(TURNS) // n]
    x0[9] = turn / cfg.dt * rng.choice([-1.0, 1.0], n)  # a roll: pitch stays small
    x0[10:] = rng.uniform(-0.2, 0.2, (2, n))
    goal = rng.uniform(0.3, 0.7, (3, n)).astype(np.float32)
    steps = rng.integers(1, T + 1, n).astype(np.int32)
    u = np.zeros((T, 4, n), np.float32)
    u[:, 0] = rng.uniform(5.0, 15.0, (T, n))
    u[:, 1:] = rng.normal(0.0, 0.005, (T, 3, n))
    boxes = W.random_boxes(rng, 20, 0.02, 0.08)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    cost, grad = A.cost_and_grad(d(u), d(x0), d(goal), d(steps), d(boxes), cfg, ap)
    cost, grad = cost.cpu().numpy(), grad.cpu().numpy()
    for k in sorted({*range(len(TURNS)), n - 1, *(int(i) for i in rng.integers(0, n, 40))}):
        t = int(steps[k])
        J, g = orc.traj_grad_f64(cfg, ap, x0[:, k], u[:t, :, k], goal[:, k], boxes)
        assert abs(cost[k] - J) <= RTOL * max(1.0, abs(J)), (k, turn[k], t, cost[k], J)
        assert np.abs(grad[:t, :, k] - g).max() <= RTOL * max(1.0, np.abs(g).max()), (k, turn[k], t)
        assert not grad[t:, :, k].any()
