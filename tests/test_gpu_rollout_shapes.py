"""The differentiable rollout at the sizes where its work splits change:
trajectory counts around one, two and four trajectories per wave, lengths
around the rounds of 4, 8 and 16 steps (and zero), box counts around the
lanes that share them, a work space of several launches; against the oracle's
FP64 cost and adjoint."""
import numpy as np
import pytest
import torch

from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W

pytestmark = pytest.mark.gpu

# FP32 cost within 1e-4 relative, gradient within 1e-4 of the trajectory's
# largest component (and of 1.0): the bounds of the parity tests of this entry
RTOL = 1e-4


def _check(orc, rb, boxes, ks, maxT):
    T, n = rb.u.shape[0], rb.u.shape[2]
    u = np.zeros((maxT, 4, n), np.float32)
    u[:T] = rb.u
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    cost, grad = A.cost_and_grad(d(u), d(rb.x0), d(rb.goal), d(rb.steps), d(boxes), rb.cfg, rb.params)
    cost, grad = cost.cpu().numpy(), grad.cpu().numpy()
    for i in ks:
        t = int(rb.steps[i])
        assert np.all(grad[t:, :, i] == 0.0), i
        if t == 0:
            J = rb.params.w_goal * float(((rb.x0[:3, i] - rb.goal[:, i]).astype(np.float64) ** 2).sum())
            assert abs(cost[i] - J) <= RTOL * max(1.0, J), i
            continue
        J, g = orc.traj_grad_f64(rb.cfg, rb.params, rb.x0[:, i], rb.u[:t, :, i], rb.goal[:, i], boxes)
        assert abs(cost[i] - J) <= RTOL * max(1.0, abs(J)), (i, t, cost[i], J)
        assert np.abs(grad[:t, :, i] - g).max() <= RTOL * max(1.0, np.abs(g).max()), (i, t)


@pytest.mark.parametrize("n,boxes", [(1, 0), (1, 1), (3, 64), (63, 65), (1024, 5), (1025, 31), (2048, 33), (2049, 15),
                                     (4099, 17)])
def test_split_edges_match_fp64(n, boxes, orc):
    print(f"rollout n={n} boxes={boxes}", flush=True)
    rb = W.make_refine_batch(n, seed=n, objective="hover")
    lengths = np.array([0, 1, 2, 3, 4, 5, 7, 8, 9, 15, 16, 17, 31, 33, 63, 64, 65, 80], np.int32)
    rb.steps = np.minimum(lengths[np.arange(n) % len(lengths)] if n > 1 else np.array([17], np.int32),
                          rb.u.shape[0]).astype(np.int32)
    rng = np.random.default_rng(n)
    b = W.random_boxes(rng, boxes, 0.02, 0.2) if boxes else np.zeros((0, 6), np.float32)
    ks = sorted({0, n - 1, n // 2, *(int(k) for k in rng.integers(0, n, 24))})
    _check(orc, rb, b, ks, rb.u.shape[0])


def test_several_launches_match_fp64(orc):
    # 5000 trajectories of up to 1200 steps: more work space than one launch takes
    n = 5000
    print("rollout in several launches", flush=True)
    rb = W.make_refine_batch(n, seed=7, objective="hover", steps_lo=1, steps_hi=9)
    b = W.random_boxes(np.random.default_rng(7), 9, 0.02, 0.2)
    _check(orc, rb, b, [0, 1, 4223, 4224, 4287, 4288, 4289, 4303, 4304, 4351, 4352, n - 1], 1200)


def test_refine_in_lanes_of_each_split_agree():
    """The same trajectories refined alone and among others (other lanes per
    trajectory) take the same steps."""
    rb = W.make_refine_batch(2100, seed=4, objective="hover", steps_lo=3, steps_hi=21)
    rb.params.iterations = 6
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    got = []
    for n in (2100, 1500, 40):
        u = d(rb.u[:, :, :n])
        h = A.refine(u, d(rb.x0[:, :n]), d(rb.goal[:, :n]), d(rb.steps[:n]), d(rb.obstacles), rb.cfg, rb.params)
        got.append((u[:, :, :40].cpu().numpy(), h[:, :40].cpu().numpy()))
    for u, h in got[1:]:
        # six steps of at most lr 1e-2 each; the splits differ by rounding
        assert np.abs(u - got[0][0]).max() <= 1e-3
        assert np.abs(h - got[0][1]).max() <= RTOL * np.maximum(1.0, np.abs(got[0][1])).max()
