"""Boxes at the ends of the range in the differentiable rollout: rows so far
away that the squared distance overflows (padding rows), faces so near that it
underflows, and boxes without end."""
import numpy as np
import pytest
import torch

from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W

pytestmark = pytest.mark.gpu

# the bounds of the parity tests of this entry
RTOL = 1e-4


def _d(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def _grad(rb, boxes, u=None):
    c, g = A.cost_and_grad(_d(rb.u if u is None else u), _d(rb.x0), _d(rb.goal), _d(rb.steps),
                           _d(np.asarray(boxes, np.float32)), rb.cfg, rb.params)
    return c.cpu().numpy(), g.cpu().numpy()


def _far(v):
    v = np.float32(v)
    return np.array([[v, v, v, v, v, v], [-v, -v, -v, -v, -v, -v], [v, 0, 0, v, 1, 1], [0, 0, -v, 1, 1, -v]], np.float32)


@pytest.mark.parametrize("v", [1e18, 2e19, 1e20, 1e30, 3.4028235e38])
@pytest.mark.parametrize("n,boxes", [(5, 0), (70, 50), (2100, 7), (70, 1490)])
def test_far_boxes_add_nothing(v, n, boxes, orc):
    """Rows past the scene, as a caller pads it: no penalty, no gradient."""
    print(f"far boxes at {v}: n={n} boxes={boxes}", flush=True)
    rb = W.make_refine_batch(n, seed=boxes, objective="hover", steps_lo=1, steps_hi=9)
    b = W.random_boxes(np.random.default_rng(3), boxes, 0.02, 0.1) if boxes else np.zeros((0, 6), np.float32)
    want, got = _grad(rb, b), _grad(rb, np.concatenate([b, _far(v)]))
    assert np.isfinite(got[0]).all() and np.isfinite(got[1]).all()
    # a row at the end adds zeros to the sums
    assert np.array_equal(want[0], got[0]) and np.array_equal(want[1], got[1])
    k, t = 1, int(rb.steps[1])
    J, g = orc.traj_grad_f64(rb.cfg, rb.params, rb.x0[:, k], rb.u[:t, :, k], rb.goal[:, k],
                             np.concatenate([b, _far(v)]))
    assert abs(got[0][k] - J) <= RTOL * max(1.0, abs(J))
    assert np.abs(got[1][:t, :, k] - g).max() <= RTOL * max(1.0, np.abs(g).max())


def test_boxes_without_end_cost_nothing():
    """(their gradient is 0 / 0, as the quotient of two infinities gives it)"""
    rb = W.make_refine_batch(70, seed=2, objective="hover", steps_lo=1, steps_hi=9)
    inf = np.full((1, 6), np.inf, np.float32)
    want, got = _grad(rb, rb.obstacles), _grad(rb, np.concatenate([rb.obstacles, inf]))
    assert np.array_equal(want[0], got[0])


@pytest.mark.parametrize("n", [3, 70])
def test_refine_keeps_controls_finite_among_far_boxes(n):
    rb = W.make_refine_batch(n, seed=5, objective="hover", steps_lo=1, steps_hi=9)
    rb.params.iterations = 4
    out = []
    for b in (rb.obstacles, np.concatenate([rb.obstacles, _far(1e20)])):
        u = _d(rb.u)
        h = A.refine(u, _d(rb.x0), _d(rb.goal), _d(rb.steps), _d(b), rb.cfg, rb.params)
        out.append((u.cpu().numpy(), h.cpu().numpy()))
    assert np.isfinite(out[1][0]).all() and np.isfinite(out[1][1]).all()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("gap", [1e-25, 1e-22, 1e-20, 1e-19, 1.1e-19, 1e-18, 1e-10])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("low", [True, False])
def test_faces_at_a_hair_from_the_position(gap, axis, low, orc):
    """A face at 0 (as a box clipped to the workspace has) and a position at
    rest just outside it, beside positions at other distances."""
    print(f"gap {gap} axis {axis} low {low}", flush=True)
    cfg = W.config("quad12d", dt=0.1, gravity=0.0)
    ap = W.refine_params(cfg, "hover")
    ap.w_effort, ap.w_goal, ap.w_obstacle, ap.margin, ap.tau = 0.0, 0.0, 1.0, 0.02, 0.01
    n = 70
    x0 = np.zeros((12, n), np.float32)
    x0[3:6] = np.array([[0.3], [-0.4], [0.7]])  # the thrust has a part on every axis
    x0[:3] = 0.05
    x0[axis] = np.where(np.arange(n) % 3 == 0, gap, 0.01 * np.arange(n)) * (-1.0 if low else 1.0)
    box = np.array([[0.0, 0.0, 0.0, 0.1, 0.1, 0.1]], np.float32)
    if not low:
        box = np.array([[0.0, 0.0, 0.0, 0.1, 0.1, 0.1]], np.float32)
        box[0, axis], box[0, 3 + axis] = -0.1, 0.0
    u, goal, steps = np.zeros((1, 4, n), np.float32), np.zeros((3, n), np.float32), np.ones(n, np.int32)
    c, g = A.cost_and_grad(_d(u), _d(x0), _d(goal), _d(steps), _d(box), cfg, ap)
    c, g = c.cpu().numpy(), g.cpu().numpy()
    for k in range(n):
        J, w = orc.traj_grad_f64(cfg, ap, x0[:, k], u[:, :, k], goal[:, k], box)
        assert abs(c[k] - J) <= RTOL * max(J, 1e-30), (k, c[k], J)
        assert np.abs(g[:, :, k] - w).max() <= RTOL * np.abs(w).max(), (k, g[:, :, k], w)


def _one_box(z, tau, margin, orc):
    """(cost, gradient, 64-bit cost, 64-bit gradient, position) of trajectories
    at rest above the face z = 0 of one box, the thrust along z."""
    cfg = W.config("quad12d", dt=0.1, gravity=0.0)
    ap = W.refine_params(cfg, "hover")
    ap.w_effort, ap.w_goal, ap.w_obstacle, ap.margin, ap.tau = 0.0, 0.0, 1.0, margin, tau
    n = len(z)
    x0 = np.zeros((12, n), np.float32)
    x0[2] = z
    box = np.array([[-1.0, -1.0, -1.0, 1.0, 1.0, 0.0]], np.float32)
    u, goal, steps = np.zeros((1, 4, n), np.float32), np.zeros((3, n), np.float32), np.ones(n, np.int32)
    c, g = A.cost_and_grad(_d(u), _d(x0), _d(goal), _d(steps), _d(box), cfg, ap)
    J, w = np.zeros(n), np.zeros(n)
    for k in range(n):
        J[k], e = orc.traj_grad_f64(cfg, ap, x0[:, k], u[:, :, k], goal[:, k], box)
        w[k] = e[0, 0]
    return c.cpu().numpy().astype(np.float64), g.cpu().numpy()[0, 0].astype(np.float64), J, w, x0[2].astype(np.float64)


@pytest.mark.parametrize("tau", [0.5, 0.05, 0.01, 0.002])
def test_one_box_to_the_last_bits(tau, orc):
    """The distance is the position: exact but for the square's rounding and
    the root's (0.75 of 2^-24), which the exponent multiplies by z; beside it a
    few roundings of 2^-24 (the exponential 2, the logarithm's quotient, its
    sum and the product with tau 1 each, for the gradient the quotient and the
    backward chain's eight products)."""
    rng = np.random.default_rng(int(1 / tau))
    z = np.exp(rng.uniform(np.log(1e-4), np.log(min(60.0 * tau, 1.0)), 3000)).astype(np.float32)
    c, g, J, w, p = _one_box(z, tau, 0.0, orc)
    ulp = 2.0**-24
    zz = p / float(np.float32(tau))
    worst = (np.abs(c - J) / J / ulp - zz).max(), (np.abs(g - w) / np.abs(w) / ulp - zz).max()
    print(f"tau {tau}: error less z, in 2^-24: cost {worst[0]:.2f}, gradient {worst[1]:.2f}", flush=True)
    assert (np.abs(c - J) <= (zz + 5.0) * ulp * J).all()
    assert (np.abs(g - w) <= (zz + 11.0) * ulp * np.abs(w)).all()


@pytest.mark.parametrize("tau,margin", [(1e-13, 0.02), (1e-39, 0.02), (1e19, 0.02), (3e38, 0.02), (0.01, 1e19),
                                        (0.01, -1e19), (0.01, 3e38)])
def test_ends_of_tau_and_margin(tau, margin, orc):
    z = np.array([1e-3, 0.01, 0.0199, 0.0201, 0.3, 2.0], np.float32)
    c, g, J, w, _ = _one_box(z, tau, margin, orc)
    # (a cost past the largest float is infinite)
    J32 = J.astype(np.float32).astype(np.float64)
    same = (c == J32) | (np.abs(c - J) <= RTOL * np.maximum(np.abs(J), 1e-30))
    assert same.all(), (c, J)
    assert (np.abs(g - w) <= RTOL * np.maximum(np.abs(w), 1e-30)).all(), (g, w)
