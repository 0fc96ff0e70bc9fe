"""A trajectory's cost, gradient and Adam steps are its own, bit for bit:
whatever stands in the controls past its length, whatever the trajectories
beside it in a wave are, and whatever the number of trajectories (which sets
the lanes that each one gets)."""
import numpy as np
import pytest
import torch

from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W

pytestmark = pytest.mark.gpu


def _d(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def _batch(n, seed=9):
    rb = W.make_refine_batch(n, seed=seed, objective="hover", steps_lo=1, steps_hi=37)
    rng = np.random.default_rng(seed)
    rb.steps[rng.integers(0, n, n // 9 + 1)] = 0
    spin = rng.integers(0, n, n // 7 + 1)  # some turn by more than 0.1 rad in a step
    rb.x0[9:12, spin] = rng.uniform(-25.0, 25.0, (3, len(spin)))
    for k, t in enumerate(rb.steps):
        rb.u[t:, :, k] = 0.0
    return rb


def _run(rb, cols, u=None, iterations=0):
    """(cost or history, gradient or controls) of the trajectories `cols`."""
    u = rb.u if u is None else u
    args = (_d(rb.x0[:, cols]), _d(rb.goal[:, cols]), _d(rb.steps[cols]), _d(rb.obstacles), rb.cfg, rb.params)
    if not iterations:
        c, g = A.cost_and_grad(_d(u[:, :, cols]), *args)
        return c.cpu().numpy()[None], g.cpu().numpy()
    rb.params.iterations = iterations
    v = _d(u[:, :, cols])
    h = A.refine(v, *args)
    return h.cpu().numpy(), v.cpu().numpy()


def _same(a, b, rb, cols):
    assert np.array_equal(a[0].view(np.uint32), b[0].view(np.uint32))
    for k, i in enumerate(cols):  # (controls past the length stay the caller's)
        t = int(rb.steps[i])
        assert np.array_equal(a[1][:t, :, k].view(np.uint32), b[1][:t, :, k].view(np.uint32)), i


@pytest.mark.parametrize("n", [3, 64, 1025, 2051])
@pytest.mark.parametrize("pad", [float("nan"), float("inf"), 3e38, 50.0])
@pytest.mark.parametrize("iterations", [0, 4])
def test_controls_past_the_length_do_not_matter(n, pad, iterations):
    print(f"padding {pad}: n={n} iterations={iterations}", flush=True)
    rb = _batch(n)
    u = rb.u.copy()
    for k, t in enumerate(rb.steps):
        u[t:, :, k] = pad
    cols = np.arange(n)
    want, got = _run(rb, cols, iterations=iterations), _run(rb, cols, u, iterations)
    _same(want, got, rb, cols)
    if iterations:
        for k, t in enumerate(rb.steps):
            assert np.array_equal(got[1][t:, :, k].view(np.uint32), u[t:, :, k].view(np.uint32))
    else:
        for k, t in enumerate(rb.steps):
            assert not got[1][t:, :, k].any()


@pytest.mark.parametrize("iterations", [0, 4])
def test_other_trajectories_and_their_number_do_not_matter(iterations):
    n = 2300
    rb = _batch(n)
    rng = np.random.default_rng(1)
    cols = np.arange(n)
    want = _run(rb, cols, iterations=iterations)
    for m in (2300, 2049, 1400, 1025, 333, 5):
        print(f"{m} of {n} trajectories, iterations={iterations}", flush=True)
        some = rng.permutation(n)[:m]
        got = _run(rb, some, iterations=iterations)
        _same((want[0][:, some], want[1][:, :, some]), got, rb, some)


@pytest.mark.parametrize("n", [2, 1030, 2060])
def test_an_infinite_start_costs_infinitely_and_stays_alone(n):
    rb = _batch(n)
    cols = np.arange(n)
    want = _run(rb, cols)
    rb.x0[0, 1] = np.inf
    got = _run(rb, cols)
    assert got[0][0, 1] == np.inf
    others = np.delete(cols, 1)
    _same((want[0][:, others], want[1][:, :, others]), (got[0][:, others], got[1][:, :, others]), rb, others)
