"""kgmt_propagate_collide at the sizes and inputs where its work splits and
its box masks could go wrong: one child to more than one launch's lanes, box
counts around a mask word, unusual boxes, parents out of range, edges of no
step, non-finite and far-away states; bit for bit against the oracle (a NaN
equals any NaN)."""
import ctypes as C

import numpy as np
import pytest

from kgmt_amd import workloads as W
from kgmt_amd.abi import dims

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")
from tests.gpu_util import call, dev, empty, host, ptr, stream  # noqa: E402
from tests.test_gpu_parity import CASES, parent_states  # noqa: E402
from tests.test_gpu_plan import _odd_boxes  # noqa: E402


def _run(cfg, pidx, X, ctrl, steps, obs):
    S, Cd, D = dims(cfg.model)
    n = len(pidx)
    out = (empty((D, n), torch.float32), empty(n, torch.uint8), empty(n, torch.int32), empty(n, torch.int32))
    d_obs = dev(obs.reshape(-1)) if len(obs) else None
    d = [dev(pidx), dev(X), dev(ctrl), dev(steps)]
    call("kgmt_propagate_collide", C.byref(cfg), ptr(d[0]), ptr(d[1]), X.shape[1], ptr(d[2]), ptr(d[3]), n, ptr(d_obs),
         len(obs), *(ptr(o) for o in out), stream())
    return [host(o) for o in out]


def _same(got, want):
    for g, w in zip(got, want):
        if g.dtype == np.float32:
            nan = np.isnan(w)
            assert np.array_equal(np.isnan(g), nan)
            assert np.array_equal(g.view(np.uint32)[~nan], w.view(np.uint32)[~nan])
        else:
            assert np.array_equal(g, w)


def _boxes(cfg, n, rng):
    span = cfg.ws_max - cfg.ws_min
    return W.random_boxes(rng, n, 0.02 * span, 0.15 * span, ws=(cfg.ws_min, cfg.ws_max), dim=cfg.wdim) if n \
        else np.zeros((0, 2 * cfg.wdim), np.float32)


@pytest.mark.parametrize("case", list(CASES))
@pytest.mark.parametrize("n,boxes", [(1, 0), (63, 1), (257, 64), (4000, 65), (3000, 129), (1500, 700)])
def test_sizes(case, n, boxes, orc):
    cfg = CASES[case]()
    rng = np.random.default_rng(n + boxes)
    npar = max(1, n // 7)
    X = parent_states(cfg, npar, seed=n)
    pidx = rng.integers(0, npar, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, n)
    obs = _boxes(cfg, boxes, rng)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), orc.propagate_children(cfg, pidx, X, ctrl, steps, obs))


@pytest.mark.parametrize("case", list(CASES))
def test_odd_inputs(case, orc):
    cfg = CASES[case]()
    S, _, D = dims(cfg.model)
    rng = np.random.default_rng(9)
    n, npar = 2000, 90
    X = parent_states(cfg, npar, seed=4)
    span = cfg.ws_max - cfg.ws_min
    X[0, 0], X[1, 1], X[S - 1, 2], X[0, 3], X[1, 4] = np.nan, np.inf, np.nan, -np.inf, 1e30
    X[0, 5] = cfg.ws_min - 3 * span  # outside the workspace
    X[3, 6] = np.nan
    pidx = rng.integers(0, npar, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, n)
    steps = steps.copy()
    steps[::17] = 0
    steps[5::31] = -3
    obs = _odd_boxes(cfg.wdim, rng)
    obs = np.where(np.isfinite(obs), obs * span + cfg.ws_min, obs).astype(np.float32)
    # the oracle's edges of no step: the state as it is, valid
    want = orc.propagate_children(cfg, pidx, X, ctrl, steps, obs)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), want)
    # parents out of range: zeros, invalid, regions -1; the others as they were
    bad = pidx.copy()
    bad[3::11] = -1
    bad[4::13] = npar
    got = _run(cfg, bad, X, ctrl, steps, obs)
    out = (bad < 0) | (bad >= npar)
    assert np.all(got[0][:, out] == 0.0) and np.all(got[1][out] == 0)
    assert np.all(got[2][out] == -1) and np.all(got[3][out] == -1)
    _same([got[0][:, ~out], got[1][~out], got[2][~out], got[3][~out]],
          [want[0][:, ~out], want[1][~out], want[2][~out], want[3][~out]])


@pytest.mark.parametrize("case,n", [("quad12d", 270001), ("di_ref", 530001)])
def test_more_children_than_lanes(case, n, orc):
    cfg = CASES[case]().replace(steps_min=1, steps_max=2)
    rng = np.random.default_rng(2)
    X = parent_states(cfg, 900, seed=4)
    pidx = rng.integers(0, 900, n).astype(np.int32)
    ctrl, steps, _ = orc.draw_children(cfg, 0, 1, 0, n)
    obs = _boxes(cfg, 5, rng)
    _same(_run(cfg, pidx, X, ctrl, steps, obs), orc.propagate_children(cfg, pidx, X, ctrl, steps, obs))
