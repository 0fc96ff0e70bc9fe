"""Device memory that the differentiable rollout takes for a call, by the
memory pool's high-water mark: no more than a trajectory's own work space for
one, and for long rollouts of many neither more than 12 floats a step and
trajectory (20 with Adam's moments; 1 GiB at least) nor so little that the call
needs more than five launches."""
import ctypes as C

import numpy as np
import pytest
import torch

from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W

pytestmark = pytest.mark.gpu

USED_HIGH = 8  # hipMemPoolAttrUsedMemHigh
STEP = 56      # floats of work space a step and trajectory, 64 with moments


def _hip():
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    return C.CDLL(path)


def _peak(call):
    hip, pool = _hip(), C.c_void_p()
    assert hip.hipDeviceGetDefaultMemPool(C.byref(pool), 0) == 0
    torch.cuda.synchronize()
    v = C.c_uint64(0)
    assert hip.hipMemPoolSetAttribute(pool, USED_HIGH, C.byref(v)) == 0
    call()
    torch.cuda.synchronize()
    assert hip.hipMemPoolGetAttribute(pool, USED_HIGH, C.byref(v)) == 0
    return v.value


@pytest.mark.parametrize("n,T,iterations", [(1, 100000, 0), (1, 30000, 1), (3, 20000, 0), (1500, 40, 0), (4099, 40, 1),
                                            (4096, 8000, 0), (1300, 9001, 1)])
def test_work_space_of_a_call(n, T, iterations):
    rb = W.make_refine_batch(n, seed=1, objective="hover", steps_lo=3, steps_hi=9)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    u = torch.full((T, 4, n), 0.0, device="cuda:0")
    u[:, 0] = 9.81
    rb.params.iterations = iterations
    args = (d(rb.x0), d(rb.goal), d(rb.steps), d(rb.obstacles), rb.cfg, rb.params)
    run = (lambda: A.refine(u, *args)) if iterations else (lambda: A.cost_and_grad(u, *args))
    _hip()
    run()  # (the runtime's own first allocations)
    peak = _peak(run)
    step, old = (STEP + 8, 20) if iterations else (STEP, 12)
    whole = 4 * step * T * n
    few = max(1 << 30, 4 * (old * T + 12) * n)
    print(f"n={n} T={T} iterations={iterations}: {peak} bytes of {whole}", flush=True)
    assert peak <= min(whole * (1 + 3 / n) if n > 1024 else whole, few) + (1 << 16)
    assert 5 * peak >= whole


@pytest.mark.parametrize("n,T", [(7, 20000), (1029, 6000), (2100, 5000)])
def test_long_rollouts_in_several_launches_agree(n, T):
    """The same trajectories in a long and in a short array."""
    rb = W.make_refine_batch(n, seed=n, objective="hover", steps_lo=1, steps_hi=33)
    d = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")
    args = (d(rb.x0), d(rb.goal), d(rb.steps), d(rb.obstacles), rb.cfg, rb.params)
    c, g = A.cost_and_grad(d(rb.u), *args)
    u = torch.zeros((T, 4, n), device="cuda:0")
    u[:rb.u.shape[0]] = d(rb.u)
    C2, G2 = A.cost_and_grad(u, *args)
    assert torch.equal(c, C2) and torch.equal(g, G2[:rb.u.shape[0]]) and not bool(G2[rb.u.shape[0]:].any())
