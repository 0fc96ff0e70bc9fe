"""Measured workloads of the framework, through its public entry points.

Kinds of case and what they stand for in use:
  plan   KGMT.plan on one planner, one query after the other: start, goal and
         obstacles in device memory, the result and the goal path read back
         (with "tree": the whole tree too, as a caller that draws or exports it
         does). Small trees of a few boxes up to the shipped tree sizes; every
         dynamics model.
  batch  BatchKGMT.plan: many independent queries served together, host
         arrays in, results and every solved query's path out.
  edges  kgmt_propagate_collide: a caller's own set of edges (parent, control,
         duration) integrated and checked against a scene.
  grad   rollout_cost forward and backward: the differentiable rollout inside a
         caller's own optimiser.
  refine refine: Adam on found control sequences in one call.

A plan is a random search whose decisions are whole numbers (tree indices,
counts), so no 64-bit value of its outputs exists; edges, gradients and short
refinements have one.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from kgmt_amd import _lib
from kgmt_amd import adjoint as A
from kgmt_amd import workloads as W
from kgmt_amd.abi import (KGMT_MAX_SAMPLE, KGMT_MODEL_DOUBLE_INTEGRATOR, KGMT_MODEL_DUBINS_5D,
                          KGMT_MODEL_DUBINS_AIRPLANE, KGMT_MODEL_UNICYCLE, dims)
from kgmt_amd.planner import KGMT, BatchKGMT

DEV = "cuda:0"


def listed():
    return [
        # a planar robot with a small tree: the shortest call, launches and host latency
        {"name": "plan_unicycle_small", "kind": "plan", "model": "unicycle2d", "capacity": 4096, "boxes": 12,
         "queries": 1, "walls": False, "tree": False},
        # the configured double integrator (20 boxes, 2^17 nodes)
        {"name": "plan_di6d", "kind": "plan", "model": "di6d", "capacity": 131072, "boxes": 20, "queries": 4,
         "walls": False, "tree": False},
        # the benchmark's queries: 5D airplane, 100 boxes, 2^18 nodes
        {"name": "plan_dubins5d", "kind": "plan", "model": "dubins5d", "capacity": 262144, "boxes": 100,
         "queries": 8, "walls": False, "tree": False},
        # the 6D airplane of the reference's configuration, odd tree size, scene and count, the tree read back
        {"name": "plan_dubins6d_tree", "kind": "plan", "model": "dubins6d", "capacity": 100003, "boxes": 333,
         "queries": 1, "walls": False, "tree": True},
        # the configured quadcopter: slotted walls and 50 boxes, 2^19 nodes
        {"name": "plan_quad12d", "kind": "plan", "model": "quad12d", "capacity": 524288, "boxes": 50, "queries": 1,
         "walls": True, "tree": False},
        # the configured batch: 512 queries, half double integrator, half quadcopter, trees of 2^12..2^17, 10..500 boxes
        {"name": "batch_512_mixed", "kind": "batch", "model": "mixed", "n": 512, "cap_lo": 4096, "cap_hi": 131072,
         "boxes_lo": 10, "boxes_hi": 500},
        # a few queries of one model served together, odd count
        {"name": "batch_33_dubins5d", "kind": "batch", "model": "dubins5d", "n": 33, "cap_lo": 8192, "cap_hi": 65536,
         "boxes_lo": 20, "boxes_hi": 150},
        # a given set of edges of one planner iteration, one scene
        {"name": "edges_quad_100003", "kind": "edges", "model": "quad12d", "n": 100003, "parents": 3200, "boxes": 200},
        # the configured refinement: 4096 sequences of 20..80 steps, 50 Adam steps, 50 boxes
        {"name": "refine_4096", "kind": "refine", "n": 4096, "steps_lo": 20, "steps_hi": 80, "iterations": 50,
         "boxes": 50, "objective": "configured"},
        # a handful of short sequences polished: too few to fill the chip
        {"name": "refine_61", "kind": "refine", "n": 61, "steps_lo": 8, "steps_hi": 24, "iterations": 50, "boxes": 50,
         "objective": "hover"},
        # one cost and gradient of a caller's own optimiser loop
        {"name": "grad_4096", "kind": "grad", "n": 4096, "steps_lo": 20, "steps_hi": 80, "boxes": 50,
         "objective": "configured"},
        {"name": "grad_333_many_boxes", "kind": "grad", "n": 333, "steps_lo": 5, "steps_hi": 61, "boxes": 301,
         "objective": "hover"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


PLAN_CAP = {"unicycle2d": 131072, "di6d": 131072, "dubins5d": 262144, "dubins6d": 262144, "quad12d": 524288}


def draw(rng):
    kind = rng.choice(["plan", "plan", "plan", "batch", "edges", "refine", "grad"])
    if kind == "plan":
        model = rng.choice(sorted(PLAN_CAP))
        quad = model == "quad12d"  # a step costs several times the other models'
        cap = _log(rng, 4096, PLAN_CAP[model] // (2 if quad else 1))
        return {"kind": kind, "model": model, "capacity": cap, "boxes": _log(rng, 10, 200 if quad else 500),
                "queries": 1 if quad else rng.randint(1, 4), "walls": False, "tree": rng.random() < 0.25}
    if kind == "batch":
        lo = _log(rng, 4096, 16384)
        hi = _log(rng, lo, 131072)
        blo = _log(rng, 10, 100)
        return {"kind": kind, "model": rng.choice(["mixed", "di6d", "dubins5d"]), "n": _log(rng, 8, 256), "cap_lo": lo,
                "cap_hi": hi, "boxes_lo": blo, "boxes_hi": rng.randint(blo, 500)}
    if kind == "edges":
        n = _log(rng, 1000, 200000)
        return {"kind": kind, "model": rng.choice(sorted(PLAN_CAP)), "n": n, "parents": max(1, n // rng.randint(1, 40)),
                "boxes": _log(rng, 10, 500)}
    lo = rng.randint(5, 40)
    case = {"kind": kind, "n": _log(rng, 30, 4096), "steps_lo": lo, "steps_hi": rng.randint(lo + 1, 80),
            "boxes": _log(rng, 5, 200 if kind == "refine" else 400), "objective": rng.choice(["configured", "hover"])}
    if kind == "refine":
        case["iterations"] = rng.randint(3, 50)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _config(model, **kw):
    if model == "dubins6d":
        # the reference's Dubins-airplane block on a unit cube
        q = math.pi / 4
        return W.config("dubins5d").replace(model=KGMT_MODEL_DUBINS_AIRPLANE, dt=0.1, steps_min=1, steps_max=10,
                                            v_min=0.0, v_max=0.3, ctrl_min=[-q, -q, -0.3, 0.0],
                                            ctrl_max=[q, q, 0.3, 0.0], r1_len=8, r2_len=2, **kw)
    return W.config(model, **kw)


# side lengths of random boxes per model
SIDES = {"unicycle2d": (0.03, 0.1), "di6d": (0.03, 0.12), "dubins5d": (0.02, 0.1), "dubins6d": (0.02, 0.08),
         "quad12d": (0.02, 0.06)}


def _boxes(rng, n, sides, clear, dim):
    """n boxes of the unit cube, drawn again while nearer than r to a (centre, r) of `clear`."""
    out = np.zeros((n, 2 * dim))
    todo = np.arange(n)
    while todo.size:
        c = rng.uniform(0.0, 1.0, (todo.size, dim))
        s = rng.uniform(sides[0], sides[1], (todo.size, dim))
        b = np.concatenate([np.clip(c - s / 2, 0.0, 1.0), np.clip(c + s / 2, 0.0, 1.0)], axis=1)
        ok = np.ones(todo.size, bool)
        for p, r in clear:
            ok &= W.box_ball_distance(b, np.asarray(p)) >= r
        out[todo[ok]] = b[ok]
        todo = todo[~ok]
    return out.astype(np.float32)


def _query(model, rng, boxes, far):
    """start, goal, boxes of one query: opposite corners, or a random pair at least 0.6 apart."""
    w = 2 if model == "unicycle2d" else 3
    if far:
        start, goal = np.full(w, 0.05), np.full(w, 0.95)
    else:
        while True:
            start, goal = rng.uniform(0.1, 0.9, w), rng.uniform(0.1, 0.9, w)
            if np.linalg.norm(start - goal) >= 0.6:
                break
    rows = _boxes(rng, boxes, SIDES[model], [(start, 0.06), (goal, 0.06)], w)
    return start, goal, rows


def _plan_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 1])
    model = case["model"]
    cfg = _config(model, capacity=case["capacity"])
    queries = []
    for _ in range(case["queries"]):
        if case["walls"]:  # three slotted walls and 50 boxes
            q = W.make_query("quad12d", int(rng.integers(1 << 30)))
            start, goal, rows = q.start, q.goal, q.obstacles
        else:
            start, goal, rows = _query(model, rng, case["boxes"], True)
        x = np.zeros(cfg.dims[2], np.float32)
        x[:len(start)] = start
        g = np.zeros(cfg.dims[2], np.float32)
        g[:len(goal)] = goal
        queries.append((int(rng.integers(1, 1 << 40)), x, g, torch.from_numpy(rows).to(DEV), len(rows)))
    planner = KGMT(cfg)
    torch.cuda.synchronize()
    s = {"planner": planner, "queries": queries, "tree": None, "paths": _path_rows(len(queries), [cfg])}
    if case["tree"]:
        cap, D = cfg.capacity, cfg.dims[2]
        s["tree"] = (np.zeros((cap, D), np.float32), np.zeros(cap, np.int32), np.zeros(cap, np.float32))
    return s


def _path_rows(n, cfgs):
    """The caller's room for n goal paths (as long as the iteration limit allows)."""
    return np.zeros((n, max(c.max_iter for c in cfgs) + 2, max(c.dims[2] for c in cfgs)), np.float32)


def _batch_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 2])
    cfgs, starts, goals, rows, offs, cnts = [], [], [], [], [], []
    at = 0
    for q in range(case["n"]):
        model = case["model"] if case["model"] != "mixed" else ("di6d" if q % 2 == 0 else "quad12d")
        cap = int(round(math.exp(rng.uniform(math.log(case["cap_lo"]), math.log(case["cap_hi"])))))
        n = int(rng.integers(case["boxes_lo"], case["boxes_hi"] + 1))
        s, g, b = _query("quad12d" if case["model"] == "mixed" else model, rng, n, False)
        cfgs.append(_config(model, capacity=cap, seed=int(rng.integers(1, 1 << 40)), query_id=q))
        for to, v in ((starts, s), (goals, g)):
            x = np.zeros(KGMT_MAX_SAMPLE, np.float32)
            x[:3] = v
            to.append(x)
        rows.append(b)
        offs.append(at)
        cnts.append(n)
        at += n
    return {"planner": BatchKGMT(cfgs), "starts": np.stack(starts), "goals": np.stack(goals),
            "rows": np.concatenate(rows), "paths": _path_rows(len(cfgs), cfgs), "offs": np.asarray(offs, np.uint32), "cnts": np.asarray(cnts, np.uint32)}


def _edge_inputs(case, seed):
    rng = np.random.default_rng([int(seed), 3])
    cfg = _config(case["model"])
    S, Cd, D = dims(cfg.model)
    n, m, w = case["n"], case["parents"], cfg.wdim
    x = np.zeros((S, m), np.float32)
    x[:w] = rng.uniform(0.05, 0.95, (w, m))
    if cfg.model == KGMT_MODEL_UNICYCLE:
        x[2], x[3] = rng.uniform(-math.pi, math.pi, m), rng.uniform(-0.6, 0.6, m)
    elif cfg.model == KGMT_MODEL_DOUBLE_INTEGRATOR:
        x[3:6] = rng.uniform(-0.5, 0.5, (3, m))
    elif cfg.model in (KGMT_MODEL_DUBINS_AIRPLANE, KGMT_MODEL_DUBINS_5D):
        x[3], x[4] = rng.uniform(-math.pi, math.pi, m), rng.uniform(-0.5, 0.5, m)
        if cfg.model == KGMT_MODEL_DUBINS_AIRPLANE:
            x[5] = rng.uniform(0.05, 0.3, m)
    else:
        x[3:6] = rng.uniform(-0.3, 0.3, (3, m))
        x[6:12] = rng.uniform(-1.0, 1.0, (6, m))
    lo, hi = np.array(cfg.ctrl_min[:Cd], np.float32), np.array(cfg.ctrl_max[:Cd], np.float32)
    u = rng.uniform(lo[:, None], hi[:, None], (Cd, n)).astype(np.float32)
    parent = np.sort(rng.integers(0, m, n)).astype(np.int32)  # children of one parent lie together
    steps = rng.integers(cfg.steps_min, cfg.steps_max + 1, n).astype(np.int32)
    boxes = _boxes(rng, case["boxes"], SIDES[case["model"]], [], w)
    d = {k: torch.from_numpy(v).to(DEV) for k, v in (("x", x), ("u", u), ("parent", parent), ("steps", steps),
                                                     ("boxes", boxes))}
    d["child"] = torch.empty((D, n), device=DEV)
    d["valid"] = torch.empty(n, dtype=torch.uint8, device=DEV)
    d["r1"], d["r2"] = (torch.empty(n, dtype=torch.int32, device=DEV) for _ in range(2))
    d["cfg"] = cfg
    return d


def _rollout_inputs(case, seed):
    """Control sequences of the refinement workload: from rest, hover thrust and noise, goals 0.05..0.15 away."""
    rng = np.random.default_rng([int(seed), 4])
    cfg = W.config("quad12d")
    n = case["n"]
    steps = rng.integers(case["steps_lo"], case["steps_hi"] + 1, n).astype(np.int32)
    T = int(steps.max())
    x0 = np.zeros((12, n), np.float32)
    x0[:3] = rng.uniform(0.25, 0.75, (3, n))
    d = rng.normal(size=(3, n))
    d /= np.linalg.norm(d, axis=0, keepdims=True)
    goal = (x0[:3] + d * rng.uniform(0.05, 0.15, n)).astype(np.float32)
    u = np.zeros((T, 4, n), np.float32)
    u[:, 0] = np.clip(9.81 + rng.normal(0.0, 1.0, (T, n)), cfg.ctrl_min[0], cfg.ctrl_max[0])
    u[:, 1:] = np.clip(rng.normal(0.0, 0.005, (T, 3, n)), cfg.ctrl_min[1], cfg.ctrl_max[1])
    boxes = _boxes(rng, case["boxes"], (0.02, 0.08), [], 3)
    params = W.refine_params(cfg, case["objective"], iterations=case.get("iterations", 50))
    s = {k: torch.from_numpy(v).to(DEV) for k, v in (("u", u), ("x0", x0), ("goal", goal), ("steps", steps),
                                                     ("boxes", boxes))}
    s["cfg"], s["params"] = cfg, params
    return s


def prepare(case, seed):
    torch.cuda.init()  # torch's runtime first: it shares the device with the library's
    torch.zeros(1, device=DEV)
    kind = case["kind"]
    make = {"plan": _plan_inputs, "batch": _batch_inputs, "edges": _edge_inputs}.get(kind, _rollout_inputs)
    s = make(case, seed)
    s["kind"] = kind
    return s


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def _outcome(results, paths):
    """Whole-number and real fields of every result, and the goal paths."""
    whole = np.array([[r.success, r.goal_index, r.iterations, r.tree_size, r.path_rows, r.expanded] for r in results],
                     np.int64)
    real = np.array([[r.path_cost, r.path_length] for r in results], np.float32)
    return {"whole": whole, "real": real, "paths": paths}


def _keep(paths, q, rows):
    paths[q, :rows.shape[0], :rows.shape[1]] = rows


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def run(s):
    kind = s["kind"]
    if kind == "plan":
        p, results = s["planner"], []
        for q, (seed, start, goal, boxes, n) in enumerate(s["queries"]):
            p.set_seed(seed)
            r = p.plan(start, goal, boxes, n)
            results.append(r)
            if r.success:
                _keep(s["paths"], q, p.h_controlPathToGoal_)
        out = _outcome(results, s["paths"])
        if s["tree"]:
            for to, v in zip(s["tree"], p.tree()):
                to[:len(v)] = v
            out["tree"] = s["tree"]
        return out
    if kind == "batch":
        b = s["planner"]
        results, _ = b.plan(s["starts"], s["goals"], s["rows"], s["offs"], s["cnts"])
        for q, r in enumerate(results):
            if r.success:
                _keep(s["paths"], q, b.path(q))
        return _outcome(results, s["paths"])
    if kind == "edges":
        cfg, n = s["cfg"], s["parent"].numel()
        stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        _lib.check(_lib.lib().kgmt_propagate_collide(
            C.byref(cfg), _ptr(s["parent"]), _ptr(s["x"]), s["x"].shape[1], _ptr(s["u"]), _ptr(s["steps"]), n,
            _ptr(s["boxes"]), s["boxes"].shape[0], _ptr(s["child"]), _ptr(s["valid"]), _ptr(s["r1"]), _ptr(s["r2"]),
            stream))
        return {"child": s["child"], "valid": s["valid"], "r1": s["r1"], "r2": s["r2"]}
    if kind == "grad":
        u = s["u"].detach().requires_grad_(True)
        cost = A.rollout_cost(u, s["x0"], s["goal"], s["steps"], s["boxes"], s["cfg"], s["params"])
        cost.sum().backward()
        return {"cost": cost.detach(), "grad": u.grad}
    u = s["u"].clone()
    history = A.refine(u, s["x0"], s["goal"], s["steps"], s["boxes"], s["cfg"], s["params"])
    return {"u": u, "history": history}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
# float operations of one integration step (RK4 stages with their sin / cos as
# one operation each, bound checks; Euler for the unicycle)
STEP_FLOPS = {"unicycle2d": 20, "di6d": 90, "dubins5d": 70, "dubins6d": 80, "quad12d": 420}


def _edges_work(model, n):
    cfg = _config(model)
    S, Cd, D = dims(cfg.model)
    mean = 0.5 * (cfg.steps_min + cfg.steps_max)
    return n * (4 * Cd + 4 + 4 + 4 * D + 9), n * mean * STEP_FLOPS[model]


def _tree_work(model, nodes):
    """A search that fills about half its tree, four children tried for each node kept: a node is written once
    (sample, parent, cost) and read once as a parent."""
    D = dims(_config(model).model)[2]
    return 0.5 * nodes * (8 * D + 8), _edges_work(model, 2.0 * nodes)[1]


def work(case):
    kind = case["kind"]
    if kind == "plan":
        b, f = _tree_work(case["model"], case["capacity"])
        return {"bytes": case["queries"] * b, "flops": case["queries"] * f}
    if kind == "batch":
        lo, hi = case["cap_lo"], case["cap_hi"]
        cap = (hi - lo) / math.log(hi / lo) if hi > lo else lo  # mean of a log-uniform size
        models = ["di6d", "quad12d"] if case["model"] == "mixed" else [case["model"]]
        per = [_tree_work(m, cap) for m in models]
        k = case["n"] / len(models)
        return {"bytes": k * sum(p[0] for p in per), "flops": k * sum(p[1] for p in per)}
    if kind == "edges":
        cfg = _config(case["model"])
        b, f = _edges_work(case["model"], case["n"])
        return {"bytes": b + 4 * cfg.dims[0] * case["parents"] + 8 * cfg.wdim * case["boxes"], "flops": f}
    T = 0.5 * (case["steps_lo"] + case["steps_hi"])
    n, m = case["n"], case["boxes"]
    # a step forward (RK4, about 25 operations for each box's penalty) and backward (stage values are kept or
    # computed again, four vector-Jacobian products, the penalty's gradient)
    forward, backward = STEP_FLOPS["quad12d"] + 25 * m, 3 * STEP_FLOPS["quad12d"] + 35 * m
    rows = case["steps_hi"] * 4 * n * 4
    if kind == "grad":
        return {"bytes": 2 * rows + 4 * 17 * n, "flops": n * T * (forward + backward)}
    it = case["iterations"]
    return {"bytes": 2 * rows + 4 * (16 + it + 1) * n, "flops": n * T * ((it + 1) * forward + it * backward)}


# ---------------------------------------------------------------------------
# 64-bit values
# ---------------------------------------------------------------------------
def _ode(cfg, s, c):
    """Quadcopter ODE of the 12 state rows `s` under the 4 control rows `c`."""
    phi, th, psi, u, v, w, p, q, r = s[3:]
    sf, cf, st, ct, sp, cp = phi.sin(), phi.cos(), th.sin(), th.cos(), psi.sin(), psi.cos()
    ix, iy, iz, g = cfg.quad_ix, cfg.quad_iy, cfg.quad_iz, cfg.gravity
    e = q * sf + r * cf
    drag = -cfg.quad_nu * _norm(u, v, w) / cfg.quad_mass
    spin = -cfg.quad_mu * _norm(p, q, r)
    return [ct * cp * u + (sf * st * cp - cf * sp) * v + (cf * st * cp + sf * sp) * w,
            ct * sp * u + (sf * st * sp + cf * cp) * v + (cf * st * sp - sf * cp) * w,
            -st * u + sf * ct * v + cf * ct * w,
            p + e * st / ct, q * cf - r * sf, e / ct,
            r * v - q * w - g * st + drag * u,
            p * w - r * u + g * ct * sf + drag * v,
            q * u - p * v + g * ct * cf + drag * w + c[0] / cfg.quad_mass,
            (iy - iz) / ix * q * r + (spin * p + c[1]) / ix,
            (iz - ix) / iy * p * r + (spin * q + c[2]) / iy,
            (ix - iy) / iz * p * q + (spin * r + c[3]) / iz]


def _norm(a, b, c):
    s = a * a + b * b + c * c
    pos = s > 0
    return torch.where(pos, torch.where(pos, s, torch.ones_like(s)).sqrt(), torch.zeros_like(s))


def _rk4(cfg, s, c):
    h = float(np.float32(cfg.dt))
    k1 = _ode(cfg, s, c)
    k2 = _ode(cfg, [a + 0.5 * h * k for a, k in zip(s, k1)], c)
    k3 = _ode(cfg, [a + 0.5 * h * k for a, k in zip(s, k2)], c)
    k4 = _ode(cfg, [a + h * k for a, k in zip(s, k3)], c)
    return [a + h / 6.0 * (x + 2.0 * y + 2.0 * z + w) for a, x, y, z, w in zip(s, k1, k2, k3, k4)]


def _cost64(u, s):
    """J of every sequence, differentiable with respect to u."""
    cfg, ap, n = s["cfg"], s["params"], u.shape[2]
    x = list(s["x0"].double())
    box, steps = s["boxes"].double(), s["steps"]
    ref = torch.tensor(list(ap.u_ref), dtype=torch.float64, device=DEV).view(4, 1)
    J = torch.zeros(n, dtype=torch.float64, device=DEV)
    last = [v for v in x[:3]]
    for t in range(u.shape[0]):
        on = t < steps
        x = _rk4(cfg, x, u[t])
        p = torch.stack(x[:3], 1)
        q = torch.maximum(box[None, :, :3] - p[:, None], p[:, None] - box[None, :, 3:])
        o = q.clamp_min(0.0)
        sd = _norm(o[..., 0], o[..., 1], o[..., 2]) + q.amax(-1).clamp_max(0.0)
        pen = ap.tau * torch.nn.functional.softplus((ap.margin - sd) / ap.tau, threshold=30.0).sum(1)
        J = J + torch.where(on, ap.w_effort * ((u[t] - ref) ** 2).sum(0) + ap.w_obstacle * pen, torch.zeros_like(J))
        last = [torch.where(on, a, b) for a, b in zip(x[:3], last)]
    g = s["goal"].double()
    return J + ap.w_goal * sum((a - b) ** 2 for a, b in zip(last, g))


def _grad64(u, s):
    u = u.detach().requires_grad_(True)
    J = _cost64(u, s)
    (g,) = torch.autograd.grad(J.sum(), u)
    return J.detach(), g


def _edges64(s):
    """The edges in 64 bits: each model's step, its bounds and the boxes; an edge stops at its first violation."""
    cfg, w = s["cfg"], s["cfg"].wdim
    h = float(np.float32(cfg.dt))
    p, u, steps = s["parent"].long(), s["u"].double(), s["steps"]
    x = [v.clone() for v in s["x"].double()[:, p]]
    box = s["boxes"].double()
    live, model = torch.ones_like(p, dtype=torch.bool), cfg.model

    def angles(y, pt, v):
        return [v * pt.cos() * y.cos(), v * pt.cos() * y.sin(), v * pt.sin()]

    for t in range(int(steps.max())):
        on = live & (t < steps)
        bad = torch.zeros_like(on)
        if model == KGMT_MODEL_UNICYCLE:
            new = [x[0] + x[3] * x[2].cos() * h, x[1] + x[3] * x[2].sin() * h,
                   x[2] + x[3] / cfg.uni_length * u[1].tan() * h, x[3] + u[0] * h]
        elif model == KGMT_MODEL_DOUBLE_INTEGRATOR:
            # the reference's position update: (5 v + 2 a h) h / 6
            new = [a + (5.0 * v + 2.0 * c * h) * h / 6.0 for a, v, c in zip(x[:3], x[3:], u)]
            new += [v + c * h for v, c in zip(x[3:], u)]
            for v in new[3:]:
                bad |= (v < cfg.v_min) | (v > cfg.v_max)
        elif model in (KGMT_MODEL_DUBINS_AIRPLANE, KGMT_MODEL_DUBINS_5D):
            five = model == KGMT_MODEL_DUBINS_5D
            a = torch.zeros_like(u[2]) if five else u[2]
            v = u[2] if five else x[5]
            y, pt = x[3], x[4]
            k = [angles(y + f * h * u[0], pt + f * h * u[1], v + f * h * a) for f in (0.0, 0.5, 0.5, 1.0)]
            new = [b + h / 6.0 * (k[0][i] + 2.0 * k[1][i] + 2.0 * k[2][i] + k[3][i]) for i, b in enumerate(x[:3])]
            new += [y + h * u[0], pt + h * u[1]] + ([] if five else [v + h * a])
            bad |= (new[4] < cfg.pitch_min) | (new[4] > cfg.pitch_max)
            if not five:
                bad |= (new[5] < cfg.v_min) | (new[5] > cfg.v_max)
        else:
            new = _rk4(cfg, x, u)
            for v in new[6:9]:
                bad |= (v < cfg.v_min) | (v > cfg.v_max)
        hit = torch.ones((p.numel(), box.shape[0]), dtype=torch.bool, device=DEV)
        for d in range(w):
            bad |= (new[d] < cfg.ws_min) | (new[d] > cfg.ws_max)
            lo, hi = torch.minimum(x[d], new[d]), torch.maximum(x[d], new[d])
            hit &= (hi[:, None] > box[None, :, d]) & (lo[:, None] < box[None, :, w + d])
        bad |= hit.any(1)
        x = [torch.where(on, b, a) for a, b in zip(x, new)]
        live = live & ~(on & bad)
    return torch.stack(x + list(u) + [h * steps.double()])


def exact(case, seed):
    kind = case["kind"]
    if kind in ("plan", "batch"):
        return None
    s = prepare(case, seed)
    if kind == "edges":
        return {"child": _edges64(s), "valid": None, "r1": None, "r2": None}
    u = s["u"].double()
    if kind == "grad":
        cost, grad = _grad64(u, s)
        return {"cost": cost, "grad": grad}
    ap, T = s["params"], u.shape[0]
    if (ap.iterations + 1) * T > 1300:
        return None
    lo, hi = (torch.tensor(list(v), dtype=torch.float64, device=DEV).view(4, 1) for v in (s["cfg"].ctrl_min,
                                                                                         s["cfg"].ctrl_max))
    on = (torch.arange(T, device=DEV)[:, None] < s["steps"][None, :])[:, None, :]
    m, v, history = torch.zeros_like(u), torch.zeros_like(u), []
    for k in range(1, ap.iterations + 1):
        J, g = _grad64(u, s)
        history.append(J)
        m = ap.beta1 * m + (1.0 - ap.beta1) * g
        v = ap.beta2 * v + (1.0 - ap.beta2) * g * g
        new = u - ap.lr * (m / (1.0 - ap.beta1 ** k)) / ((v / (1.0 - ap.beta2 ** k)).sqrt() + ap.adam_eps)
        u = torch.where(on, torch.minimum(torch.maximum(new, lo), hi), u)
    with torch.no_grad():
        history.append(_cost64(u, s))
    return {"u": u, "history": torch.stack(history)}
