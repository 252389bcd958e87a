"""Performance cases: batched evaluation, derivative sweeps and sparse solves as a program of this package runs them.

Every case is one call (or one forward and backward) through a public entry
point on inputs that are already where such a program holds them: device
tensors, except where the call itself takes host arrays.  All values are
FP64.  The Functions are the package's own workloads: the cart-pole and
quadrotor RK4 steps and the two-link arm, the cart-pole rollout cost, the
multiple-shooting quadrotor Lagrangian and the optimal-control KKT system.
"""
import functools
import math

import numpy as np
import torch

from casadi_amd import workloads as W
from casadi_amd.function import Function
from casadi_amd.hip import HipBatch, HipJacobian, HipTape
from casadi_amd.linsol import Linsol
from casadi_amd.ops import BINARY, OP
from casadi_amd.sx import gradient

F64 = torch.float64
MIXED = ("cartpole", "quadrotor", "arm")
STEPS = {"cartpole": W.cartpole_step, "quadrotor": W.quadrotor_step, "arm": W.arm_dynamics}


def listed():
    return [
        # f.map(n, "hip") in a control loop: few instances, the launch is all of it
        {"name": "map_small", "kind": "map", "f": "cartpole", "n": 1000},
        # the same map given host arrays, as a CasADi user calls it: in, evaluate, out
        {"name": "map_host", "kind": "map_host", "f": "cartpole", "n": 65536},
        # a sweep over millions of states: the streaming end of the map
        {"name": "map_large", "kind": "map", "f": "cartpole", "n": 8388608},
        # linearisation of the dynamics along many trajectories: value and Jacobian in one call
        {"name": "jacobian", "kind": "jacobian", "f": "cartpole", "n": 65536},
        # exact Lagrangian Hessians of a batch of optimal-control problems
        {"name": "hessian", "kind": "hessian", "horizon": 20, "n": 16384},
        # cost and gradient of single-shooting rollouts (the benchmark's headline)
        {"name": "rollout_grad", "kind": "rollout", "steps": 100, "ckpt": 10, "n": 32768, "engine": "jit"},
        # the same cost and gradient without run-time compilation (HipTape's default engine), a ragged batch
        {"name": "rollout_interp", "kind": "rollout", "steps": 20, "ckpt": 5, "n": 10007, "engine": "interp"},
        # training through a mapaccum in torch: forward keeps checkpoints, backward runs the reverse sweep
        {"name": "train_mapaccum", "kind": "train", "chain": "mapaccum", "steps": 100, "ckpt": 10, "n": 200003},
        # unlike Functions with their own batch sizes, forward and adjoint in one launch
        {"name": "batch_mixed", "kind": "batch", "cartpole": 40000, "quadrotor": 12000, "arm": 25000},
        # interior-point steps of a batch of control problems: factor and solve each KKT system
        {"name": "kkt_ldl", "kind": "kkt", "solver": "ldl", "horizon": 30, "n": 8192, "solves": 0},
        # the same systems by QR, which needs no quasi-definiteness
        {"name": "kkt_qr", "kind": "kkt", "solver": "qr", "horizon": 30, "n": 8192, "solves": 0},
        # gradient of a sum over samples with respect to a shared parameter
        {"name": "mapsum_grad", "kind": "mapsum", "f": "cartpole", "n": 1048576},
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over the logarithm; two in three are odd."""
    v = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return v if rng.random() < 1 / 3 else min(v | 1, hi - 1 + hi % 2)


def draw(rng):
    kind = rng.choice(["map", "map", "map_host", "jacobian", "hessian", "rollout", "rollout", "interp", "train", "train",
                       "batch", "kkt", "kkt", "mapsum"])
    f = rng.choice(sorted(STEPS))
    if kind == "map":
        return {"kind": kind, "f": f, "n": _log(rng, 64, 8388608 if f == "cartpole" else 2097152)}
    if kind == "map_host":
        return {"kind": kind, "f": f, "n": _log(rng, 16, 65536)}
    if kind == "jacobian":
        return {"kind": kind, "f": f, "n": _log(rng, 64, 524288)}
    if kind == "hessian":
        return {"kind": kind, "horizon": rng.randint(2, 20), "n": _log(rng, 64, 16384)}
    if kind == "rollout":
        steps = _log(rng, 10, 100)
        return {"kind": kind, "steps": steps, "ckpt": rng.randint(3, max(4, steps // 4)), "n": _log(rng, 64, 262144),
                "engine": "jit"}
    if kind == "interp":
        return {"kind": "rollout", "steps": _log(rng, 5, 20), "ckpt": rng.randint(2, 5), "n": _log(rng, 64, 16384),
                "engine": "interp"}
    if kind == "train":
        steps = _log(rng, 10, 100)
        return {"kind": kind, "chain": rng.choice(["mapaccum", "flat"]), "steps": steps,
                "ckpt": rng.randint(3, max(4, steps // 4)), "n": _log(rng, 64, 200003)}
    if kind == "batch":
        return {"kind": kind, "cartpole": _log(rng, 100, 40000), "quadrotor": _log(rng, 100, 12000),
                "arm": _log(rng, 100, 40000)}
    if kind == "kkt":
        return {"kind": kind, "solver": rng.choice(["ldl", "qr"]), "horizon": _log(rng, 4, 30),
                "n": _log(rng, 64, 16384), "solves": rng.choice([0, 0, 2])}
    return {"kind": kind, "f": rng.choice(["cartpole", "quadrotor"]), "n": _log(rng, 1000, 1048576)}


# ---------------------------------------------------------------- inputs ---

def _generator(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000003 * salt + seed)


def _uniform(g, rows, n, a):
    return torch.rand((rows, n), dtype=F64, device="cuda", generator=g).mul_(2 * a).sub_(a)


def _normal(g, rows, n):
    return torch.randn((rows, n), dtype=F64, device="cuda", generator=g)


def _function_inputs(f, n, seed, salt):
    """States and angles in [-1, 1]; the cart-pole's force in [-10, 10]."""
    g = _generator(seed, salt)
    return [_uniform(g, f.nnz_in(i), n, 10.0 if (f.name(), i) == ("cartpole", 1) else 1.0) for i in range(f.n_in())]


# ------------------------------------------- Functions and their handles ---
# A program makes these once and keeps them; the inputs are new each time.

@functools.lru_cache(maxsize=None)
def _step(name):
    return STEPS[name]()


@functools.lru_cache(maxsize=4)
def _map(name, n):
    return _step(name).map(n, "hip")


@functools.lru_cache(maxsize=4)
def _jacobian(name):
    return HipJacobian(_step(name), engine="jit")


@functools.lru_cache(maxsize=4)
def _lagrangian_gradient(horizon):
    w, lam, lag = W.quadrotor_ocp_lagrangian(horizon)
    return Function("grad_lag", [w, lam], [gradient(lag, w)])


@functools.lru_cache(maxsize=2)
def _hessian(horizon):
    return HipJacobian(_lagrangian_gradient(horizon), symmetric=True, first_block=True, engine="jit")


@functools.lru_cache(maxsize=8)
def _rollout(steps):
    return W.cartpole_rollout(steps)


def _rollout_every(case):
    """The checkpoint interval in tape instructions: case["ckpt"] steps."""
    segments = -(-case["steps"] // case["ckpt"])
    return -(-_rollout(case["steps"]).n_instructions() // segments)


@functools.lru_cache(maxsize=8)
def _rollout_tape(steps, engine):
    return HipTape(_rollout(steps), engine=engine)


@functools.lru_cache(maxsize=4)
def _trainable(chain, steps, ckpt, every):
    if chain == "mapaccum":
        return W.cartpole_cost_step().mapaccum("rollout", steps).to_torch(checkpoint_every=ckpt)
    return _rollout(steps).to_torch(checkpoint_every=every)


@functools.lru_cache(maxsize=4)
def _linsol(solver, horizon):
    return Linsol("kkt", solver, W.ocp_kkt_sparsity(horizon)[0])


@functools.lru_cache(maxsize=4)
def _mapsum(name, n):
    return _step(name).map("total", "hip", n, ["u"], [0])


def _inputs(case, seed):
    kind, n = case["kind"], case.get("n")
    if kind in ("map", "map_host", "jacobian"):
        args = _function_inputs(_step(case["f"]), n, seed, 1)
        return {"args": [a.cpu().numpy() for a in args] if kind == "map_host" else args}
    if kind == "hessian":
        g = _generator(seed, 2)
        f = _lagrangian_gradient(case["horizon"])
        return {"args": [_uniform(g, f.nnz_in(0), n, 1.0), _normal(g, f.nnz_in(1), n)]}
    if kind == "rollout":
        g = _generator(seed, 3)
        return {"args": [_uniform(g, 4, n, 1.0), _uniform(g, case["steps"], n, 10.0)],
                "seeds": [torch.ones((1, n), dtype=F64, device="cuda")]}
    if kind == "train":
        g = _generator(seed, 4)
        chained = case["chain"] == "mapaccum"
        x0, u = _uniform(g, 4, n, 1.0), _uniform(g, case["steps"], n, 10.0)
        if chained:  # the state carries the running cost
            x0 = torch.cat([x0, torch.zeros((1, n), dtype=F64, device="cuda")])
        return {"args": [x0.requires_grad_(), u.requires_grad_()],
                "cotangent": _normal(g, 5 * case["steps"] if chained else 1, n)}
    if kind == "batch":
        fs = [_step(name) for name in MIXED]
        return {"args": [_function_inputs(f, case[f.name()], seed, 5 + i) for i, f in enumerate(fs)],
                "seeds": [[_normal(_generator(seed, 8 + i), f.nnz_out(0), case[f.name()])] for i, f in enumerate(fs)]}
    if kind == "kkt":
        sp, a = W.ocp_kkt_batch(np.random.default_rng([seed, 11]), n, case["horizon"])
        return {"a": torch.tensor(a, device="cuda"),
                "b": [_normal(_generator(seed, 12 + i), sp.size1(), n) for i in range(max(1, case["solves"]))]}
    if kind == "mapsum":
        f = _step(case["f"])
        g = _generator(seed, 20)
        return {"args": [_uniform(g, f.nnz_in(0), n, 1.0), _uniform(g, f.nnz_in(1), 1, 1.0).reshape(-1)],
                "seeds": [_normal(g, f.nnz_out(0), 1).reshape(-1)]}
    raise ValueError(kind)


_called = set()


def prepare(case, seed):
    s = dict(_inputs(case, seed), case=case)
    kind, n = case["kind"], case.get("n")
    if kind in ("map", "map_host"):
        s["call"] = _map(case["f"], n)
    elif kind == "jacobian":
        s["call"] = _jacobian(case["f"])
    elif kind == "hessian":
        s["call"] = _hessian(case["horizon"])
    elif kind == "rollout":
        s["tape"], s["every"] = _rollout_tape(case["steps"], case["engine"]), _rollout_every(case)
    elif kind == "train":
        chained = case["chain"] == "mapaccum"
        s["call"] = _trainable(case["chain"], case["steps"], case["ckpt"], None if chained else _rollout_every(case))
    elif kind == "batch":
        s["batch"] = HipBatch([_step(name) for name in MIXED], [case[name] for name in MIXED])
        s["out"] = [s["batch"].bind(i, a, c) for i, (a, c) in enumerate(zip(s["args"], s["seeds"]))]
        s["batch"].tune(reps=3)
    elif kind == "kkt":
        s["linsol"] = _linsol(case["solver"], case["horizon"])
    elif kind == "mapsum":
        s["call"] = _mapsum(case["f"], n)
    key = tuple(sorted((k, v) for k, v in case.items() if k != "name"))
    if key not in _called:  # the first call of a handle compiles its kernels; a program makes it once
        _called.add(key)
        run(s)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind in ("map", "map_host"):
        return state["call"](*state["args"])
    if kind in ("jacobian", "hessian"):
        return state["call"](state["args"])
    if kind == "rollout":
        return state["tape"].fwd_adj(state["args"], state["seeds"], checkpoint_every=state["every"])
    if kind == "train":
        out = state["call"](*state["args"])
        return out, torch.autograd.grad(out, state["args"], state["cotangent"])
    if kind == "batch":
        state["batch"].launch(graph=None)
        return state["out"]
    if kind == "kkt":
        if case["solves"] == 0:
            return state["linsol"].solve_batch(state["a"], state["b"][0])
        state["linsol"].nfact(state["a"])
        return [state["linsol"].solve(b) for b in state["b"]]
    return state["call"].fwd_adj(state["args"], state["seeds"])


# ---------------------------------------------------------------- work ---

def _ops(f):
    """Operations of one instance: forward one per arithmetic instruction; adjoint, per operand, a partial, a product
    and a sum."""
    a = f.instructions()["op"]
    arith = a[(a != OP.CONST) & (a != OP.INPUT) & (a != OP.OUTPUT)]
    operands = np.where(np.isin(arith, [int(b) for b in BINARY]), 2, 1)
    return int(arith.size), int(3 * operands.sum())


def _io(f):
    return sum(f.nnz_in(i) for i in range(f.n_in())), sum(f.nnz_out(i) for i in range(f.n_out()))


def work(case):
    kind, n = case["kind"], case.get("n")
    if kind in ("map", "map_host"):
        f = _step(case["f"])
        return {"bytes": 8 * n * sum(_io(f)), "flops": n * _ops(f)[0]}
    if kind in ("jacobian", "hessian"):
        f = _step(case["f"]) if kind == "jacobian" else _lagrangian_gradient(case["horizon"])
        plan = f.jac_plan(kind == "hessian", kind == "hessian")
        # one product and one sum per nonzero operand tangent; a seed direction reaches about a third of the tape
        fwd, adj = _ops(f)
        return {"bytes": 8 * n * (sum(_io(f)) + plan["jsp"].nnz()), "flops": int(n * (fwd + plan["ndir"] * adj * 2 / 9))}
    if kind == "rollout":
        f = _rollout(case["steps"])
        return {"bytes": 8 * n * 2 * sum(_io(f)), "flops": n * sum(_ops(f))}
    if kind == "train":
        f, steps = _rollout(case["steps"]), case["steps"]
        out = 5 * steps if case["chain"] == "mapaccum" else 1
        return {"bytes": 8 * n * 2 * (4 + (out > 1) + steps + out), "flops": n * sum(_ops(f))}
    if kind == "batch":
        fs = [_step(name) for name in MIXED]
        return {"bytes": sum(16 * case[f.name()] * sum(_io(f)) for f in fs),
                "flops": sum(case[f.name()] * sum(_ops(f)) for f in fs)}
    if kind == "kkt":
        sp = W.ocp_kkt_sparsity(case["horizon"])[0]
        m, rhs = sp.size1(), max(1, case["solves"])
        if case["solver"] == "ldl":
            lt, _ = sp.ldl()
            length = np.diff(lt.colind)
            factor = int((2 * length[lt.row] + 3).sum())
            solve = 4 * lt.nnz() + m
        else:
            v, r, _, _ = sp.qr_sparse()
            length = np.diff(v.colind)
            above = r.row < r.get_col()
            factor = int((4 * length[r.row[above]]).sum() + 3 * length.sum())
            solve = int(4 * length.sum() + 2 * r.nnz())
        return {"bytes": 8 * n * (sp.nnz() + 2 * m * rhs), "flops": n * (factor + rhs * solve)}
    f = _step(case["f"])
    return {"bytes": 8 * n * 2 * f.nnz_in(0), "flops": n * sum(_ops(f))}


def tolerance(case):
    # FP64 with other roundings of sin and cos (1 ulp): a step, a Jacobian or a Hessian is good to a few 1e-16 of its
    # size.  A rollout is chaotic at these forces and carries a rounding on, by up to 1e5 over 100 steps (7e-11
    # against torch's reverse mode); the KKT systems' condition (their dual regularisation is 1e-8; 5e-11 against
    # block elimination) and the cancellation in sums over samples do the same.
    kind = case["kind"]
    if kind in ("rollout", "train"):
        return {"rel": 1e-9, "max": 1e-6}
    if kind == "kkt":
        return {"rel": 1e-9, "max": 1e-6}
    if kind == "mapsum":
        return {"rel": 1e-12, "max": 1e-11}
    return {"rel": 2e-15, "max": 2e-13}


# --------------------------------------------------------------- exact ---
# The same quantities in plain torch, by torch's own reverse mode.

def _cartpole_ode(x, u):
    _, th, xd, thd = x
    s, c = torch.sin(th), torch.cos(th)
    temp = (u + 0.05 * thd * thd * s) / 1.1
    thacc = (9.81 * s - c * temp) / (0.5 * (4.0 / 3.0 - 0.1 * c * c / 1.1))
    return torch.stack([xd, thd, temp - 0.05 * thacc * c / 1.1, thacc])


def _quadrotor_ode(x, u):
    phi, th, psi, p, q, r = x[6:]
    cph, sph, cth, sth, cps, sps = phi.cos(), phi.sin(), th.cos(), th.sin(), psi.cos(), psi.sin()
    zb = torch.stack([cps * sth * cph + sps * sph, sps * sth * cph - cps * sph, cth * cph])
    acc = zb * u[0] - torch.tensor([[0.0], [0.0], [9.81]], dtype=F64, device=x.device)
    rates = torch.stack([p + (q * sph + r * cph) * torch.tan(th), q * cph - r * sph, (q * sph + r * cph) / cth])
    body = torch.stack([(u[1] - 0.01 * q * r) / 0.01, (u[2] + 0.01 * r * p) / 0.01, u[3] / 0.02])
    return torch.cat([x[3:6], acc, rates, body])


def _rk4(ode, x, u, dt):
    k1 = ode(x, u)
    k2 = ode(x + dt / 2 * k1, u)
    k3 = ode(x + dt / 2 * k2, u)
    k4 = ode(x + dt * k3, u)
    return x + dt / 6 * (k1 + 2 * k2 + 2 * k3 + k4)


def _exact_cartpole(x, u):
    return _rk4(_cartpole_ode, x, u[0], 0.05)


def _exact_quadrotor(x, u):
    return _rk4(_quadrotor_ode, x, u, 0.02)


def _exact_arm(z):
    q1, q2, v1, v2, t1, t2 = z
    c2, h = torch.cos(q2), torch.sin(q2)
    m11, m12 = 3 + 2 * c2, 1 + c2
    g2 = 9.81 * torch.cos(q1 + q2)
    r1 = t1 + h * (2 * v1 * v2 + v2 * v2) - (2 * 9.81 * torch.cos(q1) + g2)
    r2 = t2 - h * v1 * v1 - g2
    det = m11 - m12 * m12
    return torch.stack([v1, v2, (r1 - m12 * r2) / det, (m11 * r2 - m12 * r1) / det])


EXACT = {"cartpole": _exact_cartpole, "quadrotor": _exact_quadrotor, "arm": _exact_arm}


def _with_gradient(fn, args, cotangent):
    args = [a.detach().clone().requires_grad_() for a in args]
    out = fn(*args)
    return out.detach(), torch.autograd.grad(out, args, cotangent)


def _exact_rollout(x, us):
    cost = 0.0
    for u in us:
        cost = cost + (x * x).sum(0) + 0.01 * u * u
        x = _rk4(_cartpole_ode, x, u, 0.05)
    return (cost + (x * x).sum(0)).reshape(1, -1)


def _exact_chain(xc, us):
    x, c, out = xc[:4], xc[4], []
    for u in us:
        c = c + (x * x).sum(0) + 0.01 * u * u
        x = _rk4(_cartpole_ode, x, u, 0.05)
        out += [x, c.reshape(1, -1)]
    return torch.cat(out)


def _derivative_rows(fn, x):
    """(rows, columns, n) derivative of fn(x) (rows, n) by the rows of x, per instance."""
    x = x.detach().clone().requires_grad_()
    y = fn(x)
    rows = [torch.autograd.grad(y[i].sum(), x, retain_graph=True, materialize_grads=True)[0] for i in range(y.shape[0])]
    return y.detach(), torch.stack(rows)


def _nonzeros(dense, pattern):
    """The entries of dense (rows, columns, n) in the order of column-compressed nonzeros."""
    col, row = torch.nonzero(pattern.T, as_tuple=True)
    return dense[row, col]


def _exact_step_jacobian(name, args):
    split = np.cumsum([a.shape[0] for a in args])[:-1].tolist()
    y, jac = _derivative_rows(lambda z: EXACT[name](*torch.tensor_split(z, split)), torch.cat(args))
    return [y], _nonzeros(jac, (jac != 0).any(2))


def _exact_hessian(horizon, w, lam):
    """The Hessian by stages: stage k's terms depend on x_k, u_k (and on x_{k+1} linearly)."""
    n = w.shape[1]
    stages = w[:16 * horizon].reshape(horizon, 16, n).transpose(0, 1).reshape(16, horizon * n)
    mult = lam.reshape(horizon, 12, n).transpose(0, 1).reshape(12, horizon * n)

    def grad(z):
        with torch.enable_grad():
            value = (z[:12] ** 2).sum() + 0.1 * (z[12:] ** 2).sum() + (mult * _exact_quadrotor(z[:12], z[12:])).sum()
            return torch.autograd.grad(value, z, create_graph=True)[0]

    g, block = _derivative_rows(grad, stages)
    block = block.reshape(16, 16, horizon, n)
    pattern = (block != 0).any(3).any(2)
    blocks = [_nonzeros(block[:, :, k], pattern) for k in range(horizon)]
    last = torch.full((12, n), 2.0, dtype=F64, device=w.device)
    g = g.reshape(16, horizon, n).transpose(0, 1).reshape(16 * horizon, n)
    g = torch.cat([g, 2 * w[16 * horizon:]])
    for k in range(horizon):  # the multiplier's term -lam_k^T x_{k+1}
        g[16 * (k + 1):16 * (k + 1) + 12] -= lam[12 * k:12 * (k + 1)]
    return [g], torch.cat(blocks + [last])


def _exact_kkt(case, a, b):
    """Block elimination along the horizon: a block holds a stage's multipliers, state and control."""
    horizon, n = case["horizon"], a.shape[1]
    nw, dim = 5 * horizon, 9 * horizon + 4
    pattern = torch.zeros((dim, dim), dtype=torch.bool, device=a.device)
    for k in range(horizon):
        pattern[5 * k:5 * k + 5, 5 * k:5 * k + 5] = True
        pattern[nw + 4 * (k + 1):nw + 4 * (k + 2), 5 * k:5 * k + (9 if k + 1 < horizon else 5)] = True
    pattern[nw:nw + 4, 0:4] = True
    pattern |= pattern.T.clone()
    pattern |= torch.eye(dim, dtype=torch.bool, device=a.device)
    col, row = torch.nonzero(pattern.T, as_tuple=True)
    dense = torch.zeros((n, dim, dim), dtype=F64, device=a.device)
    dense[:, row, col] = a.T
    at = [list(range(nw + 4 * k, nw + 4 * k + 4)) + (list(range(5 * k, 5 * k + 5)) if k < horizon else [])
          for k in range(horizon + 1)]

    def block(i, j):
        r, c = (torch.tensor(at[q], device=a.device) for q in (i, j))
        return dense[:, r][:, :, c]

    rhs = torch.stack(b, 2).transpose(0, 1)                      # (n, dim, right-hand sides)
    diag, y = [block(0, 0)], [rhs[:, at[0]]]
    for k in range(1, horizon + 1):
        low = torch.linalg.solve(diag[-1].transpose(1, 2), block(k, k - 1).transpose(1, 2)).transpose(1, 2).contiguous()
        diag.append(block(k, k) - low @ block(k - 1, k).contiguous())
        y.append(rhs[:, at[k]] - low @ y[-1].contiguous())
    x = torch.empty_like(rhs)
    nxt = None
    for k in range(horizon, -1, -1):
        r = y[k] if nxt is None else y[k] - block(k, k + 1).contiguous() @ nxt
        nxt = torch.linalg.solve(diag[k], r)
        x[:, at[k]] = nxt
    return [x[:, :, i].T.contiguous() for i in range(x.shape[2])]


def exact(case, seed):
    kind = case["kind"]
    s = _inputs(case, seed)
    args = s.get("args")
    if kind == "map":
        return EXACT[case["f"]](*args)
    if kind == "map_host":
        return EXACT[case["f"]](*[torch.tensor(a, device="cuda") for a in args]).cpu().numpy()
    if kind == "jacobian":
        return _exact_step_jacobian(case["f"], args)
    if kind == "hessian":
        return _exact_hessian(case["horizon"], *args)
    if kind == "rollout":
        out, grad = _with_gradient(_exact_rollout, args, s["seeds"][0])
        return [out], grad
    if kind == "train":
        return _with_gradient(_exact_chain if case["chain"] == "mapaccum" else _exact_rollout, args, s["cotangent"])
    if kind == "batch":
        out = []
        for name, a, c in zip(MIXED, args, s["seeds"]):
            y, grad = _with_gradient(EXACT[name], a, c[0])
            out.append(([y], grad))
        return out
    if kind == "kkt":
        x = _exact_kkt(case, s["a"], s["b"])
        return x if case["solves"] else (x[0], None)
    n = case["n"]
    shared = args[1].reshape(-1, 1).expand(-1, n).contiguous()
    y, (gx, gu) = _with_gradient(EXACT[case["f"]], [args[0], shared], s["seeds"][0].reshape(-1, 1).expand(-1, n))
    return [y.sum(1)], [gx, gu.sum(1)]
