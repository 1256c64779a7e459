"""What a user of lineax_amd has it do: the calls whose speed is watched.

Every case goes through the package's public entry points (``linear_solve``
with a solver, ``UnevenBatch.cholesky_solve``, ``SolveServer.run``), from a
single system of a dozen unknowns to one LU of order 8192, in float32 and
float64, batched and not, with odd orders, forward and with gradients.  Sizes
are those of the benchmark configurations and the tests, or generic.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  the operators and vectors on the GPU
    run(state)           one pass
    work(case)           the bytes and flops no implementation can avoid
    tolerance(case)      how far two correct implementations may differ
    exact(case, seed)    the same answer in 64 bits by plain torch
"""

from __future__ import annotations

import math

import numpy as np
import torch

import lineax_amd as lx
from lineax_amd.batch import UnevenBatch
from lineax_amd.serving import Request, SolveServer, request_flops
from lineax_amd.stencil import StencilOperator, convection_diffusion_coeffs, poisson2d

DEVICE = "cuda"
DTYPES = {"f32": torch.float32, "f64": torch.float64}


def listed():
    return [
        # one small system: the linear solve inside an implicit ODE or Newton
        # step of a dozen unknowns, where launches and host time are everything
        {"name": "lu_one", "kind": "dense", "solver": "lu", "dtype": "f64", "batch": 1, "m": 12, "n": 12, "rhs": 1,
         "grad": False},
        # the small-LU configuration: 1024 systems of order 32
        {"name": "lu_small", "kind": "dense", "solver": "lu", "dtype": "f32", "batch": 1024, "m": 32, "n": 32,
         "rhs": 1, "grad": False},
        # a batch of medium systems inside a differentiated program: the solve
        # and the gradients of operator and right-hand side
        {"name": "lu_mid_grad", "kind": "dense", "solver": "lu", "dtype": "f32", "batch": 200, "m": 100, "n": 100,
         "rhs": 1, "grad": True},
        # the large-LU configuration: one operator of order 8192, 4 right-hand sides
        {"name": "lu_large", "kind": "dense", "solver": "lu", "dtype": "f32", "batch": 1, "m": 8192, "n": 8192,
         "rhs": 4, "grad": False},
        # a batch of float64 covariance-like systems (Gaussian processes, Gauss-Newton steps)
        {"name": "chol_mid", "kind": "dense", "solver": "chol", "dtype": "f64", "batch": 256, "m": 150, "n": 150,
         "rhs": 1, "grad": False},
        # one larger SPD system
        {"name": "chol_one", "kind": "dense", "solver": "chol", "dtype": "f32", "batch": 1, "m": 1000, "n": 1000,
         "rhs": 1, "grad": False},
        # the uneven-batch configuration: 20,000 SPD systems of orders 8..256
        {"name": "chol_uneven", "kind": "uneven", "count": 20000, "n_min": 8, "n_max": 256},
        # a batch of least-squares problems
        {"name": "qr_batch", "kind": "dense", "solver": "qr", "dtype": "f32", "batch": 256, "m": 512, "n": 256,
         "rhs": 1, "grad": False},
        # one tall regression in float64, odd sizes
        {"name": "qr_tall", "kind": "dense", "solver": "qr", "dtype": "f64", "batch": 1, "m": 3001, "n": 391,
         "rhs": 1, "grad": False},
        # the CG configuration's operator, grid and right-hand sides over a fixed step budget
        {"name": "cg_poisson", "kind": "cg", "grid": 2048, "rhs": 16, "steps": 60},
        # the GMRES configuration's operator, grid and right-hand sides over three restart cycles
        {"name": "gmres_convdiff", "kind": "gmres", "grid": 1024, "rhs": 16, "restart": 30, "cycles": 3},
        # a burst of mixed requests through the request loop (the serving configuration's size ranges)
        {"name": "serving_burst", "kind": "serving", "requests": 40, "m_max": 4096, "n_max": 1024},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _dense(solver, dtype, batch, m, n, rhs=1, grad=False):
    return {"kind": "dense", "solver": solver, "dtype": dtype, "batch": batch, "m": m, "n": n, "rhs": rhs,
            "grad": grad}


def draw(rng):
    kind = rng.choice(["lu_few", "lu_small", "lu_mid", "lu_mid", "lu_large", "chol_small", "chol_mid", "chol_one",
                       "chol_one", "uneven", "qr_batch", "qr_batch", "qr_tall", "cg", "gmres", "serving"])
    dtype = rng.choice(["f32", "f64"])
    if kind == "lu_few":
        n = _log_int(rng, 2, 64)
        return _dense("lu", dtype, rng.randint(1, 8), n, n)
    if kind == "lu_small":
        n = _log_int(rng, 4, 64)
        return _dense("lu", dtype, _log_int(rng, 64, 4096), n, n, 1, rng.random() < 0.3)
    if kind == "lu_mid":
        n = rng.randint(65, 255)
        return _dense("lu", dtype, _log_int(rng, 4, 256), n, n, 1, rng.random() < 0.5)
    if kind == "lu_large":
        n = _log_int(rng, 256, 8192)
        return _dense("lu", "f32", 1, n, n, rng.randint(1, 8))
    if kind == "chol_small":
        n = _log_int(rng, 4, 64)
        return _dense("chol", dtype, _log_int(rng, 1, 2048), n, n)
    if kind == "chol_mid":
        n = rng.randint(65, 256)
        return _dense("chol", dtype, _log_int(rng, 4, 512), n, n, 1, rng.random() < 0.3)
    if kind == "chol_one":
        n = _log_int(rng, 257, 1000)
        return _dense("chol", dtype, _log_int(rng, 1, 16), n, n)
    if kind == "uneven":
        lo = _log_int(rng, 2, 64)
        return {"kind": "uneven", "count": _log_int(rng, 500, 20000), "n_min": lo, "n_max": rng.randint(lo, 256)}
    if kind == "qr_batch":
        m = _log_int(rng, 32, 512)
        return _dense("qr", dtype, _log_int(rng, 8, 256), m, rng.randint(max(1, m // 8), max(1, m // 2)))
    if kind == "qr_tall":
        m = _log_int(rng, 400, 4000)
        return _dense("qr", dtype, rng.randint(1, 4), m, rng.randint(20, 400))
    if kind == "cg":
        return {"kind": "cg", "grid": _log_int(rng, 128, 2048), "rhs": rng.randint(1, 16),
                "steps": rng.randint(31, 60)}
    if kind == "gmres":
        return {"kind": "gmres", "grid": _log_int(rng, 128, 1024), "rhs": rng.randint(1, 16),
                "restart": rng.randint(10, 30), "cycles": rng.randint(1, 3)}
    return {"kind": "serving", "requests": rng.randint(12, 40), "m_max": _log_int(rng, 1024, 4096),
            "n_max": _log_int(rng, 300, 1024)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _spd(g, batch, n, dtype):
    """A = M M^T / n + 0.1 I, built in float64."""
    m = torch.randn((batch, n, n), generator=g, device=DEVICE, dtype=torch.float64)
    a = torch.bmm(m, m.mT.contiguous()) / n + 0.1 * torch.eye(n, device=DEVICE, dtype=torch.float64)
    return (0.5 * (a + a.mT)).to(dtype)


def _dense_inputs(case, seed):
    g = _generator(seed)
    dt = DTYPES[case["dtype"]]
    batch, m, n = case["batch"], case["m"], case["n"]
    if case["solver"] == "chol":
        a = _spd(g, batch, n, dt)
    elif case["solver"] == "lu" and n < 256:
        # the Newton matrices of implicit steps: the identity plus a Jacobian
        a = torch.eye(n, device=DEVICE, dtype=dt) + 0.3 / math.sqrt(n) * torch.randn(
            (batch, n, n), generator=g, device=DEVICE, dtype=dt)
    else:
        a = torch.randn((batch, m, n), generator=g, device=DEVICE, dtype=dt)
    if batch == 1:
        a = a[0]
    lead = () if batch == 1 else (batch,)
    if case["rhs"] > 1:
        lead = (case["rhs"],)
    b = torch.randn((*lead, m), generator=g, device=DEVICE, dtype=dt)
    ct = torch.randn((*lead, n), generator=g, device=DEVICE, dtype=dt) if case["grad"] else None
    return a, b, ct


def _uneven_inputs(case, seed):
    """Orders on the host; matrices packed back to back in system order, on the GPU."""
    # the orders belong to the case, the numbers to the seed
    rng = np.random.default_rng([case["count"], case["n_min"], case["n_max"]])
    ns = rng.integers(case["n_min"], case["n_max"] + 1, size=case["count"]).astype(np.int32)
    a_off = np.concatenate(([0], np.cumsum(ns.astype(np.int64) ** 2)))
    b_off = np.concatenate(([0], np.cumsum(ns.astype(np.int64))))
    g = _generator(seed)
    a = torch.empty(int(a_off[-1]), device=DEVICE, dtype=torch.float32)
    for n in np.unique(ns):
        n = int(n)
        idx = np.flatnonzero(ns == n)
        block = _spd(g, len(idx), n, torch.float32).reshape(len(idx), n * n)
        at = torch.from_numpy(a_off[idx]).to(DEVICE)[:, None] + torch.arange(n * n, device=DEVICE)
        a[at] = block
    b = torch.randn(int(b_off[-1]), generator=g, device=DEVICE, dtype=torch.float32)
    return ns, a_off[:-1], a, b_off[:-1], b


def _serving_inputs(case, seed):
    """Half least squares (m x n, n from m / 4 to m), half SPD; a tenth reuse
    an earlier operator with a new right-hand side; all waiting at the start."""
    # the mix of sizes belongs to the case, the numbers to the seed
    rng = np.random.default_rng([case["requests"], case["m_max"], case["n_max"]])
    g = _generator(seed)
    reqs, ops = [], {}
    for i in range(case["requests"]):
        earlier = [r for r in reqs if r.a is not None]
        if earlier and rng.random() < 0.1:
            old = earlier[int(rng.integers(len(earlier)))]
            kind, m, n, op_id, a, reuse = old.kind, old.m, old.n, old.op_id, None, True
        else:
            op_id, reuse = i, False
            if rng.random() < 0.5:
                kind, m = "qr", int(rng.integers(64, case["m_max"] + 1))
                # down from square by a few rows: an exactly square Gaussian
                # operator's conditioning has no bound to hold answers to
                n = int(rng.integers(-(-m // 4), m - m // 8 + 1))
                a = torch.randn((m, n), generator=g, device=DEVICE, dtype=torch.float32)
            else:
                kind, m = "chol", int(rng.integers(16, case["n_max"] + 1))
                n = m
                a = _spd(g, 1, n, torch.float32)[0]
            ops[op_id] = a
        b = torch.randn((m,), generator=g, device=DEVICE, dtype=torch.float32)
        reqs.append(Request(rid=i, kind=kind, arrival=0.0, m=m, n=n, op_id=op_id, reuse=reuse, a=a, b=b))
    return reqs, ops


def _grid_rhs(case, seed):
    n = case["grid"]
    # smooth sources with noise, float32 data held in float64 (the solve's dtype)
    g = _generator(seed)
    x = torch.linspace(0.0, 1.0, n, device=DEVICE, dtype=torch.float64)
    amp = torch.randn((case["rhs"], 3), generator=g, device=DEVICE, dtype=torch.float64)
    smooth = sum(amp[:, k, None, None] * torch.sin((k + 1) * math.pi * x)[:, None] * torch.sin((k + 2) * math.pi * x)
                 for k in range(3))
    noise = torch.randn((case["rhs"], n, n), generator=g, device=DEVICE, dtype=torch.float32)
    return (smooth + 0.1 * noise.double()).float().double()


def prepare(case, seed):
    if case["kind"] == "dense":
        a, b, ct = _dense_inputs(case, seed)
        if case["grad"]:
            a.requires_grad_(True)
            b.requires_grad_(True)
        solver = {"lu": lx.LU, "chol": lx.Cholesky, "qr": lx.QR}[case["solver"]]()
        return {"kind": "dense", "a": a, "b": b, "ct": ct, "solver": solver,
                "tags": lx.positive_semidefinite_tag if case["solver"] == "chol" else ()}
    if case["kind"] == "uneven":
        ns, a_off, a, b_off, b = _uneven_inputs(case, seed)
        batch = UnevenBatch(ns, a_off, a.cpu().numpy(), b_off, b.cpu().numpy(), device=DEVICE)
        return {"kind": "uneven", "batch": batch}
    if case["kind"] == "cg":
        solver = lx.CG(rtol=1e-6, atol=1e-6, max_steps=case["steps"], working_dtype=torch.float32)
        return {"kind": "krylov", "op": poisson2d(case["grid"], device=DEVICE), "b": _grid_rhs(case, seed),
                "solver": solver}
    if case["kind"] == "gmres":
        n = case["grid"]
        op = StencilOperator(n, n, convection_diffusion_coeffs(n), device=DEVICE)
        # the first step only forms the residual
        solver = lx.GMRES(rtol=1e-6, atol=1e-6, restart=case["restart"], max_steps=case["cycles"] + 1,
                          working_dtype=torch.float32)
        return {"kind": "krylov", "op": op, "b": _grid_rhs(case, seed), "solver": solver}
    reqs, ops = _serving_inputs(case, seed)
    return {"kind": "serving", "requests": reqs, "ops": ops,
            "server": SolveServer(DEVICE, hbm_budget=6 << 30, resident_budget=2 << 30)}


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(state):
    if state["kind"] == "dense":
        a, b = state["a"], state["b"]
        x = lx.linear_solve(lx.MatrixLinearOperator(a, state["tags"]), b, state["solver"]).value
        if state["ct"] is None:
            return x
        ga, gb = torch.autograd.grad(x, (a, b), state["ct"])
        return {"x": x, "grad_a": ga, "grad_b": gb}
    if state["kind"] == "uneven":
        sol = state["batch"].cholesky_solve()
        return {"x": sol.x, "result": sol.result}
    if state["kind"] == "krylov":
        # a fixed budget of steps: stopping at it is the expected end
        sol = lx.linear_solve(state["op"], state["b"], state["solver"], throw=False)
        return {"x": sol.value, "result": sol.result, "steps": sol.stats["num_steps"]}
    state["server"].run(state["requests"], state["ops"])
    return [r.x for r in state["requests"]]


# ---------------------------------------------------------------------------
# unavoidable work
# ---------------------------------------------------------------------------


def _mix(case):
    """Sums over an uneven batch's orders: n (n + 1) / 2, n and flops."""
    rng = np.random.default_rng([case["count"], case["n_min"], case["n_max"]])
    ns = rng.integers(case["n_min"], case["n_max"] + 1, size=case["count"]).astype(np.float64)
    return float(np.sum(ns * (ns + 1) / 2)), float(np.sum(ns)), float(np.sum(ns ** 3 / 3 + 2 * ns ** 2))


def work(case):
    if case["kind"] == "dense":
        e = 4 if case["dtype"] == "f32" else 8
        batch, m, n, rhs = case["batch"], float(case["m"]), float(case["n"]), case["rhs"]
        vec = max(batch, rhs) if batch == 1 else batch
        factor = {"lu": 2 * n ** 3 / 3, "chol": n ** 3 / 3, "qr": 2 * m * n * n - 2 * n ** 3 / 3}[case["solver"]]
        solve = 4 * m * n if case["solver"] == "qr" else 2 * n * n
        matrix = n * (n + 1) / 2 if case["solver"] == "chol" else m * n
        nbytes = e * (batch * matrix + vec * (m + n))
        flops = batch * factor + vec * solve
        if case["grad"]:  # one more solve, the operator's gradient written, cotangent read, gradient of b written
            nbytes += e * (batch * m * n + vec * (m + n))
            flops += vec * (solve + m * n)
        return {"bytes": nbytes, "flops": flops}
    if case["kind"] == "uneven":
        upper, total, flops = _mix(case)
        return {"bytes": 4 * upper + (4 + 8) * total, "flops": flops}
    points = float(case.get("grid", 0)) ** 2 * case.get("rhs", 0)
    if case["kind"] == "cg":
        # nine float32 vector passes per step
        return {"bytes": 36.0 * points * case["steps"], "flops": 20.0 * points * case["steps"]}
    if case["kind"] == "gmres":
        # the basis read once per Arnoldi step and once for the update
        m = case["restart"]
        return {"bytes": 4.0 * points * (m * (m + 1) / 2 + 4 * m) * case["cycles"],
                "flops": 4.0 * points * m * (m + 3) / 2 * case["cycles"]}
    rng = np.random.default_rng([case["requests"], case["m_max"], case["n_max"]])
    nbytes, flops, seen = 0.0, 0.0, []
    for _ in range(case["requests"]):
        if seen and rng.random() < 0.1:
            kind, m, n = seen[int(rng.integers(len(seen)))]
            reuse = True
        else:
            reuse = False
            if rng.random() < 0.5:
                kind, m = "qr", int(rng.integers(64, case["m_max"] + 1))
                n = int(rng.integers(-(-m // 4), m - m // 8 + 1))
            else:
                kind, m = "chol", int(rng.integers(16, case["n_max"] + 1))
                n = m
            seen.append((kind, m, n))
            nbytes += 4.0 * m * n
        nbytes += 4.0 * m + 8.0 * n
        flops += request_flops(Request(0, kind, 0.0, m, n, 0, reuse, None, None))
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# tolerances and 64-bit answers
# ---------------------------------------------------------------------------


def tolerance(case):
    """From the errors measured against ``exact``: 32-bit dense answers up to
    2.5e-6, 64-bit ones 6e-15; refined answers (uneven batches, serving) 2e-12."""
    if case["kind"] == "dense":
        if case["dtype"] == "f64":
            return {"rel": 1e-12}
        if case["solver"] == "lu" and case["n"] >= 256:
            # refined until the backward error is at float32 epsilon: Gaussian
            # operators' conditioning, of about their order, times that
            return {"rel": 1e-3}
        return {"rel": 1e-5}
    if case["kind"] == "uneven":
        return {"rel": 1e-10}
    if case["kind"] == "cg":
        return {"rel": 1e-6}
    if case["kind"] == "gmres":
        return {"rel": 1e-5}
    return {"rel": 1e-10}


def _lstsq(a, b):
    q, r = torch.linalg.qr(a)
    return torch.linalg.solve_triangular(r, q.mT @ b[..., None], upper=True)[..., 0]


def _exact_dense(case, seed):
    a, b, ct = _dense_inputs(case, seed)
    a, b = a.double().cpu(), b.double().cpu()
    if case["solver"] == "qr":
        return _lstsq(a, b)
    if case["solver"] == "chol":
        a = torch.triu(a) + torch.triu(a, 1).mT
    if case["rhs"] > 1:
        return torch.linalg.solve(a, b.mT.contiguous()).mT.contiguous()
    x = torch.linalg.solve(a, b)
    if ct is None:
        return x
    lam = torch.linalg.solve(a.mT.contiguous(), ct.double().cpu())
    return {"x": x, "grad_a": -lam[..., :, None] * x[..., None, :], "grad_b": lam}


def _exact_uneven(case, seed):
    ns, a_off, a, b_off, b = _uneven_inputs(case, seed)
    x = torch.empty(b.numel(), device=DEVICE, dtype=torch.float64)
    for n in np.unique(ns):
        n = int(n)
        idx = np.flatnonzero(ns == n)
        at = torch.from_numpy(a_off[idx]).to(DEVICE)[:, None] + torch.arange(n * n, device=DEVICE)
        bt = torch.from_numpy(b_off[idx]).to(DEVICE)[:, None] + torch.arange(n, device=DEVICE)
        m = a[at].double().reshape(-1, n, n)
        m = torch.triu(m) + torch.triu(m, 1).mT
        x[bt] = torch.linalg.solve(m, b[bt].double())
    return {"x": x, "result": None}


def _five_point(u, coeffs):
    c, w, e, s, n = coeffs
    y = c * u
    y[..., :, 1:] += w * u[..., :, :-1]
    y[..., :, :-1] += e * u[..., :, 1:]
    y[..., 1:, :] += s * u[..., :-1, :]
    y[..., :-1, :] += n * u[..., 1:, :]
    return y


def _dot(u, v):
    return (u * v).sum(dim=(-2, -1), keepdim=True)


def _exact_cg(case, seed):
    coeffs = (4.0, -1.0, -1.0, -1.0, -1.0)
    b = _grid_rhs(case, seed)
    x = torch.zeros_like(b)
    r, p = b.clone(), b.clone()
    g = _dot(r, r)
    for _ in range(case["steps"]):
        q = _five_point(p, coeffs)
        alpha = g / _dot(p, q)
        x += alpha * p
        r -= alpha * q
        g, old = _dot(r, r), g
        p = r + (g / old) * p
    return {"x": x, "result": None, "steps": None}


def _exact_gmres(case, seed):
    coeffs = convection_diffusion_coeffs(case["grid"])
    b_all = _grid_rhs(case, seed)
    m, out = case["restart"], []
    for b in b_all:  # one right-hand side at a time: the float64 basis is large
        x = torch.zeros_like(b)
        for _ in range(case["cycles"]):
            r = b - _five_point(x, coeffs)
            beta = r.norm()
            basis = torch.empty((m + 1, b.numel()), device=DEVICE, dtype=torch.float64)
            basis[0] = (r / beta).reshape(-1)
            hess = torch.zeros((m + 1, m), device=DEVICE, dtype=torch.float64)
            for j in range(m):
                w = _five_point(basis[j].reshape(b.shape), coeffs).reshape(-1)
                for _ in range(2):
                    h = basis[: j + 1] @ w
                    w = w - h @ basis[: j + 1]
                    hess[: j + 1, j] += h
                hess[j + 1, j] = w.norm()
                basis[j + 1] = w / hess[j + 1, j]
            hc = hess.cpu()
            rhs = torch.zeros(m + 1, 1, dtype=torch.float64)
            rhs[0] = float(beta)
            z = torch.linalg.lstsq(hc, rhs).solution[:, 0].to(DEVICE)
            x = x + (z @ basis[:m]).reshape(b.shape)
        out.append(x)
    return {"x": torch.stack(out), "result": None, "steps": None}


def _exact_serving(case, seed):
    reqs, ops = _serving_inputs(case, seed)
    out = []
    for r in reqs:
        a, b = ops[r.op_id].double(), r.b.double()
        if r.kind == "qr":
            # the normal equations in float64, refined once: ample for these operators
            gram = torch.linalg.cholesky(a.mT @ a)
            x = torch.cholesky_solve((a.mT @ b)[:, None], gram)[:, 0]
            x = x + torch.cholesky_solve((a.mT @ (b - a @ x))[:, None], gram)[:, 0]
        else:
            a = torch.triu(a) + torch.triu(a, 1).mT
            x = torch.linalg.solve(a, b)
        out.append(x)
    return out


def exact(case, seed):
    if case["kind"] == "dense":
        return _exact_dense(case, seed)
    if case["kind"] == "uneven":
        return _exact_uneven(case, seed)
    if case["kind"] == "cg":
        return _exact_cg(case, seed)
    if case["kind"] == "gmres":
        return _exact_gmres(case, seed)
    return _exact_serving(case, seed)
