"""The work that programs built on this framework have it do, as cases to measure.

Four kinds of work, each through the package's own Python view (mnc.py) or, where
the arrays already live on the GPU, through the C entry points it binds:

  batch  the entropy closure on a batch of moment vectors (mnc_opt_batch on device
         arrays, mnc_opt_batch_noalloc for serving loops, Context.opt_batch_host as
         the drop-in for a host solver's arrays)
  optcb  the change-of-basis optimiser on host arrays
  step   Heun steps of the moment solver: the state goes in, a program's interval
         between two outputs is advanced, the state comes back for writing
  sn     the discrete-ordinates solver, the independent truth for the closures
  mlp    training of the learned warm start's network

Inputs are made from the seed alone: smooth closures from known multipliers
(u = <m exp(alpha.m)>), near-boundary closures as narrow beams, grids as the
decks' initial conditions with a smooth random modulation of the density.
exact() evaluates the same mathematics in float64 with plain torch and numpy.
"""
import ctypes
import importlib.util
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SQRT_PI = math.sqrt(math.pi)
DEV = "cuda"


def _package():
    name = "closures2d_amd_mnc"
    if name not in sys.modules:
        path = os.path.join(ROOT, "closures-2d_amd", "mnc.py")
        spec = importlib.util.spec_from_file_location(name, path)
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


# ---- the cases --------------------------------------------------------------------

def listed():
    return [
        # a serving loop's call on a handful of M2 closures: launches and latency only
        dict(name="batch-m2-60", kind="batch", entry="noalloc", order=2, quad=12, gaunt=False, cells=60,
             precision="fp64", start="isotropic", beams=0.0, kappa=0.0, tol=1e-8),
        # one subdomain's closures of a time step, started from the previous step's multipliers
        dict(name="batch-m4-2049-warm", kind="batch", entry="device", order=4, quad=16, gaunt=False, cells=2049,
             precision="fp64", start="previous", beams=0.0, kappa=0.0, tol=1e-8),
        # a host solver's arrays handed over once per solve, the Gaunt form of the Hessian
        dict(name="batch-m3-gaunt-30011-host", kind="batch", entry="host", order=3, quad=20, gaunt=True, cells=30011,
             precision="fp64", start="isotropic", beams=0.0, kappa=0.0, tol=1e-6),
        # a large cold batch in mixed precision
        dict(name="batch-m4-200003-mixed", kind="batch", entry="device", order=4, quad=16, gaunt=False, cells=200003,
             precision="mixed", start="isotropic", beams=0.0, kappa=0.0, tol=1e-8),
        # a fifth of the closures near the realizability boundary: uneven iteration counts, some regularized
        dict(name="batch-m4-beams-150001", kind="batch", entry="device", order=4, quad=16, gaunt=False,
             cells=150001, precision="fp64", start="isotropic", beams=0.2, kappa=40.0, tol=1e-8),
        # the change-of-basis optimiser on host arrays
        dict(name="optcb-m4-5003", kind="optcb", order=4, quad=16, cells=5003, bfgs=False, tol=1e-8),
        # the plain M2 Gaussian pulse, ten steps to the next output
        dict(name="step-m2-gauss-50", kind="step", order=2, quad=12, ppn=False, nx=50, ny=50, ic=0, sigma=0.1,
             floor=1e-4, precision="fp64", steps=10),
        # an M4 lattice of a convergence study (ragged), plain double precision
        dict(name="step-m4-lattice-133x101", kind="step", order=4, quad=16, ppn=False, nx=133, ny=101, ic=1,
             sigma=0.0, floor=1e-6, precision="fp64", steps=16),
        # the full-size M4 lattice in mixed precision, at the regression decks' floor
        dict(name="step-m4-lattice-280-mixed", kind="step", order=4, quad=16, ppn=False, nx=280, ny=280, ic=1,
             sigma=0.0, floor=1e-4, precision="mixed", steps=24),
        # the high-order closure on a smooth periodic grid
        dict(name="step-m8-periodic-96", kind="step", order=8, quad=32, ppn=False, nx=96, ny=96, ic=2, sigma=0.0,
             floor=0.0, precision="fp64", steps=2),
        # the discrete-ordinates truth of a convergence study
        dict(name="sn-192-q12", kind="sn", quad=12, nx=192, ny=192, ic=2, steps=84),
        # the warm start's network: minibatches of 4,096 pairs out of a harvested set
        dict(name="mlp-train-4096", kind="mlp", pairs=100000, batch=4096, steps=100),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["batch"] * 5 + ["step"] * 4 + ["optcb", "sn", "mlp"])
    if kind == "batch":
        order, gaunt = rng.choice([1, 2, 3, 4, 4, 4]), rng.random() < 0.25
        cells = _log_int(rng, 50, 200000)
        limits = (("noalloc", 16384), ("host", 50000), ("device", 1 << 30))
        entry = rng.choice([e for e, most in limits if cells <= most])
        c = dict(kind="batch", entry=entry, order=order, quad=rng.choice([12, 14, 16]), gaunt=gaunt, cells=cells,
                 precision=rng.choice(["fp64", "mixed"]), start=rng.choice(["isotropic", "previous"]), beams=0.0,
                 kappa=0.0, tol=1e-6 if gaunt else 1e-8)
        if order == 4 and not gaunt and rng.random() < 0.35:
            c.update(precision="fp64", quad=16, cells=min(cells, 150000), start="isotropic",
                     beams=rng.choice([0.05, 0.1, 0.2]), kappa=rng.choice([10.0, 20.0, 40.0]))
        elif c["precision"] == "fp64":
            c["quad"] = rng.choice([12, 14, 16, 20])
        return c
    if kind == "optcb":
        order = rng.choice([2, 3, 4])
        return dict(kind="optcb", order=order, quad=rng.choice([12, 16]), cells=_log_int(rng, 200, 20000),
                    bfgs=rng.random() < 0.3, tol=1e-8)
    if kind == "step":
        order = rng.choice([1, 2, 3, 4, 4, 4, 8])
        if order == 8:
            return dict(kind="step", order=8, quad=32, ppn=False, nx=_log_int(rng, 24, 96), ny=_log_int(rng, 24, 96),
                        ic=2, sigma=0.0, floor=0.0, precision="fp64", steps=rng.choice([1, 2]))
        nx, ny = _log_int(rng, 24, 280), _log_int(rng, 24, 280)
        ppn = rng.random() < 0.2
        ic = rng.choice([0, 2]) if ppn else rng.choice([0, 1, 2])
        precision = "fp64" if ppn else rng.choice(["fp64", "mixed"])
        return dict(kind="step", order=order, quad=rng.choice([12, 16]), ppn=ppn, nx=nx, ny=ny, ic=ic,
                    sigma=rng.choice([0.1, 0.2]) if ic == 0 else 0.0,
                    floor=rng.choice([1e-4, 1e-6]) if ic == 1 and precision == "fp64" else 1e-4,
                    precision=precision, steps=rng.randint(4, 20))
    if kind == "sn":
        return dict(kind="sn", quad=rng.choice([8, 10, 12, 16]), nx=_log_int(rng, 48, 192), ny=_log_int(rng, 48, 192),
                    ic=rng.choice([1, 2]), steps=rng.randint(20, 84))
    return dict(kind="mlp", pairs=_log_int(rng, 20000, 100000), batch=rng.choice([1000, 2048, 4096, 5000]),
                steps=rng.randint(20, 100))


# ---- the mathematics' own tables (numpy, float64) -------------------------------------

_table_cache = {}


def _legendre(l, m, x):
    """Fully normalised associated Legendre function with the Condon-Shortley sign."""
    s = np.sqrt((1.0 - x) * (1.0 + x))
    p = np.full_like(x, 1.0 / math.sqrt(4.0 * math.pi))
    for k in range(1, m + 1):
        p = -p * s * math.sqrt((2.0 * k + 1.0) / (2.0 * k))
    below = np.zeros_like(x)
    for ll in range(m + 1, l + 1):
        a = math.sqrt((4.0 * ll * ll - 1.0) / (ll * ll - m * m))
        b = math.sqrt(((ll - 1.0) ** 2 - m * m) / (4.0 * (ll - 1.0) ** 2 - 1.0))
        p, below = a * (x * p - b * below), p
    return p


def _tables(order, quad):
    """(w[nq], p[nq][n], xi[nq], eta[nq]) of the mu < 0 hemisphere, as CPU tensors."""
    if (order, quad) not in _table_cache:
        mu, wg = np.polynomial.legendre.leggauss(quad)
        for _ in range(3):           # polished to the last bits
            c = np.zeros(quad + 1)
            c[quad] = 1.0
            pn = np.polynomial.legendre.legval(mu, c)
            dpn = np.polynomial.legendre.legval(mu, np.polynomial.legendre.legder(c))
            mu = mu - pn / dpn
        wg = 2.0 / ((1.0 - mu * mu) * dpn * dpn)
        mu, wg = mu[:quad // 2], wg[:quad // 2]
        phi = (np.arange(2 * quad) + 0.5) * math.pi / quad
        mq, pq = np.repeat(mu, 2 * quad), np.tile(phi, quad // 2)
        w = np.repeat(2.0 * math.pi / quad * wg, 2 * quad)
        st = np.sqrt(1.0 - mq * mq)
        cols = []
        for l in range(order + 1):
            for m in range(-l, l + 1):
                if (l + m) % 2 == 0:
                    y = _legendre(l, abs(m), mq)
                    cols.append(y if m == 0 else math.sqrt(2.0) * (np.sin if m < 0 else np.cos)(m * pq) * y)
        _table_cache[order, quad] = tuple(torch.from_numpy(np.ascontiguousarray(a)) for a in (
            w, np.stack(cols, axis=1), st * np.cos(pq), st * np.sin(pq)))
    return _table_cache[order, quad]


def _moments_of(alpha, w, p):
    """u = <m exp(alpha.m)>, in slices that keep the quadrature values small."""
    return torch.cat([torch.exp(a @ p.T) @ (w[:, None] * p) for a in alpha.split(65536)])


# ---- batches ----------------------------------------------------------------------------

def _batch_inputs(case, seed):
    """(u, alpha passed in, alpha of u; NaN rows for beams) on the GPU."""
    w, p, xi, eta = (t.to(DEV) for t in _tables(case["order"], case["quad"]))
    n, nm = case["cells"], p.shape[1]
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    f64 = dict(dtype=torch.float64, device=DEV, generator=g)
    k = torch.arange(nm, dtype=torch.float64, device=DEV)
    true = torch.randn(n, nm, **f64) * (3.0 / (1.0 + k))
    true[:, 0] = torch.rand(n, **f64) * 4.0 - 2.0
    u = _moments_of(true, w, p)
    if case.get("beams"):            # one to three beams of angular width kappa^-1/2
        rows = torch.randperm(n, device=DEV, generator=g)[:int(round(case["beams"] * n))]
        nb = len(rows)
        om = torch.stack([xi, eta, -torch.sqrt((1.0 - xi * xi - eta * eta).clamp(min=0.0))], dim=1)
        count = torch.randint(1, 4, (nb, 1), device=DEV, generator=g)
        c = (0.1 + 0.9 * torch.rand(nb, 3, **f64)) * (torch.arange(3, device=DEV)[None, :] < count)
        z, ph = -torch.rand(nb, 3, **f64), 2.0 * math.pi * torch.rand(nb, 3, **f64)
        r = torch.sqrt(1.0 - z * z)
        axis = torch.stack([r * torch.cos(ph), r * torch.sin(ph), z], dim=2)
        f = torch.zeros(nb, len(w), dtype=torch.float64, device=DEV)
        for j in range(3):
            f += c[:, j:j + 1] * torch.exp(case["kappa"] * (axis[:, j] @ om.T - 1.0))
        u[rows] = f @ (w[:, None] * p)
        true[rows] = math.nan
    if case.get("start") == "previous":
        start = true + 0.02 * torch.randn(n, nm, **f64) / (1.0 + k)
    else:                            # the multipliers of the isotropic state of the same density
        start = torch.zeros_like(true)
        start[:, 0] = 2.0 * SQRT_PI * (torch.log(u[:, 0]) - math.log(2.0 * SQRT_PI))
    return u, start, true


def _prepare_batch(case, seed):
    mnc = _package()
    u, start, _ = _batch_inputs(case, seed)
    ctx = mnc.Context(case["order"], case["quad"], use_gaunt=case["gaunt"])
    opt = mnc.options(tol=case["tol"], line_search=mnc.LS_ROBUST,
                      precision=mnc.PREC_MIXED if case["precision"] == "mixed" else mnc.PREC_FP64)
    s = dict(case=case, ctx=ctx, opt=opt)
    if case["entry"] == "host":
        s.update(u=u.cpu().numpy(), alpha=start.cpu().numpy())
    else:
        s.update(u=u, alpha=start, u_io=torch.empty_like(u), alpha_io=torch.empty_like(start))
    torch.cuda.synchronize()
    return s


def _run_batch(s):
    ctx, case = s["ctx"], s["case"]
    if case["entry"] == "host":
        _, u, alpha, _, _, _ = ctx.opt_batch_host(s["u"], s["alpha"], s["opt"])
        return {"u": u, "alpha": alpha}
    lib = _package().lib()
    call = lib.mnc_opt_batch_noalloc if case["entry"] == "noalloc" else lib.mnc_opt_batch
    s["u_io"].copy_(s["u"])
    s["alpha_io"].copy_(s["alpha"])
    torch.cuda.current_stream().synchronize()      # the context solves on its own stream
    st = call(ctx.h, case["cells"], s["u_io"].data_ptr(), s["alpha_io"].data_ptr(), ctypes.byref(s["opt"]), None)
    if st != 0:
        raise RuntimeError("closure solve failed (status %d)" % st)
    return {"u": s["u_io"], "alpha": s["alpha_io"]}


def _prepare_optcb(case, seed):
    mnc = _package()
    u, _, _ = _batch_inputs(dict(case, start="isotropic"), seed)
    ctx = mnc.Context(case["order"], case["quad"])
    n, nm = u.shape
    a0 = np.zeros((n, nm))
    a0[:, 0] = 2.0 * SQRT_PI * math.log(0.5 / SQRT_PI)
    opt = mnc.options(tol=case["tol"], line_search=mnc.LS_ROBUST,
                      opt_type=mnc.OPT_BFGS if case["bfgs"] else mnc.OPT_CHANGE_BASIS)
    return dict(case=case, ctx=ctx, opt=opt, u=u.cpu().numpy(),
                basis=np.tile(np.eye(nm).reshape(1, -1), (n, 1)), alpha=a0)


def _run_optcb(s):
    _, u, basis, alpha_p, alpha_m, _, _, _ = s["ctx"].optcb_batch_host(s["u"], s["basis"], s["alpha"], s["opt"])
    return {"u": u, "basis": basis, "alpha_p": alpha_p, "alpha_m": alpha_m}


def _exact_optcb(case, seed):
    # the basis ends as the Cholesky factor of the scaled problem's Hessian at
    # the solution (only Newton's own move of the basis ends there exactly)
    u, _, true = _batch_inputs(dict(case, start="isotropic"), seed)
    if case["bfgs"]:
        return {"u": u, "basis": None, "alpha_p": None, "alpha_m": true}
    w, p, _, _ = (t.to(DEV) for t in _tables(case["order"], case["quad"]))
    a = true.clone()
    a[:, 0] -= 2.0 * SQRT_PI * torch.log(u[:, 0])
    L = torch.linalg.cholesky(_hessian(torch.exp(a @ p.T) * w, p).cpu()).to(DEV)
    return {"u": u, "basis": L.transpose(1, 2).reshape(len(u), -1),
            "alpha_p": (L.transpose(1, 2) * a[:, None, :]).sum(dim=2), "alpha_m": true}


# ---- Heun steps of the moment solver -------------------------------------------------------

LATTICE = ((2, 2), (2, 0), (2, -2), (1, 1), (1, -1), (0, -2), (-1, 1), (-1, -1), (-2, 2), (-2, 0), (-2, -2))
THETA, CFL, DELTA_PPN = 2.0, 0.9, 1e-10


def _grid(case, seed):
    """Cell sizes, cross sections and density of the deck's initial condition (two
    ghost layers), the density modulated smoothly at random."""
    nx, ny, ic = case["nx"], case["ny"], case["ic"]
    half = 3.5 if ic == 1 else 1.0
    dx, dy = 2.0 * half / nx, 2.0 * half / ny
    x = (-half + (np.arange(nx + 4) - 2) * dx + dx / 2.0)[:, None]
    y = (-half + (np.arange(ny + 4) - 2) * dy + dy / 2.0)[None, :]
    inner = np.zeros((nx + 4, ny + 4), dtype=bool)
    inner[2:-2, 2:-2] = True
    sig_t, sig_s = np.ones((nx + 4, ny + 4)), np.ones((nx + 4, ny + 4))
    if ic == 0:
        s2 = case["sigma"] ** 2
        pulse = np.maximum(np.exp(-(x * x + y * y) / (2.0 * s2)) / (2.0 * math.pi * s2), case["floor"])
        rho = np.where(inner, pulse, case["floor"])
    elif ic == 1:
        rho = np.full((nx + 4, ny + 4), case["floor"])
        block = np.zeros_like(inner)
        for cx, cy in LATTICE:
            block |= (np.abs(x - cx) < 0.5) & (np.abs(y - cy) < 0.5)
        sig_t[block & inner], sig_s[block & inner] = 10.0, 0.0
    else:
        rho = 1.0 + 0.5 * np.sin(math.pi * x) * np.sin(math.pi * y)
    rng = np.random.default_rng(seed)
    ph = rng.uniform(0.0, 2.0 * math.pi, (3, 2))
    for i, (kx, ky) in enumerate(((1, 1), (2, 1), (1, 3))):
        wave = np.sin(kx * math.pi * x / half + ph[i, 0]) * np.sin(ky * math.pi * y / half + ph[i, 1])
        rho = rho * (1.0 + 0.1 * wave)
    return half, dx, dy, sig_t, sig_s, rho


def _isotropic_state(rho, nm, ppn):
    m, a = np.zeros(rho.shape + (nm,)), np.zeros(rho.shape + (nm,))
    m[..., 0] = 2.0 * SQRT_PI * rho
    a[..., 0] = m[..., 0] - 4.0 * math.pi * DELTA_PPN / m[..., 0] if ppn else 2.0 * SQRT_PI * np.log(rho)
    return m, a


def _time_step(dx, dy):
    return CFL * (2.0 / (2.0 + THETA)) * (dx * dy) / (dx + dy)


def _prepare_step(case, seed):
    mnc = _package()
    half, dx, dy, sig_t, sig_s, rho = _grid(case, seed)
    ctx = mnc.Context(case["order"], case["quad"], moment_type=mnc.MOMENT_PPN if case["ppn"] else mnc.MOMENT_MN)
    m, a = _isotropic_state(rho, ctx.nm, case["ppn"])
    delta = DELTA_PPN if case["ppn"] else 0.0
    ctx.grid_create(case["nx"], case["ny"], dx, dy, -half, -half, case["ic"], THETA, m, a, sig_t, sig_s,
                    delta_ppn=delta)
    opt = mnc.options(tol=1e-8, line_search=mnc.LS_ROBUST, delta_ppn=delta,
                      precision=mnc.PREC_MIXED if case["precision"] == "mixed" else mnc.PREC_FP64)
    return dict(case=case, ctx=ctx, opt=opt, m=m, a=a, dt=_time_step(dx, dy))


def _run_step(s):
    ctx = s["ctx"]
    ctx.grid_set(s["m"], s["a"])
    for _ in range(s["case"]["steps"]):
        ctx.update(s["dt"], s["opt"])
    m, a = ctx.grid_get()
    return {"moments": m, "alpha": a}


def _hessian(we, p):
    """sum_q we_q p_q p_q^T per cell, from the products of the columns."""
    n = p.shape[1]
    i, j = torch.tril_indices(n, n, device=p.device)
    low = we @ (p[:, i] * p[:, j])
    H = torch.empty(len(we), n, n, dtype=p.dtype, device=p.device)
    H[:, i, j] = low
    H[:, j, i] = low
    return H


def _spd_solve(H, g):
    """H^-1 g for a batch, the factor formed column by column."""
    n = g.shape[1]
    L = torch.zeros_like(H)
    y = g.clone()
    for j in range(n):
        c = H[:, j:, j] - (L[:, j:, :j] * L[:, j:j + 1, :j]).sum(dim=2)
        L[:, j:, j] = c / torch.sqrt(c[:, :1])
        y[:, j] = (y[:, j] - (L[:, j, :j] * y[:, :j]).sum(dim=1)) / L[:, j, j]
    for j in range(n - 1, -1, -1):
        y[:, j] = (y[:, j] - (L[:, j + 1:, j] * y[:, j + 1:]).sum(dim=1)) / L[:, j, j]
    return y


def _ansatz(z, delta):
    """(value, its derivative, the dual integrand) of the closure's ansatz at z."""
    if delta is None:
        e = torch.exp(z)
        return e, e, e
    t = 0.5 * z
    r = torch.sqrt(t * t + delta)
    G = torch.where(t < 0.0, -delta / (t - r), t + r)
    return G, 0.5 * G / r, t * G - 0.5 * delta + delta * torch.log(G)


def _solve_exact(u, a, w, p, ppn):
    """The dual problem to convergence: damped Newton on the u0 = 1 problem."""
    u0 = u[:, :1]
    us, al = u / u0, a.clone()
    if ppn:
        al /= u0
    else:
        al[:, :1] -= 2.0 * SQRT_PI * torch.log(u0)
    todo = torch.arange(len(u), device=u.device)
    for _ in range(80):
        if not len(todo):
            break
        left = []
        for rows in todo.split(16384):
            A, U = al[rows], us[rows]
            delta = DELTA_PPN / u0[rows] ** 2 if ppn else None
            value, slope, dual = _ansatz(A @ p.T, delta)
            g = (value * w) @ p - U
            d = -_spd_solve(_hessian(slope * w, p), g)
            f = (dual * w).sum(dim=1) - (A * U).sum(dim=1)
            gd, scale = (g * d).sum(dim=1), 1.0 + f.abs()
            t = torch.ones(len(rows), 1, dtype=u.dtype, device=u.device)
            for _ in range(30):
                B = A + t * d
                fn = (_ansatz(B @ p.T, delta)[2] * w).sum(dim=1) - (B * U).sum(dim=1)
                bad = ~((fn <= f + 1e-3 * t[:, 0] * gd) | (-gd <= 1e-11 * scale))
                if not bad.any():
                    break
                t = torch.where(bad[:, None], 0.5 * t, t)
            al[rows] = A + t * d
            left.append(rows[(t * d).abs().amax(dim=1) > 1e-11 * (1.0 + A.abs().amax(dim=1))])
        todo = torch.cat(left)
    if ppn:
        return al * u0
    al[:, :1] += 2.0 * SQRT_PI * torch.log(u0)
    return al


def _minmod(a, b):
    s = torch.where(a >= 0.0, 1.0, -1.0)
    return s * torch.minimum(a.abs(), b * s).clamp(min=0.0)


def _slope(l, c, r):
    return _minmod(THETA * (r - c), _minmod(0.5 * (r - l), THETA * (c - l)))


def _upwind(E, axis, positive):
    """F(i+1/2) - F(i-1/2) over the interior of `axis` for one sign of the speed."""
    n = E.shape[axis]
    lo, hi = (0, n - 1) if positive else (1, n)      # the cells whose edge values the faces take
    E = E.narrow(axis, lo, hi - lo)
    k = E.shape[axis]
    s = _slope(E.narrow(axis, 0, k - 2), E.narrow(axis, 1, k - 2), E.narrow(axis, 2, k - 2))
    edge = E.narrow(axis, 1, k - 2) + (0.5 if positive else -0.5) * s
    return edge.narrow(axis, 1, k - 3) - edge.narrow(axis, 0, k - 3)


def _flux_term(E, xi, eta, dx, dy):
    """Upwind divergence of xi E_x + eta E_y on the interior, E[i][j][q]."""
    out = torch.zeros(E.shape[0] - 4, E.shape[1] - 4, E.shape[2], dtype=E.dtype, device=E.device)
    for speed, axis, h in ((xi, 0, dx), (eta, 1, dy)):
        for positive in (True, False):
            q = torch.nonzero(speed > 0.0 if positive else speed < 0.0)[:, 0]
            if len(q):
                part = E[:, 2:-2, q] if axis == 0 else E[2:-2, :, q]
                out[:, :, q] += _upwind(part, axis, positive) * speed[q] / h
    return out


def _periodic(f):
    f[:2, 2:-2], f[-2:, 2:-2] = f[-4:-2, 2:-2].clone(), f[2:4, 2:-2].clone()
    f[2:-2, :2], f[2:-2, -2:] = f[2:-2, -4:-2].clone(), f[2:-2, 2:4].clone()


def _exact_step(case, seed):
    half, dx, dy, sig_t, sig_s, rho = _grid(case, seed)
    w, p, xi, eta = (t.to(DEV) for t in _tables(case["order"], case["quad"]))
    m, a = (torch.from_numpy(v).to(DEV) for v in _isotropic_state(rho, p.shape[1], case["ppn"]))
    st, ss = torch.from_numpy(sig_t).to(DEV), torch.from_numpy(sig_s).to(DEV)
    nx, ny, nm, dt = case["nx"], case["ny"], p.shape[1], _time_step(dx, dy)
    source = np.zeros((nx, ny))
    if case["ic"] == 1:              # a unit isotropic source where the cell's left edge is inside the centre block
        source[np.ix_(np.abs(-half + np.arange(nx) * dx) < 0.5, np.abs(-half + np.arange(ny) * dy) < 0.5)] = 1.0
    source = torch.from_numpy(source).to(DEV) * 2.0 * SQRT_PI
    mass = torch.zeros(nm, dtype=torch.float64, device=DEV)
    mass[0] = 1.0
    I = (slice(2, -2), slice(2, -2))
    for _ in range(case["steps"]):
        old = m.clone()
        for stage in (1, 2):
            if case["ic"] == 2:
                _periodic(m)
            a = _solve_exact(m.reshape(-1, nm), a.reshape(-1, nm), w, p, case["ppn"]).reshape(m.shape)
            F = torch.zeros(nx, ny, nm, dtype=torch.float64, device=DEV)
            for q in torch.arange(len(w), device=DEV).split(64):
                u0 = m.reshape(-1, nm)[:, :1]
                z = (a.reshape(-1, nm)) @ p[q].T
                E = _ansatz(z, DELTA_PPN if case["ppn"] else None)[0].reshape(nx + 4, ny + 4, len(q))
                F += (_flux_term(E, xi[q], eta[q], dx, dy) * w[q]) @ p[q]
            v = m[I] * (1.0 - dt * st[I])[:, :, None] - dt * F + (dt * ss[I] * m[I][:, :, 0])[:, :, None] * mass
            v += (dt * source)[:, :, None] * mass
            m[I] = v if stage == 1 else 0.5 * (v + old[I])
    return {"moments": m, "alpha": a}


# ---- discrete ordinates ----------------------------------------------------------------------

def _sn_inputs(case, seed):
    half, dx, dy, sig_t, sig_s, rho = _grid(dict(case, floor=1e-4, sigma=0.1), seed)
    f = np.repeat(rho[:, :, None], case["quad"] ** 2, axis=2)
    return half, dx, dy, sig_t, sig_s, f, 0.5 * CFL * (dx * dy) / (dx + dy)


def _prepare_sn(case, seed):
    half, dx, dy, sig_t, sig_s, f, dt = _sn_inputs(case, seed)
    return dict(case=case, half=half, dx=dx, dy=dy, sig_t=sig_t, sig_s=sig_s, f=f, dt=dt)


def _run_sn(s):
    c = s["case"]
    f, _ = _package().sn_run(s["f"], s["sig_t"], s["sig_s"], c["quad"], s["dx"], s["dy"], -s["half"], -s["half"],
                             c["ic"], s["dt"], c["steps"])
    return {"f": f}


def _exact_sn(case, seed):
    half, dx, dy, sig_t, sig_s, f, dt = _sn_inputs(case, seed)
    w, _, xi, eta = (t.to(DEV) for t in _tables(1, case["quad"]))
    f, st, ss = (torch.from_numpy(v).to(DEV) for v in (f, sig_t, sig_s))
    nx, ny = case["nx"], case["ny"]
    source = np.zeros((nx, ny))
    if case["ic"] == 1:              # the solver takes the cell's index with its ghosts here
        source[np.ix_(np.abs(-half + np.arange(2, nx + 2) * dx) < 0.5,
                      np.abs(-half + np.arange(2, ny + 2) * dy) < 0.5)] = 1.0
    source = torch.from_numpy(source).to(DEV)
    I = (slice(2, -2), slice(2, -2))

    def stage(g):
        v = g[I]
        scatter = (v @ w) * ss[I] / (4.0 * math.pi) + source
        return v - dt * st[I][:, :, None] * v + dt * scatter[:, :, None] - dt * _flux_term(g, xi, eta, dx, dy)

    for _ in range(case["steps"]):
        old = f[I].clone()
        for k in (0, 1):
            if case["ic"] == 2:
                _periodic(f)
            v = stage(f)
            f[I] = v if k == 0 else 0.5 * (v + old)
    return {"f": f}


# ---- the learned warm start's network -----------------------------------------------------------

LAYERS = (15, 128, 128, 128, 15)


def _mlp_inputs(case, seed):
    """Pairs (u/u0, scaled alpha) of smooth M4 closures, and the state of a fresh
    network: weights, biases, then the pairs' standardisation."""
    u, _, true = _batch_inputs(dict(order=4, quad=16, cells=case["pairs"]), seed)
    us = u / u[:, :1]
    al = true.clone()
    al[:, 0] -= 2.0 * SQRT_PI * torch.log(u[:, 0])
    rng = np.random.default_rng(seed)
    parts = []
    for i, o in zip(LAYERS[:-1], LAYERS[1:]):
        b = math.sqrt(6.0 / (i + o))
        parts += [rng.uniform(-b, b, i * o), np.zeros(o)]
    us, al = us.cpu().numpy(), al.cpu().numpy()
    for v in (us, al):
        sd = v.std(axis=0)
        parts += [v.mean(axis=0), np.where(sd > 1e-6, sd, 1.0)]
    return us, al, np.concatenate(parts).astype(np.float32)


def _prepare_mlp(case, seed):
    us, al, params = _mlp_inputs(case, seed)
    return dict(case=case, ctx=_package().Context(4, 16), us=us, al=al, params=params)


def _run_mlp(s):
    ctx, c = s["ctx"], s["case"]
    ctx.mlp_set_params(s["params"])
    loss = ctx.mlp_train(s["us"], s["al"], c["steps"], batch=c["batch"], lr=1e-3, seed=1)
    return {"params": ctx.mlp_params(), "loss": loss}


def _splitmix(x):
    with np.errstate(over="ignore"):
        x = x + np.uint64(0x9e3779b97f4a7c15)
        x = (x ^ (x >> np.uint64(30))) * np.uint64(0xbf58476d1ce4e5b9)
        x = (x ^ (x >> np.uint64(27))) * np.uint64(0x94d049bb133111eb)
        return x ^ (x >> np.uint64(31))


def _exact_mlp(case, seed):
    us, al, params = _mlp_inputs(case, seed)
    flat = torch.from_numpy(params).to(DEV, torch.float64)
    np_ = sum((i + 1) * o for i, o in zip(LAYERS[:-1], LAYERS[1:]))
    stats = flat[np_:].reshape(4, 15)
    X = (torch.from_numpy(us).to(DEV) - stats[0]) / stats[1]
    T = (torch.from_numpy(al).to(DEV) - stats[2]) / stats[3]
    theta = flat[:np_].clone().requires_grad_(True)
    m, v = torch.zeros_like(theta), torch.zeros_like(theta)
    losses = []
    for k in range(1, case["steps"] + 1):
        with np.errstate(over="ignore"):
            sk = (np.uint64(0x9e3779b97f4a7c15) ^ np.uint64(k) ^ np.uint64(0x5bd1e995)) | np.uint64(1)
            i = np.arange(case["batch"], dtype=np.uint64) * np.uint64(0xd1b54a32d192ed03)
        rows = torch.from_numpy((_splitmix(sk ^ i) % np.uint64(case["pairs"])).astype(np.int64)).to(DEV)
        h, at = X[rows], 0
        for j, (ni, no) in enumerate(zip(LAYERS[:-1], LAYERS[1:])):
            h = h @ theta[at:at + ni * no].reshape(ni, no) + theta[at + ni * no:at + (ni + 1) * no]
            at += (ni + 1) * no
            if j < 3:
                h = 0.5 * h * (1.0 + torch.erf(h / math.sqrt(2.0)))
        loss = ((h - T[rows]) ** 2).mean()
        (grad,) = torch.autograd.grad(loss, theta)
        losses.append(loss.detach())
        with torch.no_grad():
            m = 0.9 * m + 0.1 * grad
            v = 0.999 * v + 0.001 * grad * grad
            theta -= 1e-3 * (m / (1.0 - 0.9 ** k)) / (torch.sqrt(v / (1.0 - 0.999 ** k)) + 1e-8)
    return {"params": torch.cat([theta.detach(), flat[np_:]]), "loss": torch.stack(losses)}


# ---- what is measured ---------------------------------------------------------------------------

_PREPARE = dict(batch=_prepare_batch, optcb=_prepare_optcb, step=_prepare_step, sn=_prepare_sn, mlp=_prepare_mlp)
_RUN = dict(batch=_run_batch, optcb=_run_optcb, step=_run_step, sn=_run_sn, mlp=_run_mlp)


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def run(state):
    return _RUN[state["case"]["kind"]](state)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        if case["beams"]:            # the beams are solved regularized, along the solver's own ladder
            return None
        u, _, true = _batch_inputs(case, seed)
        return {"u": u, "alpha": true}
    return dict(optcb=_exact_optcb, step=_exact_step, sn=_exact_sn, mlp=_exact_mlp)[kind](case, seed)


def work(case):
    """Bytes: every input once, every output once.  Flops: per closure the
    iterations its start needs (from isotropic about 6, a beam about 20, from
    the previous step's multipliers 2), each alpha.m, the sums of H and one
    factorisation; fluxes and ordinates per point."""
    kind = case["kind"]
    if kind == "mlp":
        per_row = 2 * sum(i * o for i, o in zip(LAYERS[:-1], LAYERS[1:]))
        return {"bytes": case["pairs"] * 240.0, "flops": 3.0 * per_row * case["batch"] * case["steps"]}
    if kind == "sn":
        points = float(case["nx"] * case["ny"] * case["quad"] ** 2)
        return {"bytes": 16.0 * points, "flops": 2.0 * case["steps"] * 60.0 * points}
    n, nq = (case["order"] + 1) * (case["order"] + 2) // 2, case["quad"] ** 2
    iteration = 2.0 * n * nq + n * (n + 1) * nq + 2.0 * nq + n ** 3 / 3.0 + 2.0 * n * n
    if kind == "step":
        cells = float((case["nx"] + 4) * (case["ny"] + 4))
        per_stage = 2.0 * iteration + (6.0 * n + 30.0) * nq
        return {"bytes": 32.0 * n * cells, "flops": 2.0 * case["steps"] * cells * per_stage}
    cells = float(case["cells"])
    if kind == "optcb":
        return {"bytes": cells * 8.0 * (5 * n + 2 * n * n), "flops": 6.0 * cells * (iteration + n * n * nq)}
    each = 2.0 if case["start"] == "previous" else 6.0 + case["beams"] * 15.0
    return {"bytes": 32.0 * n * cells, "flops": each * cells * iteration}
