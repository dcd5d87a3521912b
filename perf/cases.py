"""The work that users of this framework have it do, as timed cases.

Each case is one call, or one short program, through the public entry points
(ast-grid_amd/astg over include/astg.h): short smoke simulations, pressure
projections of caller-owned fields, one transport step, the CSR solver seam,
batched solves, the uniform-layout AST projection and a differentiable rollout.
Scenes and sizes are those of astg.scenes, bench.py and the tests (32^3 to
256^3 effective octrees, 192x384 and 64^3 uniform grids), and ragged sizes in
between.

A case is a dict of plain values. "seed" arguments select the inputs (fields,
right-hand sides, sources); the layout of a case is part of the case.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ast-grid_amd"))

import astg  # noqa: E402
from astg import diff, scenes, uniform  # noqa: E402


# ---- the cases --------------------------------------------------------------
def listed():
    return [
        # The everyday loop: a 64^3 smoke simulation from scratch (context,
        # layout, 6 steps with tilt adaptivity), reference settings in FP64.
        dict(name="smoke_64", kind="smoke", R=64, levels=3, steps=6, precision="fp64", tol=1e-5, collider=False),
        # The same around a sphere collider, at another size.
        dict(name="smoke_collider_96", kind="smoke", R=96, levels=4, steps=4, precision="fp64", tol=1e-5,
             collider=True),
        # project(dt) on the caller's device fields: the smallest scene, where
        # latency and launches count.
        dict(name="project_fp64_32", kind="project", R=32, levels=3, precision="fp64", tol=1e-5),
        # A large projection in the reference's own arithmetic and numbering.
        dict(name="project_fp64_192", kind="project", R=192, levels=4, precision="fp64", tol=1e-6),
        # Ordinary and largest mixed-precision projections (bench.py's headline
        # workload is the second: 256^3 effective, 3.5 M unknowns).
        dict(name="project_mixed_96", kind="project", R=96, levels=4, precision="mixed", tol=1e-6),
        dict(name="project_mixed_256", kind="project", R=256, levels=4, precision="mixed", tol=1e-6),
        # The step after a projection: constraint, ghosts, dual grid, advection
        # of density, heat and velocity.
        dict(name="transport_192", kind="transport", R=192, levels=4),
        # The CUDA-solver seam: one host CSR system of a cut-cell Poisson
        # problem, a ragged box, the reference's FP64 solver.
        dict(name="csr_fp64", kind="csr", nx=61, ny=47, nz=53, precision="fp64", tol=1e-8),
        # Uneven independent systems in one batched call, mixed precision.
        dict(name="batch_mixed", kind="batch", count=6, lo=12, hi=56, layout=3, precision="mixed", tol=1e-6),
        # The reference's uniform 2D example size, its own settings.
        dict(name="ast2_fp64", kind="ast", nx=192, ny=384, nz=0, precision="fp64"),
        # The uniform 3D solver in the mixed form.
        dict(name="ast3_mixed", kind="ast", nx=64, ny=64, nz=64, precision="mixed"),
        # A training-like pass: differentiable rollout and its gradient.
        dict(name="grad_64", kind="grad", R=64, levels=3, steps=3, every=2, precision="mixed", tol=1e-8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _log_size(rng, lo, hi, unit):
    return min(hi, max(lo, int(round(_log_int(rng, lo, hi) / unit)) * unit))


def draw(rng):
    kind = rng.choice(["smoke", "project", "project", "project", "transport", "csr", "batch", "ast", "ast", "grad"])
    if kind == "smoke":
        levels = rng.choice([3, 4])
        collider = rng.random() < 0.4
        return dict(kind="smoke", R=_log_size(rng, 32, 96, 1 << (levels - 1)), levels=levels, steps=rng.randint(2, 5),
                    precision="fp64" if collider else rng.choice(["fp64", "mixed"]),
                    tol=rng.choice([1e-5, 1e-6]), collider=collider)
    if kind == "project":
        precision = rng.choice(["fp64", "mixed", "mixed"])
        levels = rng.choice([3, 4, 4])
        hi = 160 if precision == "fp64" else 224
        R = _log_size(rng, 32, hi if levels == 4 else 128, 1 << (levels - 1))
        return dict(kind="project", R=R, levels=levels, precision=precision,
                    tol=1e-6 if precision == "mixed" else rng.choice([1e-5, 1e-6]))
    if kind == "transport":
        levels = rng.choice([3, 4, 4])
        return dict(kind="transport", R=_log_size(rng, 40, 192 if levels == 4 else 128, 1 << (levels - 1)),
                    levels=levels)
    if kind == "csr":
        return dict(kind="csr", nx=rng.randint(14, 66), ny=rng.randint(14, 60), nz=rng.randint(14, 56),
                    precision=rng.choice(["fp64", "fp64", "mixed"]), tol=1e-8)
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(2, 9), lo=rng.randint(8, 20), hi=rng.randint(24, 52),
                    layout=rng.randint(0, 9999), precision=rng.choice(["fp64", "mixed"]), tol=1e-6)
    if kind == "ast":
        precision = rng.choice(["fp64", "mixed"])
        if rng.random() < 0.5:
            return dict(kind="ast", nx=_log_int(rng, 33, 192), ny=_log_int(rng, 40, 384), nz=0, precision=precision)
        nx = rng.randint(18, 64)
        return dict(kind="ast", nx=nx, ny=rng.randint(16, nx), nz=rng.randint(15, 64), precision=precision)
    return dict(kind="grad", R=_log_size(rng, 24, 64, 4), levels=3, steps=rng.randint(1, 3), every=rng.randint(1, 3),
                precision=rng.choice(["fp64", "mixed"]), tol=1e-8)


# ---- inputs -----------------------------------------------------------------
def _params(case, **kw):
    prec = astg.PREC_MIXED if case["precision"] == "mixed" else astg.PREC_FP64
    return astg.default_params(tol=case["tol"], max_iterations=3000, precision=prec, **kw)


def _normal(n, seed, stream, scale=1.0):
    """N(0,1) drawn in FP32 and widened, as astg.scenes.velocity_frames."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * seed + stream)
    return torch.randn(n, generator=g, device="cuda", dtype=torch.float32).double().mul_(scale)


@functools.lru_cache(maxsize=8)
def _octree_split(R, levels):
    """The six-sphere layout of astg.scenes.projection_256 at any size."""
    split, spheres = scenes.projection_256_split(0, R, levels, scenes.BAND_256[:levels - 1])
    return split, spheres


def _octree(case):
    R, levels = case["R"], case["levels"]
    split, spheres = _octree_split(R, levels)
    ctx = astg.Context(0)
    ctx.set_topology(split, R, levels, scenes.CLOSED_XY)
    xyz, _ = ctx.nodes(0)
    leaf = xyz[:ctx.level_info(0)[1]]
    inside = np.zeros(len(leaf), np.uint8)
    p = leaf.astype(np.float32) / np.float32(R)
    for s in spheres.astype(np.float32):
        d = p - s[:3]
        inside |= ((d * d).sum(axis=1) < s[3] * s[3]).astype(np.uint8)
    ctx.set_tilt_open(0, inside)
    return ctx


def _prepare_smoke(case, seed):
    R, levels = case["R"], case["levels"]
    rng = np.random.default_rng([seed, 11])
    h = 1.0 / R
    source = (0.5, 0.5, 0.12, 0.08)
    band = [4 * h]
    for l in range(1, levels - 1):
        band.append(band[-1] + 8 * h * (1 << l))
    # finest cells at the source and, with a collider, around it
    fine = [source] + ([(0.5, 0.5, 0.45, 0.1)] if case["collider"] else [])
    st = dict(split=astg.split_spheres(R, levels, np.array(fine).ravel(), band), source=source,
              density=float(rng.uniform(0.8, 1.0)), speed=float(rng.uniform(0.7, 1.3)),
              buoyancy=float(rng.uniform(0.8, 1.2)), prm=_params(case))
    if case["collider"]:
        st["sdf"] = astg.sphere_sdf(R, (0.5, 0.5, 0.45), 0.1)
    return st


def _run_smoke(case, st):
    R, levels = case["R"], case["levels"]
    ctx = astg.Context(0)
    ctx.set_topology(st["split"], R, levels, scenes.CLOSED_XY)
    if case["collider"]:
        ctx.set_boundary_sdf(st["sdf"])
    ctx.set_tilt_adaptivity(True)
    cx, cy, cz, r = st["source"]
    dt = 0.5 / R
    for k in range(case["steps"]):
        ctx.apply_sphere_source((cx, cy, cz), r, st["density"], 1.0, st["speed"], update_ghost=k == 0)
        if case["collider"]:
            ctx.wipe_boundary()
        ctx.add_force(dt, st["buoyancy"], 0.0)
        ctx.step(dt, 2.0, st["prm"])
    G, _ = ctx.field_layout()
    new = lambda m: torch.empty(m * G, dtype=torch.float64, device="cuda")
    out = dict(mac=new(3), tilt=new(8), density_cell=new(1), density_vert=new(1), heat_cell=new(1), heat_vert=new(1))
    ctx.download_fields(**out)
    ctx.close()
    return out


def _prepare_project(case, seed):
    ctx = _octree(case)
    G, _ = ctx.field_layout()
    return dict(ctx=ctx, prm=_params(case), mac=_normal(3 * G, seed, 1), tilt=_normal(8 * G, seed, 2))


def _run_project(case, st):
    mac, tilt = st["mac"].clone(), st["tilt"].clone()
    st["ctx"].project_fields(0.5 / case["R"], 2.0, st["prm"], mac, tilt)
    return dict(mac=mac, tilt=tilt)


def _prepare_transport(case, seed):
    ctx = _octree(case)
    G, _ = ctx.field_layout()
    st = dict(ctx=ctx, fields=dict(mac=_normal(3 * G, seed, 1, 0.5), tilt=_normal(8 * G, seed, 2, 0.5)))
    for j, k in enumerate(("density_cell", "density_vert", "heat_cell", "heat_vert")):
        st["fields"][k] = _normal(G, seed, 3 + j).abs_()
    st["out"] = {k: torch.empty_like(v) for k, v in st["fields"].items()}
    return st


def _run_transport(case, st):
    ctx = st["ctx"]
    ctx.upload_fields(**st["fields"])
    ctx.post_project()
    ctx.advect(0.5 / case["R"])
    ctx.download_fields(**st["out"])
    return st["out"]


class _Poisson:
    """A cut-cell Poisson problem on an nx x ny x nz box, x fastest: face
    weights 1 in most places and U[0.05, 1] in a shell (cut faces), closed x
    and y walls, open z walls."""

    def __init__(self, nx, ny, nz, rng):
        self.shape = (nz, ny, nx)
        Z, Y, X = np.meshgrid(*[(np.arange(s) + 0.5) / s for s in self.shape], indexing="ij")
        c = rng.uniform(0.3, 0.7, 3)
        dist = np.abs(np.sqrt((X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2) - 0.25)
        cutcell = dist < 1.5 / min(self.shape)
        w = np.where(cutcell, rng.uniform(0.05, 1.0, self.shape), 1.0)
        # weight of the face between a cell and its upper neighbour, per axis
        self.w = [np.minimum(w[1:], w[:-1]), np.minimum(w[:, 1:], w[:, :-1]), np.minimum(w[:, :, 1:], w[:, :, :-1])]
        d = np.zeros(self.shape)
        d[1:] += self.w[0]
        d[:-1] += self.w[0]
        d[:, 1:] += self.w[1]
        d[:, :-1] += self.w[1]
        d[:, :, 1:] += self.w[2]
        d[:, :, :-1] += self.w[2]
        d[0] += 1.0
        d[-1] += 1.0
        self.diag = d
        # a velocity field's divergence on the same faces
        u = [rng.standard_normal(f.shape) * f for f in self.w]
        b = np.zeros(self.shape)
        b[1:] += u[0]
        b[:-1] -= u[0]
        b[:, 1:] += u[1]
        b[:, :-1] -= u[1]
        b[:, :, 1:] += u[2]
        b[:, :, :-1] -= u[2]
        self.b = b

    def csr(self):
        nz, ny, nx = self.shape
        n = nx * ny * nz
        cand = np.full((n, 7), -1, np.int64)
        vals = np.zeros((n, 7))
        idx = np.arange(n).reshape(self.shape)
        lo = [np.s_[1:], np.s_[:, 1:], np.s_[:, :, 1:]]
        up = [np.s_[:-1], np.s_[:, :-1], np.s_[:, :, :-1]]
        for a in range(3):
            cand[idx[lo[a]].ravel(), a] = idx[up[a]].ravel()
            vals[idx[lo[a]].ravel(), a] = -self.w[a].ravel()
            cand[idx[up[a]].ravel(), 6 - a] = idx[lo[a]].ravel()
            vals[idx[up[a]].ravel(), 6 - a] = -self.w[a].ravel()
        cand[:, 3] = np.arange(n)
        vals[:, 3] = self.diag.ravel()
        keep = cand >= 0
        rs = np.concatenate([[0], np.cumsum(keep.sum(axis=1))]).astype(np.int32)
        return rs, cand[keep].astype(np.int32), vals[keep], self.b.ravel().copy()

    def solve(self):
        w = [torch.from_numpy(x) for x in self.w]
        d = torch.from_numpy(self.diag)

        def A(p):
            q = d * p
            q[1:] -= w[0] * p[:-1]
            q[:-1] -= w[0] * p[1:]
            q[:, 1:] -= w[1] * p[:, :-1]
            q[:, :-1] -= w[1] * p[:, 1:]
            q[:, :, 1:] -= w[2] * p[:, :, :-1]
            q[:, :, :-1] -= w[2] * p[:, :, 1:]
            return q

        return _cg(A, torch.from_numpy(self.b), 1.0 / d).ravel()


def _cg(A, b, minv):
    """Jacobi-preconditioned conjugate gradients in FP64 to rounding."""
    x = torch.zeros_like(b)
    r = b.clone()
    z = minv * r
    s = z.clone()
    rho = (z * r).sum()
    target = 1e-13 * float(b.abs().max())
    for _ in range(20000):
        q = A(s)
        alpha = rho / (s * q).sum()
        x += alpha * s
        r -= alpha * q
        if float(r.abs().max()) <= target:
            break
        z = minv * r
        new = (z * r).sum()
        s = z + (new / rho) * s
        rho = new
    return x


def _csr_problem(case, seed):
    return _Poisson(case["nx"], case["ny"], case["nz"], np.random.default_rng([seed, 21]))


def _prepare_csr(case, seed):
    return dict(ctx=astg.Context(0), system=_csr_problem(case, seed).csr(), prm=_params(case))


def _run_csr(case, st):
    x, _ = st["ctx"].pcg_solve_csr(*st["system"], st["prm"])
    return x


def _batch_problems(case, seed):
    rng = np.random.default_rng([case["layout"], 31])
    shapes = [[int(v) for v in np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), 3))]
              for _ in range(case["count"])]
    rng = np.random.default_rng([seed, 32])
    return [_Poisson(*s, rng) for s in shapes]


def _prepare_batch(case, seed):
    return dict(ctx=astg.Context(0), systems=[p.csr() for p in _batch_problems(case, seed)], prm=_params(case))


def _run_batch(case, st):
    xs, _ = st["ctx"].pcg_solve_batch(st["systems"], st["prm"])
    return xs


# The uniform-layout solver's inputs as bench.py's: 30 % of the tilt nodes open
# (the boundary ones are held closed), N(0,1) velocities, dt 0.025, rho 2.
AST_DT, AST_RHO = 0.025, 2.0


def _ast_res(case):
    return (case["nx"], case["ny"]) if case["nz"] == 0 else (case["nx"], case["ny"], case["nz"])


def _ast_inputs(case, seed):
    res = _ast_res(case)
    d = len(res)
    rng = np.random.default_rng([seed, 41])
    nt = int(np.prod([r + 1 for r in res]))
    open_ = (rng.random(nt) < 0.3).astype(np.uint8)
    mac = [rng.standard_normal(int(np.prod([r + (i == a) for i, r in enumerate(res)]))) for a in range(d)]
    tilt = rng.standard_normal((nt, 4 if d == 2 else 8))
    return res, open_, mac, tilt


def _prepare_ast(case, seed):
    res, open_, mac, tilt = _ast_inputs(case, seed)
    ast = uniform.ASTSolver(len(res), res, 1.0 / res[0])
    ast.set_layout(open_)
    prec = astg.PREC_MIXED if case["precision"] == "mixed" else astg.PREC_FP64
    tau = dict(mic_tau=astg.TAU_AUTO) if case["precision"] == "mixed" else {}
    return dict(ast=ast, mac=mac, tilt=tilt, prm=uniform.default_params(precision=prec, **tau))


def _run_ast(case, st):
    ast = st["ast"]
    ast.set_velocity(st["mac"], st["tilt"])
    ast.project(AST_DT, AST_RHO, st["prm"])
    mac, tilt = ast.velocity()
    return dict(mac=mac, tilt=tilt)


def _exact_ast(case, seed):
    """The same projection written as operators on the cell and node grids.

    An open node couples with its 2^d cells at distance half * sqrt(d) over a
    face of area `ta`, and takes `cut` from every MAC face it touches; the y
    walls are Dirichlet faces; the other walls carry no flux."""
    res, open_, mac, tilt = _ast_inputs(case, seed)
    d = len(res)
    dx = 1.0 / res[0]
    half = dx / 2.0
    dist = half * math.sqrt(d)
    ta, cut, full = (half * math.sqrt(2.0), half, dx) if d == 2 else (math.sqrt(3.0) * 0.5 * half * half,
                                                                      0.5 * half * half, dx * dx)
    cshape = tuple(reversed(res))
    tshape = tuple(s + 1 for s in cshape)
    op = open_.reshape(tshape).astype(np.float64)
    for ax in range(d):
        op[(slice(None),) * ax + ([0, -1],)] = 0.0
    # slot k of a node: the cell on its (lower 0 / upper 1) side per axis x, y, z
    side = [(1, 1), (1, 0), (0, 0), (0, 1)]
    slots = side if d == 2 else [s + (1,) for s in side] + [s + (0,) for s in side]
    nk = len(slots)
    up = lambda k: -1.0 if k < nk // 2 else 1.0
    opposite = lambda k: slots.index(tuple(1 - v for v in slots[k]))

    def nodes_of_cells(s):
        """Node-grid view of the cells' corner nodes for which the cell is on side s."""
        return tuple(slice(0, n) if v else slice(1, n + 1) for v, n in zip(reversed(s), cshape))

    def axis_slice(ax, sl):
        return (slice(None),) * (d - 1 - ax) + (sl,)

    # open area of every MAC face: a face of axis ax is touched by 2^(d-1) nodes
    area = []
    for ax in range(d):
        a = np.full(tuple(n + (i == d - 1 - ax) for i, n in enumerate(cshape)), full)
        corners = op
        for o in range(d):
            if o != ax:
                lo, hi = corners[axis_slice(o, slice(0, -1))], corners[axis_slice(o, slice(1, None))]
                corners = lo + hi
        a -= cut * corners
        a[a <= np.finfo(np.float64).eps] = 0.0
        area.append(a)
    inner = [area[ax][axis_slice(ax, slice(1, -1))] / dx for ax in range(d)]
    ct = ta / dist
    diag = np.zeros(cshape)
    b = np.zeros(cshape)
    vel = [mac[ax].reshape(area[ax].shape) for ax in range(d)]
    tu = tilt.reshape(tshape + (nk,))
    tb = np.zeros(tshape)
    for ax in range(d):
        lo, hi = axis_slice(ax, slice(0, -1)), axis_slice(ax, slice(1, None))
        flux = area[ax] * vel[ax]
        coef = area[ax] / dx
        if ax != 1:
            for wall in (0, -1):
                flux[axis_slice(ax, wall)] = 0.0
                coef[axis_slice(ax, wall)] = 0.0
        b += flux[lo] - flux[hi]
        diag += coef[lo] + coef[hi]
    for k, s in enumerate(slots):
        # slot k of a node faces the cell on side slots[k]; seen from that cell the node is the opposite corner
        sl = nodes_of_cells(s)
        diag += ct * op[sl]
        b += up(opposite(k)) * ta * op[sl] * tu[sl + (k,)]
        tb += up(k) * ta * op * tu[..., k]
    diag[diag < np.finfo(np.float64).eps] = 1.0
    scale = AST_RHO / AST_DT
    nc = int(np.prod(cshape))
    inner = [torch.from_numpy(np.ascontiguousarray(w)) for w in inner]
    top = torch.from_numpy(op)
    tdiag = torch.from_numpy(diag)

    def A(x):
        p, t = x[:nc].reshape(cshape), x[nc:].reshape(tshape)
        q, r = tdiag * p, nk * ct * t
        for ax in range(d):
            lo, hi = axis_slice(ax, slice(0, -1)), axis_slice(ax, slice(1, None))
            q[hi] -= inner[ax] * p[lo]
            q[lo] -= inner[ax] * p[hi]
        for s in slots:
            sl = nodes_of_cells(s)
            q -= ct * top[sl] * t[sl]
            r[sl] -= ct * p
        r = torch.where(top > 0, r, t)
        return torch.cat([q.reshape(-1), r.reshape(-1)])

    rhs = torch.cat([torch.from_numpy(b * scale).reshape(-1), torch.from_numpy(tb * scale).reshape(-1)])
    minv = torch.cat([1.0 / tdiag.reshape(-1), torch.where(top > 0, 1.0 / (nk * ct), 1.0).reshape(-1)])
    x = _cg(A, rhs, minv).numpy()
    p, t = x[:nc].reshape(cshape), x[nc:].reshape(tshape)
    tout = tu.copy()
    for k, s in enumerate(slots):
        sl = nodes_of_cells(s)
        tout[sl + (k,)] += up(k) * AST_DT / AST_RHO * op[sl] * (p - t[sl]) / dist
    mout = []
    for ax in range(d):
        pad = np.zeros(tuple(n + 2 * (i == d - 1 - ax) for i, n in enumerate(cshape)))
        pad[axis_slice(ax, slice(1, -1))] = p
        v = vel[ax] - AST_DT / AST_RHO * (pad[axis_slice(ax, slice(1, None))] - pad[axis_slice(ax, slice(0, -1))]) / dx
        if ax == 0:
            v[axis_slice(0, [0, -1])] = 0.0
        if ax == 1 and d == 3:  # closed for x below the y resolution
            v[:, [0, -1], :res[1]] = 0.0
        mout.append(v.ravel())
    return dict(mac=mout, tilt=tout.reshape(-1, nk))


def _prepare_grad(case, seed):
    ctx, info = scenes.diff_smoke(device=0, R=case["R"], levels=case["levels"])
    sim = diff.DiffSim(ctx, info["dt"], info["rho"], _params(case))
    target = torch.as_tensor(info["target"], device="cuda")
    leaf = torch.as_tensor(info["leaf_cells"], device="cuda")
    return dict(sim=sim, state0=sim.get_state(), u0=_normal(3 * info["G"], seed, 1, 0.1), target=target, leaf=leaf)


def _run_grad(case, st):
    u = st["u0"].clone().requires_grad_(True)
    rho = diff.rollout(u, st["sim"], st["state0"], case["steps"], case["every"])
    loss = ((rho - st["target"]).square() * st["leaf"]).sum()
    loss.backward()
    return dict(density=rho.detach(), grad=u.grad)


# ---- the interface ----------------------------------------------------------
_PREPARE = dict(smoke=_prepare_smoke, project=_prepare_project, transport=_prepare_transport, csr=_prepare_csr,
                batch=_prepare_batch, ast=_prepare_ast, grad=_prepare_grad)
_RUN = dict(smoke=_run_smoke, project=_run_project, transport=_run_transport, csr=_run_csr, batch=_run_batch,
            ast=_run_ast, grad=_run_grad)


def prepare(case, seed):
    st = _PREPARE[case["kind"]](case, seed)
    st["case"] = dict(case)
    return st


def run(state):
    return _RUN[state["case"]["kind"]](state["case"], state)


def _nodes(case):
    """Leaves of the case's octree, and with them its node count (leaves plus
    about an eighth of ghosts)."""
    if case["kind"] in ("project", "transport"):
        leaves = scenes.leaf_count(_octree_split(case["R"], case["levels"])[0])
    else:
        leaves = scenes.leaf_count(scenes.smoke_64_split(case["R"], case["levels"]))
    return leaves * 1.13


def work(case):
    """Bytes and operations one pass cannot do without: its inputs read once,
    its outputs written once; operations of one product with the system."""
    kind = case["kind"]
    if kind == "smoke":  # per step: velocity, both scalars, the layout
        G = _nodes(case)
        return dict(bytes=case["steps"] * G * (2 * 15 * 8 + 16), flops=case["steps"] * G * 8 * 2)
    if kind == "project":
        G = _nodes(case)
        return dict(bytes=G * (2 * 11 * 8 + 16), flops=G * 8 * 2)
    if kind == "transport":
        G = _nodes(case)
        return dict(bytes=G * (2 * 15 * 8 + 16), flops=G * 5 * 100)
    if kind == "grad":
        G = _nodes(case)
        return dict(bytes=case["steps"] * 2 * G * 2 * 19 * 8, flops=case["steps"] * 2 * G * 8 * 2)
    if kind == "csr":
        n = case["nx"] * case["ny"] * case["nz"]
        return dict(bytes=n * (7 * 12 + 4 + 16), flops=n * 14)
    if kind == "batch":
        rng = np.random.default_rng([case["layout"], 31])
        n = sum(int(np.prod([int(v) for v in np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), 3))]))
                for _ in range(case["count"]))
        return dict(bytes=n * (7 * 12 + 4 + 16), flops=n * 14)
    res = _ast_res(case)
    d = len(res)
    nc = int(np.prod(res))
    nt = int(np.prod([r + 1 for r in res]))
    return dict(bytes=2 * 8 * (d * nc + nt * (4 if d == 2 else 8)) + nt, flops=2 * nc * (2 * d + 3))


def tolerance(case):
    """What two correct solvers stopped at the case's residual tolerance differ
    by: about four times the largest distance measured between the result, the
    same case at a thousandth of its tolerance, its other precision and
    exact(). (The error behind a residual of `tol` exceeds `tol` by the
    conditioning that the preconditioner leaves.)"""
    kind = case["kind"]
    if kind == "project":
        return dict(rel=6e-4 if case["tol"] > 2e-6 else 1.5e-4)
    if kind == "ast":
        return dict(rel=5e-5 if case["nz"] == 0 else 8e-4)
    return dict(rel=dict(smoke=1e-5, transport=1e-10, csr=1e-6, batch=5e-5, grad=2e-7)[kind])


def exact(case, seed):
    """The results in plain FP64, for the solver cases on structured grids.
    The octree cases have none: their discretisation (T-junctions, half-tilts,
    ghost rules, samplers) written row by row in plain Python takes minutes."""
    if case["kind"] == "csr":
        return _csr_problem(case, seed).solve().numpy()
    if case["kind"] == "batch":
        return [p.solve().numpy() for p in _batch_problems(case, seed)]
    if case["kind"] == "ast":
        return _exact_ast(case, seed)
    return None
