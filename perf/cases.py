"""The workloads this framework's speed is measured on.

Each case is one call (or one solve) that a program built on ``apple_amd``
makes over and over, through the public entry points: the element passes of
the potentials (``fused``, ``hess_prod``, ``mixed_derivative_prod``), the
static solve (``DeviceSolver.solve``, what ``Forward.step`` and the inverse
loop call), the batched solve (``Batch.solve``) and the adjoint solve
(``DeviceSolver.cg``).  ``exact`` restates the same quantities in plain torch,
in 64 bits.

Meshes are the package's cubes (n^3 cells of five tets) with their vertices
moved by a tenth of a cell, so that no two tets are alike.  ``order`` "morton"
is the order that ``mesh.cube`` and ``mesh.reorder`` give, "lex" that of a
mesh from a generator which sweeps it plane by plane.  Displacements are a
smooth bend, twist and sag of the whole body plus a per-vertex part of a few
percent of a cell (what a trial point of a solve looks like).
"""

from __future__ import annotations

import functools
import math

import numpy as np
import torch

from apple_amd import _lib, batch, fem
from apple_amd.mesh import Region, cube
from apple_amd.potential import gravity_from_potential
from apple_amd.solver import DeviceSolver, PncgConfig, mask_bits

DEVICE = "cuda"
LAWS = {"snh": fem.StableNeoHookean, "arap": fem.Arap, "muscle": fem.StableNeoHookeanMuscle}
DTYPES = {"f32": torch.float32, "f64": torch.float64}


# ---------------------------------------------------------------- the cases


def listed():
    def case(name, kind, law, n, dtype="f32", order="morton", **more):
        return {"name": name, "kind": kind, "law": law, "n": n, "dtype": dtype, "order": order, **more}

    return [
        # one evaluation of E, dE/du and diag H of a small body (5,000 tets):
        # a host-driven optimizer's step, bound by launches
        case("snh_fused_n10", "fused", "snh", 10),
        # the same at the benchmark's size (1.31M tets)
        case("snh_fused_n64", "fused", "snh", 64),
        # the law whose pass needs a 3x3 SVD per tet
        case("arap_fused_n64", "fused", "arap", 64),
        # muscle tissue with a per-tet activation
        case("muscle_fused_n45", "fused", "muscle", 45),
        # the FP64 element pass: reference runs and the residuals of refined FP32 solves
        case("snh_fused_n37_f64", "fused", "snh", 37, dtype="f64"),
        # one Hessian-vector product of a caller's own Krylov solver, on a mesh in generator order
        case("snh_hess_prod_n51_lex", "hess_prod", "snh", 51, order="lex"),
        # the parameter gradients of one inverse step: p^T d(grad)/d(activation, mu, lambda)
        case("muscle_mixed_n32", "mixed", "muscle", 32),
        # static equilibrium of a small body under its own weight, start to finish (launch-bound)
        case("snh_solve_n10", "solve", "snh", 10, density=1e3),
        # ... of a large one
        case("snh_solve_n64", "solve", "snh", 64, density=1e2),
        # ... with the ARAP law at the size of the differentiation benchmark
        case("arap_solve_n32", "solve", "arap", 32, density=1e2),
        # many uneven bodies solved in one set of launches
        case("snh_batch_solve", "batch", "snh", 28, meshes=48, least=6),
        # the adjoint system H y = rhs of one equilibrium
        case("snh_adjoint_n32", "adjoint", "snh", 32),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fused", "fused", "hess_prod", "mixed", "solve", "batch", "adjoint"])
    law = rng.choice(["snh", "arap", "muscle"])
    case = {"kind": kind, "law": law, "dtype": rng.choice(["f32", "f32", "f64"]),
            "order": rng.choice(["morton", "morton", "lex"])}
    if kind in ("fused", "hess_prod", "mixed"):
        case["n"] = _log_int(rng, 6, 64)
    elif kind == "batch":
        case.update(law="snh", dtype="f32", order="morton", least=rng.randint(5, 8), n=rng.randint(12, 28),
                    meshes=_log_int(rng, 6, 48))
    elif kind == "adjoint":
        case.update(dtype="f32", n=_log_int(rng, 6, 40))
    else:
        case.update(law=rng.choice(["snh", "arap"]), dtype="f32", n=_log_int(rng, 6, 40), density=round(rng.uniform(50, 150), 1))
    return case


# ---------------------------------------------------------------- inputs


@functools.lru_cache(maxsize=8)
def _cube(n, order):
    return cube(n, order=order)


@functools.lru_cache(maxsize=64)
def _region(n):
    return Region.from_mesh(_cube(n, "morton"))


def _mesh(case, rng):
    """The cube with its inner vertices moved and per-tet materials:
    mu lognormal (median 1e4, sigma 0.5), lambda = 10 mu, activation ~ 0.1 N(0, 1)."""
    n = case["n"]
    base = _cube(n, case["order"])
    m = base.copy()
    inner = np.all((base.points > 1e-9) & (base.points < 1 - 1e-9), axis=1)
    m.points[inner] += (0.1 / n) * (2 * rng.random((int(inner.sum()), 3)) - 1)
    mu = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    m.cell_data["mu"] = mu
    m.cell_data["lambda"] = 10 * mu
    if case["law"] == "muscle":
        m.cell_data["activation"] = 0.1 * rng.standard_normal((m.n_cells, 6))
    return m


def _displacement(points, n, rng):
    """Twist about z, bend, sag and a per-vertex part of 4 % of a cell."""
    x, y, z = points[:, 0] - 0.5, points[:, 1] - 0.5, points[:, 2]
    a = (0.6 + 0.3 * rng.random()) * z
    c, s = np.cos(a), np.sin(a)
    u = np.stack([c * x - s * y - x + 0.15 * z * z, s * x + c * y - y, -0.12 * z + 0.05 * np.sin(3 * x)], axis=1)
    return u + (0.04 / n) * rng.standard_normal(points.shape)


def _tensor(a, dtype):
    return torch.as_tensor(a, dtype=dtype, device=DEVICE).contiguous()


def _pinned(points):
    fixed = np.zeros(points.shape, bool)
    fixed[points[:, 2] < 1e-9] = True
    return fixed


def _host_inputs(case, seed):
    """Mesh, displacement and direction of a single-body case, made from the seed alone."""
    rng = np.random.default_rng([int(seed), 17])
    m = _mesh(case, rng)
    if case["kind"] == "solve":
        u = (0.1 / case["n"]) * rng.standard_normal(m.points.shape)
        u[_pinned(m.points)] = 0.0
    elif case["kind"] == "adjoint":
        # a stable state: stretched along z, a little narrower
        u = np.zeros(m.points.shape)
        u[:, 2] = 0.04 * m.points[:, 2] * (2 - m.points[:, 2])
        u[:, :2] = -0.02 * m.points[:, 2:] * (m.points[:, :2] - 0.5)
    else:
        u = _displacement(m.points, case["n"], rng)
    return m, u, rng.standard_normal(m.points.shape)


def _batch_sizes(case, rng):
    sizes = rng.integers(case["least"], case["n"] + 1, case["meshes"])
    sizes[0], sizes[-1] = case["n"], case["least"]  # the spread is the case's, the order the seed's
    return rng.permutation(sizes)


def _batch_instances(case, seed):
    """Bodies of uneven sizes (the same for every seed), each with its own mu ~ U[1e4, 1e5]
    and nu ~ U[0.3, 0.45], under a light lumped gravity, pinned at z = 0, noisy start."""
    sizes = _batch_sizes(case, np.random.default_rng([case["n"], case["meshes"], case["least"]]))
    rng = np.random.default_rng([int(seed), 23])
    out = []
    for n in sizes:
        region = _region(int(n))
        m = region.mesh
        mu0, nu = rng.uniform(1e4, 1e5), rng.uniform(0.3, 0.45)
        mu = np.full(m.n_cells, mu0)
        f = np.zeros(m.points.shape)
        f[:, 2] = np.bincount(m.cells.reshape(-1), np.repeat(-9.8 * 2e2 * region.dV / 4, 4), m.n_points)
        fixed = _pinned(m.points)
        x0 = (0.1 / int(n)) * rng.standard_normal(m.points.shape)
        x0[fixed] = 0.0
        out.append(batch.Instance(region, mu, mu * 2 * nu / (1 - 2 * nu), f, fixed, x0))
    return out


# ---------------------------------------------------------------- the framework's side


def prepare(case, seed):
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "batch":
        b = batch.Batch(_batch_instances(case, seed), _lib.APL_SNH, dtype=dtype, device=DEVICE)
        b.solver()
        return {"case": case, "batch": b, "x": torch.empty_like(b.x0), "config": PncgConfig(rtol=1e-6, max_steps=20000)}
    m, u, v = _host_inputs(case, seed)
    pot = LAWS[case["law"]].from_pyvista(m, dtype=dtype, device=DEVICE, setup="device")
    s = {"case": case, "pot": pot, "u": _tensor(u, dtype), "v": _tensor(v, dtype)}
    if case["kind"] in ("solve", "adjoint"):
        s["solver"] = DeviceSolver(pot)
        s["mask"] = mask_bits(_pinned(m.points), DEVICE)
        s["x"] = torch.empty_like(s["u"])
        if case["kind"] == "solve":
            s["force"] = gravity_from_potential(pot, case["density"]).force
        s["config"] = PncgConfig(rtol=1e-6, max_steps=20000)
    else:
        s["energy"] = torch.zeros(1, dtype=torch.float64, device=DEVICE)
        s["a"], s["b"] = torch.empty_like(s["u"]), torch.empty_like(s["u"])
    return s


def run(state):
    kind = state["case"]["kind"]
    if kind == "batch":
        state["x"].copy_(state["batch"].x0)
        x, _ = state["batch"].solve(state["x"], state["config"])
        return x
    pot, u, v = state["pot"], state["u"], state["v"]
    if kind == "fused":
        pot.fused(u, state["energy"], state["a"], state["b"], accumulate=False)
        # the energy in the working precision, to be added to other loss terms
        return {"energy": state["energy"].to(u.dtype), "grad": state["a"], "hess_diag": state["b"]}
    if kind == "hess_prod":
        out = state["a"].zero_()
        pot.hess_prod(u, v, out)
        return out
    if kind == "mixed":
        return pot.mixed_derivative_prod(u, v)
    if kind == "solve":
        x = state["x"].copy_(u)
        state["solver"].solve(x, state["force"], state["mask"], state["config"])
        return x
    y = state["x"]
    state["solver"].cg(u, v, y, state["mask"], rtol=1e-6, max_iters=20000)
    return y


# ---------------------------------------------------------------- compulsory work


def work(case):
    """Bytes: cells 16 B, nine inverse rest shape entries, the volume and the
    materials per tet, and each vertex vector once; a solve or an adjoint
    solve has to read that once and write the answer, whatever its iterations
    do.  Flops: the algebra of one evaluation per tet."""
    r = 8 if case["dtype"] == "f64" else 4
    mats = {"snh": 2, "arap": 1, "muscle": 8}[case["law"]]
    flops = {"snh": 300, "arap": 900, "muscle": 360}[case["law"]]
    if case["kind"] == "batch":
        sizes = [int(n) for n in _batch_sizes(case, np.random.default_rng([case["n"], case["meshes"], case["least"]]))]
    else:
        sizes = [case["n"]]
    tets = sum(5 * n**3 for n in sizes)
    verts = sum((n + 1) ** 3 for n in sizes)
    vectors = {"fused": 3, "hess_prod": 3, "mixed": 2}.get(case["kind"], 3)
    per_tet = 16 + (10 + mats) * r
    if case["kind"] == "mixed":
        per_tet += mats * r
    return {"bytes": tets * per_tet + verts * 3 * r * vectors, "flops": tets * flops}


# ---------------------------------------------------------------- the same in plain torch, 64 bits


def _rounded(a, dtype):
    """The values the framework was given, in 64 bits."""
    return torch.as_tensor(a, device=DEVICE).to(dtype).to(torch.float64)


class _Body:
    """F, stresses and Hessian terms of one mesh in FP64, every tet at once."""

    def __init__(self, case, m):
        dtype = DTYPES[case["dtype"]]
        self.law = case["law"]
        self.cells = torch.as_tensor(m.cells, device=DEVICE).long()
        self.n_points = m.n_points
        X = torch.as_tensor(m.points, device=DEVICE)[self.cells]
        M = (X[:, 1:] - X[:, :1]).transpose(1, 2)
        B = torch.linalg.inv(M)
        self.d = torch.cat([-B.sum(1, keepdim=True), B], 1)  # (T, 4, 3)
        self.dV = torch.linalg.det(M) / 6
        self.mu = _rounded(m.cell_data["mu"], dtype)
        self.lam = _rounded(m.cell_data["lambda"], dtype)
        self.A = None
        if self.law == "muscle":
            self.act = _rounded(m.cell_data["activation"], dtype)
            self.A = _stretch(self.act)

    def grad_u(self, u):
        """sum_a u_a (x) d_a"""
        return u[self.cells].transpose(1, 2) @ self.d

    def scatter(self, per_corner):
        out = torch.zeros(self.n_points, 3, dtype=torch.float64, device=DEVICE)
        return out.index_add_(0, self.cells.reshape(-1), per_corner.reshape(-1, 3))

    def shape(self):
        """Shape gradients in the stretched configuration."""
        return self.d if self.A is None else self.d @ self.A

    def deformation(self, u):
        F = self.grad_u(u) + torch.eye(3, dtype=torch.float64, device=DEVICE)
        return F if self.A is None else F @ self.A


def _stretch(act):
    a = act
    rows = [a[:, 0], a[:, 3], a[:, 4], a[:, 3], a[:, 1], a[:, 5], a[:, 4], a[:, 5], a[:, 2]]
    return torch.stack(rows, 1).reshape(-1, 3, 3) + torch.eye(3, dtype=torch.float64, device=a.device)


def _cross_columns(F, H):
    """The derivative of the cofactor at F in direction H (bilinear: _cross_columns(F, F) = 2 cof F)."""
    f, h = F.unbind(2), H.unbind(2)
    cr = torch.linalg.cross
    return torch.stack([cr(f[1], h[2]) + cr(h[1], f[2]), cr(f[2], h[0]) + cr(h[2], f[0]),
                        cr(f[0], h[1]) + cr(h[0], f[1])], 2)


def _svd(F):
    """Rotation-variant SVD by one-sided Jacobi: U, V rotations, the sign of det F on the smallest value."""
    W = F.clone()
    V = torch.eye(3, dtype=F.dtype, device=F.device).expand_as(F).clone()
    for _ in range(10):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            wp, wq = W[:, :, p].clone(), W[:, :, q].clone()
            g = (wp * wq).sum(1)
            z = ((wq * wq).sum(1) - (wp * wp).sum(1)) / torch.where(g == 0, torch.ones_like(g), 2 * g)
            t = torch.where(z >= 0, 1.0, -1.0) / (z.abs() + torch.sqrt(1 + z * z))
            t = torch.where(g == 0, torch.zeros_like(t), t)
            c = 1 / torch.sqrt(1 + t * t)
            s = (c * t)[:, None]
            c = c[:, None]
            W[:, :, p], W[:, :, q] = c * wp - s * wq, s * wp + c * wq
            vp, vq = V[:, :, p].clone(), V[:, :, q].clone()
            V[:, :, p], V[:, :, q] = c * vp - s * vq, s * vp + c * vq
    sv = W.norm(dim=1)
    at = sv.argsort(1, descending=True)
    sv = sv.gather(1, at)
    W = W.gather(2, at[:, None, :].expand_as(W))
    V = V.gather(2, at[:, None, :].expand_as(V))
    V[:, :, 2] *= torch.sign(torch.linalg.det(V))[:, None]
    U = W / sv[:, None, :]
    U[:, :, 2] = torch.linalg.cross(U[:, :, 0], U[:, :, 1])
    sv[:, 2] *= torch.where(torch.linalg.det(F) < 0, -1.0, 1.0)
    return U, sv, V


def _twists(U, sv, V):
    """The three twist modes (T, 3, 3, 3) and their clamped eigenvalues (T, 3)."""
    pairs = ((1, 0, 0, 1), (1, 2, 2, 1), (0, 2, 2, 0))
    Q = [(U[:, :, a, None] * V[:, None, :, b] - U[:, :, c, None] * V[:, None, :, d]) / math.sqrt(2)
         for a, b, c, d in pairs]
    sums = torch.stack([sv[:, 0] + sv[:, 1], sv[:, 1] + sv[:, 2], sv[:, 2] + sv[:, 0]], 1)
    return torch.stack(Q, 1), 2 / sums.clamp(min=2.0)


def _energy_gradient(body, u):
    """Total energy and dE/du."""
    F = body.deformation(u)
    if body.law == "arap":
        U, sv, V = _svd(F)
        psi = body.mu / 2 * ((sv - 1) ** 2).sum(1)
        P = body.mu[:, None, None] * (F - U @ V.transpose(1, 2))
    else:
        C = _cross_columns(F, F) / 2
        J = torch.linalg.det(F)
        psi = body.mu / 2 * ((F * F).sum((1, 2)) - 3) - body.mu * (J - 1) + body.lam / 2 * (J - 1) ** 2
        P = body.mu[:, None, None] * (F - C) + (body.lam * (J - 1))[:, None, None] * C
    g = (body.dV[:, None, None] * P) @ body.shape().transpose(1, 2)  # (T, 3, 4)
    return (psi * body.dV).sum(), body.scatter(g.transpose(1, 2))


def _diagonal(body, u):
    """Per-tet Hessian diagonals, clamped at zero, summed."""
    F, D = body.deformation(u), body.shape()
    t = (D * D).sum(2)[:, :, None]
    if body.law == "arap":
        Q, lam = _twists(*_svd(F))
        qd = torch.einsum("tkij,taj->taki", Q, D)
        h = body.mu[:, None, None] * (t - (lam[:, None, :, None] * qd * qd).sum(2))
    else:
        w = D @ (_cross_columns(F, F) / 2).transpose(1, 2)
        h = body.lam[:, None, None] * w * w + body.mu[:, None, None] * t
    return body.scatter((body.dV[:, None, None] * h).clamp(min=0))


def _hessian(body, u):
    """v -> H(u) v (ARAP: with the clamped twist eigenvalues)."""
    F, D = body.deformation(u), body.shape()
    mu, lam = body.mu[:, None, None], body.lam[:, None, None]
    if body.law == "arap":
        Q, tw = _twists(*_svd(F))
    else:
        C = _cross_columns(F, F) / 2
        s = lam * (torch.linalg.det(F) - 1)[:, None, None] - mu

    def times(v):
        dF = body.grad_u(v)
        if body.A is not None:
            dF = dF @ body.A
        if body.law == "arap":
            T = mu * (dF - torch.einsum("tk,tkij->tij", tw * torch.einsum("tkij,tij->tk", Q, dF), Q))
        else:
            T = lam * (C * dF).sum((1, 2))[:, None, None] * C + mu * dF + s * _cross_columns(F, dF)
        return body.scatter(((body.dV[:, None, None] * T) @ D.transpose(1, 2)).transpose(1, 2))

    return times


def _conjugate_gradients(times, diag, rhs, free, rtol, most):
    """H y = rhs on the free entries, Jacobi-preconditioned; stops at negative curvature."""
    y, r = torch.zeros_like(rhs), rhs * free
    z = r / diag
    d, rz, stop = z.clone(), float((r * z).sum()), rtol * float(r.norm())
    for _ in range(most):
        q = times(d) * free
        dq = float((d * q).sum())
        if dq <= 0:
            break
        a = rz / dq
        y += a * d
        r -= a * q
        if float(r.norm()) <= stop:
            break
        z = r / diag
        rz, old = float((r * z).sum()), rz
        d = z + (rz / old) * d
    return y


def _equilibrium(body, u, force, free):
    """Newton's method from u, each step by conjugate gradients, halved while the energy rises."""
    e, g = _energy_gradient(body, u)
    e = float(e - (force * u).sum())
    first = float(((g - force) * free).norm())
    for _ in range(40):
        r = (force - g) * free
        if float(r.norm()) <= 1e-11 * first:
            break
        dg = _diagonal(body, u)
        near = float(r.norm()) < 1e-3 * first
        step = _conjugate_gradients(_hessian(body, u), torch.where(dg > 0, dg, dg.mean()), r, free,
                                    1e-6 if near else 1e-2, 4000)
        a = 1.0
        while True:
            trial = u + a * step
            et, g = _energy_gradient(body, trial)
            et = float(et - (force * trial).sum())
            if near or et <= e or a < 1e-6:
                break
            a /= 2
        u, e = trial, et
    return u


def exact(case, seed):
    kind = case["kind"]
    # a solve's equilibrium takes minutes here beyond these sizes (and ARAP's projected Hessian
    # has no Newton step that gets to 64 bits): those answers have no value to be held against
    if kind == "batch" or (kind == "solve" and (case["law"] != "snh" or case["n"] > 24)):
        return None
    m, u, v = _host_inputs(case, seed)
    dtype = DTYPES[case["dtype"]]
    body = _Body(case, m)
    u, v = _rounded(u, dtype), _rounded(v, dtype)
    if kind == "fused":
        e, g = _energy_gradient(body, u)
        return {"energy": e.reshape(1), "grad": g, "hess_diag": _diagonal(body, u)}
    if kind == "hess_prod":
        return _hessian(body, u)(v)
    if kind == "mixed":
        return _mixed(body, u, v)
    free = torch.as_tensor(~_pinned(m.points), device=DEVICE).double()
    if kind == "solve":
        vol = torch.zeros(m.n_points, dtype=torch.float64, device=DEVICE)
        vol.index_add_(0, body.cells.reshape(-1), (body.dV / 4).repeat_interleave(4))
        force = torch.zeros_like(u)
        force[:, 2] = -9.8 * case["density"] * vol
        return _equilibrium(body, u, force, free)
    return _conjugate_gradients(_hessian(body, u), _diagonal(body, u), v, free, 1e-11, 20000)


def _mixed(body, u, p):
    """Per tet: the derivatives of dE/du : p with respect to its materials."""
    Fu = body.grad_u(u) + torch.eye(3, dtype=torch.float64, device=DEVICE)
    dF = body.grad_u(p)
    if body.law == "arap":
        U, _, V = _svd(Fu)
        return {"mu": body.dV * ((Fu - U @ V.transpose(1, 2)) * dF).sum((1, 2))}
    mats = {"mu": body.mu.clone().requires_grad_(), "lambda": body.lam.clone().requires_grad_()}
    A = torch.eye(3, dtype=torch.float64, device=DEVICE).expand_as(Fu)
    if body.law == "muscle":
        mats["activation"] = body.act.clone().requires_grad_()
        A = _stretch(mats["activation"])
    F = Fu @ A
    C = _cross_columns(F, F) / 2
    J = (F[:, :, 0] * C[:, :, 0]).sum(1)
    P = mats["mu"][:, None, None] * (F - C) + (mats["lambda"] * (J - 1))[:, None, None] * C
    total = (body.dV * (P * (dF @ A)).sum((1, 2))).sum()
    return dict(zip(mats, torch.autograd.grad(total, list(mats.values()))))
