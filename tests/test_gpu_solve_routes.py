"""The solver's routes compared where a rule on sizes changes them, for every
law and precision, and the vertices that no tet touches."""

import numpy as np
import pytest
import torch

from apple_amd import _lib, batch, fem
from apple_amd.mesh import Mesh, Region, cube
from apple_amd.model import DeviceModel
from apple_amd.solver import DeviceSolver, PncgConfig, mask_bits
from oracle import fem as of

pytestmark = pytest.mark.gpu

# element blocks up to which a single instance's step length rides in its trial
# pass (and d.Hd's sum in its CG update); vertex blocks up to which its decision
# rides in the direction pass, and the CG's beta
BLOCKS, VBLOCKS, CG_VBLOCKS = 2048, 192, 1024


def _case(n, seed=0):
    m = cube(n)
    rng = np.random.default_rng(seed)
    mu = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    m.cell_data["mu"] = mu
    m.cell_data["lambda"] = 10 * mu
    m.cell_data["activation"] = 0.05 * rng.standard_normal((m.n_cells, 6))
    fixed = np.zeros((m.n_points, 3), bool)
    fixed[m.points[:, 2] == 0.0] = True
    x0 = 0.1 / n * rng.standard_normal((m.n_points, 3))
    x0[fixed] = 0.0
    f = np.zeros((m.n_points, 3))
    f[:, 2] = -1.0 / m.n_points
    return m, fixed, x0, f


LAWS = {"snh": (fem.StableNeoHookean, _lib.APL_SNH), "arap": (fem.Arap, _lib.APL_ARAP),
        "muscle": (fem.StableNeoHookeanMuscle, _lib.APL_SNH_MUSCLE)}


def _potential(law, m, dtype):
    if law != "model":
        return LAWS[law][0].from_region(Region.from_mesh(m), dtype=dtype, device="cuda")
    r = Region.from_mesh(m)
    return DeviceModel([LAWS[w][0].from_region(r, dtype=dtype, device="cuda") for w in LAWS], m.n_points, dtype=dtype)


def _instance(law, m, fixed, x0, f):
    r, c = Region.from_mesh(m), m.cell_data
    if law != "model":
        return batch.Instance(r, c["mu"], c["lambda"], f, fixed, x0, c["activation"])
    parts = [batch.Part(k, r.cells, r.dminv, r.dV, c["mu"], c["lambda"], c["activation"]) for _, k in LAWS.values()]
    return batch.Instance(None, f_ext=f, fixed_mask=fixed, x0=x0, parts=parts, n_points=m.n_points)


def _same(a, b, names):
    assert [getattr(a, k) for k in names] == [getattr(b, k) for k in names]


def _compare(law, dtype, n, steps, cg_iters):
    """PNCG and CG of a mesh alone and as an instance of a batch; returns the mesh's block counts."""
    m, fixed, x0, f = _case(n)
    m2, fixed2, x2, f2 = _case(3, seed=1)
    t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda").contiguous()  # noqa: E731
    pot = _potential(law, m, dtype)
    solver, mask = DeviceSolver(pot), mask_bits(fixed, "cuda")
    cfg = PncgConfig(rtol=1e-12, max_steps=steps)
    x = t(x0)
    st = solver.solve(x, t(f), mask, cfg)[0]
    rng = np.random.default_rng(4)
    rhs, rhs2 = t(rng.standard_normal(x0.shape)), t(rng.standard_normal(x2.shape))
    y = torch.empty_like(rhs)
    kw = dict(rtol=1e-12, max_iters=cg_iters)
    sc = solver.cg(t(0.1 * x0), rhs, y, mask, **kw)[0]
    b = batch.Batch([_instance(law, m2, fixed2, x2, f2), _instance(law, m, fixed, x0, f)],
                    _lib.APL_MODEL if law == "model" else LAWS[law][1], dtype=dtype, device="cuda")
    xb, stb = b.solve(config=cfg)
    yb = torch.empty_like(b.x0)
    scb = b.solver().cg(torch.cat([t(0.1 * x2), t(0.1 * x0)]), torch.cat([rhs2, rhs]), yb, b.mask, **kw)
    assert st.n_steps == steps and sc.n_steps == cg_iters and torch.isfinite(y).all() and torch.isfinite(x).all()
    assert torch.equal(b.split(xb)[1], x) and torch.equal(b.split(yb)[1], y)
    _same(st, stb[1], ("result", "n_steps", "n_evals", "f", "grad_norm", "alpha", "beta"))
    _same(sc, scb[1], ("result", "n_steps", "f", "grad_norm", "alpha", "beta"))
    info = pot.mesh.info()
    return info["n_blocks"], info["n_vertex_blocks"]


# on both sides of the three limits: a change of the block size or of a limit
# that takes a size to the other side fails here
@pytest.mark.parametrize("n,blocks,vblocks,cg_vblocks", [
    (35, True, True, True), (36, True, False, True), (47, True, False, True), (48, False, False, True),
    (63, False, False, True), (64, False, False, False)])
def test_both_sides_of_the_limits(n, blocks, vblocks, cg_vblocks):
    print(f"[routes] n = {n}", flush=True)
    nb, nvb = _compare("snh", torch.float32, n, 5, 4)
    assert (nb <= BLOCKS, nvb <= VBLOCKS, nvb <= CG_VBLOCKS) == (blocks, vblocks, cg_vblocks)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("law", [*LAWS, "model"])
def test_every_law_and_precision(law, dtype):
    print(f"[routes] {law} {dtype}", flush=True)
    nb, nvb = _compare(law, dtype, 6, 5, 4)
    assert nb <= BLOCKS and nvb <= VBLOCKS


def test_a_model_past_the_limits():
    print("[routes] model, 36^3", flush=True)
    nb, nvb = _compare("model", torch.float32, 36, 3, 3)
    assert nb > BLOCKS and nvb > VBLOCKS


def _with_isolated(m, fixed, x0, f, extra, force):
    """The mesh with vertices that no tet touches, pulled along z."""
    mi = Mesh(np.concatenate([m.points, np.random.default_rng(2).random((extra, 3))]), m.cells, {}, m.cell_data)
    pad = lambda a, v: np.concatenate([a, np.full((extra, 3), v, a.dtype)])  # noqa: E731
    f = pad(f, 0.0)
    f[m.n_points:, 2] = force
    return mi, pad(fixed, False), pad(x0, 0.25), f


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_isolated_vertices_of_a_batch_are_stepped_with_their_own_instance(dtype):
    """Their gradient is minus their force and their preconditioner the mean: they move, each at its instance's pace."""
    print(f"[routes] isolated vertices, batch, {dtype}", flush=True)
    cases = [_with_isolated(*_case(n, seed=n), extra, force) for n, extra, force in ((4, 17, -0.5), (5, 300, 0.25))]
    cfg = PncgConfig(rtol=1e-12, max_steps=4)
    t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda").contiguous()  # noqa: E731
    b = batch.Batch([_instance("snh", *c) for c in cases], _lib.APL_SNH, dtype=dtype, device="cuda")
    xb, stb = b.solve(config=cfg)
    for k, (m, fixed, x0, f) in enumerate(cases):
        x = t(x0)
        st = DeviceSolver(_potential("snh", m, dtype)).solve(x, t(f), mask_bits(fixed, "cuda"), cfg)[0]
        assert torch.equal(b.split(xb)[k], x)
        _same(st, stb[k], ("result", "n_steps", "f", "grad_norm", "alpha", "beta"))
        touched = np.zeros(m.n_points, bool)
        touched[m.cells.reshape(-1)] = True
        moved = (x.cpu().numpy() - t(x0).cpu().numpy())[~touched]
        assert (moved[:, :2] == 0).all() and (moved[:, 2] * np.sign(f[-1, 2]) > 0).all()


# FP32: some tens of roundings of 2^-24 per iteration, relative to the largest entry
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 1e-5), (torch.float64, 1e-12)])
def test_cg_directions_of_isolated_vertices(dtype, tol):
    """A right-hand side on vertices no tet touches: H is zero there and the
    preconditioner the mean diagonal, so the direction takes part in every
    later update.  Against a CG on the host with the oracle's Hessian."""
    print(f"[routes] isolated vertices, CG, {dtype}", flush=True)
    m, fixed, x0, f = _with_isolated(*_case(4), 30, 0.0)
    pot = _potential("snh", m, dtype)
    t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda").contiguous()  # noqa: E731
    rng = np.random.default_rng(6)
    rhs = t(rng.standard_normal(x0.shape)).double().cpu().numpy()
    r0 = Region.from_mesh(m)
    rounded = lambda a: t(a).double().cpu().numpy()  # noqa: E731
    ref = of.FemPotential(of.SNH, m.cells, r0.dhdX, r0.dV, rounded(m.cell_data["mu"]), rounded(m.cell_data["lambda"]))
    u = np.zeros_like(x0)
    diag = ref.hess_diag(u)
    free = ~fixed
    mean = diag[free & (diag > 0)].mean()
    P = np.where(diag > 0, 1 / np.where(diag > 0, diag, 1), 1 / mean)
    iters = 3
    r = np.where(free, rhs, 0.0)
    y, d, rz = np.zeros_like(r), np.zeros_like(r), 1.0
    for k in range(iters):
        z = np.where(free, P * r, 0.0)
        rz, old = (r * z).sum(), rz
        d = z + (rz / old if k else 0.0) * d
        q = np.where(free, ref.hess_prod(u, d), 0.0)
        a = rz / (d * q).sum()
        y, r = y + a * d, r - a * q
    out = torch.full_like(t(x0), 7.0)
    st = DeviceSolver(pot).cg(t(u), t(rhs), out, mask_bits(fixed, "cuda"), rtol=1e-12, max_iters=iters)[0]
    assert st.n_steps == iters
    assert np.abs(y[-30:]).max() > 0.01 * np.abs(y).max()
    assert np.abs(out.double().cpu().numpy() - y).max() <= tol * np.abs(y).max()
