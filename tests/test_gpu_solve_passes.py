"""The solver's element passes that carry the vector updates and, for a
single instance, the scalar steps.

* A single instance takes its scalar steps inside the element passes up to
  fixed table sizes, a batch in kernels of their own: the same iterate, bit
  for bit, on both sides of those sizes.
* Vertices that no tet touches are stepped outside the blocks: they change
  nothing for the others and stay where they are when nothing pulls at them.
"""

import numpy as np
import pytest
import torch

from apple_amd import _lib, batch, fem
from apple_amd.mesh import Mesh, Region, cube
from apple_amd.solver import DeviceSolver, PncgConfig, mask_bits

pytestmark = pytest.mark.gpu


def _case(n, seed=0):
    m = cube(n)
    rng = np.random.default_rng(seed)
    mu = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    m.cell_data["mu"] = mu
    m.cell_data["lambda"] = 10 * mu
    fixed = np.zeros((m.n_points, 3), bool)
    fixed[m.points[:, 2] == 0.0] = True
    x0 = 0.1 / n * rng.standard_normal((m.n_points, 3))
    x0[fixed] = 0.0
    f = np.zeros((m.n_points, 3))
    f[:, 2] = -1.0 / m.n_points
    return m, fixed, x0, f


# one block; the largest and the next size with the decision in the pass
# (192 vertex blocks), with the step length in the pass (2,048 element blocks)
@pytest.mark.parametrize("n", [2, 35, 36, 46, 47])
def test_single_instance_equals_the_same_instance_of_a_batch(n):
    print(f"[passes] n = {n}", flush=True)
    m, fixed, x0, f = _case(n)
    r = Region.from_mesh(m)
    m2, fixed2, x2, f2 = _case(3, seed=1)
    r2 = Region.from_mesh(m2)
    cfg = PncgConfig(rtol=1e-9, max_steps=9)
    pot = fem.StableNeoHookean.from_region(r, device="cuda")
    x = torch.as_tensor(x0, dtype=torch.float32, device="cuda")
    st = DeviceSolver(pot).solve(x, torch.as_tensor(f, dtype=torch.float32, device="cuda"), mask_bits(fixed, "cuda"), cfg)[0]
    insts = [batch.Instance(r, m.cell_data["mu"], m.cell_data["lambda"], f, fixed, x0),
             batch.Instance(r2, m2.cell_data["mu"], m2.cell_data["lambda"], f2, fixed2, x2)]
    b = batch.Batch(insts, _lib.APL_SNH, device="cuda")
    xb, stb = b.solve(config=cfg)
    assert torch.equal(b.split(xb)[0], x)
    assert (st.n_steps, st.n_evals, st.f, st.grad_norm, st.alpha, st.beta) == (
        stb[0].n_steps, stb[0].n_evals, stb[0].f, stb[0].grad_norm, stb[0].alpha, stb[0].beta)


# likewise the CG: the step from the blocks' d.Hd (2,048 element blocks), beta
# from two columns per vertex block (1,024 of them), and the normal equations
@pytest.mark.parametrize("n,normal", [(2, False), (46, False), (47, False), (63, False), (64, False), (6, True)])
def test_single_cg_equals_the_same_instance_of_a_batch(n, normal):
    print(f"[passes] CG n = {n} normal {normal}", flush=True)
    m, fixed, x0, f = _case(n)
    m2, fixed2, x2, f2 = _case(3, seed=1)
    r, r2 = Region.from_mesh(m), Region.from_mesh(m2)
    pot = fem.StableNeoHookean.from_region(r, device="cuda")
    t = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    rhs, rhs2 = t(np.random.default_rng(4).standard_normal(x0.shape)), t(np.random.default_rng(5).standard_normal(x2.shape))
    kw = dict(rtol=1e-12, max_iters=7, normal=normal)
    y = torch.empty_like(rhs)
    st = DeviceSolver(pot).cg(t(0.1 * x0), rhs, y, mask_bits(fixed, "cuda"), **kw)[0]
    b = batch.Batch([batch.Instance(r2, m2.cell_data["mu"], m2.cell_data["lambda"], f2, fixed2, x2),
                     batch.Instance(r, m.cell_data["mu"], m.cell_data["lambda"], f, fixed, x0)], _lib.APL_SNH, device="cuda")
    yb = torch.empty_like(b.x0)
    stb = b.solver().cg(t(torch.cat([t(0.1 * x2), t(0.1 * x0)])), torch.cat([rhs2, rhs]), yb, b.mask, **kw)[1]
    assert st.n_steps == 7 and torch.isfinite(y).all()
    assert torch.equal(b.split(yb)[1], y)
    assert (st.result, st.n_steps, st.f, st.grad_norm, st.alpha, st.beta) == (
        stb.result, stb.n_steps, stb.f, stb.grad_norm, stb.alpha, stb.beta)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("cls", [fem.StableNeoHookean, fem.Arap])
def test_vertices_without_tets(cls, dtype):
    print(f"[passes] isolated vertices {cls.__name__} {dtype}", flush=True)
    m, fixed, x0, f = _case(5)
    extra = 30  # 216 + 30 vertices: the same vertex blocks with and without
    mi = Mesh(np.concatenate([m.points, np.random.default_rng(2).random((extra, 3))]), m.cells, {}, m.cell_data)
    pad = lambda a, v: np.concatenate([a, np.full((extra, 3), v, a.dtype)])  # noqa: E731
    out = []
    for mesh, fx, x_, f_ in ((m, fixed, x0, f), (mi, pad(fixed, False), pad(x0, 0.25), pad(f, 0.0))):
        pot = cls.from_pyvista(mesh, dtype=dtype, device="cuda", setup="device")
        s = DeviceSolver(pot)
        t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda").contiguous()  # noqa: E731
        x, mask = t(x_), mask_bits(fx, "cuda")
        st = s.solve(x, t(f_), mask, PncgConfig(rtol=1e-5))[0]
        rhs = t(np.concatenate([np.random.default_rng(3).standard_normal((m.n_points, 3)),
                                np.zeros((mesh.n_points - m.n_points, 3))]))
        y = torch.full_like(x, 7.0)
        sc = s.cg(x, rhs, y, mask, rtol=1e-5)[0]
        out.append((x, y, st, sc))
    (xa, ya, sa, ca), (xb, yb, sb, cb) = out
    assert torch.equal(xb[: m.n_points], xa) and torch.equal(yb[: m.n_points], ya)
    assert torch.equal(xb[m.n_points:], torch.full_like(xb[m.n_points:], 0.25))
    assert not yb[m.n_points:].any()
    assert (sa.n_steps, sa.result, ca.n_steps, ca.result) == (sb.n_steps, sb.result, cb.n_steps, cb.result)


def test_a_mesh_without_tets_ends_at_once():
    m = Mesh(np.zeros((5, 3)), np.zeros((0, 4), np.int32), {}, {"mu": np.zeros(0), "lambda": np.zeros(0)})
    pot = fem.StableNeoHookean.from_pyvista(m, device="cuda", setup="device")
    x = torch.full((5, 3), 0.5, device="cuda")
    st = DeviceSolver(pot).solve(x, None, None, PncgConfig())[0]
    assert st.success and st.n_steps == 0
    assert torch.equal(x, torch.full_like(x, 0.5))


# the evaluation's vertex sums: one block, the largest and the next size whose partials are all in flight at
# once (two vertex blocks per CU: 512), against the loop that a batch takes: the same sums, bit for bit
@pytest.mark.parametrize("n", [2, 49, 50])
def test_single_evaluation_equals_the_same_instance_of_a_batch(n):
    print(f"[passes] evaluation n = {n}", flush=True)
    m, fixed, x0, f = _case(n)
    m2, fixed2, x2, f2 = _case(3, seed=1)
    r, r2 = Region.from_mesh(m), Region.from_mesh(m2)
    t = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    b = batch.Batch([batch.Instance(r2, m2.cell_data["mu"], m2.cell_data["lambda"], f2, fixed2, x2),
                     batch.Instance(r, m.cell_data["mu"], m.cell_data["lambda"], f, fixed, x0)], _lib.APL_SNH, device="cuda")
    pot = fem.StableNeoHookean.from_region(r, device="cuda")
    g, h = torch.empty_like(t(x0)), torch.empty_like(t(x0))
    pot.fused(t(x0), None, g, h, accumulate=False)
    gb, hb = torch.empty_like(b.x0), torch.empty_like(b.x0)
    b.mesh.eval(_lib.APL_SNH, b.mu, b.lam, torch.cat([t(x2), t(x0)]), grad=gb, hess_diag=hb)
    assert torch.equal(b.split(gb)[1], g) and torch.equal(b.split(hb)[1], h)
    assert g.abs().max() > 0 and h.abs().max() > 0
