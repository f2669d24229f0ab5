"""The CG's step length a = r.z / d.Hd: d.Hd is formed and added in FP64, also
on FP32 meshes.

At rest, on cells of unit size with moduli and directions that are small whole
numbers, every FP32 factor (stress increment, direction gradient, residual) is
exact, and the products and their sum are whole multiples of 1/4 below 2^53:
FP64 gives them exactly, in any order, and FP32 does not (products of more
than 24 bits)."""

import numpy as np
import pytest
import torch

from apple_amd import _lib, batch, fem
from apple_amd.mesh import Region, cube
from apple_amd.solver import DeviceSolver, mask_bits

pytestmark = pytest.mark.gpu


def _region(n):
    m = cube(n, 0.0, float(n))
    rng = np.random.default_rng(n)
    m.cell_data["mu"] = rng.integers(1, 5, m.n_cells).astype(float)
    m.cell_data["lambda"] = rng.integers(4, 9, m.n_cells).astype(float)
    r = Region.from_mesh(m)
    r.dminv = np.round(2 * r.dminv) / 2  # entries 0, +-1/2, +-1
    r.dV = np.round(6 * r.dV)  # six times the volume: 1 or 2
    r.dhdX = np.concatenate([-r.dminv.sum(1, keepdims=True), r.dminv], 1)
    return r


def _d_h_d(r, d):
    """d.H(0)d of stable Neo-Hookean in whole numbers: dP = mu (dF + dF^T) + (lambda - mu) tr(dF) I."""
    m = r.mesh
    dF = np.einsum("tai,taj->tij", d[m.cells], r.dhdX)
    mu, lam = m.cell_data["mu"][:, None, None], m.cell_data["lambda"][:, None, None]
    tr = np.trace(dF, axis1=1, axis2=2)[:, None, None]
    dP = mu * (dF + dF.transpose(0, 2, 1)) + (lam - mu) * tr * np.eye(3)
    return float((4 * r.dV[:, None, None] * dP * dF).sum()) / 4


# a block per 256 tets, and blocks whose threads take two and four tets
@pytest.mark.parametrize("chunks", [1, 2, 4])
@pytest.mark.parametrize("batched", [False, True])
def test_step_length_is_formed_in_fp64(chunks, batched):
    print(f"[cg step] chunks {chunks} batched {batched}", flush=True)
    rng = np.random.default_rng(0)
    regions = [_region(n) for n in ((6, 3) if batched else (6,))]
    ks, fixed = [], []
    for r in regions:
        k = rng.integers(-2047, 2048, r.mesh.points.shape).astype(float)
        k[r.mesh.points[:, 2] == 0.0] = 0.0
        ks.append(k)
        fixed.append(np.repeat(r.mesh.points[:, 2:3] == 0.0, 3, axis=1))
    t = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    if batched:
        b = batch.Batch([batch.Instance(r, r.mesh.cell_data["mu"], r.mesh.cell_data["lambda"], None, f, None)
                         for r, f in zip(regions, fixed)], _lib.APL_SNH, device="cuda", chunks=chunks)
        mesh, solver, mask, mu, lam = b.mesh, b.solver(), b.mask, b.mu, b.lam
    else:
        pot = fem.StableNeoHookean.from_region(regions[0], device="cuda", chunks=chunks)
        mesh, solver, mask = pot.mesh, DeviceSolver(pot), mask_bits(fixed[0], "cuda")
        mu, lam = pot.materials["mu"], pot.materials["lambda"]
    x, diag, k = t(np.zeros((mesh.n_verts, 3))), t(np.zeros((mesh.n_verts, 3))), t(np.concatenate(ks))
    mesh.eval(_lib.APL_SNH, mu, lam, x, hess_diag=diag)
    rhs = diag * k  # so that the first direction, rhs / diag, is k
    stats = solver.cg(x, rhs, torch.empty_like(x), mask, rtol=0.0, max_iters=1)
    start = 0
    for r, kk, st in zip(regions, ks, stats):
        rows = rhs[start : start + len(kk)].double().cpu().numpy()
        start += len(kk)
        dhd, rz = _d_h_d(r, kk), float((4 * rows * kk).sum()) / 4
        assert dhd != float(np.float32(dhd)) and dhd > 0
        assert st.n_steps == 1 and st.alpha == rz / dhd
