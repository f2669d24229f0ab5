"""A step-wise solve with other calls of the same solver and mesh between its steps."""

import numpy as np
import pytest
import torch

from apple_amd import _lib, batch
from apple_amd.mesh import Region, cube
from apple_amd.solver import DeviceSolver, PncgConfig

pytestmark = pytest.mark.gpu


def _instance(n):
    m = cube(n)
    rng = np.random.default_rng(n)
    mu = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    fixed = np.repeat(m.points[:, 2:] == 0.0, 3, axis=1)
    x0 = np.where(fixed, 0.0, 0.1 / n * rng.standard_normal((m.n_points, 3)))
    f = np.zeros((m.n_points, 3))
    f[:, 2] = -1.0 / m.n_points
    return batch.Instance(Region.from_mesh(m), mu, 10 * mu, f, fixed, x0)


@pytest.mark.parametrize("sizes", [(5,), (5, 3)])
@pytest.mark.parametrize("iters", [7, 8])
def test_other_calls_between_the_steps_of_a_solve(sizes, iters):
    """An adjoint solve by the same solver and evaluations on the same mesh
    leave a step-wise solve as it is (either parity of the CG's own buffers)."""
    print(f"[between] sizes {sizes}, {iters} iterations", flush=True)
    b = batch.Batch([_instance(n) for n in sizes], _lib.APL_SNH, device="cuda")
    cfg = PncgConfig(rtol=1e-12, max_steps=50)
    rhs = torch.as_tensor(np.random.default_rng(1).standard_normal(b.x0.shape), dtype=torch.float32, device="cuda")

    def solve(between):
        s = DeviceSolver(b.potential)
        x, seen = b.x0.clone(), []
        s.begin(x, b.f_ext, b.mask, cfg)
        for k in range(4):
            at = torch.empty_like(x)
            opt = s.advance(1, x_out=at)
            seen.append((at, [(o.n_steps, o.convergence_state.grad_norm, o.beta) for o in opt]))
            if between:
                s.cg(at, rhs, torch.empty_like(x), b.mask, rtol=1e-12, max_iters=iters)
                b.mesh.eval(_lib.APL_SNH, b.mu, b.lam, at, rhs, grad=torch.empty_like(x), hess_prod=torch.empty_like(x))
        st = s.end()
        return x, seen, [(q.n_steps, q.f, q.grad_norm) for q in st]

    x, seen, st = solve(False)
    xc, seenc, stc = solve(True)
    for (a, oa), (c, oc) in zip(seen, seenc):
        assert torch.equal(a, c) and oa == oc
    assert torch.equal(x, xc) and st == stc
    assert torch.equal(x, seen[-1][0]) and not torch.equal(seen[0][0], seen[-1][0])
