"""Calls straight from torch tensors: a plain tensor of the right form takes
the native path, anything else the checked one, with the results and errors
that it always had."""

import numpy as np
import pytest
import torch

from apple_amd import _lib, fem
from apple_amd.mesh import Region, cube


class _Sub(torch.Tensor):
    pass


def test_what_is_not_a_plain_device_tensor_is_declined():
    """No entry is called (its address here is not one): None comes back."""
    mod = _lib.calls()[0]
    spec = (0, 0, 1, 1, 1)
    for t in (torch.zeros(1), torch.zeros(1).as_subclass(_Sub), torch.zeros(1, device="meta"), 3, "x"):
        assert mod.elem_eval(1, 1, 0, spec, 0, False, t, *[None] * 10) is None
        assert mod.elem_mixed_activation(1, 1, 0, spec, False, t, *[None] * 6) is None
        assert mod.set_activation(1, 1, 0, spec, t) is None
    for bad in ((), (1, 1), (1, 0, 0, spec, None), (1, 1, 0, spec[:4], None), ("1", 1, 0, spec, None)):
        assert mod.set_activation(*bad) is None


FORMS = {
    "plain": (lambda t: t, None),
    "parameter": (lambda t: torch.nn.Parameter(t, requires_grad=True), None),
    "subclass": (lambda t: t.as_subclass(_Sub), None),
    "view of a larger one": (lambda t: torch.cat([t, t])[: t.shape[0]], None),
    "other dtype": (lambda t: t.double() if t.dtype == torch.float32 else t.float(), TypeError),
    "host": (lambda t: t.cpu(), ValueError),
    "flat": (lambda t: t.reshape(-1), ValueError),
    "too many rows": (lambda t: torch.cat([t, t]), ValueError),
    "transposed strides": (lambda t: t.t().contiguous().t(), ValueError),
    "no tensor": (lambda t: t.tolist(), TypeError),
}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("form", FORMS)
def test_forms_are_taken_or_refused_as_before(form, dtype):
    m = cube(3)
    rng = np.random.default_rng(0)
    m.cell_data["mu"] = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    m.cell_data["lambda"] = 10 * m.cell_data["mu"]
    m.cell_data["activation"] = 0.1 * rng.standard_normal((m.n_cells, 6))
    pot = fem.StableNeoHookeanMuscle.from_region(Region.from_mesh(m), dtype=dtype, device="cuda")
    t = lambda a: torch.as_tensor(a, dtype=dtype, device="cuda")  # noqa: E731
    u, p = t(0.01 * rng.standard_normal(m.points.shape)), t(rng.standard_normal(m.points.shape))
    make, error = FORMS[form]

    def calls(w, act):
        g = torch.zeros_like(u)
        pot.grad(w, g)
        pot.mesh.set_activation(act)
        return [g, *(pot.mixed_derivative_prod(w, p)[k] for k in ("mu", "lambda", "activation"))]

    act = pot.materials["activation"]
    if error is None:
        for a, b in zip(calls(make(u), make(act)), calls(u, act)):
            assert torch.equal(a, b) and a.abs().max() > 0
    else:
        with pytest.raises(error):
            pot.grad(make(u), torch.zeros_like(u))
        with pytest.raises(error):
            pot.mixed_derivative_prod(make(u), p)
        with pytest.raises(error):
            pot.mesh.set_activation(make(act))
        with pytest.raises(error):
            pot.grad(u, make(torch.zeros_like(u)))
