"""The FP32 ARAP passes choose the route of the SVD by wave (64 tets): one
inverted or drawn-out tet sends its wave the other way.  Per-tet results of
every tet of a wave, with such tets at its edges, against FP64."""

import numpy as np
import pytest
import torch

from apple_amd import _lib
from apple_amd.runtime import DeviceMesh

pytestmark = pytest.mark.gpu


def _rotations(rng, n):
    q, r = np.linalg.qr(rng.standard_normal((n, 3, 3)))
    q *= np.sign(np.einsum("tii->ti", r))[:, None, :]
    q[np.linalg.det(q) < 0, :, 2] *= -1
    return q


@pytest.mark.parametrize("n", [1, 63, 64, 65, 257, 700])
@pytest.mark.parametrize("shape", ["inverted", "drawn out", "flat"])
@pytest.mark.parametrize("where", ["none", "first", "last", "some", "all"])
def test_every_tet_of_a_mixed_wave(n, shape, where):
    print(f"[arap waves] {n} tets, {shape}, {where}", flush=True)
    rng = np.random.default_rng(n)
    k = np.arange(n)
    odd = {"none": k < 0, "first": k % 64 == 0, "last": (k % 64 == 63) | (k == n - 1), "some": k % 37 == 5, "all": k >= 0}[where]
    s = rng.uniform(0.7, 1.4, (n, 3))
    s[odd] = {"inverted": (1.3, 1.0, -0.6), "drawn out": (6.0, 1.1, 0.8), "flat": (1.5, 1.2, 0.005)}[shape]
    U, V = _rotations(rng, n), _rotations(rng, n)
    F = U * s[:, None, :] @ V.transpose(0, 2, 1)
    # a tet of its own per F: the unit one, displaced by (F - I) X
    X = np.concatenate([np.zeros((1, 3)), np.eye(3)])
    u = (np.einsum("tij,aj->tai", F - np.eye(3), X)).astype(np.float32)
    p = rng.standard_normal((n, 4, 3)).astype(np.float32)
    mesh = DeviceMesh(np.arange(4 * n).reshape(n, 4), np.broadcast_to(np.eye(3), (n, 3, 3)), np.ones(n), 4 * n, device="cuda")
    t = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda").contiguous()  # noqa: E731
    dmu = torch.empty(n, device="cuda")
    mesh.eval(_lib.APL_ARAP, t(np.ones(n)), None, t(u.reshape(-1, 3)), t(p.reshape(-1, 3)), dmu=dmu)
    # (F - R) : dF of the F that FP32 holds, R = U V^T with the sign of det F on the smallest singular value
    Fd = np.eye(3) + (u[:, 1:] - u[:, :1]).astype(float).transpose(0, 2, 1)
    dF = (p[:, 1:].astype(float) - p[:, :1]).transpose(0, 2, 1)
    a, sv, b = np.linalg.svd(Fd)
    a[:, :, 2] *= np.where(np.linalg.det(a) * np.linalg.det(b) < 0, -1.0, 1.0)[:, None]
    P = Fd - a @ b
    # the stress to 5e-6 of its largest entry (what the host harness holds the
    # SVD to), the nine products with dF rounded to FP32
    bound = 9 * (5e-6 + 2e-6) * np.abs(P).max((1, 2)) * np.abs(dF).max((1, 2))
    err = np.abs(dmu.double().cpu().numpy() - (P * dF).sum((1, 2)))
    assert (err <= bound).all(), (err / bound).max()
