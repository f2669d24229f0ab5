"""The extension module that calls the library from torch tensors is an
accelerator: without it the library builds and every call takes the checked
Python path, as it did before there was one."""

import ctypes
import os
import subprocess
import sys
import warnings

import numpy as np
import pytest
import torch

from apple_amd import _lib, build, fem
from apple_amd.mesh import Region, cube

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_a_library_without_the_module_is_used_as_it_is(tmp_path, monkeypatch):
    monkeypatch.setattr(_lib, "LIB_PATH", str(tmp_path / "libapple_amd.so"))
    monkeypatch.setattr(_lib, "_calls", None)
    with pytest.warns(RuntimeWarning, match="tensor_calls.so is missing"):
        assert not _lib.calls()
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        assert not _lib.calls()  # said once


@pytest.mark.gpu
def test_calls_without_the_module_give_the_same(monkeypatch):
    m = cube(3)
    rng = np.random.default_rng(0)
    m.cell_data["mu"] = 1e4 * np.exp(0.5 * rng.standard_normal(m.n_cells))
    m.cell_data["lambda"] = 10 * m.cell_data["mu"]
    m.cell_data["activation"] = 0.1 * rng.standard_normal((m.n_cells, 6))
    pot = fem.StableNeoHookeanMuscle.from_region(Region.from_mesh(m), device="cuda")
    t = lambda a: torch.as_tensor(a, dtype=torch.float32, device="cuda")  # noqa: E731
    u, p = t(0.01 * rng.standard_normal(m.points.shape)), t(rng.standard_normal(m.points.shape))

    def calls():
        g, e = torch.zeros_like(u), torch.zeros(1, dtype=torch.float64, device="cuda")
        pot.fused(u, e, g, None)
        return [g, e, *pot.mixed_derivative_prod(u, p).values()]

    native = calls()
    monkeypatch.setattr(_lib, "_calls", ())
    for a, b in zip(native, calls()):
        assert torch.equal(a, b) and a.abs().max() > 0


def test_import_without_the_raw_stream_lookup():
    """A PyTorch without CUDA or ROCm has no torch._C._cuda_getCurrentRawStream: the package imports there."""
    code = ("import torch\n"
            "if hasattr(torch._C, '_cuda_getCurrentRawStream'):\n"
            "    del torch._C._cuda_getCurrentRawStream\n"
            "import apple_amd.runtime, apple_amd.fem, apple_amd.mesh\n"
            "print('imported')\n")
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300, cwd=ROOT)
    assert r.returncode == 0 and r.stdout.strip().endswith("imported"), r.stderr


def test_the_library_is_linked_whatever_becomes_of_the_module(tmp_path, monkeypatch):
    """The C ABI needs neither PyTorch's nor Python's headers."""
    src = tmp_path / "one.cpp"
    src.write_text('extern "C" int one() { return 1; }\n')
    monkeypatch.setattr(build, "LIBDIR", str(tmp_path / "lib"))
    monkeypatch.setattr(build, "OBJDIR", str(tmp_path / "lib" / "obj"))
    monkeypatch.setattr(build, "sources", lambda: [str(src)])
    lib = tmp_path / "lib" / build.LIBNAME

    def fails():
        raise RuntimeError("compile failed: no headers")

    monkeypatch.setattr(build, "_build_module", fails)
    with pytest.raises(RuntimeError, match="no headers"):  # said, and the library is there
        build.build(verbose=False)
    assert ctypes.CDLL(str(lib)).one() == 1
    lib.unlink()

    def no_torch():
        raise ImportError("no module named torch")

    monkeypatch.setattr(build, "_build_module", no_torch)
    assert build.build(verbose=False) == str(lib) and lib.exists()
