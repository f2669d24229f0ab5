"""The ARAP kernels' SVD over the shapes that decide its route (squeezed, drawn
out, flattened elements), compiled for the host: no less accurate than FP32
Jacobi sweeps for every element, against the FP64 SVD."""

import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def rows(tmp_path_factory):
    cxx = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(cxx):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("arap") / "arap_ranges")
    subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(HERE, "host", "arap_ranges.cpp"), "-o", exe],
                   check=True, capture_output=True)
    out = subprocess.run([exe], check=True, capture_output=True, text=True).stdout
    return {line.split()[0]: np.array([float(x) for x in line.split()[1:]]) for line in out.strip().splitlines()}


def test_sigma_minus_one_takes_the_correctly_rounded_root(rows):
    exact, approximate = rows["sqrt"]
    assert exact == 5 and approximate == 0


# The root mean squares of two formulas of one precision over 20,000 samples
# agree to about a hundredth when they are equally good; the worst of 20,000
# scatters by some tens of per cent.
def _no_less_accurate(rows, names):
    for name in names:
        sweeps, fast = rows[name][:4], rows[name][4:]
        for k in (0, 2):
            assert fast[k] <= 1.5 * sweeps[k], (name, fast, sweeps)
            assert fast[k + 1] <= 1.02 * sweeps[k + 1], (name, fast, sweeps)


def test_squeezed_and_moderate_elements(rows):
    names = [n for n in rows if n.startswith(("all_", "strain_"))] + ["any_1.25", "any_2", "long_1.5", "long_2", "flat_2"]
    assert len(names) == 20
    _no_less_accurate(rows, names)


# Drawn out or flattened, the error of the rotation about the long axis (or in
# the flat plane) grows with sigma_0^2 / (sigma_1 (sigma_1 + sigma_2)).
def test_drawn_out_and_flattened_elements(rows):
    names = [n for n in rows if n.startswith(("long_", "flat_", "any_"))]
    assert len(names) == 19
    _no_less_accurate(rows, names)
    # singular values drawn log-uniformly from [0.1, 10]: the extreme ones among
    # them finish in FP64, the others keep what FP32 loses up to the threshold
    assert rows["any_10"][4] <= 1e-5 and rows["any_10"][6] <= 2e-5
