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
