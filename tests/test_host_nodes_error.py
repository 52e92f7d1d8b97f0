"""Rounding errors of the node kernels' waveform (node_values) on the CPU: A, dA/du, Psi and dPsi/du of
every mode are no further from the same formulas in extended precision than the dual-number waveform,
which takes each elementary function per frequency.

rms errors over 24,000 random binaries and frequencies per mode and range (from the early inspiral to the
ringdown); two rms values of that many draws differ by about 1% by chance, 5% is allowed.
"""

import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++" if os.path.exists("/opt/rocm/llvm/bin/clang++") else shutil.which("clang++")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if CXX is None:
        pytest.skip("no clang++")
    from pespace_amd.build import gen_qnm_inc
    gen_qnm_inc()
    exe = str(tmp_path_factory.mktemp("nodes") / "host_node_error")
    # contraction as in device code
    subprocess.run([CXX, "-std=c++17", "-O2", "-ffp-contract=fast", "-mfma", "-I",
                    os.path.join(ROOT, "tests", "host_kernel", "stub"), "-I", os.path.join(ROOT, "pespace_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host_kernel", "host_node_error.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("x_lo,x_hi", [(1e-5, 0.005), (2e-4, 0.9), (5e-3, 0.9), (0.02, 0.25)])
def test_node_values_as_accurate_as_the_dual_waveform(driver, x_lo, x_hi):
    out = subprocess.run([driver, "1", str(x_lo), str(x_hi)], check=True, capture_output=True, text=True).stdout
    v = np.array(out.split(), dtype=float).reshape(6, 4, 2)
    print(v)
    assert np.all(v > 0.1) and np.all(v[:, :, 0] <= 1.05 * v[:, :, 1])
