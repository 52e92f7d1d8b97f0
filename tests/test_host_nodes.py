"""The node kernels' waveform (node_values: powers of the frequency from a table) and its adjoint
(node_adjoint) against the dual-number waveform (Phenom::amp_phase), on the CPU: every mode, every
region of the ansatz and both sides of each region's edge, equal and unequal masses."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = "/opt/rocm/llvm/bin/clang++" if os.path.exists("/opt/rocm/llvm/bin/clang++") else shutil.which("clang++")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if CXX is None:
        pytest.skip("no clang++")
    from pespace_amd.build import gen_qnm_inc
    gen_qnm_inc()
    exe = str(tmp_path_factory.mktemp("nodes") / "host_nodes")
    subprocess.run([CXX, "-std=c++17", "-O2", "-I", os.path.join(ROOT, "tests", "host_kernel", "stub"),
                    "-I", os.path.join(ROOT, "pespace_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host_kernel", "host_nodes.cpp"), "-o", exe], check=True)
    return exe


@pytest.mark.parametrize("seed", [1, 2])
def test_nodes_against_dual_waveform(driver, seed):
    out = subprocess.run([driver, str(seed)], check=True, capture_output=True, text=True).stdout.split()
    # sums of at most ~30 roundings of 1.1e-16 (the ninth power of the cube root among them) of terms
    # that cancel by at most two orders of magnitude: 30 * 1.1e-16 * 100 = 3e-13; the gradients' terms
    # cancel by one order more (the alignment's t0 against the phase's slope)
    assert all(float(v) < 1e-12 for v in out[:4]), out
    assert all(float(v) < 1e-11 for v in out[4:]), out
