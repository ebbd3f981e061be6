"""Coefficients with which the batched solver adds up an inner solve's
correction from its kept preconditioned residuals (CPU; the device kernels
call the same helper)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")


@pytest.fixture(scope="module")
def driver(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = str(tmp_path_factory.mktemp("combination") / "combination_check")
    src = os.path.join(ROOT, "tests", "native", "combination_check.cpp")
    subprocess.run([HIPCC, "-O2", "-std=c++17", f"-I{ROOT}/include", f"-I{ROOT}/tetmag_amd/csrc", src, "-o", exe],
                   check=True, capture_output=True)
    return exe


@pytest.mark.parametrize("K", [1, 2, 7, 40])
@pytest.mark.parametrize("stride", [1, 64])
def test_coefficients_of_the_iterations_that_ran(driver, K, stride):
    """c_i = sum_{k >= i} alpha_k beta_{i+1} ... beta_k.  The V-cycle after the
    last iteration is left out, so beta_K is never written and must not be read:
    it is NaN here."""
    c = np.array(subprocess.run([driver, str(K), str(stride)], check=True, capture_output=True,
                                text=True).stdout.split(), float)
    alpha, beta = 1.0 / np.arange(1, K + 1), np.arange(K) / 8.0
    # the sum over the directions p_k = sum_i P[k, i] z_i themselves
    P = np.eye(K)
    for k in range(1, K):
        P[k] += beta[k] * P[k - 1]
    ref = alpha @ P
    # K products and sums each way, all terms positive
    np.testing.assert_allclose(c, ref, rtol=4 * K * 2.3e-16, atol=0)
