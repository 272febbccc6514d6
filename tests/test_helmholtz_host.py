"""Host set-up of the diagonalised wall-normal solves (csrc/helmholtz.h),
compiled with g++: each half system's v and omega_y solution against the dense
collocation systems of the oracle (get_coef_v, get_coef_omegay, folded by
parity), over degrees, time-step coefficients and wavenumbers."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import cf_oracle as O

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("hh") / "libhh.so"
    subprocess.run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "native", "helmholtz_harness.cpp"), "-o", str(out)], check=True,
                   capture_output=True)
    l = ctypes.CDLL(str(out))
    dp = ctypes.POINTER(ctypes.c_double)
    l.helmholtz_c.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_double, ctypes.c_double, dp, dp]
    return l


# The dense inverse's own error is cond(A) eps, at most 2e-11 of the solution
# over these systems against an extended-precision solve; the bar leaves it a factor of 5.
@pytest.mark.parametrize("N,c", [(4, 1e-3), (5, 1e-3), (7, 1e-5), (16, 1e-4), (21, 1.4e-6), (32, 1.7e-7),
                                 (33, 1e-6), (64, 5e-5), (100, 1e-7), (129, 1e-7), (192, 1.6e-8), (256, 1e-8)])
def test_half_systems_match_dense(lib, N, c):
    t0, _, t2, t4 = O.scheb(N)
    dp = ctypes.POINTER(ctypes.c_double)
    rng = np.random.default_rng(N)
    for par in (0, 1):
        n = N // 2 + 1 if par == 0 else (N + 1) // 2
        l = 2 * np.arange(n) + par
        for is_v in (0, 1):
            for k2 in (0.25, 5.0, 1.0e3, 8.0e4) if is_v else (0.0, 1.0, 8.0e4):
                if is_v:
                    rows = (-c * t4 + (1 + 2 * c * k2) * t2 - k2 * (1 + c * k2) * t0)[2:n][:, l]
                    a = np.vstack([np.ones(n), l.astype(float) ** 2, rows]) if n >= 2 else np.ones((1, 1))
                else:
                    a = np.vstack([np.ones(n), (-c * t2 + (1 + c * k2) * t0)[1:n][:, l]])
                f = np.zeros(max(n - 1, 1))
                f[is_v:n - 1] = rng.standard_normal(max(n - 1 - is_v, 0))
                x = np.full(n, np.nan)
                rc = lib.helmholtz_c(N, par, is_v, c, k2, f.ctypes.data_as(dp), x.ctypes.data_as(dp))
                assert rc == 0, (par, is_v, k2, rc)
                rhs = np.zeros(n)
                rhs[1 + is_v:] = f[is_v:n - 1]
                ref = np.linalg.solve(a, rhs)
                err = np.abs(x - ref).max()
                assert err <= 1e-10 * np.abs(ref).max(), (par, is_v, k2, err, np.abs(ref).max())
