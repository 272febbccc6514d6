"""Acceptance of the diagonalised solves (csrc/helmholtz.h, compiled with g++): every
degree of the library is accepted, and solutions off by 5e-12 are refused, those off
by 5e-13 not (the bar is 1e-12; the solves come within 1e-13 at every degree)."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def accept(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("ha") / "libha.so"
    subprocess.run([cxx, "-O2", "-std=c++17", "-shared", "-fPIC",
                    os.path.join(HERE, "native", "helmholtz_accept_harness.cpp"), "-o", str(out)], check=True,
                   capture_output=True)
    f = ctypes.CDLL(str(out)).accept_c
    f.argtypes = [ctypes.c_int, ctypes.c_int] + 4 * [ctypes.c_double]
    return f


@pytest.mark.parametrize("N", [4, 5, 16, 33, 96, 193, 256])
def test_bar(accept, N):
    for par in (0, 1):
        if (N // 2 + 1 if par == 0 else (N + 1) // 2) < 3:
            continue  # no interior row of v
        assert accept(N, par, 1e-6, 0.25, 5e3, 5e-12) == 0, par
        assert accept(N, par, 1e-6, 0.25, 5e3, 5e-13) == 1, par


def test_every_degree_is_accepted(accept):
    for N in range(4, 257):
        for par in (0, 1):
            assert accept(N, par, 10.0 ** -(3 + N % 6), 0.0625, 1e5, 0.0) == 1, (N, par)
