"""The register DFTs with a factor 5 (the wall-normal FFTs of degrees such as 50,
100, 150, 160, 200), and the radices 9 and 18 beside them, compiled for the host:
every unit impulse in both directions and both precisions against the exact
exponentials, within rounding."""
import ctypes
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
RADICES = [5, 9, 10, 15, 18, 20]

SOURCE = """
#include "%s"
template <int R, int S, class V>
static void run(double* x) {
  V v[R];
  for (int i = 0; i < R; ++i) { v[i].x = x[2 * i]; v[i].y = x[2 * i + 1]; }
  chf::Dft<R, S, V>::run(v);
  for (int i = 0; i < R; ++i) { x[2 * i] = v[i].x; x[2 * i + 1] = v[i].y; }
}
template <int R>
static void all(int s, int f, double* x) {
  if (f) { if (s > 0) run<R, 1, float2>(x); else run<R, -1, float2>(x); }
  else { if (s > 0) run<R, 1, double2>(x); else run<R, -1, double2>(x); }
}
extern "C" void dft(int r, int s, int f, double* x) {
  switch (r) { %s }
}
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    hipcc = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)
    if hipcc is None:
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("dft5")
    header = os.path.join(os.path.dirname(HERE), "channel_flow_amd", "csrc", "fftreg.h")
    src = d / "dft5.hip"
    src.write_text(SOURCE % (header, " ".join(f"case {r}: all<{r}>(s, f, x); break;" for r in RADICES)))
    out = d / "libdft5.so"
    subprocess.run([hipcc, "-O2", "-std=c++17", "-shared", "-fPIC", "--offload-arch=gfx950",
                    "-Wno-unused-command-line-argument", str(src), "-o", str(out)], check=True, capture_output=True)
    return ctypes.CDLL(str(out))


@pytest.mark.parametrize("r", RADICES)
@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("fp32", [0, 1])
def test_impulses(lib, r, sign, fp32):
    for n in range(r):
        x = np.zeros(2 * r)
        x[2 * n] = 1.0
        lib.dft(r, sign, fp32, x.ctypes.data_as(ctypes.c_void_p))
        exact = np.exp(sign * 2j * np.pi * (n * np.arange(r) % r) / r)
        # two rounded twiddles and up to three levels of sums on values of modulus 1
        assert np.max(np.abs(x[0::2] + 1j * x[1::2] - exact)) < 8 * np.finfo(np.float32 if fp32 else np.float64).eps
