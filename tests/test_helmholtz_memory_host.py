"""Host set-up of the diagonalised solves (csrc/helmholtz.h) without memory: a set-up
whose n-th allocation fails is refused (the stored inverses are the fallback), never
verified on what is missing, and the next one over the same half system, as a second
ensemble member of the degree makes it, is whole."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def harness(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("hm") / "hm"
    subprocess.run([cxx, "-O2", "-std=c++17", os.path.join(HERE, "native", "helmholtz_memory_harness.cpp"), "-o", str(out)],
                   check=True, capture_output=True)
    return str(out)


@pytest.mark.parametrize("N,par", [(5, 1), (12, 0), (13, 1)])
def test_failed_allocations(harness, N, par):
    r = subprocess.run([harness, str(N), str(par)], capture_output=True, text=True)
    assert r.returncode == 0, (r.returncode, r.stdout[-300:], r.stderr)
    rows = [line.split() for line in r.stdout.splitlines()]
    assert len(rows) > 20
    for n, first, empty, second, diff in rows:
        assert (first, empty, second, float(diff)) == ("0", "0", "1", 0.0), n
