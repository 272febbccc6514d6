"""Copies between device and host arrays (csrc/hostcopy.hip, compiled with g++ over
host stand-ins for the HIP calls) without memory: whichever allocation fails, the
start of a helper thread among them, the copy is whole, nothing is thrown, and the
pool's lanes serve the next copy."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_failed_allocations(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "hostcopy")
    native = os.path.join(HERE, "native")
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-x", "c++", "-I" + os.path.join(native, "hipstub"),
                    os.path.join(native, "hostcopy_harness.cpp"), "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-500:])
    rows = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert {d for d, _, _ in rows} == {0, 1} and max(n for _, n, _ in rows) >= 5, rows
    assert all(lanes == 6 for _, _, lanes in rows), rows
