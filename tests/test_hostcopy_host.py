"""Copies between device and host arrays (csrc/hostcopy.hip, compiled with g++ over
host stand-ins for the HIP calls): without memory, whichever allocation fails, the
start of a helper thread among them, the copy is whole, nothing is thrown, and the
pool's lanes serve the next copy; copies of one or two lanes make no streams; and a
context of another device than the caller's current one copies as well."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


def test_copies(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    exe = str(tmp_path / "hostcopy")
    native = os.path.join(HERE, "native")
    subprocess.run([cxx, "-O1", "-std=c++17", "-pthread", "-x", "c++", "-I" + os.path.join(native, "hipstub"),
                    os.path.join(native, "hostcopy_harness.cpp"), "-o", exe], check=True, capture_output=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, (r.returncode, r.stdout[-500:], r.stderr[-500:])
    head, loads, *lines = r.stdout.splitlines()
    # 5 MB: one lane; 12 MB: two, on the context's own streams; 100 MB: all six
    assert head == "streams 0 0 4", head
    # loads of 3 MB with two contexts alive, 14 MB with one and with two, 50 MB with one
    assert loads == "lanes 0 0 2 6", loads
    rows = [tuple(map(int, line.split())) for line in lines]
    assert {d for d, _, _ in rows} == {0, 1} and max(n for _, n, _ in rows) >= 5, rows
    assert all(lanes == 6 for _, _, lanes in rows), rows
