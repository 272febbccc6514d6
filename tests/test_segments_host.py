"""The rule for the passes along the degree (csrc/segments.h, compiled with g++): the
form whose steps were the faster ones, summed over the degrees timed, is taken."""
import ctypes
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

# (columns, mixed form with FFTs): (step us with the pass in segments, serial) per degree timed
KINEMATICS = {
    (18432, 0): [(320.4, 323.0), (517.1, 521.0)],
    (20736, 0): [(353.0, 348.3), (651.8, 655.1), (963.8, 970.8), (498.7, 498.3)],
    (23328, 0): [(1433.5, 1442.6)],
    (16384, 1): [(178.5, 178.5), (589.8, 594.5), (929.1, 938.7)],
    (24576, 1): [(266.1, 260.1), (941.3, 939.7), (1509.9, 1518.9), (2096.3, 2061.3)],
    (32768, 0): [(214.0, 154.0)],  # the launch alone
}
HASSEMBLE = {
    (18432, 0): [(195.8, 196.4), (320.0, 320.4), (515.2, 517.1)],
    (20736, 0): [(354.8, 353.0), (653.4, 651.8), (967.4, 963.8), (1621.1, 1616.9)],
    (23328, 0): [(1440.7, 1433.5)],
    (24576, 0): [(418.3, 415.5), (1143.6, 1137.0), (1437.0, 1431.2), (1924.5, 1917.4), (3010.5, 2989.7)],
    (16384, 1): [(12.1, 16.8), (37.4, 49.3), (62.1, 87.3)],  # the launch alone
    (24576, 1): [(16.3, 18.1), (29.0, 31.4), (50.8, 52.6), (91.1, 97.0)],
}


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no g++")
    out = tmp_path_factory.mktemp("seg") / "libseg.so"
    subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", os.path.join(HERE, "native", "segments_harness.cpp"),
                    "-o", str(out)], check=True, capture_output=True)
    l = ctypes.CDLL(str(out))
    for f in (l.kinematics_c, l.hassemble_c):
        f.argtypes = [ctypes.c_long, ctypes.c_int]
    return l


@pytest.mark.parametrize("name,timed", [("kinematics_c", KINEMATICS), ("hassemble_c", HASSEMBLE)])
def test_the_faster_form_is_taken(lib, name, timed):
    for (ncol, f32), rows in timed.items():
        segments, serial = map(sum, zip(*rows))
        assert bool(getattr(lib, name)(ncol, f32)) == (segments < serial), (ncol, f32)
