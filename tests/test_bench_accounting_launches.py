"""bench.py's algorithmic HBM bytes per launch (kernel_work, with the FFT transforms and
the shared diagonalisation) against the HBM traffic that the FETCH_SIZE and
WRITE_SIZE counters measured for the same launches at 256x193x256
(bench.py --launch-probe: every launch alone and over all planes; the committed
summaries under profiles/, scaled by a device copy of known size).  A class outside
[0.97, 1.15] would mean a field counted at the wrong precision, or counted twice or
not at all.  The two right-hand sides share a kernel, and so do the two solves: an
average over their dispatches is that of the pair."""
import json
import os

import pytest

import bench
from channel_flow_amd import ic

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CONFIG = "retau395_256x193x256"

# kernel symbol -> the classes its dispatches are, in equal numbers
LAUNCHES = {
    "mixed": {"void k_xpass_st<": ("xpass",), "void k_hassemble<true>": ("hassemble",),
              "void k_kinematics<true>": ("kinematics",), "void k_yrhs<16, 24, ": ("rhs_v", "rhs_o"),
              "void k_hsolve<": ("solve", "wsolve"), "void k_zfft_pair<16, 24, 8, true>": ("zfft_inv",),
              "void k_zfft_pair<16, 24, 8, false>": ("zfft_fwd",),
              "void k_ycheb<16, 24, float2, float2, float2, true": ("analysis",)},
    "fp64": {"void k_xpass_st<": ("xpass",), "void k_hassemble<false>": ("hassemble",),
             "void k_kinematics<false>": ("kinematics",), "void k_yrhs<16, 24, ": ("rhs_v", "rhs_o"),
             "void k_hsolve<": ("solve", "wsolve"), "void k_zfft_reg<16, 24, 8, true": ("zfft_inv",),
             "void k_zfft_reg<16, 24, 8, false": ("zfft_fwd",),
             "void k_ycheb<16, 24, double2, double2, double2, true": ("analysis",),
             "void k_ycheb<16, 24, double2, double2, double2, false": ("synth_padded",)},
}


def measured(form):
    with open(os.path.join(ROOT, "profiles", f"hbm_launches_{CONFIG}_{form}.json")) as f:
        return json.load(f)["kernels"]


def traffic(data, prefix):
    hits = [v for k, v in data.items() if k.startswith(prefix)]
    assert len(hits) == 1, (prefix, list(data))
    return hits[0]["fetch_bytes"] + hits[0]["write_bytes"], hits[0]["dispatches"]


@pytest.mark.parametrize("form", ["mixed", "fp64"])
def test_algorithmic_bytes_match_measured_traffic(form):
    work = bench.kernel_work(bench.dims(dict(ic.CONFIGS[CONFIG])), form, yfft=True, diag=True)
    data = measured(form)
    for prefix, classes in LAUNCHES[form].items():
        got, dispatches = traffic(data, prefix)
        assert dispatches % len(classes) == 0, prefix
        ratio = got / (sum(work[c][0] for c in classes) / len(classes))
        assert 0.97 <= ratio <= 1.15, (form, classes, round(ratio, 4))


def test_mixed_synthesis_reads_its_fp32_fields():
    """u, w, omega_x, omega_z come from their FP32 copies: four of the six fields of
    a step, in a launch of their own."""
    d = bench.dims(dict(ic.CONFIGS[CONFIG]))
    got, _ = traffic(measured("mixed"), "void k_ycheb<16, 24, float2, float2, float2, false")
    S, Y = d["Ny"] * d["ncol"] * 8, d["Py"] * d["ncol"] * 8
    assert 0.97 <= got / (4 * (S + Y)) <= 1.15


@pytest.mark.parametrize("form", ["mixed", "fp64"])
def test_reported_traffic_is_of_these_launches(form):
    """The traffic beside bench.py's roofline is the streamwise pass's own, from the
    summary that names the present kernel."""
    got, _ = traffic(measured(form), "void k_xpass_st<")
    assert bench.measured_traffic(CONFIG, form, "xpass") == int(got)
    assert bench.measured_traffic(CONFIG, form, "solve") is None  # two classes, one kernel
