"""Ensemble steps whose members are in different phases on the GPU: a record
loaded into one member between steps (its h point values formed, the others'
pending), fields read between steps, a member stepped on its own: every member
bit-identical to a lone channel taken through the same calls."""
import numpy as np
import pytest

from channel_flow_amd import ic

from .helpers import STATE_KEYS

pytestmark = pytest.mark.gpu

MEMBERS = [dict(nnx=32, nny=32, nnz=32, precision="mixed"), dict(nnx=32, nny=16, nnz=48, precision="fp64"),
           dict(nnx=32, nny=32, nnz=24, precision="mixed"), dict(nnx=64, nny=64, nnz=64, precision="mixed")]


def test_mixed_phases(require_gpu):
    from channel_flow_amd.channel import Channel
    from channel_flow_amd.ensemble import Ensemble
    full = [dict(m, aphi=1.0, beta=0.5, dt=1.0e-3, re=3000.0, re_p=2.0 / 3000.0) for m in MEMBERS]
    start = [ic.seeded_ic(m["nnx"], m["nny"], m["nnz"], 1.0, 0.5, 1.0, 0.1, 6.0, -4.0 / 3.0, 60 + i)
             for i, m in enumerate(full)]
    record = {}

    def script(chans, step_all):
        for c, s in zip(chans, start):
            c.initial(*s)
        step_all(2)
        for i in (0, 1):
            record.setdefault(i, chans[i].get_state())
        step_all(1)
        for i in (0, 1):
            chans[i].set_state(record[i])
        read = [chans[2].fields(), chans[3].plane_statistics()]
        step_all(2)
        chans[3].step(1)
        step_all(3)
        return [c.get_state() for c in chans], [c.fields() for c in chans], read

    with Ensemble(full) as ens:
        got = script([ens.member(i) for i in range(len(full))], ens.step)
    lone = [Channel(**m) for m in full]
    ref = script(lone, lambda n: [c.step(n) for c in lone])
    for c in lone:
        c.close()
    for i in range(len(full)):
        for k in STATE_KEYS:
            np.testing.assert_array_equal(got[0][i][k], ref[0][i][k], err_msg=f"{i} {k}")
        for k in got[1][i]:
            np.testing.assert_array_equal(got[1][i][k], ref[1][i][k], err_msg=f"{i} {k}")
    for k in got[2][0]:
        np.testing.assert_array_equal(got[2][0][k], ref[2][0][k])
    np.testing.assert_array_equal(got[2][1], ref[2][1])
