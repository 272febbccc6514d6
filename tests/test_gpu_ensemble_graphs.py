"""Graphs of an ensemble on the GPU: reading members between steps captures none,
loading the same ones again captures none, members stepped by themselves leave
their number bounded, and every member stays bit-identical to a lone channel
taken through the same calls."""
import numpy as np
import pytest

from channel_flow_amd import ic

from .helpers import STATE_KEYS

pytestmark = pytest.mark.gpu


def members(sizes):
    return [dict(nnx=nx, nny=nz, nnz=n, precision=form, aphi=1.0, beta=0.5, dt=1.0e-3, re=3000.0, re_p=2.0 / 3000.0)
            for nx, nz, n, form in sizes]


def starts(full):
    return [ic.seeded_ic(m["nnx"], m["nny"], m["nnz"], 1.0, 0.5, 1.0, 0.1, 6.0, -4.0 / 3.0, 80 + i)
            for i, m in enumerate(full)]


def test_reading_and_repeated_loading_capture_nothing(require_gpu):
    from channel_flow_amd.channel import Channel
    from channel_flow_amd.ensemble import Ensemble
    full = members([(32, 32, 32, "mixed"), (16, 16, 48, "fp64"), (32, 32, 24, "mixed"), (32, 16, 64, "fp64")])
    fields = starts(full)

    def script(chans, step_all, after=lambda: None):
        for c, f in zip(chans, fields):
            c.initial(*f)
        step_all(2)
        records = [c.get_state() for c in chans]
        for read in ((0,), (1, 3), (2,), (0, 1, 2, 3), (3,)):
            for i in read:
                chans[i].get_state()
            step_all(1)
            after()
        for load in ((1,), (0, 2), (1,), (0, 2)):
            for i in load:
                chans[i].set_state(records[i])
            step_all(2)
            after()
        return [c.get_state() for c in chans]

    counts = []
    with Ensemble(full) as ens:
        got = script([ens.member(i) for i in range(4)], ens.step, lambda: counts.append(ens.graph_count()))
    assert counts[:5] == [2] * 5, counts
    assert counts[5:] == [3, 4, 4, 4], counts  # one per set of members loaded
    lone = [Channel(**m) for m in full]
    ref = script(lone, lambda n: [c.step(n) for c in lone])
    for c in lone:
        c.close()
    for i in range(4):
        for k in STATE_KEYS:
            np.testing.assert_array_equal(got[i][k], ref[i][k], err_msg=f"{i} {k}")


def test_graphs_are_bounded(require_gpu):
    """Each member stepped by itself flips its history phase: 2^6 combinations."""
    from channel_flow_amd.channel import Channel
    from channel_flow_amd.ensemble import Ensemble
    full = members([(16, 16, 32, "fp64")] * 6)
    fields = starts(full)
    order = [(j ^ (j >> 1) ^ ((j - 1) ^ ((j - 1) >> 1))).bit_length() - 1 for j in range(1, 65)]  # a Gray code's flips
    with Ensemble(full) as ens, Channel(**full[0]) as lone:
        for i, f in enumerate(fields):
            ens.member(i).initial(*f)
        lone.initial(*fields[0])
        for i in order:
            ens.member(min(i, 5)).step(1)
            ens.step(1)
            lone.step(2 if i == 0 else 1)
            assert ens.graph_count() <= 32
        got, ref = ens.member(0).get_state(), lone.get_state()
    for k in STATE_KEYS:
        np.testing.assert_array_equal(got[k], ref[k], err_msg=k)
