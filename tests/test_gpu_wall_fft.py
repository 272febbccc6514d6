"""The wall-normal FFTs of every degree whose split has a factor 5, 9 or an odd
row count, on the GPU: initial() and three steps in FP64 against the oracle at
the trajectory bar, the same of the mixed form against the FP64 form at the bars
of the mixed form at N = 192, and the unpadded v (the point values) of the cold
start against the oracle's."""
import numpy as np
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [40, 50, 60, 72, 80, 90, 100, 120, 144, 150, 160, 180, 200, 216, 240])
def test_degree(require_gpu, nnz):
    from channel_flow_amd.channel import Channel
    cfg = dict(nnx=32, nny=8, nnz=nnz, aphi=1.0, beta=0.5, re=7940.0, re_p=2.0 / 7940.0, dt=2.5e-4, u_c=1.0, rms=0.1,
               kmax=6.0, slope=-4.0 / 3.0, seed=23)
    p = params_of(cfg)
    arrays = ic_of(cfg)
    st = O.initial_presolve_state(*arrays, p)
    O.Stepper(p).step(st, 3)
    args = (32, 8, nnz, 1.0, 0.5, 2.5e-4, 7940.0, 2.0 / 7940.0)
    with Channel(*args) as ch, Channel(*args, precision="mixed") as mx:
        ch.initial(*arrays)
        got_v = ch.physical("v")
        ch.step(3)
        for k, e in state_errors(ch.get_state(), st).items():
            assert e < 1e-9, (k, e)
        mx.initial(*arrays)
        mx.step(3)
        a, b = mx.get_state(), ch.get_state()
        e = state_errors(a, b)
        for k in ("vnp1", "omegaynp1"):
            assert e[k] < 1e-5, ("mixed", k, e[k])
        for k in ("au0", "w0"):
            assert e[k] < 1e-9, ("mixed", k, e[k])
    ref = O.physical_field(arrays[0], p)
    assert np.max(np.abs(got_v - ref)) < 1e-11 * np.max(np.abs(ref))
