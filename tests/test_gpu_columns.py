"""Kinematics and h assembly in segments on the GPU: degrees at and past the
ends of a segment count (56, 112, 168, 224 coefficients fill 28 segments of 2,
4, 6, 8): initial() and three steps against the oracle, at the trajectory bar
and on the inputs of the parity tests at other degrees."""
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [4, 5, 55, 56, 111, 112, 167, 168, 223, 224, 256])
def test_segment_ends(require_gpu, nnz):
    from channel_flow_amd.channel import Channel
    cfg = dict(nnx=16, nny=8, nnz=nnz, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-3, u_c=1.0, rms=0.1,
               kmax=6.0, slope=-4.0 / 3.0, seed=23)
    p = params_of(cfg)
    arrays = ic_of(cfg)
    st = O.initial_presolve_state(*arrays, p)
    O.Stepper(p).step(st, 3)
    with Channel(16, 8, nnz, 1.0, 0.5, 1.0e-3, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(*arrays)
        ch.step(3)
        got = ch.get_state()
    for k, e in state_errors(got, st).items():
        assert e < 1e-9, (k, e)
