"""The span pass that exchanges its lines in two halves (576 and 768 padded points)
on the GPU, on column counts that leave its tiles partial, full and
both: initial() and two steps in FP64 against the oracle at the trajectory bar,
and the mixed form against the FP64 form at the bars of the mixed form."""
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnx,nny,mixed", [(4, 384, False), (16, 384, False), (4, 512, False), (16, 512, False),
                                           (24, 512, False), (32, 512, True), (96, 512, True)])
def test_columns(require_gpu, nnx, nny, mixed):
    from channel_flow_amd.channel import Channel
    cfg = dict(nnx=nnx, nny=nny, nnz=10, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4, u_c=1.0,
               rms=0.1, kmax=float(nny), slope=-4.0 / 3.0, seed=31)
    p = params_of(cfg)
    arrays = ic_of(cfg)
    st = O.initial_presolve_state(*arrays, p)
    O.Stepper(p).step(st, 2)
    args = (nnx, nny, 10, 1.0, 0.5, 1.0e-4, 3000.0, 2.0 / 3000.0)
    with Channel(*args) as ch:
        ch.initial(*arrays)
        ch.step(2)
        got = ch.get_state()
    for k, e in state_errors(got, st).items():
        assert e < 1e-9, (k, e)
    if not mixed:
        return
    with Channel(*args, precision="mixed") as mx:
        mx.initial(*arrays)
        mx.step(2)
        e = state_errors(mx.get_state(), got)
    for k in ("vnp1", "omegaynp1"):
        assert e[k] < 1e-5, (k, e[k])
    for k in ("au0", "w0"):
        assert e[k] < 1e-9, (k, e[k])
