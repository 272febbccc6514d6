"""Padded Fourier lengths of the FP64 form on the GPU: every length that has a
register FFT of its own, streamwise and spanwise, on column counts that fill
the kernels' tiles partly; initial() and two steps against the oracle.  The
tolerance is the trajectory bar of the parity tests (two steps of operations
that agree to 1e-13, through solves that amplify to at most 1e-10)."""
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of, state_errors

pytestmark = pytest.mark.gpu

# n with 3n/2 = 18, 36, 54, 72, 108, 162, 216, 288, 324, 432, 576, 768
LENGTHS = [12, 24, 36, 48, 72, 108, 144, 192, 216, 288, 384, 512]


@pytest.mark.parametrize("direction", ["stream", "span"])
@pytest.mark.parametrize("n", LENGTHS)
def test_padded_length_matches_oracle(require_gpu, n, direction):
    from channel_flow_amd.channel import Channel
    nnx, nny = (n, 8) if direction == "stream" else (12, n)
    cfg = dict(nnx=nnx, nny=nny, nnz=10, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4, u_c=1.0,
               rms=0.1, kmax=float(n), slope=-4.0 / 3.0, seed=31)
    p = params_of(cfg)
    arrays = ic_of(cfg)
    st = O.initial_presolve_state(*arrays, p)
    O.Stepper(p).step(st, 2)
    with Channel(nnx, nny, 10, 1.0, 0.5, 1.0e-4, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(*arrays)
        ch.step(2)
        got = ch.get_state()
    for k, e in state_errors(got, st).items():
        assert e < 1e-9, (k, e)
