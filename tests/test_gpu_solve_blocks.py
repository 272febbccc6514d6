"""Per-mode solves on the GPU at the ends of a row-block count (a half system of
the even degrees has N / 2 rows, 16 to a block), with a last column tile that is
part full (12 x 12 grids: 72 columns): initial() and two steps against the
oracle, at the trajectory bar of the parity tests."""
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of, state_errors

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nnz", [32, 33, 34, 64, 66, 96, 98, 128, 130, 160, 162, 192, 194, 224, 226, 255])
def test_row_block_ends(require_gpu, nnz):
    from channel_flow_amd.channel import Channel
    cfg = dict(nnx=12, nny=12, nnz=nnz, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-3, u_c=1.0, rms=0.1,
               kmax=6.0, slope=-4.0 / 3.0, seed=31)
    p = params_of(cfg)
    arrays = ic_of(cfg)
    st = O.initial_presolve_state(*arrays, p)
    O.Stepper(p).step(st, 2)
    with Channel(12, 12, nnz, 1.0, 0.5, 1.0e-3, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(*arrays)
        ch.step(2)
        got = ch.get_state()
    for k, e in state_errors(got, st).items():
        assert e < 1e-9, (k, e)
