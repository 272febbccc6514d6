"""The unpadded physical transform and the plane statistics on the GPU over the
lengths that have a register form of their own (streamwise, spanwise), column
and line counts that fill the kernels' tiles partly, and lengths without one,
against the oracle.  Both are FP64 sums of at most 600 terms of order one: 1e-12
of the field's largest value, and of the variance's."""
import numpy as np
import pytest

from oracle import cf_oracle as O

from .helpers import ic_of, params_of

pytestmark = pytest.mark.gpu

SIZES = [(16, 8, 8), (24, 12, 9), (32, 16, 32), (36, 24, 5), (48, 36, 12), (64, 32, 7), (72, 48, 6), (96, 64, 8),
         (108, 72, 6), (128, 96, 16), (144, 108, 5), (192, 128, 8), (216, 144, 6), (256, 192, 5), (288, 16, 4),
         (384, 24, 4), (512, 32, 4), (16, 216, 6), (16, 256, 6), (16, 288, 5), (16, 384, 5), (16, 512, 4), (4, 4, 6),
         (12, 324, 4), (324, 8, 4), (8, 8, 64)]


@pytest.mark.parametrize("nnx,nny,nnz", SIZES)
def test_physical_and_statistics(require_gpu, nnx, nny, nnz):
    from channel_flow_amd.channel import Channel
    cfg = dict(nnx=nnx, nny=nny, nnz=nnz, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4, u_c=1.0,
               rms=0.1, kmax=float(max(nnx, nny)), slope=-1.0, seed=77)
    p = params_of(cfg)
    v, oy, au0, w0 = ic_of(cfg)
    st = O.zero_state(p)
    st.update(vnp1=v, omegaynp1=oy, au0=au0, w0=w0)
    O.kinematics_all(st, p)
    ref = [O.physical_field(st[k], p) for k in ("unp1", "vnp1", "wnp1")]
    stats = O.plane_statistics(*ref)
    with Channel(nnx, nny, nnz, 1.0, 0.5, 1.0e-4, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(v, oy, au0, w0)
        got = [ch.physical(f) for f in ("u", "v", "w")]
        gs = ch.plane_statistics()
        again = ch.plane_statistics()
    for g, r in zip(got, ref):
        assert np.abs(g - r).max() <= 1e-12 * np.abs(ref[0]).max()
    np.testing.assert_array_equal(gs, again)
    for i in range(12):
        scale = np.abs(ref[0]).max() if i < 3 or i > 8 else np.abs(stats[3:6]).max()
        assert np.abs(gs[i] - stats[i]).max() <= 1e-12 * scale, i
