"""Planes a multiple of 512 KB apart (ncol values of 16 or 8 bytes) are padded at
the padded wall-normal points when the transforms run as FFTs: two steps against
the cos-table form, whose planes are not padded, from the same state."""
import numpy as np
import pytest

from channel_flow_amd import ic
from channel_flow_amd.channel import Channel

pytestmark = pytest.mark.gpu


# the FP64 bound is the parity tests' per-trajectory bar, the mixed form's that of
# its v and omega_y (its h terms are k^2 times FP32 roundings, with no bar of their own)
@pytest.mark.parametrize("form,nnx,nny,nnz,bound,names", [
    ("fp64", 256, 256, 32, 1e-9, ("vnp1", "omegaynp1", "rhsvn", "rhsomegayn")),
    ("fp64", 128, 512, 40, 1e-9, ("vnp1", "omegaynp1", "rhsvn", "rhsomegayn")),
    ("mixed", 512, 256, 32, 1e-5, ("vnp1", "omegaynp1"))])
def test_padded_planes(require_gpu, monkeypatch, form, nnx, nny, nnz, bound, names):
    cfg = dict(nnx=nnx, nny=nny, nnz=nnz, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4, precision=form)
    fields = ic.seeded_ic(nnx, nny, nnz, 1.0, 0.5, 1.0, 5e-2, 4.0, 0.0, 7)
    out = []
    for transforms in ("", "matrix"):
        monkeypatch.setenv("CHF_Y_TRANSFORMS", transforms)
        with Channel(**cfg) as ch:
            ch.initial(*fields)
            ch.step(2)
            out.append(ch.get_state())
    for k in names:
        a, b = out[0][k], out[1][k]
        e = np.abs(a - b).max() / np.abs(b).max()
        assert e < bound, (k, e)
