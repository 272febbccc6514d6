"""Grids large enough for the padded transforms to run in slabs of wall-normal
planes: every plane's values are the ones that the launches over all planes (with
timing on) give, bit for bit, and the two forms may follow one another."""
import numpy as np
import pytest

from channel_flow_amd import ic
from channel_flow_amd.channel import Channel

pytestmark = pytest.mark.gpu


# a last slab shorter than the others, an odd degree, and a span length without
# a register FFT (3 nny / 2 = 972); the six padded fields take more than 1 GiB
@pytest.mark.parametrize("form,nnx,nny,nnz", [
    ("fp64", 256, 256, 128), ("mixed", 256, 512, 128), ("fp64", 512, 128, 131), ("mixed", 512, 512, 64),
    ("fp64", 128, 648, 101)])
def test_slabs_are_the_whole_launches(form, nnx, nny, nnz):
    cfg = dict(nnx=nnx, nny=nny, nnz=nnz, aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4,
               precision=form)
    fields = ic.seeded_ic(nnx, nny, nnz, 1.0, 0.5, 1.0, 5e-2, 4.0, 0.0, 7)
    with Channel(**cfg) as slabs, Channel(**cfg) as whole:
        whole.set_timing(True)
        for ch in (slabs, whole):
            ch.initial(*fields)
            ch.step(2)
        whole.set_timing(False)
        slabs.set_timing(True)
        for ch in (slabs, whole):
            ch.step(1)
        a, b = slabs.get_state(), whole.get_state()
    assert np.abs(a["rhsvn"]).max() > 0
    for k in a:
        assert np.array_equal(a[k], b[k]), k
