"""Plane statistics of a state that is not finite on the GPU: a plane mean is NaN
exactly where the mean of the plane's physical values is, whichever mode holds
the NaN or the infinity."""
import numpy as np
import pytest

from channel_flow_amd import ic

pytestmark = pytest.mark.gpu


# nnx / 2 = 16, 64: sums from the lines in registers (one and several blocks a plane);
# 162: no register split, sums over the stored physical fields
@pytest.mark.parametrize("nnx,nny,nnz", [(32, 16, 32), (128, 96, 24), (324, 8, 16)])
@pytest.mark.parametrize("field,value", [("vnp1", np.nan), ("omegaynp1", np.nan), ("omegaynp1", np.inf), ("au0", np.nan)])
def test_plane_means_show_it(require_gpu, nnx, nny, nnz, field, value):
    from channel_flow_amd import runtime
    from channel_flow_amd.channel import Channel
    with Channel(nnx, nny, nnz, 1.0, 0.5, 1.0e-3, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(*ic.seeded_ic(nnx, nny, nnz, 1.0, 0.5, 1.0, 0.1, 6.0, -4.0 / 3.0, 5))
        state = ch.get_state()
        state[field][(2, 3, 5) if state[field].ndim == 3 else 2] = value
        with pytest.raises(runtime.ChfNonFinite):
            ch.set_state(state)
        stats = ch.plane_statistics()
        with np.errstate(invalid="ignore"):
            for q in range(3):
                mean = ch.physical(q).mean(axis=(1, 2))
                np.testing.assert_array_equal(np.isnan(stats[q]), np.isnan(mean), err_msg=f"field {q}")
        assert np.isnan(stats[0]).any()
