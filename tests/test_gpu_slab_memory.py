"""Which grids run in slabs of planes on the GPU, by the padded planes a context
holds: a large one's two slabs, so that turning the timing on (all planes at once)
adds the others; all planes from the start in a smaller one and in an ensemble."""
import pytest

pytestmark = pytest.mark.gpu

RE = dict(aphi=1.0, beta=0.5, re=3000.0, re_p=2.0 / 3000.0, dt=1.0e-4)


def planes_added(ch, nnx, nny, form):
    """Bytes of one wall-normal plane of the six padded fields; those that timing adds."""
    before = ch.device_bytes()
    ch.set_timing(True)
    added = ch.device_bytes() - before
    ch.set_timing(True)
    assert ch.device_bytes() == before + added
    return 6 * (16 if form == "fp64" else 8) * (3 * nny // 2) * (nnx // 2), added


# the grids on which the slabs are compared with the launches over all planes
@pytest.mark.parametrize("form,nnx,nny,nnz", [
    ("fp64", 256, 256, 128), ("mixed", 256, 512, 128), ("fp64", 512, 128, 131), ("mixed", 512, 512, 64),
    ("fp64", 128, 648, 101)])
def test_large_grids_hold_two_slabs(require_gpu, form, nnx, nny, nnz):
    from channel_flow_amd.channel import Channel
    with Channel(nnx=nnx, nny=nny, nnz=nnz, precision=form, **RE) as ch:
        plane, added = planes_added(ch, nnx, nny, form)
    held = plane * (2 * nnz + 1) - added
    assert added > 0 and added % plane == 0
    assert 0 < held <= 2 * (160 << 20)
    assert held // plane % 2 == 0  # two slabs of as many planes


@pytest.mark.parametrize("form,nnx,nny,nnz", [("fp64", 128, 128, 128), ("mixed", 256, 256, 128)])
def test_smaller_grids_hold_all_planes(require_gpu, form, nnx, nny, nnz):
    from channel_flow_amd.channel import Channel
    with Channel(nnx=nnx, nny=nny, nnz=nnz, precision=form, **RE) as ch:
        assert planes_added(ch, nnx, nny, form)[1] == 0


def test_ensemble_members_hold_all_planes(require_gpu):
    from channel_flow_amd.ensemble import Ensemble
    m = dict(nnx=256, nny=256, nnz=128, precision="fp64", **RE)
    with Ensemble([m]) as ens:
        assert planes_added(ens.member(0), 256, 256, "fp64")[1] == 0
