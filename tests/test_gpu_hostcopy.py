"""State exchange through the staged host copies on the GPU: records whose
arrays lie below, at and past a chunk, with remainders, from one and from two
threads at once: what is loaded is what is read back, bit for bit."""
import threading

import numpy as np
import pytest

from channel_flow_amd import runtime as rt

pytestmark = pytest.mark.gpu

# field bytes: 2.13 MB (one chunk and a rest), 2.1 MB * 4, 1.07 MB (plain copies), 17 MB + rest
SIZES = [(64, 64, 64), (128, 128, 64), (64, 32, 64), (128, 128, 128), (96, 96, 100)]


def make(nnx, nny, nnz):
    from channel_flow_amd.channel import Channel
    return Channel(nnx, nny, nnz, 1.0, 0.5, 1.0e-4, 3000.0, 2.0 / 3000.0)


def record(ch, seed):
    rng = np.random.default_rng(seed)
    out = {}
    for k in rt.STATE_FIELDS:
        shape = (ch.Ny,) if k in rt.MEAN_FIELDS else ch.field_shape
        out[k] = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    return out


def roundtrip(ch, seed, errors):
    st = record(ch, seed)
    for _ in range(3):
        ch.set_state(st)
        got = ch.get_state()
        errors += [k for k in st if not np.array_equal(got[k], st[k])]


@pytest.mark.parametrize("size", SIZES)
def test_roundtrip(require_gpu, size):
    errors = []
    with make(*size) as ch:
        roundtrip(ch, 5, errors)
    assert not errors


def test_two_threads(require_gpu):
    errors = [[], []]
    with make(128, 128, 64) as a, make(128, 128, 128) as b:
        threads = [threading.Thread(target=roundtrip, args=(c, s, errors[s])) for s, c in enumerate((a, b))]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
    assert errors == [[], []]
