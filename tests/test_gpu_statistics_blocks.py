"""Blocks of the plane statistics on the GPU: as many a plane as fill the chip with
16 lines each, but none without lines (the partial results, 12 values per block and
plane, are part of the context's device memory), and the statistics of the physical
fields whichever number that is."""
import numpy as np
import pytest

from channel_flow_amd import ic

pytestmark = pytest.mark.gpu


# lines a block takes at a time: 64, 32, 16 and 10 by the split of nnx / 2 points; one
# block, some with a remainder of lines, and a plane whose blocks take several turns
@pytest.mark.parametrize("nnx,nny,nnz,lines", [(16, 512, 32, 64), (64, 64, 32, 32), (64, 8, 8, 32), (256, 24, 16, 16),
                                               (384, 64, 12, 10), (384, 96, 200, 10)])
def test_blocks_have_lines(require_gpu, nnx, nny, nnz, lines):
    from channel_flow_amd.channel import Channel
    with Channel(nnx, nny, nnz, 1.0, 0.5, 1.0e-3, 3000.0, 2.0 / 3000.0) as ch:
        ch.initial(*ic.seeded_ic(nnx, nny, nnz, 1.0, 0.5, 1.0, 0.1, 6.0, -4.0 / 3.0, 9))
        before = ch.device_bytes()
        stats = ch.plane_statistics()
        ny = nnz + 1
        partial = ch.device_bytes() - before - 3 * 16 * ny * nny * (nnx // 2) - 8 * 12 * ny
        u, v, w = (ch.physical(i) for i in range(3))
    blocks = min(1536 // ny, nny // 16, -(-nny // lines))
    assert partial == 8 * 12 * ny * max(1, blocks)
    mean = [f.mean(axis=(1, 2)) for f in (u, v, w)]
    du = [f - m[:, None, None] for f, m in zip((u, v, w), mean)]
    pairs = [(0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)]
    ref = mean + [(du[a] * du[b]).mean(axis=(1, 2)) for a, b in pairs] + [np.abs(f).max(axis=(1, 2)) for f in (u, v, w)]
    # sums of up to 512 x 96 values of O(1): 1e-13 is 500 roundings of the largest
    assert np.abs(stats - np.array(ref)).max() <= 1e-13
