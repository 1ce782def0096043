"""Batches whose tiles are put in address order: shapes for which the order
is only estimated (several dimensions, reversed rows, one long row), buffers
far apart, and tile counts around the split over XCDs.  Every packed byte and
every byte of the unpacked buffers against the oracle."""
import numpy as np
import pytest

import tempi_amd as ta
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

SPAN = 4 << 20
SB = ta.StridedBlock.make
SHAPES = {
    # one tile each, too few for the split
    "tiny": [SB(16 * i, 64, [8, 3], [1, 16]) for i in range(9)],
    # rows in reverse, planes forward, and planes in reverse
    "reversed": [SB(3 << 20, 64, [24, 900], [1, -1072]), SB(1 << 20, 64, [24, 30, 40], [1, 96, -4000]),
                 SB(0, 64, [12, 50, 60], [1, 20, 30000])] + [SB(64 * i, 64, [5, 7], [1, 9])
                                                            for i in range(8)],
    # one row of 3 MiB, cut into segments, among short ones
    "one long row": [SB(7, 64, [3 << 20], [1])] + [SB(300000 * i, 64, [4, 2000], [1, 100])
                                                   for i in range(12)],
    # the same bytes packed several times, and blocks between others' rows
    "shared": [SB(100, 64, [64, 20000], [1, 192])] * 3 + [
        SB(164 + 8 * i, 64, [8, 20000], [1, 192]) for i in range(9)],
}


@pytest.mark.parametrize("name", sorted(SHAPES))
def test_batches_in_address_order(name):
    blocks = SHAPES[name]
    n = len(blocks)
    hosts = [orc.splitmix_bytes(SPAN, 60 + i) for i in range(2)]
    srcs = [ta.DeviceBuffer(SPAN) for _ in hosts]
    apart = ta.DeviceBuffer(512 << 20)  # keeps the buffers' addresses apart
    dsts = [ta.DeviceBuffer(SPAN) for _ in range(n)]
    for s, h in zip(srcs, hosts):
        s.upload(h)
    for d in dsts:
        d.fill(0xAB)
    packed = ta.DeviceBuffer(sum(sb.size() for sb in blocks) + n)
    packed.fill(0x5A)
    packs, unpacks, at = [], [], []
    off = 0
    for i, sb in enumerate(blocks):
        at.append(off)
        packs.append((sb, srcs[i % 2].addr(), packed.addr(off), 1, ta.DIR_PACK))
        unpacks.append((sb, dsts[i].addr(), packed.addr(off), 1, ta.DIR_UNPACK))
        off += sb.size() + 1  # a byte between the packed ranges
    ta.Batch(packs).launch()
    ta.synchronize()
    got = packed.download()
    ta.Batch(unpacks).launch()
    ta.synchronize()
    for i, sb in enumerate(blocks):
        desc = orc.sb_desc(*sb.as_tuple())
        want = orc.sb_pack(desc, hosts[i % 2], 0, 1)
        assert (got[at[i]:at[i] + sb.size()] == want).all(), (name, i)
        assert got[at[i] + sb.size()] == 0x5A, (name, i)
        ref = np.full(SPAN, 0xAB, np.uint8)
        orc.sb_unpack(desc, want, ref, 0, 1)
        assert (dsts[i].download() == ref).all(), (name, i)
    apart.free()
