"""Rows that end inside a word: each kernel variant at row lengths around the
edges of its words, of its lanes and of its segments, where the lane and the
segment that move a row's last bytes change."""
import numpy as np
import pytest

import tempi_amd as ta
from oracle import oracle as orc

ROWS, BASE_S, BASE_P = 5, 1 << 40, 1 << 41


def lengths(variant):
    """Row lengths one word, one row of lanes and one or two segments long,
    with every kind of tail the word allows."""
    v = ta.variant_info(variant)
    w, seg = v["word_bytes"], v["lanes_per_row"] * v["word_bytes"] * v["unroll"]
    tails = sorted({0, 1, w // 2, w - 1} & set(range(w)))
    edges = (0, w, v["lanes_per_row"] * w, seg - w, seg, 2 * seg)
    return sorted({e + t for e in edges for t in tails if e + t > 0})


def block(length):
    return ta.StridedBlock.make(2, 2 + ROWS * (length + 7), [length, ROWS], [1, length + 7])


@pytest.mark.parametrize("variant", range(19))
def test_tails_are_stored_once(variant):
    for length in lengths(variant):
        for direction in (ta.DIR_PACK, ta.DIR_UNPACK):
            e = ta.copy_emulate(block(length), 1, BASE_S + 3, BASE_P + 5, direction, variant)
            assert e["exact"] == 1 and e["bytes_read"] == e["bytes_written"] == ROWS * length, \
                (variant, length, direction, e)


@pytest.mark.gpu
@pytest.mark.parametrize("variant", range(19))
def test_tails_match_the_oracle(variant):
    sizes = lengths(variant)
    room = block(max(sizes)).extent + 64
    host = orc.splitmix_bytes(room, 300 + variant)
    src, dst = ta.DeviceBuffer(room), ta.DeviceBuffer(room)
    packed = ta.DeviceBuffer(ROWS * max(sizes) + 64)
    src.upload(host)
    for length in sizes:
        sb = block(length)
        desc, size = orc.sb_desc(*sb.as_tuple()), sb.size()
        packed.fill(0x5A)
        dst.fill(0xAB)
        ta.pack_sb(sb, src.addr(3), 1, packed.addr(), size + 5, 5, variant)
        ta.unpack_sb(sb, packed.addr(), size + 5, dst.addr(3), 1, 5, variant)
        ta.synchronize()
        want = orc.sb_pack(desc, host, 3, 1)
        got = packed.download()
        assert (got[5:5 + size] == want).all(), (variant, length)
        assert (got[:5] == 0x5A).all() and (got[5 + size:] == 0x5A).all(), (variant, length)
        ref = np.full(room, 0xAB, np.uint8)
        orc.sb_unpack(desc, want, ref, 3, 1)
        assert (dst.download() == ref).all(), (variant, length)
