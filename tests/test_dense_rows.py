"""The choice for copies whose short rows share lines with each other: the
12-B words' kernel, or for 16-B rows the 8-B words', and never several lanes to
a row; rows further apart, or few of them, keep the others.  Each pick stores
exactly the copy's bytes (checked on fewer rows of the same layout)."""
import pytest

import tempi_amd as ta

MIB = 1 << 20


def pick(length, stride, rows, direction, planes=1):
    counts, strides = [length, rows], [1, stride]
    if planes > 1:
        counts, strides = counts + [planes], strides + [rows * stride + 1000]
    sb = ta.StridedBlock.make(0, planes * (rows * stride + 1000), counts, strides)
    v = ta.select_variant(sb, 1, 1 << 40, 1 << 41, direction, ta.SELECT_HEURISTIC)
    small = ta.StridedBlock.make(0, 40 * stride, [length, 17, 2], [1, stride, 20 * stride])
    for offset in (0, 5):
        e = ta.copy_emulate(small, 2, (1 << 40) + offset, (1 << 41) + 3, direction, v)
        assert e["exact"] == 1, (length, stride, v, e)
    return v


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
def test_rows_that_share_lines(direction):
    for length in (1, 2, 3, 4, 5, 6, 7, 8, 12):
        for gap in (1, 4, 8):
            stride = length + gap
            rows = 80 * MIB // stride
            want = 16 if length in (1, 2, 4, 8, 12) or stride < 16 else None
            v = pick(length, stride, rows, direction)
            assert v == want or want is None and v in (9, 11, 12, 8), (length, stride, v)
            assert pick(length, stride, rows // 8, direction, planes=8) == v
    for stride in (17, 20, 31):
        assert pick(16, stride, 80 * MIB // stride, direction) == 18
    # below 64 MiB of lines: rows under 8 B, from 4 Mi rows on
    for length in range(1, 8):
        for rows in (4 * MIB, 5 * MIB):
            assert pick(length, length + 4, rows, direction) == (12 if rows * (length + 4) <
                                                                 64 * MIB else 16)
        assert pick(length, length + 4, 4 * MIB - 1, direction) in (9, 11)
        assert pick(length, 40, 1 * MIB, direction) in (9, 11)


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
def test_other_short_rows(direction):
    for length in (1, 2, 4, 8):
        for stride in (32, 64, 127, 1000):
            assert pick(length, stride, 80 * MIB // min(length + 127, stride) + 1, direction) == 18
        # few rows to a run share lines with nobody
        assert pick(length, length + 2, 8, direction, planes=4 * MIB) != 16
    for length, streamed in ((12, 16), (24, 17)):
        for stride in (64, 95, 128, 500):
            assert pick(length, stride, 300 * MIB // min(length + 127, stride), direction) == streamed
        for stride in (96, 127):
            v = pick(length, stride, 300 * MIB // stride, direction)
            assert not ta.variant_info(v)["nontemporal_loads"], (length, stride, v)
            assert pick(length, stride, 200 * MIB // stride, direction) == streamed
