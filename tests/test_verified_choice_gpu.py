"""The variant kept for a large copy is kept for what it was timed on: rows
that cut sectors at another address are timed for themselves, and a batch's
pack to host memory leaves no entry for copies on the device."""
import pytest

import tempi_amd as ta

pytestmark = pytest.mark.gpu

L, STRIDE, ROWS = 64, 192, (1 << 20) + 8  # 64 MiB packed, 191 MiB of lines
SB = ta.StridedBlock.make(0, ROWS * STRIDE, [L, ROWS], [1, STRIDE])


def pick(strided, packed, direction):
    return ta.select_variant(SB, 1, strided, packed, direction, ta.SELECT_DEFAULT)


def test_rows_that_cut_sectors_are_timed_for_themselves():
    grid, packed = ta.DeviceBuffer(ROWS * STRIDE + 64), ta.DeviceBuffer(ROWS * L)
    for offset in (0, 16, 32, 48, 0):
        ta.unpack_sb(SB, packed.addr(), ROWS * L, grid.addr(offset), 1)
        ta.synchronize()
        v = pick(grid.addr(offset), packed.addr(), ta.DIR_UNPACK)
        # the strided stores go nontemporal where rows are whole sectors only
        assert ta.variant_info(v)["nontemporal_stores"] == (offset == 0), (offset, v)


def test_a_batch_to_host_memory_is_not_timed_on_the_device():
    grid = ta.DeviceBuffer(ROWS * STRIDE)
    mapped, packed = ta.DeviceBuffer(ROWS * L, mapped=True), ta.DeviceBuffer(ROWS * L)
    timed = ta.counters()["verified_choices"]
    b = ta.Batch([(SB, grid.addr(), mapped.addr(), 1, ta.DIR_PACK)])
    assert ta.counters()["verified_choices"] == timed
    b.destroy()
    ta.pack_sb(SB, grid.addr(), 1, packed.addr(), ROWS * L)
    ta.synchronize()
    assert ta.counters()["verified_choices"] == timed + 1
