"""Copies of 512 KiB and more to or from host memory take the variant for the
link, smaller ones that for copies bound by their launch."""
import pytest

import tempi_amd as ta

pytestmark = pytest.mark.gpu

KIB = 1 << 10


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
@pytest.mark.parametrize("length", [64, 128, 256, 1024, 4096])
def test_the_link_comes_first(length, direction):
    assert ta.device_count() > 0
    strided, packed = ta.DeviceBuffer(64 << 20), ta.DeviceBuffer(8 << 20, mapped=True)
    device = ta.DeviceBuffer(8 << 20)

    def pick(kib, buf):
        rows = kib * KIB // length
        sb = ta.StridedBlock.make(0, rows * (length + 100), [length, rows], [1, length + 100])
        return ta.select_variant(sb, 1, strided.addr(), buf.addr(), direction, ta.SELECT_DEFAULT)

    link = pick(8192, packed)
    for kib in (512, 640, 768, 1024, 1025, 4096):
        assert pick(kib, packed) == link, kib
    for kib in (16, 256, 508):
        assert pick(kib, packed) == pick(kib, device), kib
    if direction == ta.DIR_UNPACK:
        assert link != pick(512, device)
