"""Copies of more workgroups than one grid holds (65 536) loop over their
units; a synchronous one returns on the signal kernel behind it, with every
byte there for a copy on the null stream."""
import ctypes

import numpy as np
import pytest

import tempi_amd as ta
import typecatalog as tc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

ROWS, STRIDE = (65536 + 100) * 256 + 3, 9


def fetch(buf, n):
    hip = ctypes.CDLL("libamdhip64.so")
    out = np.empty(n, np.uint8)
    assert hip.hipMemcpy(ctypes.c_void_p(out.ctypes.data), ctypes.c_void_p(buf.addr()),
                         ctypes.c_size_t(n), 2) == 0
    return out


@pytest.mark.parametrize("length,variant", [(4, 9), (3, 11), (5, 8), (8, 7), (4, 12)])
def test_a_grid_that_loops(length, variant):
    rows = ROWS * 4 if variant == 12 else ROWS  # four rows to a lane
    stride = length + 1
    sb = ta.StridedBlock.make(0, rows * stride, [length, rows], [1, stride])
    host = orc.splitmix_bytes(rows * stride, 5)
    want = host.reshape(rows, stride)[:, :length].reshape(-1)
    src, packed = ta.DeviceBuffer(rows * stride), ta.DeviceBuffer(rows * length)
    src.upload(host)
    packed.fill(0xAB)
    ta.pack_sb(sb, src.addr(), 1, packed.addr(), rows * length, 0, variant)
    ta.synchronize()
    assert (packed.download() == want).all()
    src.fill(0xAB)
    ta.unpack_sb(sb, packed.addr(), rows * length, src.addr(), 1, 0, variant)
    ta.synchronize()
    got = src.download().reshape(rows, stride)
    assert (got[:, :length].reshape(-1) == want).all() and (got[:, length:] == 0xAB).all()


def test_the_signal_kernel_behind_a_large_grid(mpi):
    h = mpi.type_from_spec(("vector", ROWS, 4, STRIDE, tc.BYTE))
    sb, size = mpi.strided_block(h)
    src, packed = ta.DeviceBuffer(ROWS * STRIDE), ta.DeviceBuffer(size)
    for it in range(2):
        host = orc.splitmix_bytes(ROWS * STRIDE, 70 + it)
        want = host.reshape(ROWS, STRIDE)[:, :4].reshape(-1)
        src.upload(host)
        packed.fill(0xAB)
        before = ta.signals()
        assert mpi.pack(src.addr(), 1, h, packed.addr(), size) == (0, size)
        assert (fetch(packed, size) == want).all(), it
        assert [b - a for a, b in zip(before, ta.signals())] == [1, 1]
        src.fill(0xAB)
        assert mpi.unpack(packed.addr(), size, src.addr(), 1, h) == (0, size)
        got = fetch(src, ROWS * STRIDE).reshape(ROWS, STRIDE)
        assert (got[:, :4].reshape(-1) == want).all() and (got[:, 4:] == 0xAB).all()
    mpi.free(h)
