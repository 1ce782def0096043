"""Synchronous copies of more workgroups than signal for themselves return on
a signal kernel behind the copy, before the runtime reports the copy done.
The bytes must be there then: each round reads the result right after the
call with a plain hipMemcpy on the null stream, which does not wait for the
library's stream, beside small copies that signal for themselves."""
import ctypes

import numpy as np
import pytest

import tempi_amd as ta
import typecatalog as tc
from conftest import signalled
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def fetch(buf, n):
    hip = ctypes.CDLL("libamdhip64.so")
    out = np.empty(n, np.uint8)
    assert hip.hipMemcpy(ctypes.c_void_p(out.ctypes.data), ctypes.c_void_p(buf.addr()),
                         ctypes.c_size_t(n), 2) == 0  # device to host
    return out


@pytest.mark.parametrize("rows,block,stride,rounds", [
    (1 << 16, 64, 96, 40),     # 4 MiB
    (70001, 100, 131, 20),     # rows that end inside a word
    (1 << 19, 64, 80, 4),      # 32 MiB, the largest grid of one launch
])
def test_bytes_are_there_when_a_large_call_returns(mpi, rows, block, stride, rounds):
    spec, small = ("vector", rows, block, stride, tc.BYTE), ("vector", 64, 4, 12, tc.FLOAT)
    h, hs = mpi.type_from_spec(spec), mpi.type_from_spec(small)
    sb, size = mpi.strided_block(h)
    o = orc.OracleType(spec)
    span = o.span(1)[1]
    src, dst = ta.DeviceBuffer(span), ta.DeviceBuffer(span)
    packed, scratch = ta.DeviceBuffer(size), ta.DeviceBuffer(4096)
    assert not (signalled(sb, src.addr(), packed.addr(), ta.DIR_PACK)
                and signalled(sb, dst.addr(), packed.addr(), ta.DIR_UNPACK))
    for it in range(rounds):
        host = orc.splitmix_bytes(span, 4000 + it)
        src.upload(host)
        dst.fill(0xAB)
        assert mpi.pack(src.addr(), 1, h, packed.addr(), size) == (0, size)
        want = o.pack(host, 0, 1)
        assert (fetch(packed, size) == want).all(), it
        assert mpi.pack(src.addr(), 1, hs, scratch.addr(), 4096)[0] == 0
        assert mpi.unpack(packed.addr(), size, dst.addr(), 1, h) == (0, size)
        ref = np.full(span, 0xAB, np.uint8)
        o.unpack(want, ref, 0, 1)
        assert (fetch(dst, span) == ref).all(), it
    mpi.free(h)
    mpi.free(hs)
