"""Each completion signal has a number of its own, whatever error an
application has left unread in its thread (the runtime reports it to the next
hipGetLastError of anyone): a copy that waited for another's number would
return before it is done."""
import ctypes

import numpy as np
import pytest

import tempi_amd as ta
import typecatalog as tc
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

INVALID_DEVICE = 101


def hip():
    lib = ctypes.CDLL("libamdhip64.so")
    lib.hipMemcpy.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int]
    return lib


def fetch(lib, buf, n):
    """A plain hipMemcpy on the null stream: it does not wait for the library's."""
    out = np.empty(n, np.uint8)
    assert lib.hipMemcpy(out.ctypes.data, buf.addr(), n, 2) == 0
    return out


@pytest.mark.parametrize("rows,block,stride", [
    (1 << 16, 64, 96),    # 4 MiB: a signal kernel behind the copy
    (1 << 20, 64, 80),    # 64 MiB
])
def test_an_unread_error_of_the_application(mpi, rows, block, stride):
    lib = hip()
    big, small = ("vector", rows, block, stride, tc.BYTE), ("vector", 512, 256, 512, tc.BYTE)
    hb, hs = mpi.type_from_spec(big), mpi.type_from_spec(small)
    ob, os_ = orc.OracleType(big), orc.OracleType(small)
    nb, ns = ob.span(1)[1], os_.span(1)[1]
    src, packed = ta.DeviceBuffer(nb), ta.DeviceBuffer(ob.size())
    src2, packed2 = ta.DeviceBuffer(ns), ta.DeviceBuffer(os_.size())
    host = orc.splitmix_bytes(nb, 81)
    src.upload(host)
    want = ob.pack(host, 0, 1)
    assert mpi.pack(src.addr(), 1, hb, packed.addr(), ob.size())[0] == 0  # the pick is made
    for it in range(10):
        host2 = orc.splitmix_bytes(ns, 900 + it)
        src2.upload(host2)
        packed.fill(0xAB)
        packed2.fill(0xAB)
        assert lib.hipSetDevice(9999) == INVALID_DEVICE  # never read
        n0, k0 = ta.signals()
        assert mpi.pack(src.addr(), 1, hb, packed.addr(), ob.size()) == (0, ob.size())
        n1, k1 = ta.signals()
        assert mpi.pack(src2.addr(), 1, hs, packed2.addr(), os_.size()) == (0, os_.size())
        got2 = fetch(lib, packed2, os_.size())
        n2, k2 = ta.signals()
        assert (n1 - n0, k1 - k0, n2 - n1, k2 - k1) == (1, 1, 1, 0)
        assert (got2 == os_.pack(host2, 0, 1)).all(), it
        assert (fetch(lib, packed, ob.size()) == want).all(), it
        assert lib.hipGetLastError() == INVALID_DEVICE  # still the application's
    mpi.free(hb)
    mpi.free(hs)
