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


@pytest.mark.parametrize("block,rows,mapped,own", [
    (24, 21845, True, False),   # 512 KiB of lane-per-row stores over the link
    (100, 13107, True, False),  # 1.25 MiB in 103 workgroups of four lanes a row
    (24, 4096, True, True),     # 96 KiB in 16 workgroups
    (256, 1024, True, True),    # 32 workgroups, whole lines
    (256, 1024, False, True),
    (12, 21845, False, None),   # either, by the pick
    (4096, 8192, True, False),  # 32 MiB
])
def test_the_copy_signals_itself_where_that_is_the_shorter_wait(mpi, block, rows, mapped, own):
    """... and its bytes are there, in mapped memory for the host itself to
    read, when the call returns."""
    spec = ("vector", rows, block, block + 100, tc.BYTE)
    h = mpi.type_from_spec(spec)
    o = orc.OracleType(spec)
    n, size = o.span(1)[1], o.size()
    src, dst = ta.DeviceBuffer(n), ta.DeviceBuffer(n)
    packed = ta.DeviceBuffer(size, mapped=mapped)
    lib = hip()
    for it in range(20 if size < (1 << 21) else 3):
        host = orc.splitmix_bytes(n, 300 + it)
        want = o.pack(host, 0, 1)
        src.upload(host)
        dst.fill(0xAB)
        n0, k0 = ta.signals()
        assert mpi.pack(src.addr(), 1, h, packed.addr(), size) == (0, size)
        if mapped:
            got = np.ctypeslib.as_array((ctypes.c_uint8 * size).from_address(packed.addr()))
        else:
            got = fetch(lib, packed, size)
        assert (got == want).all(), it
        n1, k1 = ta.signals()
        assert n1 - n0 == 1
        if own is not None:
            assert k1 - k0 == (0 if own else 1)
        assert mpi.unpack(packed.addr(), size, dst.addr(), 1, h) == (0, size)
        ref = np.full(n, 0xAB, np.uint8)
        o.unpack(want, ref, 0, 1)
        assert (fetch(lib, dst, n) == ref).all(), it
    mpi.free(h)


@pytest.mark.parametrize("rows,kernels", [(64, 2), (256, 1), (2048, 1)])
def test_a_copy_by_the_dma_engine_has_no_signal_kernel_behind_it(mpi, rows, kernels):
    """STAGED: the send waits for its copy to the host with the stream where
    that copy is larger than 16 KiB; the receive's unpack signals."""
    ta.lib().tempi_set_datatype_method(3)
    spec = ("vector", rows, 256, 300, tc.BYTE)
    h = mpi.type_from_spec(spec)
    o = orc.OracleType(spec)
    n = o.span(1)[1]
    src, dst = ta.DeviceBuffer(n), ta.DeviceBuffer(n)
    try:
        for it in range(5):
            host = orc.splitmix_bytes(n, 500 + it)
            src.upload(host)
            dst.fill(0xAB)
            ref = np.full(n, 0xAB, np.uint8)
            o.unpack(o.pack(host, 0, 1), ref, 0, 1)
            err, rr = mpi.irecv(dst.addr(), 1, h, 0, 91)
            assert err == 0
            k0 = ta.signals()[1]
            if it % 2:
                err, sr = mpi.isend(src.addr(), 1, h, 0, 91)
                assert err == 0 and mpi.wait(sr, h)[0] == 0
            else:
                assert mpi.send(src.addr(), 1, h, 0, 91) == 0
            assert mpi.wait(rr, h)[0] == 0
            assert ta.signals()[1] - k0 == kernels, it
            assert (dst.download() == ref).all(), it
    finally:
        ta.lib().tempi_set_datatype_method(-1)
    mpi.free(h)
