"""Requests and calls without completion signals (TEMPI_NO_SIGNAL; the same
path a device without them takes): a request completes when its own copy is
done, whatever is on the library's stream behind it."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = r"""
import ctypes, sys
sys.path[:0] = ["tests", "."]
import numpy as np
import tempi_amd as ta
import typecatalog as tc
from oracle import oracle as orc
from tempi_amd import mpi as tmpi

hip = ctypes.CDLL("libamdhip64.so")
hip.hipStreamQuery.argtypes = [ctypes.c_void_p]
mpi = tmpi.get()
method = int(sys.argv[1])
ta.lib().tempi_set_datatype_method(method)
large = ta.StridedBlock.make(0, 1 << 30, [1 << 30], [1])
a, b = ta.DeviceBuffer(1 << 30), ta.DeviceBuffer(1 << 30)
for spec in (("vector", 300, 3, 7, tc.FLOAT), ("vector", 4096, 256, 300, tc.BYTE)):
    h = mpi.type_from_spec(spec)
    o = orc.OracleType(spec)
    n = o.span(1)[1]
    src, dst, packed = ta.DeviceBuffer(n), ta.DeviceBuffer(n), ta.DeviceBuffer(o.size())
    for it in range(3):
        host = orc.splitmix_bytes(n, 60 + it)
        ref = np.full(n, 0xAB, np.uint8)
        o.unpack(o.pack(host, 0, 1), ref, 0, 1)
        src.upload(host)
        dst.fill(0xAB)
        err, rr = mpi.irecv(dst.addr(), 1, h, 0, 11)
        assert err == 0
        err, sr = mpi.isend(src.addr(), 1, h, 0, 11)
        assert err == 0
        for _ in range(400):  # about 0.15 s of copies behind the pack
            ta.pack_sb(large, a.addr(), 1, b.addr(), 1 << 30, 0, 1)
        assert mpi.wait(sr, h)[0] == 0
        busy = hip.hipStreamQuery(ta.stream())
        assert busy == 600, busy  # the copies still run: the request did not wait for them
        assert mpi.wait(rr, h)[0] == 0
        assert (dst.download() == ref).all(), (spec, it)
        assert mpi.pack(src.addr(), 1, h, packed.addr(), o.size()) == (0, o.size())
        assert (packed.download() == o.pack(host, 0, 1)).all()
    mpi.free(h)
assert ta.signals() == (0, 0) and ta.counters()["signalled_waits"] == 0
print("done")
"""


@pytest.mark.parametrize("method", [2, 3], ids=["oneshot", "staged"])
def test_requests_wait_for_their_own_copy(method):
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(method)], cwd=ROOT, text=True,
                       capture_output=True, timeout=110,
                       env=dict(os.environ, TEMPI_NO_SIGNAL="1"))
    assert r.returncode == 0 and "done" in r.stdout, r.stdout + r.stderr
