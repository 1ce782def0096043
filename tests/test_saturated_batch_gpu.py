"""Batches with more tiles than the grid runs at once, whose variants follow
from the row length: every length at which the rule changes its variant and
its neighbours, both directions, at odd addresses and at one multiple of 16,
against the oracle; and batches past the tiles one launch can start."""
import numpy as np
import pytest

import tempi_amd as ta
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

LENGTHS = [1, 2, 3, 7, 8, 12, 15, 16, 19, 20, 23, 24, 25, 31, 32, 40, 47, 48,
           63, 64, 127, 128, 200, 255, 256, 257, 512, 513, 600]
ROWS = 40000
# (least length, variant): packs, unpacks
RULE = {ta.DIR_PACK: [(513, 3), (256, 4), (128, 5), (48, 6), (24, 17), (20, 12), (16, 7), (1, 12)],
        ta.DIR_UNPACK: [(256, 4), (128, 5), (48, 6), (24, 7), (20, 12), (16, 7), (1, 12)]}


@pytest.mark.parametrize("align,entry,mapped", [(1, "batch", False), (16, "batch", False),
                                                (1, "noalloc", False), (16, "noalloc", False),
                                                (1, "batch", True)])
def test_rule_moves_every_row_length(align, entry, mapped):
    blocks, offs, poffs, at, pat = [], [], [], 0, 0
    for i, L in enumerate(LENGTHS):
        stride = -(-(L + 5 + i) // align) * align
        start = 3 if align == 1 else 16
        # rows forward, in reverse, and in two dimensions
        if i % 3 == 1:
            sb = ta.StridedBlock.make(start + (ROWS - 1) * stride, 0, [L, ROWS], [1, -stride])
        elif i % 3 == 2:
            sb = ta.StridedBlock.make(start, 0, [L, ROWS // 50, 50],
                                      [1, stride, stride * (ROWS // 50) + 32])
        else:
            sb = ta.StridedBlock.make(start, 0, [L, ROWS], [1, stride])
        blocks.append(sb)
        offs.append(at)
        poffs.append(pat)
        at += -(-(start + ROWS * stride + 50 * 32 + 64) // 16) * 16
        pat += -(-(sb.size() + align) // align) * align
    host = orc.splitmix_bytes(at, 71)
    src, dst = ta.DeviceBuffer(at), ta.DeviceBuffer(at)
    packed = ta.DeviceBuffer(pat, mapped=mapped)
    src.upload(host)
    dst.fill(0xAB)
    packed.fill(0x5A)
    packs = [(sb, src.addr(o), packed.addr(p), 1, ta.DIR_PACK)
             for sb, o, p in zip(blocks, offs, poffs)]
    unpacks = [(sb, dst.addr(o), packed.addr(p), 1, ta.DIR_UNPACK)
               for sb, o, p in zip(blocks, offs, poffs)]
    for reqs in (packs, unpacks):
        if entry == "batch":
            b = ta.Batch(reqs)
            assert [b.variant(i) for i in range(len(reqs))] == [
                9 if mapped else next(v for least, v in RULE[reqs[0][4]] if L >= least) for L in LENGTHS]
            b.launch()
        else:
            ta.batch_run_noalloc(reqs)
        ta.synchronize()
    got = packed.download()
    ref = np.full(at, 0xAB, np.uint8)
    want = np.full(pat, 0x5A, np.uint8)
    for sb, o, p in zip(blocks, offs, poffs):
        desc = orc.sb_desc(*sb.as_tuple())
        want[p:p + sb.size()] = orc.sb_pack(desc, host[o:], 0, 1)
        orc.sb_unpack(desc, want[p:p + sb.size()], ref[o:], 0, 1)
    assert (got == want).all()
    assert (dst.download() == ref).all()


@pytest.mark.parametrize("extra", [0, 8])
def test_more_tiles_than_one_launch_starts(extra):
    # 2^23 tiles is the largest grid: these make the workgroups loop, in the
    # kernel for at most eight requests and in the one for more
    torch = pytest.importorskip("torch")
    rows = 1 << 30
    n = 5
    sb = ta.StridedBlock.make(1, 0, [1, rows], [1, 2])
    src = torch.randint(0, 256, (2 * rows,), dtype=torch.uint8, device="cuda")
    out = torch.zeros(n, rows, dtype=torch.uint8, device="cuda")
    small = torch.zeros(8, 64, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    reqs = [(sb, src.data_ptr(), out[i].data_ptr(), 1, ta.DIR_PACK) for i in range(n)]
    reqs += [(ta.StridedBlock.make(0, 0, [8, 8], [1, 16]), src.data_ptr(),
              small[i].data_ptr(), 1, ta.DIR_PACK) for i in range(extra)]
    b = ta.Batch(reqs)
    assert b.info()["tiles"] > 1 << 23
    b.launch()
    ta.synchronize()
    want = src[1::2]
    for i in range(n):
        assert torch.equal(out[i], want), i
    for i in range(extra):
        assert torch.equal(small[i], src[:128].view(8, 16)[:, :8].reshape(-1)), i
