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
RULE = {ta.DIR_PACK: [(256, 4), (128, 5), (48, 6), (24, 7), (20, 12), (16, 7), (1, 12)],
        ta.DIR_UNPACK: [(513, 3), (256, 4), (128, 5), (48, 6), (24, 17), (20, 12), (16, 7),
                        (1, 12)]}


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
    # the byte variant: 256 rows a tile
    reqs = [(sb, src.data_ptr(), out[i].data_ptr(), 1, ta.DIR_PACK, 11) for i in range(n)]
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


@pytest.mark.parametrize("L", [12, 13])
@pytest.mark.parametrize("variant", [12, 16])
def test_few_requests_of_one_word_units(L, variant):
    # two or four rows per lane, by the request's rows against 3/4 of a tile of
    # 1 024 per CU (256 CUs: 196 608); and a request of less than one tile
    rows = [196607, 196608, 196609, 600]
    span = max(rows) * 24 + 64
    host = orc.splitmix_bytes(span, 73)
    src = ta.DeviceBuffer(span)
    src.upload(host)
    packed = [ta.DeviceBuffer(n * L + 16) for n in rows]
    dsts = [ta.DeviceBuffer(span) for _ in rows]
    blocks = [ta.StridedBlock.make(4, 0, [L, n], [1, 24]) for n in rows]
    for b in packed:
        b.fill(0x5A)
    for b in dsts:
        b.fill(0xAB)
    ta.Batch([(sb, src.addr(), p.addr(), 1, ta.DIR_PACK, variant)
              for sb, p in zip(blocks, packed)]).launch()
    ta.Batch([(sb, d.addr(), p.addr(), 1, ta.DIR_UNPACK, variant)
              for sb, d, p in zip(blocks, dsts, packed)]).launch()
    ta.synchronize()
    for sb, p, d, n in zip(blocks, packed, dsts, rows):
        desc = orc.sb_desc(*sb.as_tuple())
        want = np.full(n * L + 16, 0x5A, np.uint8)
        want[:n * L] = orc.sb_pack(desc, host, 0, 1)
        assert (p.download() == want).all(), n
        ref = np.full(span, 0xAB, np.uint8)
        orc.sb_unpack(desc, want[:n * L], ref, 0, 1)
        assert (d.download() == ref).all(), n


def test_noalloc_takes_fewer_tiles_before_it_refuses():
    # 9 x 35 M rows of a byte: 615 000 tiles of the rule's 512 rows are past
    # the 524 288 the array holds, those of 1 024 rows are not
    rows, n = 35_000_000, 9
    host = orc.splitmix_bytes(2 * rows, 79)
    src, out = ta.DeviceBuffer(2 * rows), ta.DeviceBuffer(n * rows)
    src.upload(host)
    sb = ta.StridedBlock.make(1, 0, [1, rows], [1, 2])
    reqs = [(sb, src.addr(), out.addr(i * rows), 1, ta.DIR_PACK) for i in range(n)]
    ta.batch_run_noalloc(reqs)
    ta.synchronize()
    got = out.download().reshape(n, rows)
    for i in range(n):
        assert (got[i] == host[1::2]).all(), i
    with pytest.raises(ta.TempiError) as e:
        ta.batch_run_noalloc(reqs * 2)
    assert e.value.code == ta.TEMPI_ERR_UNSUPPORTED


def test_few_requests_from_host_memory():
    # unpacks of 512 KiB and more read mapped memory lane apart, in dwords
    sizes = [(12, 50000, 100), (1024, 700, 1100), (100, 100, 130)]  # the last is small
    blocks = [ta.StridedBlock.make(5, 0, [L, n], [1, st]) for L, n, st in sizes]
    span = max(n * st for _, n, st in sizes) + 64
    packed = ta.DeviceBuffer(sum(sb.size() for sb in blocks) + 3, mapped=True)
    host = orc.splitmix_bytes(packed.nbytes, 83)
    packed.upload(host)
    dsts = [ta.DeviceBuffer(span) for _ in blocks]
    reqs, at = [], 0
    for sb, d in zip(blocks, dsts):
        d.fill(0xAB)
        reqs.append((sb, d.addr(), packed.addr(at), 1, ta.DIR_UNPACK))
        at += sb.size() + 1  # odd packed addresses
    b = ta.Batch(reqs)
    assert [b.variant(i) for i in range(2)] == [9, 9]
    b.launch()
    ta.synchronize()
    at = 0
    for sb, d in zip(blocks, dsts):
        ref = np.full(span, 0xAB, np.uint8)
        orc.sb_unpack(orc.sb_desc(*sb.as_tuple()), host[at:at + sb.size()], ref, 0, 1)
        assert (d.download() == ref).all()
        at += sb.size() + 1
