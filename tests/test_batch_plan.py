"""The tile plan of a batch, on the host: every tile of every request runs
exactly once, and each of the eight XCDs gets an eighth of the cost (to one
tile) wherever the requests' buffers lie."""
import random

import pytest

import tempi_amd as ta

GIB = 1 << 30


def rows2d(length, rows, stride, start=0):
    return ta.StridedBlock.make(start, start + max(rows * abs(stride), length), [length, rows],
                                [1, stride])


def far_grids(gap):
    """52 requests on two grids of 20 MiB: 26 faces of 40 tiles each."""
    sb = rows2d(512, 1280, 600)
    return [(sb, (1 << 40) + g * gap + k * (20 << 20) // 26, (1 << 45) + k * GIB, 1, ta.DIR_PACK)
            for g in (0, 1) for k in range(26)]


def one_window():
    """100 packs of the same 4 KiB, sixteen times over (stride 0)."""
    sb = rows2d(4096, 16, 0)
    return [(sb, 1 << 40, (1 << 45) + (k << 20), 1, ta.DIR_PACK) for k in range(100)]


def same_face():
    sb = rows2d(2048, 512, 4096)
    return [(sb, 1 << 40, (1 << 45) + (k << 20), 1, ta.DIR_PACK) for k in range(26)]


def sparse_and_dense():
    """One request across 256 GiB, the others close together inside it."""
    reqs = [(rows2d(64, 1 << 12, 1 << 26), 1 << 40, 1 << 45, 1, ta.DIR_PACK)]
    sb = rows2d(256, 4096, 320)
    return reqs + [(sb, (1 << 40) + 100 * GIB + (k << 20) * 2, (1 << 46) + (k << 20), 1,
                    ta.DIR_UNPACK) for k in range(60)]


def mixed():
    rng = random.Random(7)
    reqs = []
    for k in range(300):
        length = rng.choice((1, 4, 12, 24, 100, 512, 4096))
        rows = rng.randint(1, 3000)
        stride = rng.choice((length, length + rng.randint(1, 500), -(length + 64)))
        start = rows * abs(stride) if stride < 0 else 0
        at = (1 << 40) + rng.randrange(1 << rng.choice((20, 30, 38)))
        reqs.append((rows2d(length, rows, stride, start), at, (1 << 46) + (k << 24), 1,
                     rng.choice((ta.DIR_PACK, ta.DIR_UNPACK))))
    return reqs


# bound of one tile's cost: 1024 rows of a line each, both sides, half as much again
LARGEST_TILE = 1.5 * (1024 * (128 + 128) + 2 * 65536)


def long_and_tiny_rows():
    """Half of the tiles hold 4-KiB rows, the other half 1-B rows."""
    long, tiny = rows2d(4096, 512, 4160), rows2d(1, 512 * 128, 2)
    return [(sb, (1 << 40) + k * (4 << 20), (1 << 45) + (k << 22), 1, ta.DIR_PACK)
            for k, sb in enumerate([long] * 20 + [tiny] * 20)]


@pytest.mark.parametrize("make", [
    lambda: far_grids(16 * GIB), lambda: far_grids(100 * GIB), lambda: far_grids(-(1 << 39)),
    one_window, same_face, sparse_and_dense, mixed, long_and_tiny_rows,
], ids=["16GiB", "100GiB", "below", "one_window", "same_face", "sparse", "mixed", "long_tiny"])
def test_every_xcd_gets_its_share(make):
    reqs = make()
    e = ta.batch_emulate(reqs)
    assert e["exact"] == 1 and e["requests"] == len(reqs)
    assert sum(e["xcd_tiles"]) == e["tiles"] >= 64
    assert e["grid"] == 8 * max(e["xcd_tiles"])
    total = sum(e["xcd_cost"])
    assert max(e["xcd_cost"]) <= total / 8 + LARGEST_TILE
    assert min(e["xcd_cost"]) >= total / 8 - LARGEST_TILE


def test_a_workgroup_costs_something():
    """Tiles of 1-B rows move 2 KiB and take a quarter of the time of 32-KiB ones."""
    e = ta.batch_emulate(long_and_tiny_rows())
    assert max(e["xcd_tiles"]) <= 5 * min(e["xcd_tiles"])


@pytest.mark.parametrize("n", [1, 8, 9])
def test_few_requests(n):
    for rows in (1, 2, 63, 1000):
        reqs = [(rows2d(12, rows, 24), (1 << 40) + (k << 30), (1 << 45) + (k << 20), 1,
                 ta.DIR_UNPACK) for k in range(n)]
        e = ta.batch_emulate(reqs)
        assert e["exact"] == 1 and sum(e["xcd_tiles"]) == e["tiles"]
    assert ta.batch_emulate([])["exact"] == 1


# -- what a batch takes ---------------------------------------------------------
#
# Sizes whose work units would reach 2^31 with the variant that is fastest:
# the plan takes one that holds them.  (No table of these sizes fits the static
# array, which the plan reports and does not refuse.)

SMALL = [(rows2d(64, 64, 128), (1 << 40) + (k << 20), (1 << 44) + (k << 20), 1, ta.DIR_PACK)
         for k in range(12)]


def plan_of_large(length, rows, direction, host=False, variant=-1):
    large = (rows2d(length, rows, length + 8), 1 << 46, 1 << 47, 1, direction, variant)
    e = ta.batch_emulate(SMALL + [large], packed_on_host=host)
    assert e["exact"] == 1 and e["requests"] == len(SMALL) + 1
    return e


@pytest.mark.parametrize("length,rows,direction,host", [
    (4096, 1 << 23, ta.DIR_PACK, True),    # 32 GiB in 4-KiB rows of host memory
    (4096, 1 << 23, ta.DIR_UNPACK, True),
    (40, 1 << 30, ta.DIR_UNPACK, False),   # 40-B rows: two units of 32 B
    (100, 1 << 29, ta.DIR_PACK, True),
])
def test_large_requests_are_taken(length, rows, direction, host):
    plan_of_large(length, rows, direction, host)


@pytest.mark.parametrize("variant,length,rows", [
    (12, 24, 1 << 30), (16, 48, 1 << 29), (17, 64, 1 << 30),
])
def test_large_requests_of_a_given_variant_are_taken(variant, length, rows):
    plan_of_large(length, rows, ta.DIR_PACK, variant=variant)


def test_rows_beyond_the_limit_stay_refused():
    for host in (False, True):
        with pytest.raises(ta.TempiError):
            plan_of_large(16, 1 << 31, ta.DIR_PACK, host)
    for variant in (7, 9, 12, 16, 17):
        with pytest.raises(ta.TempiError):
            plan_of_large(16, 1 << 31, ta.DIR_PACK, variant=variant)


@pytest.mark.parametrize("variant", [-1, 0, 1, 2, 3, 4, 5, 6, 7, 13, 14, 15, 16, 17])
def test_static_tables_hold_large_batches(variant):
    """7.5 GiB in 4-KiB rows are 480 Ki tiles of 16 KiB: they fit the static
    tables with each variant whose tiles are that large, and with 16 and 17,
    which give way to one of them."""
    reqs = [(rows2d(4096, 160 << 10, 4160), (1 << 40) + (k << 30), (1 << 44) + (k << 30), 1,
             ta.DIR_PACK, variant) for k in range(12)]
    e = ta.batch_emulate(reqs)
    assert e["exact"] == 1 and e["fits_static_tables"] == 1
