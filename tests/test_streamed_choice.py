"""The closed-form choice for copies whose strided side touches more than the
caches hold: cached accesses below the threshold, nontemporal ones above it,
and whatever the row length, stride and alignment the chosen variant stores
exactly the copy's bytes (checked on fewer rows of the same layout)."""
import pytest

import tempi_amd as ta

LENGTHS = [*range(1, 37), 40, 48, 60, 63, 64, 80, 100, 112, 127, 128, 129, 144, 256, 300, 511,
           512, 513, 528, 1000, 1024, 4096, 5001]
MIB = 1 << 20


def pick(length, stride, mib, direction, offset):
    """The rule's variant for rows touching about `mib` MiB of lines."""
    touched = min(length + 127, max(length, abs(stride)))
    rows = mib * MIB // touched + 1
    sb = ta.StridedBlock.make(0, rows * abs(stride), [length, rows], [1, stride])
    return ta.select_variant(sb, 1, (1 << 40) + offset, 1 << 41, direction, ta.SELECT_HEURISTIC)


def nontemporal(variant, direction):
    info = ta.variant_info(variant)
    strided_side = bool(info["nontemporal_stores"])
    loads = bool(info["nontemporal_loads"]) and not (strided_side and direction == ta.DIR_UNPACK)
    return loads, strided_side and direction == ta.DIR_UNPACK


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
@pytest.mark.parametrize("gap", [3, 64, 1000, -200])
def test_streamed_choice(direction, gap):
    kinds = set()
    for length in LENGTHS:
        stride = -(length - gap) if gap < 0 else length + gap
        for offset in (0, 5):
            assert nontemporal(pick(length, stride, 32, direction, offset), direction) == \
                (False, False), length
            for mib in (70, 200, 600):
                v = pick(length, stride, mib, direction, offset)
                loads, stores = nontemporal(v, direction)
                kinds.add((loads, stores))
                if stores:  # never where a row's bytes are few or the cache holds the lines
                    assert length >= 16 and mib > 128, (length, mib)
                small = ta.StridedBlock.make(9 * abs(stride), 20 * abs(stride), [length, 9],
                                             [1, stride])
                e = ta.copy_emulate(small, 2, (1 << 40) + offset, (1 << 41) + 3, direction, v)
                assert e["exact"] == 1, (length, stride, offset, mib, v, e)
    assert (True, False) in kinds and ((False, True) in kinds) == (direction == ta.DIR_UNPACK)
