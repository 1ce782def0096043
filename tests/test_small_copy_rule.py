"""The closed-form choice for copies bound by their launch: whatever the row
length, strides and alignment, its variant stores exactly the copy's bytes,
in a single launch."""
import random

import pytest

import tempi_amd as ta


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
def test_the_choice_copies_every_shape(direction):
    rng = random.Random(11)
    picks = set()
    for length in [*range(1, 70), 96, 100, 127, 128, 200, 256, 300, 1000, 1024, 5000]:
        for stride in (length, length + 3, -(length + 16)):
            sb = ta.StridedBlock.make(6 * abs(stride), 14 * abs(stride) + length,
                                      [length, 5, 2], [1, stride, 7 * abs(stride)])
            at, to = (1 << 40) + rng.randrange(16), (1 << 41) + rng.randrange(16)
            v = ta.select_variant(sb, 2, at, to, direction, ta.SELECT_DEFAULT)
            e = ta.copy_emulate(sb, 2, at, to, direction, v)
            assert e["exact"] == 1 and e["launches"] == 1, (length, stride, v, e)
            picks.add(v)
    assert len(picks) >= 6  # every branch of the rule
