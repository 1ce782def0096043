"""The closed-form choice for copies bound by their launch takes each of its
variants for the row lengths it says, in both directions."""
import pytest

import tempi_amd as ta

PICKS = {4: (256, 300, 1024, 5000), 5: (128, 200, 255), 6: (48, 64, 96, 100, 127),
         7: (16, 17, 32, 33, 62), 8: (8, 24, 40, 56), 9: (1, 3, 4, 13, 20, 28, 44, 52),
         12: (12, 36, 60)}


@pytest.mark.parametrize("direction", [ta.DIR_PACK, ta.DIR_UNPACK])
def test_each_variant_of_the_rule(direction):
    for variant, lengths in PICKS.items():
        for length in lengths:
            sb = ta.StridedBlock.make(0, 9 * (length + 5), [length, 9], [1, length + 5])
            v = ta.select_variant(sb, 1, 1 << 40, 1 << 41, direction, ta.SELECT_DEFAULT)
            assert v == variant, length
