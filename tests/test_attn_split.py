"""How decode attention cuts a row into splits (host-only entry point, no GPU call)."""
import pytest


@pytest.mark.parametrize("least", [1, 2, 7, 8, 32])
def test_splits_cover_a_row_and_keep_their_bounds(least):
    """Every key in one of at most `num_splits` splits, whole 32-key steps, none empty; until they are as many as the plan has they hold the plan's units at
    most (rounded up to a step) and more than half as many."""
    from pie_amd import ops

    for num in (1, 2, 3, 16, 64):
        for units in list(range(1, 140)) + [255, 256, 257, 1000]:
            each = ops.attn_row_split(units * 16 - 5, least, num)
            splits = -(-units // each)
            assert 1 <= splits <= num and (splits - 1) * each < units
            if num == 1:
                assert each == units
                continue
            assert each % 2 == 0
            if -(-units // least) <= num:
                assert each <= least + least % 2 and (splits == 1 or 2 * each > least)
    assert ops.attn_row_split(0, least, 4) >= 1
    assert ops.attn_row_split(9 * 16, 8, 4) == 6
    assert ops.attn_row_split(-1, least, 4) == ops.attn_row_split(16, 0, 4) == ops.attn_row_split(16, least, 0) == 0
