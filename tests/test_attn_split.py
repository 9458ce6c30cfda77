"""How decode attention cuts a row into splits (host-only entry point, no GPU call)."""
import numpy as np
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


def test_a_half_more_times_the_reciprocal_has_the_whole_part_of_a_quotient():
    """What the kernels divide by: floor((a + 1/2) * r) in fp32 for a below 2^20, with r the reciprocal of b and its neighbours one place off (the
    hardware's has an error of one)."""
    rng = np.random.default_rng(7)
    for b in [*range(1, 140), 255, 256, 1000, 4095, 65535, 1 << 19]:
        whole = np.arange(0, 1 << 20, b, dtype=np.int64)
        a = np.concatenate([whole, whole[1:] - 1, whole + b // 2, rng.integers(0, 1 << 20, 2000)])
        a = a[a < 1 << 20]
        r = np.float32(1.0) / np.float32(b)
        for near in (np.nextafter(r, np.float32(0)), r, np.nextafter(r, np.float32(2))):
            assert np.array_equal(((a.astype(np.float32) + np.float32(0.5)) * near).astype(np.int64), a // b), b
