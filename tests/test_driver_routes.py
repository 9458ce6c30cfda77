"""The driver's rules that choose a kernel (host-only entry points of libpie_driver_hip.so, no GPU call)."""
import numpy as np
import pytest


def skinny_us(M, N, K, tile_major):
    """The estimate the line of the int4 rule is drawn with: side-by-side passes of 32 rows, a fifth pass as dear as eight."""
    data = N * K / 2
    if not tile_major:
        return 5.0 + data / 2.8e6 * (1.0 + 0.85 * (-(-M // 16) - 1))
    passes = -(-M // 32)
    p2 = 1 << (passes - 1).bit_length()
    return 5.0 + data / 3.8e6 * 1.38 * (1.0 + 0.52 * (p2 - 1) if p2 <= 8 else (1.0 + 0.52 * 7) * passes / 8.0)


def tiles_us(M, N, K):
    return 2.0 + K // 64 * 0.68 * max(1.0, -(-N // 128) * -(-M // 128) / 512.0)


@pytest.mark.parametrize("tile_major", [True, False])
def test_int4_prompts_keep_fp32_scales_where_the_skinny_gemm_reaches(tile_major):
    """The skinny GEMM scales int4 groups in fp32, the blocks round each code times its scale to bf16: a matrix is not moved
    from the first to the second because the second is a little faster."""
    from pie_amd import driver as drv

    for N, K, last in [(4096, 14336, 768), (6144, 4096, 480), (4096, 4096, 704), (28672, 4096, 128)]:
        for M in (129, 200, last - 32, last, last + 1, last + 64):
            if tile_major and M > 128 and M <= last:
                assert drv.linear_route("int4b8", M, N, K, 128) == "skinny", (M, N, K)
    rng = np.random.default_rng(11)
    for _ in range(400):
        M, N, K = int(rng.integers(129, 2048)), int(rng.integers(8, 1800)) * 16, int(rng.integers(2, 120)) * 128
        route = drv.linear_route("int4b8", M, N, K, 128, tile_major)
        if skinny_us(M, N, K, tile_major) <= tiles_us(M, N, K):
            assert route == "skinny", (M, N, K)
        assert route in ("skinny", "tiled", "wide")


def test_formats_whose_scales_wait_for_the_sum_take_the_blocks():
    """One-byte and bf16 weights enter the blocks' products exactly: the faster estimate decides."""
    from pie_amd import driver as drv

    for kind in ("int8", "fp8", "bf16"):
        assert drv.linear_route(kind, 381, 28672, 4096) in ("wide", "tiled")
        assert drv.linear_route(kind, 2048, 4096, 4096) in ("wide", "tiled")
    assert drv.linear_route("int4b8", 2048, 28672, 4096, 128) == "wide"
    assert drv.linear_route("int4b8", 40, 28672, 4096, 128) == "wide"    # (its columns form: groups scaled in fp32)
    assert drv.linear_route("int4b8", 1, 4096, 4096, 128) == "gemv"


@pytest.mark.parametrize("experts", [8, 128])
def test_int4_experts_keep_fp32_scales(experts):
    """The passes of 16 routes scale int4 groups in fp32, the blocks of routes round each code times its scale to bf16."""
    from pie_amd import driver as drv

    for each in (1, 15, 16, 17, 88, 500, 4096):
        assert not drv.experts_in_blocks("int4b8", each * experts, experts)
    for kind, first in (("fp8", 16), ("int8", 16), ("bf16", 12)):
        assert [drv.experts_in_blocks(kind, n * experts, experts) for n in (first - 1, first, 500)] == [False, True, True]


def test_workspace_of_shares_is_what_the_shares_take():
    """With the bytes the library names no row count up to the limit is estimated slower than with all the memory there is, and
    they are no more than 32 MiB, none where no shape takes shares."""
    from pie_amd import ops

    rng = np.random.default_rng(12)
    assert ops.gemm_mfma_tiled_workspace_bytes(2048, 4096, 4096) == 32 << 20
    assert ops.gemm_mfma_tiled_workspace_bytes(128, 4096, 4096) == 0          # (no prompts)
    assert ops.gemm_mfma_tiled_workspace_bytes(4096, 28672, 4096) == 0        # (more than half a round of blocks in one row of them)
    for _ in range(60):
        top, N, K = int(rng.integers(129, 4097)), int(rng.integers(1, 1200)) * 16, int(rng.integers(4, 240)) * 64
        named = ops.gemm_mfma_tiled_workspace_bytes(top, N, K)
        assert named <= 32 << 20
        for M in rng.integers(129, top + 1, 20):
            for kind in ("int8", "bf16"):
                assert ops.gemm_mfma_us(kind, int(M), N, K, 0, True, named) == ops.gemm_mfma_us(kind, int(M), N, K, 0, True, 1 << 40)


# microseconds of one layer's attention over a bf16 cache on an MI355X, row by row and as tiles: a portion of 32, 64, 112, 160 and 256
# rows by (query heads, kv heads, head size) and cached tokens
MEASURED_ROWS = (32, 64, 112, 160, 256)
MEASURED = {
    ((32, 8, 128), 0): [(4.4, 5.3), (5.1, 6.1), (9.6, 7.9), (14.4, 8.3), (22.1, 10.5)],
    ((32, 8, 128), 256): [(7.5, 11.1), (11.1, 11.8), (19.7, 12.8), (25.0, 13.7), (37.5, 15.4)],
    ((32, 8, 128), 1000): [(15.2, 26.5), (24.6, 27.0), (56.2, 27.4), (73.4, 28.6), (105.1, 30.3)],
    ((32, 8, 128), 2000): [(23.7, 45.7), (40.5, 46.7), (86.6, 46.4), (116.2, 47.9), (164.1, 50.5)],
    ((32, 4, 128), 0): [(5.0, 5.3), (5.4, 6.1), (7.0, 7.9), (11.3, 8.3), (14.8, 10.4)],
    ((32, 4, 128), 256): [(8.2, 11.1), (8.7, 11.8), (12.6, 12.8), (19.4, 13.9), (24.4, 15.6)],
    ((32, 4, 128), 1000): [(15.8, 26.2), (16.7, 26.7), (24.9, 27.6), (50.3, 28.5), (74.0, 30.1)],
    ((32, 4, 128), 2000): [(20.1, 45.6), (25.2, 46.6), (40.7, 46.9), (82.0, 47.9), (111.7, 49.8)],
    ((32, 8, 64), 0): [(3.4, 4.1), (3.7, 4.9), (6.0, 6.2), (7.5, 6.6), (12.7, 8.0)],
    ((32, 8, 64), 256): [(5.2, 8.5), (7.0, 8.8), (11.3, 9.6), (14.0, 10.4), (21.2, 11.8)],
    ((32, 8, 64), 1000): [(9.9, 20.4), (15.7, 20.8), (31.5, 21.1), (42.0, 22.2), (58.2, 23.3)],
    ((32, 8, 64), 2000): [(15.4, 35.1), (25.8, 35.7), (47.9, 36.0), (60.4, 36.7), (89.7, 38.2)],
}


def taken(requests, heads, one_byte=False):
    """Indices of the requests whose rows are tiled; checks that every row is in one tile or one run, once."""
    from pie_amd import driver as drv

    cut = drv.attention_cut(requests, *heads, one_byte)
    first = np.concatenate([[0], np.cumsum([n for _, n in requests])])
    seen, tiled = np.zeros(first[-1], int), set()
    for a, n in cut["tiles"]:
        r = int(np.searchsorted(first, a, side="right")) - 1
        assert 0 < n <= cut["tile_rows"] and a + n <= first[r + 1]   # (one request's rows)
        seen[a:a + n] += 1
        tiled.add(r)
    for a, n, _ in cut["runs"]:
        seen[a:a + n] += 1
    assert (seen == 1).all()
    return sorted(tiled)


def test_measured_portions_take_their_faster_form():
    for (heads, history), times in MEASURED.items():
        for n, (rows, tiles) in zip(MEASURED_ROWS, times):
            us = tiles if taken([(history, n)], heads) else rows
            assert us <= 1.08 * min(rows, tiles), (heads, history, n, us)


@pytest.mark.parametrize("heads", [(32, 8, 128), (32, 4, 128), (32, 8, 64), (8, 8, 128), (16, 8, 128), (8, 2, 64), (32, 32, 128)])
@pytest.mark.parametrize("history", [0, 60, 256, 1000, 2000, 8000])
def test_longer_portions_do_not_fall_back_to_rows(heads, history):
    """A portion takes tiles from some number of rows on, not here and there, and about where its rows fill a round of blocks."""
    tiles = [bool(taken([(history, n)], heads)) for n in range(8, 800)]
    first = tiles.index(True) + 8
    assert all(tiles[first - 8:])
    assert (512 if history < 4000 else 440) < first * heads[1] <= 1024


def test_portions_behind_a_context_beside_decoded_tokens_take_tiles():
    decoded = [(700 + 40 * i, 1) for i in range(8)]
    assert taken(decoded + [(2000, 100)], (32, 8, 128)) == [8]
    assert taken(decoded + [(2000, 30)], (32, 8, 128)) == []
    assert taken(decoded + [(0, 400), (0, 20)], (32, 8, 128)) == [8, 9]     # (the shorter one rides along)
    assert taken([(0, 400), (4000, 16)], (32, 8, 128)) == [0]               # (and a few rows behind many keys do not)
    assert taken([(900, 1)] * 64, (32, 8, 128)) == []
    # (64 rows behind 4000 keys, row by row and as tiles: 104 and 86 us, over a one-byte cache 88 and 91)
    assert taken([(4000, 64)], (32, 8, 128)) == [0] and taken([(4000, 64)], (32, 8, 128), one_byte=True) == []
    assert taken([(500, 60)] * 4, (32, 8, 64)) == [0, 1, 2, 3]


@pytest.mark.parametrize("heads", [(32, 8, 128), (32, 4, 128), (32, 8, 64)])
def test_long_portions_take_tiles_in_whatever_order_requests_come(heads):
    """Every run of rows between portions is another launch, which is priced (measured: 105 us in rows and 58 cut, 65 and 55, 55 and 40;
    the last batch, five runs around short portions: 42 and 56, 30 and 57, 23 and 45)."""
    assert taken([(800, 1)] * 20 + [(0, 500), (900, 1), (0, 400), (700, 1)], heads) == [20, 22]
    assert taken([(800, 1)] * 20 + [(0, 500), (0, 400), (900, 1), (700, 1)], heads) == [20, 21]
    assert taken([(500, 1), (0, 130)] * 4 + [(400, 1)], heads) == []


@pytest.mark.parametrize("seed", range(8))
def test_every_row_is_attended_once(seed):
    rng = np.random.default_rng(300 + seed)
    for _ in range(60):
        requests = [(int(rng.integers(0, 3000)), int(1 if rng.random() < 0.5 else rng.integers(1, 300))) for _ in range(int(rng.integers(1, 20)))]
        taken(requests, [(32, 8, 128), (32, 4, 128), (32, 8, 64), (32, 32, 128), (12, 2, 128), (14, 2, 64)][seed % 6])
