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
