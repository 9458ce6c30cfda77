"""The estimates that choose a GEMM's kernel, its blocks and its shares of K, against times measured on an MI355X with each call's weights
out of HBM (host-only entry points, no GPU call)."""
import pytest

WORKSPACE = 32 << 20

# (format, rows, N, K): microseconds in blocks of 256 rows, and in blocks of (rows, shares of K) for every way within an eighth of the fastest.
# On the long K of these, a few blocks without shares wait for HBM at each of 128 and 224 steps and take up to 1.45 times as long.
ONE_BYTE = {
    ("int8", 256, 4096, 14336): (45.2, {(64, 4): 45.1, (96, 5): 46.1, (128, 4): 46.9, (64, 6): 48.1, (128, 6): 50.1, (96, 4): 50.3}),
    ("int8", 800, 2048, 8192): (45.3, {(96, 3): 41.5, (128, 4): 42.8, (64, 2): 44.6, (96, 4): 44.7, (64, 3): 45.2, (96, 5): 45.6, (64, 4): 46.0}),
    ("int8", 192, 8192, 8192): (48.6, {(96, 4): 40.3, (96, 3): 43.3, (64, 4): 44.5, (128, 4): 45.3}),
    ("int8", 256, 8192, 8192): (48.3, {(128, 4): 49.2, (64, 2): 49.2, (128, 2): 50.8, (64, 3): 51.5, (128, 3): 52.8, (96, 2): 53.5, (96, 4): 54.3}),
    ("int8", 400, 5120, 8192): (54.4, {(128, 3): 52.8, (96, 2): 53.7, (64, 2): 54.8, (96, 3): 56.5, (64, 3): 57.1, (128, 4): 59.4}),
    ("fp8", 1024, 2048, 8192): (47.0, {(128, 4): 45.2, (64, 2): 45.2, (64, 3): 46.3, (128, 2): 47.1, (128, 3): 48.9, (96, 4): 49.8, (96, 2): 50.1, (96, 3): 50.1}),
    ("fp8", 256, 4096, 14336): (44.6, {(96, 5): 44.0, (128, 4): 44.6, (64, 4): 45.0, (64, 6): 47.6, (96, 4): 47.8, (128, 6): 48.8}),
    ("fp8", 512, 3072, 8192): (41.6, {(96, 3): 39.5, (64, 4): 40.3, (128, 5): 40.6, (128, 4): 41.9, (64, 5): 44.0, (64, 3): 44.2, (64, 2): 44.4}),
    ("fp8", 400, 5120, 8192): (54.0, {(128, 3): 50.4, (64, 2): 50.5, (96, 2): 50.6, (32, 1): 54.0, (96, 3): 54.3, (64, 3): 54.5, (128, 4): 56.6}),
    ("fp8", 700, 2048, 14336): (55.5, {(96, 4): 51.1, (128, 5): 54.2, (96, 3): 55.5, (64, 4): 55.7}),
    ("fp8", 1300, 2048, 4096): (43.8, {(32, 1): 33.3, (64, 1): 35.9, (96, 2): 37.0, (96, 1): 37.0}),
    ("fp8", 1300, 5120, 2048): (37.3, {(128, 1): 33.8, (64, 1): 34.5, (96, 1): 35.2}),
    ("fp8", 400, 5120, 2048): (30.9, {(32, 1): 17.0}),
    ("fp8", 320, 28672, 4096): (109.2, {(128, 1): 83.7, (64, 1): 86.0, (96, 1): 87.6}),
    ("int8", 1300, 6144, 4096): (103.5, {(96, 1): 70.0, (64, 1): 72.7}),
}


@pytest.mark.parametrize("shape", ONE_BYTE, ids=str)
def test_one_byte_prompts_take_a_way_within_an_eighth_of_the_fastest(shape):
    from pie_amd import ops

    kind, M, N, K = shape
    tall, ways = ONE_BYTE[shape]
    fastest = min(tall, *ways.values())
    us = ops.gemm_rows_us(kind, M, N, K, WORKSPACE)
    if us < ops.gemm_mfma_us(kind, M, N, K, 0, True, WORKSPACE):
        plan = ops.gemm_rows_plan(kind, M, N, K, WORKSPACE)
        assert plan in ways and abs(us / ways[plan] - 1) < 0.2
    else:
        assert tall <= 1.125 * fastest


# bf16 rows, N, K: microseconds in blocks of 128 columns and two heights (the faster is the entry's choice), and of 256 rows of 8 waves by 128 or 256 columns
SHORT_K = {(500, 2048, 256): (8.9, 10.0), (300, 14336, 256): (15.8, 11.9), (2011, 8192, 256): (30.8, 20.4), (2011, 14336, 256): (55.0, 34.7), (3000, 4096, 256): (26.1, 19.2),
           (2011, 8192, 512): (38.7, 25.6), (2011, 14336, 512): (70.4, 46.1), (1000, 4096, 512): (12.0, 14.2), (700, 8192, 768): (21.5, 18.1),
           (1000, 2048, 1024): (14.4, 18.3), (2011, 4096, 1024): (26.8, 22.6), (3000, 16384, 1024): (147.8, 101.2), (2011, 2176, 1536): (29.7, 25.6),
           (4000, 6144, 2048): (112.5, 95.1), (2011, 8192, 4096): (127.4, 100.2), (200, 4096, 4096): (37.4, 51.7), (2011, 2176, 4096): (58.1, 50.9)}


@pytest.mark.parametrize("shape", SHORT_K, ids=str)
def test_bf16_prompts_of_short_k_are_priced_at_the_faster_form(shape):
    from pie_amd import ops

    assert abs(ops.gemm_mfma_us("bf16", *shape, 0, False) / min(SHORT_K[shape]) - 1) < 0.2


# fp8 rows, N, K: microseconds in blocks of 32 rows and of the faster of 64 and 96, none in shares of K
THIN = {(1250, 2048, 4096): (33.6, 36.3), (900, 3072, 2048): (18.6, 21.0), (900, 3072, 4096): (32.8, 37.5), (600, 4096, 4096): (31.5, 35.1),
        (448, 5120, 2048): (17.5, 19.4), (448, 6144, 1024): (12.3, 13.5), (1400, 3072, 1024): (17.4, 16.2), (700, 6144, 1024): (18.3, 16.7)}


@pytest.mark.parametrize("shape", THIN, ids=str)
def test_fp8_prompts_take_blocks_of_32_rows_where_they_are_faster(shape):
    from pie_amd import ops

    thin, others = THIN[shape]
    rows, shares = ops.gemm_rows_plan("fp8", *shape, WORKSPACE)
    assert shares == 1 and (rows == 32) == (thin < others)


# (format, experts, hidden, inner): microseconds of gate|up and down by routes, in passes of 16 and in blocks of 32
FEW_ROUTES = {
    ("fp8", 8, 4096, 14336): {2: (76, 151), 4: (143, 192), 8: (162, 219), 32: (243, 248), 64: (245, 250)},
    ("int8", 8, 4096, 14336): {2: (81, 179), 4: (147, 222), 8: (165, 248), 32: (244, 278), 64: (246, 281)},
    ("fp8", 128, 2048, 768): {8: (21, 18), 16: (24, 21), 32: (39, 31), 128: (83, 75), 256: (110, 102)},
    ("int8", 128, 2048, 768): {8: (25, 22), 16: (27, 25), 32: (43, 33), 128: (84, 79), 256: (109, 106)},
    ("fp8", 16, 4096, 2048): {2: (28, 31), 4: (30, 32), 8: (39, 36), 32: (66, 64), 64: (70, 66)},
    ("int8", 16, 4096, 2048): {2: (32, 38), 4: (33, 39), 8: (45, 41), 32: (67, 67), 64: (70, 67)},
    ("fp8", 32, 1024, 256): {4: (11, 13), 8: (11, 13), 16: (12, 13), 64: (13, 14), 128: (14, 15)},
    ("int8", 32, 1024, 256): {4: (12, 14), 8: (12, 15), 16: (12, 15), 64: (14, 15), 128: (14, 16)},
    ("fp8", 64, 2048, 1024): {8: (21, 19), 16: (27, 25), 32: (44, 35), 128: (71, 66), 256: (80, 74)},
    ("int8", 64, 2048, 1024): {8: (26, 23), 16: (29, 27), 32: (47, 37), 128: (72, 67), 256: (79, 77)},
    ("fp8", 8, 2048, 4096): {2: (21, 35), 4: (28, 36), 8: (30, 40), 32: (42, 46), 64: (43, 45)},
    ("int8", 8, 2048, 4096): {2: (22, 41), 4: (30, 42), 8: (32, 46), 32: (43, 52), 64: (44, 51)},
    ("fp8", 16, 4096, 6400): {2: (41, 79), 4: (66, 86), 8: (104, 114), 32: (199, 192), 64: (209, 198)},
    ("int8", 16, 4096, 6400): {2: (52, 88), 4: (68, 94), 8: (101, 124), 32: (194, 202), 64: (201, 205)},
}


@pytest.mark.parametrize("mixture", FEW_ROUTES, ids=str)
def test_few_routes_per_expert_leave_the_passes_only_where_blocks_are_no_slower(mixture):
    from pie_amd import driver as drv

    kind, experts, hidden, inner = mixture
    for routes, (passes, blocks) in FEW_ROUTES[mixture].items():
        taken = blocks if drv.experts_in_blocks(kind, routes, experts, hidden, inner) else passes
        assert taken <= 1.06 * passes and taken <= 1.3 * blocks, (routes, passes, blocks)


# (rows, N, K): microseconds of int4 weights in the skinny GEMM's passes and in blocks that scale groups in fp32
INT4 = {
    (2, 8192, 8192): (9.9, 11.4), (2, 8192, 1024): (4.1, 6.2), (3, 5120, 8192): (8.2, 10.4), (4, 6144, 14336): (11.9, 14.3),
    (4, 28672, 4096): (18.3, 13.7), (8, 8192, 1024): (4.5, 5.7), (16, 28672, 4096): (19.8, 13.8), (16, 2048, 2048): (5.7, 7.5),
    (17, 3072, 2048): (5.4, 7.4), (24, 4096, 8192): (10.2, 11.7), (32, 28672, 4096): (21.9, 17.4), (40, 2048, 2048): (6.9, 7.8),
    (64, 6144, 4096): (12.3, 12.7), (96, 28672, 4096): (47.4, 34.5),
}
# (rows, N, K): the faster of both and the norm behind it, and in shares of K that meet in the norm's kernel
INT4_SHARES = {
    (16, 4096, 14336): (21.5, 13.0), (64, 4096, 14336): (21.8, 19.5), (64, 4096, 4096): (13.3, 11.8), (96, 8192, 8192): (28.2, 25.1),
    (128, 4096, 8192): (21.9, 19.9), (200, 4096, 4096): (19.8, 20.3), (256, 4096, 4096): (20.1, 21.0), (400, 2048, 2048): (13.6, 15.9),
    (400, 1024, 8192): (20.9, 19.3),
}


@pytest.mark.parametrize("shape", INT4, ids=str)
def test_int4_rows_leave_the_passes_only_for_faster_blocks(shape):
    from pie_amd import driver as drv

    M, N, K = shape
    passes, blocks = INT4[shape]
    forms = drv.linear_forms("int4b8", M, N, K, 128)
    assert not forms["rows"]
    taken = blocks if forms["groups"] else passes
    assert taken <= 1.06 * passes and taken <= 1.15 * blocks


@pytest.mark.parametrize("shape", INT4_SHARES, ids=str)
def test_int4_projections_meet_in_the_norm_where_that_is_no_slower(shape):
    from pie_amd import driver as drv

    M, N, K = shape
    apart, met = INT4_SHARES[shape]
    taken = met if drv.linear_forms("int4b8", M, N, K, 128)["shares"] else apart
    assert taken <= 1.06 * apart and taken <= 1.15 * met


@pytest.mark.parametrize("M", [17, 32, 40, 48])
def test_few_int4_rows_have_one_estimate(M):
    """The wide GEMM runs 17 to 48 rows of int4 weights in the blocks that scale groups in fp32: either way to them costs the same."""
    from pie_amd import driver as drv, ops

    for N, K in ((28672, 4096), (6144, 4096), (4096, 14336), (2048, 2048)):
        for ws in (0, WORKSPACE):
            assert ops.gemm_mfma_us("int4b8", M, N, K, 128, True, ws) == ops.gemm_groups_us(M, N, K, 128, ws)
        if drv.linear_route("int4b8", M, N, K, 128) == "wide":
            assert drv.linear_forms("int4b8", M, N, K, 128)["groups"]


def test_a_measurement_decides_the_forms_of_up_to_128_int4_rows():
    """What the start-up measurement found goes before the estimates, where the form takes the shape at all."""
    from pie_amd import driver as drv

    for M, N, K in ((17, 2048, 2048), (40, 4096, 14336), (128, 4096, 4096)):
        for form in ("groups", "shares"):
            got = [drv.linear_forms("int4b8", M, N, K, 128, **{f"measured_{form}": v})[form] for v in (0, 1)]
            assert got == [False, True], (M, N, K, form)
            assert not drv.linear_forms("int4b8", M, N, K, 64, **{f"measured_{form}": 1})[form]   # (groups of half a step)
    assert not drv.linear_forms("int4b8", 40, 4096, 14336, 128, workspace_bytes=0, measured_shares=1)["shares"]
    assert not drv.linear_forms("int4b8", 40, 16400, 16384, 128, measured_shares=1)["shares"]   # (a row the norm's kernel does not hold)
    for v in (0, 1):   # (more rows are not measured)
        assert drv.linear_forms("int4b8", 129, 4096, 14336, 128, measured_groups=v, measured_shares=v) == drv.linear_forms("int4b8", 129, 4096, 14336, 128)


def test_blocks_of_tile_major_experts_have_the_rows_that_were_asked_for():
    from pie_amd import ops

    assert [ops.moe_block_rows(each * 8, 8) for each in (1, 24, 25, 54, 55, 84, 85, 4000)] == [32, 32, 64, 64, 96, 96, 128, 128]
    assert all(ops.moe_block_rows(each * 8, 8, 128) == 128 for each in (1, 50, 500))
    assert [ops.moe_block_rows(80, 8, rows) for rows in (16, 64, 96, 256)] == [0] * 4
