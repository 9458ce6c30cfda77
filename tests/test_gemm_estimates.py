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
    low, wide = SHORT_K[shape]
    assert (wide if ops.gemm_bf16_wide(*shape) else low) <= 1.05 * min(low, wide)


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


# (format, rows, N, K): microseconds in the skinny GEMM's passes, in blocks whose waves take the steps of K in turn, and in what else takes the shape (int4 blocks that scale groups,
# one-byte blocks of 32 to 128 rows, the wide GEMM, the tiled GEMM and its shares of K); "rows" behind a format: row-major.
FORMS = {
    ("int8", 8, 9216, 3584): dict(passes=13.6, waves=11.6),
    ("int8", 20, 2048, 2048): dict(passes=5.9, waves=5.3, wide=11.8, tiled=20.7, shares=12.0),
    ("int8", 40, 5120, 5120): dict(passes=17.6, waves=12.0, wide=24.6, tiled=44.0, shares=25.7),
    ("int8", 72, 14336, 1024): dict(passes=17.1, waves=10.8, rows=11.6, wide=11.7, tiled=17.7, shares=23.2),
    ("int8", 112, 16384, 2048): dict(passes=26.2, waves=21.9, rows=19.6, wide=20.1, tiled=27.1),
    ("int8", 128, 28672, 4096): dict(passes=70.2, waves=60.0, rows=42.4, wide=62.4, tiled=49.3),
    ("int8", 160, 2560, 7168): dict(passes=21.1, waves=17.3, rows=21.2, wide=26.9, tiled=73.0),
    ("int8", 192, 8192, 512): dict(passes=13.7, waves=9.8, rows=8.0, wide=13.8, tiled=13.2),
    ("int8", 192, 10240, 2560): dict(passes=28.9, waves=24.9, rows=23.4, wide=28.9, tiled=31.9),
    ("int8", 320, 5120, 5120): dict(passes=43.5, waves=35.9, rows=33.2, wide=38.3, tiled=54.1),
    ("fp8", 12, 9216, 3584): dict(passes=13.9, waves=12.0),
    ("fp8", 17, 2048, 8192): dict(passes=8.6, waves=9.8, wide=23.2, tiled=56.5, shares=16.0),
    ("fp8", 24, 4096, 4096): dict(passes=8.7, waves=8.2, wide=14.3, tiled=31.7, shares=20.1),
    ("fp8", 56, 28672, 4096): dict(passes=40.1, waves=34.8, wide=33.7, tiled=36.4, shares=49.8),
    ("fp8", 80, 5120, 5120): dict(passes=16.6, waves=13.9, rows=18.1, wide=31.2, tiled=50.6, shares=30.6),
    ("fp8", 128, 16384, 2048): dict(passes=24.5, waves=21.6, rows=17.4, wide=20.4, tiled=26.0),
    ("fp8", 144, 6144, 4096): dict(passes=21.4, waves=18.6, rows=20.7, wide=26.3, tiled=40.0),
    ("fp8", 240, 2048, 2048): dict(passes=10.2, waves=7.9, rows=13.8, wide=21.5, tiled=24.0),
    ("fp8", 304, 9216, 3584): dict(passes=53.2, waves=39.8, rows=33.7, wide=49.5, tiled=37.7),
    ("fp8", 448, 3072, 2048): dict(passes=19.6, waves=19.8, rows=13.7, wide=24.7, tiled=23.9),
    ("int4b8", 6, 4096, 14336): dict(passes=12.6, waves=12.1, groups=13.1),
    ("int4b8", 12, 1536, 8960): dict(waves=8.6, groups=10.4),   # (the passes refuse parts of a step of K)
    ("int4b8", 24, 1536, 8960): dict(waves=9.5, groups=11.0, wide=11.0, tiled=77.8, shares=16.8),
    ("int4b8", 16, 6144, 4096): dict(passes=8.2, waves=7.3, groups=9.7),
    ("int4b8", 28, 9216, 3584): dict(passes=13.5, waves=10.8, groups=11.6, wide=11.7, tiled=33.8, shares=26.8),
    ("int4b8", 36, 14336, 1024): dict(passes=9.6, waves=7.9, groups=7.0, wide=7.0, tiled=14.0, shares=16.9),
    ("int4b8", 80, 6144, 2048): dict(passes=12.0, waves=9.1, groups=8.1, wide=19.9, tiled=26.8, shares=25.0),
    ("int4b8", 96, 4096, 4096): dict(passes=11.9, waves=10.2, groups=12.5, wide=23.9, tiled=47.8, shares=28.8),
    ("int4b8", 112, 6144, 2048): dict(passes=12.2, waves=11.4, groups=10.0, wide=21.8, tiled=27.4, shares=29.2),
    ("int4b8", 128, 3072, 2048): dict(passes=8.7, waves=7.4, groups=7.8, wide=19.0, tiled=27.7, shares=18.7),
    ("int4b8", 192, 5120, 5120): dict(passes=21.2, waves=18.5, groups=19.7, wide=28.4, tiled=59.1),
    ("int4b8", 256, 2048, 2048): dict(passes=8.5, waves=7.3, groups=7.7, wide=20.3, tiled=26.8),
    ("bf16", 8, 16384, 2048): dict(passes=18.0, waves=15.5),
    ("bf16", 16, 2048, 2048): dict(passes=6.7, waves=5.9),
    ("bf16", 40, 5120, 5120): dict(passes=23.6, waves=20.5, tiled=42.9, shares=24.5),
    ("bf16", 72, 2560, 7168): dict(passes=17.7, waves=15.8, tiled=61.2, shares=25.0),
    ("bf16", 112, 9216, 3584): dict(passes=45.8, waves=31.4, tiled=39.5),
    ("bf16", 136, 16384, 2048): dict(passes=50.9, waves=31.1, tiled=24.8),
    ("bf16", 144, 9216, 3584): dict(passes=45.1, waves=32.5, tiled=28.6),
    ("bf16", 160, 14336, 1024): dict(passes=31.1, waves=19.3, tiled=16.0),
    ("bf16", 192, 4096, 4096): dict(passes=28.4, waves=18.3, tiled=23.5),
    ("bf16", 256, 2560, 7168): dict(passes=42.2, waves=26.2, tiled=28.9),
    ("bf16", 384, 4096, 4096): dict(passes=46.1, waves=32.1, tiled=29.0),
    ("bf16", 448, 2048, 8192): dict(passes=45.5, waves=34.6, tiled=30.6),
    ("bf16 rows", 10, 128, 2048): dict(passes=6.8, waves=4.2),
    ("bf16 rows", 16, 32000, 4096): dict(passes=53.1, waves=47.8),
    ("bf16 rows", 24, 48000, 2048): dict(passes=71.5, waves=43.3, tiled=48.3, shares=49.7),
    ("bf16 rows", 40, 32000, 4096): dict(passes=124.4, waves=52.8, tiled=61.8, shares=67.1),
    ("bf16 rows", 96, 512, 4096): dict(passes=10.6, waves=7.6, tiled=38.0, shares=14.6),
    ("bf16 rows", 128, 5120, 5120): dict(passes=66.1, waves=24.9, tiled=58.3),
    ("bf16 rows", 192, 384, 4096): dict(passes=15.9, waves=8.5, tiled=17.4),
    ("bf16 rows", 288, 2048, 2048): dict(passes=29.9, waves=10.5, tiled=20.7),
    ("bf16 rows", 136, 16384, 2048): dict(passes=83.5, waves=31.5, tiled=25.0),
    ("bf16 rows", 288, 8192, 512): dict(passes=46.6, waves=14.4, tiled=11.2),
    ("bf16 rows", 288, 2048, 8192): dict(passes=96.1, waves=26.0, tiled=29.7),
    ("bf16 rows", 352, 4096, 512): dict(passes=30.0, waves=12.2, tiled=11.2),
    ("bf16 rows", 448, 4096, 512): dict(passes=38.4, waves=13.7, tiled=11.0),
    ("bf16 rows", 224, 6144, 1536): dict(passes=51.7, waves=18.4, tiled=20.4),
    ("bf16 rows", 480, 128, 2048): dict(passes=7.1, waves=8.0, tiled=15.5),
}
# (matrices that no estimate was fitted to: over 4030 points of 42 matrices the form taken is 1.01 - 1.03 of the fastest on average by format, 157 are more than a tenth over)
NOT_FITTED = {(1536, 8960), (5120, 5120), (9216, 3584), (2560, 7168), (6144, 2048), (10240, 2560), (48000, 2048), (8192, 512), (512, 4096), (384, 4096), (128, 2048)}


@pytest.mark.parametrize("shape", FORMS, ids=str)
def test_few_rows_take_a_form_near_the_fastest(shape):
    from pie_amd import driver as drv

    kind, M, N, K = shape
    kind, tiled, group = kind.split()[0], not kind.endswith("rows"), 128 if kind == "int4b8" else 0
    route, forms = drv.linear_route(kind, M, N, K, group, tile_major=tiled), drv.linear_forms(kind, M, N, K, group, tile_major=tiled)
    taken = {"skinny": "waves" if forms["waves"] else "groups" if forms["groups"] else "passes", "wide": "rows" if forms["rows"] and M > 64 else "wide",
             "tiled": "tiled", "tiled in shares": "shares"}[route]
    us = FORMS[shape]
    assert us[taken] <= (1.26 if (N, K) in NOT_FITTED else 1.12) * min(us.values()), taken


# (format, rows, N, K): the fastest product with the norm behind it, and in shares of K that meet in the norm's kernel
NORM_SHARES = {
    ("int8", 16, 2048, 8192): (12.4, 9.4),
    ("int8", 24, 4096, 14336): (20.7, 17.7),
    ("int8", 40, 2048, 2048): (8.2, 8.0),
    ("int8", 64, 5120, 5120): (19.3, 16.5),
    ("int8", 96, 4096, 4096): (14.7, 14.6),
    ("int8", 128, 2048, 8192): (17.4, 15.7),
    ("int8", 256, 4096, 14336): (46.2, 50.7),
    ("fp8", 12, 4096, 4096): (11.4, 9.3),
    ("fp8", 40, 2560, 7168): (15.0, 12.2),
    ("fp8", 64, 2048, 2048): (8.0, 7.9),
    ("fp8", 80, 4096, 14336): (28.7, 25.6),
    ("fp8", 128, 5120, 5120): (21.4, 24.4),
    ("fp8", 192, 2048, 8192): (20.9, 17.4),
    ("bf16", 8, 4096, 14336): (27.3, 26.2),
    ("bf16", 24, 2048, 2048): (8.5, 7.9),
    ("bf16", 40, 5120, 5120): (24.2, 18.7),
    ("bf16", 64, 4096, 4096): (16.1, 14.7),
    ("bf16", 96, 2048, 8192): (19.5, 16.6),
    ("bf16", 128, 2560, 7168): (23.6, 19.7),
}


@pytest.mark.parametrize("shape", NORM_SHARES, ids=str)
def test_projections_meet_in_the_norm_where_that_is_no_slower(shape):
    from pie_amd import driver as drv

    apart, met = NORM_SHARES[shape]
    taken = met if drv.linear_forms(*shape)["shares"] else apart
    assert taken <= 1.1 * min(apart, met)


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


LADDER = (2, 3, 4, 17, 24, 32, 33, 40, 48, 56, 64, 65, 72, 80, 88, 96, 97, 104, 112, 120, 128)   # (row counts of the start-up measurement)


@pytest.mark.parametrize("kind", ["int4b8", "int8", "fp8", "bf16"])
def test_a_start_measures_the_two_forms_that_it_names(kind):
    """Where a start times a pair of forms, each setting runs a form of its own, none of them blocks whose waves take the steps of K in turn: those are by
    estimate alone, so that two starts of one driver run the same ones."""
    from pie_amd import driver as drv

    group, pairs = 128 if kind == "int4b8" else 0, {"groups": 0, "shares": 0}
    for N, K in ((6144, 4096), (28672, 4096), (4096, 4096), (4096, 14336), (3072, 2048), (2048, 2048), (16384, 2048), (2048, 8192), (14336, 2048), (8192, 8192)):
        for M in LADDER:
            for name, timed in drv.measured_forms(kind, M, N, K, group).items():
                if not timed:
                    continue
                pairs[name] += 1
                got = [drv.linear_forms(kind, M, N, K, group, **{f"measured_{name}": v}) for v in (0, 1)]
                assert [f[name] for f in got] == [False, True] and not any(f["waves"] for f in got), (name, M, N, K)
    assert (pairs["groups"] > 0) == (kind == "int4b8")
    assert kind == "int4b8" or pairs["shares"] == 0


def test_blocks_of_tile_major_experts_have_the_rows_that_were_asked_for():
    from pie_amd import ops

    assert [ops.moe_block_rows(each * 8, 8) for each in (1, 24, 25, 54, 55, 84, 85, 4000)] == [32, 32, 64, 64, 96, 96, 128, 128]
    assert all(ops.moe_block_rows(each * 8, 8, 128) == 128 for each in (1, 50, 500))
    assert [ops.moe_block_rows(80, 8, rows) for rows in (16, 64, 96, 256)] == [0] * 4


# (format, activation rows, N, K, pairs): microseconds of a GEMV with four weight rows a step and two waves a SIMD, with two and two, and with two and four
GEMV_ROWS = {
    ('int4b8', 1, 8192, 4096, 0): (7.2, 6.4, 7.2), ('int4b8', 1, 9216, 4096, 0): (9.4, 7.8, 8.4), ('int4b8', 1, 12288, 2048, 0): (7.0, 6.2, 7.0),
    ('int4b8', 1, 14336, 14336, 0): (21.6, 24.7, 22.1), ('int4b8', 1, 14336, 4096, 1): (9.8, 9.5, 9.8), ('int4b8', 2, 14336, 11008, 0): (24.5, 27.2, 24.4),
    ('int4b8', 4, 14336, 18944, 0): (117.8, 127.0, 112.9), ('int4b8', 1, 17408, 4096, 0): (11.8, 10.6, 10.0), ('int4b8', 1, 28672, 4096, 1): (14.4, 14.2, 13.2),
    ('int4b8', 1, 32000, 512, 0): (8.5, 9.5, 8.5), ('int4b8', 2, 32768, 1024, 0): (11.7, 12.4, 11.5), ('int4b8', 4, 43008, 2048, 0): (25.9, 24.8, 22.3),
    ('int4b8', 1, 65536, 2048, 0): (15.4, 16.5, 14.6), ('int4b8', 1, 128256, 2048, 0): (26.1, 29.5, 25.5), ('int8', 1, 8192, 2048, 0): (6.3, 5.8, 6.6),
    ('int8', 1, 12288, 4096, 0): (13.1, 11.2, 11.9), ('int8', 1, 14336, 14336, 0): (35.5, 38.1, 35.0), ('int8', 1, 16384, 4096, 0): (15.9, 13.6, 15.4),
    ('int8', 1, 22016, 1536, 0): (9.4, 9.9, 9.2), ('int8', 1, 28672, 512, 0): (7.2, 7.8, 7.2), ('int8', 1, 28672, 4096, 0): (23.7, 21.7, 22.1),
    ('int8', 1, 32000, 512, 0): (7.5, 8.2, 7.3), ('int8', 2, 14336, 4096, 0): (15.4, 16.0, 14.5), ('int8', 2, 14336, 7168, 1): (22.8, 24.4, 22.4),
    ('int8', 2, 28672, 4096, 1): (27.1, 26.4, 23.3), ('int8', 4, 32000, 2048, 0): (20.1, 22.2, 17.7),
    ('fp8', 1, 9216, 2048, 0): (7.6, 6.8, 7.1), ('fp8', 1, 14336, 14336, 0): (34.9, 36.9, 34.2), ('fp8', 1, 32000, 512, 0): (7.2, 8.0, 7.1),
    ('fp8', 2, 14336, 4096, 0): (15.0, 14.8, 13.7), ('fp8', 2, 22016, 4096, 1): (20.9, 21.2, 19.4), ('bf16', 1, 8192, 2048, 0): (9.2, 8.8, 9.2),
    ('bf16', 1, 12288, 4096, 0): (19.4, 18.0, 18.8), ('bf16', 1, 13312, 3072, 0): (15.5, 16.2, 15.3), ('bf16', 1, 14336, 4096, 0): (21.0, 21.3, 22.8),
    ('bf16', 1, 15360, 7168, 0): (34.7, 35.3, 35.0), ('bf16', 1, 20480, 2048, 0): (17.3, 16.0, 16.1), ('bf16', 1, 32000, 1024, 0): (13.1, 13.9, 12.8),
    ('bf16', 1, 32768, 1024, 0): (13.5, 15.0, 13.0), ('bf16', 1, 16384, 8192, 0): (47.9, 49.9, 61.5), ('bf16', 2, 16384, 4096, 0): (26.1, 24.9, 27.0),
    ('bf16', 2, 28672, 4096, 0): (40.0, 37.2, 39.5), ('bf16', 4, 14336, 2048, 0): (14.9, 14.6, 13.9),
    ('bf16', 1, 16384, 2048, 1): (14.4, 13.4, 14.4), ('bf16', 2, 14336, 512, 1): (7.3, 6.6, 7.0), ('bf16', 1, 22016, 3072, 1): (22.8, 23.7, 22.9),
    ('int4b8', 1, 17408, 512, 0): (7.2, 7.2, 6.7), ('int4b8', 1, 51200, 1024, 0): (12.0, 13.5, 11.1), ('int8', 1, 22016, 4096, 1): (18.8, 18.0, 18.3),
    ('fp8', 1, 24576, 4096, 0): (20.0, 19.0, 18.6),
}


@pytest.mark.parametrize("shape", GEMV_ROWS, ids=str)
def test_gemvs_leave_four_rows_a_step_only_for_a_faster_form(shape):
    from pie_amd import ops

    forms = dict(zip(((4, 2), (2, 2), (2, 4)), GEMV_ROWS[shape]))
    taken = forms[ops.gemv_plan(*shape)]
    assert taken <= 1.04 * forms[4, 2] and taken <= 1.1 * min(forms.values())


def test_the_plan_of_a_gemv_is_by_the_rows_of_a_pass():
    """Rows too long for several activation rows in one pass are planned as one; pairs are walked two or four at a time."""
    from pie_amd import ops

    assert ops.gemv_plan("int8", 4, 28672, 14336) == ops.gemv_plan("int8", 1, 28672, 14336) == (2, 2)
    assert ops.gemv_plan("int8", 4, 28672, 4096) == (2, 4)
    for kind in ("int4b8", "int8", "fp8", "bf16"):
        for N in (2, 62, 2048, 4100, 6144, 6146, 8192, 14336, 28672, 70000):
            assert ops.gemv_plan(kind, 1, N, 4096, True)[0] in (2, 4)
            assert ops.gemv_plan(kind, 2, N, 4096)[0] in (1, 2, 3, 4)
