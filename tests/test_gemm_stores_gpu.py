"""GPU: the stores of the GEMMs' blocks.  Activations and codes are small whole numbers and scales powers of two, so that every sum is exact in
fp32 whatever its order and each epilogue has one right answer, bit for bit.  A y on 16 bytes (and whole pairs of column tiles) takes stores of 16 bytes a
lane, one on 8 bytes those of 8, columns off a pair of tiles the same."""
import numpy as np
import pytest

from gpu_util import dev

pytestmark = pytest.mark.gpu

RULES = dict(limit=7.0, alpha=1.702, shift=1.0)


def exact_problem(gpu, kind, M, N, K, seed):
    """Activations, tile-major weights (bf16: row-major) and the products in fp32."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(seed)
    act = dev(rng.integers(-1, 2, (M, K)).astype(np.float32), gpu).bfloat16()
    codes = rng.integers(-8, 8, (N, K))
    wide = dev(codes.astype(np.float32), gpu)
    row_scale = 2.0 ** -rng.integers(5, 8, N).astype(np.float32)
    if kind == "int4b8":
        packed = sum((codes[:, i::8] + 8).astype(np.uint32) << np.uint32(4 * i) for i in range(8))
        G = 128 if K % 256 else 256
        w = ops.WeightView(kind, dev(packed, gpu), dev(np.repeat(row_scale[:, None], K // G, axis=1), gpu).bfloat16(), G, N, K)
    elif kind == "bf16":
        w = ops.WeightView(kind, (wide * dev(row_scale, gpu)[:, None]).bfloat16(), None, 0, N, K)
    else:
        data = wide.to(torch.int8) if kind == "int8" else wide.to(torch.float8_e4m3fn).view(torch.uint8)
        w = ops.WeightView(kind, data, dev(row_scale, gpu).bfloat16(), 0, N, K)
    sums = (act.double() @ wide.double().T * dev(row_scale, gpu).double()).float()
    return act, w if kind == "bf16" else ops.repack_mfma_tiles(w), sums


def check_stores(gpu, call, sums, seed):
    """call(y, beta, epilogue, rule) fills y [M, N] (gated: [M, N / 2])."""
    import torch
    from pie_amd import ops

    M, N = sums.shape
    g = torch.Generator(device=gpu).manual_seed(seed)
    y0 = torch.randn(M, N, generator=g, device=gpu).bfloat16()
    bias = torch.randint(-8, 9, (N,), generator=g, device=gpu).float() / 4
    gated = {}
    for name, rule, add in (("plain", ops.glu(), 0.0), ("biased", ops.glu(**RULES), bias)):
        gated[name] = ops.glu_f32((sums + add).bfloat16().float().contiguous(), rule).bfloat16()
    gelu = None
    for offset in (0, 4):   # (elements: y on 16 bytes, on 8)
        def run(cols, beta, epilogue, rule=None):
            y = torch.empty(M * cols + 8, device=gpu, dtype=torch.bfloat16)[offset:offset + M * cols].view(M, cols)
            if beta:
                y.copy_(y0)
            else:
                y.fill_(float("nan"))
            assert y.data_ptr() % 16 == 2 * offset
            call(y, beta, epilogue, rule)
            return y

        assert torch.equal(run(N, 0, 0), sums.bfloat16())
        assert torch.equal(run(N, 1, 0), (sums + y0.float()).bfloat16())
        assert torch.equal(run(N, 0, 2), sums.clamp(min=0).square().bfloat16())
        assert torch.equal(run(N // 2, 0, 1), gated["plain"])
        assert torch.equal(run(N // 2, 0, 1, ops.glu(bias=bias, **RULES)), gated["biased"])
        y = run(N, 0, 3)
        assert gelu is None or torch.equal(y, gelu)
        gelu = y
    want = torch.nn.functional.gelu(sums.double())
    # (rounding, and of the sum half of 1.5e-7, the error function's approximation, and what fp32 leaves of its factors)
    assert ((gelu.double() - want).abs() <= 2.0 ** -8 * want.abs() + 4e-7 * sums.double().abs()).all()


@pytest.mark.parametrize("kind", ["int4b8", "int8", "fp8", "bf16"])
@pytest.mark.parametrize("M,N,K,shares", [(129, 32, 256, False), (255, 160, 384, False), (257, 288, 512, False), (300, 16672, 256, False), (600, 23040, 384, False),
                                          (255, 272, 384, False), (160, 4128, 4096, True)])
def test_wide_blocks(gpu, kind, M, N, K, shares):
    """Whole pairs of column tiles, off a block and on one, in one round of blocks and two, and one width off a pair; the last in K shares."""
    import torch
    from pie_amd import ops

    act, w, sums = exact_problem(gpu, kind, M, N, K, 900 + M + N)
    ws = torch.full((8 << 20,), float("nan"), device=gpu) if shares else None
    if shares:
        assert ops.gemm_mfma_us(kind, M, N, K, w.group_size, True, 32 << 20) < ops.gemm_mfma_us(kind, M, N, K, w.group_size, True, 0)
    check_stores(gpu, lambda y, beta, epilogue, rule: ops.gemm_mfma_tiled(act, w, y=y, beta=beta, epilogue=epilogue, rule=rule, workspace=ws), sums, 900 + M)


# (rows, N, K, rows of a block, shares of K): each height by itself and in shares whose last is the shortest, columns on a pair of tiles and off
# one, step counts that leave one to three of those in flight
GROUPS = [(15, 144, 640, 16, 1), (16, 160, 896, 16, 1), (30, 16432, 384, 32, 1), (23, 16416, 640, 32, 1), (45, 16432, 256, 48, 1), (47, 16416, 896, 48, 1),
          (61, 16432, 384, 64, 1), (61, 16416, 384, 64, 1), (12, 48, 2176, 16, 6), (24, 4112, 2944, 32, 6), (33, 4112, 2944, 48, 6), (49, 4112, 4480, 64, 7)]


@pytest.mark.parametrize("M,N,K,rows,shares", GROUPS)
def test_blocks_that_scale_groups_in_fp32(gpu, M, N, K, rows, shares):
    import torch
    from pie_amd import ops

    ws = torch.full((4 << 20,), float("nan"), device=gpu) if shares > 1 else None
    assert ops.gemm_groups_plan(M, N, K, 128, 0 if ws is None else ws.numel() * 4) == (rows, shares)
    act, w, sums = exact_problem(gpu, "int4b8", M, N, K, 920 + M + N)
    if w.group_size != 128:
        assert ops.gemm_groups_plan(M, N, K, w.group_size, 0 if ws is None else ws.numel() * 4) == (rows, shares)
    check_stores(gpu, lambda y, beta, epilogue, rule: ops.gemm_groups_tiled(act, w, y=y, beta=beta, epilogue=epilogue, rule=rule, workspace=ws), sums, 920 + M)


# (as above, of one-byte weights by format)
ROWS = {"int8": [(33, 16, 320, 32, 1), (33, 1056, 320, 32, 1), (300, 8208, 320, 64, 1), (300, 8224, 320, 64, 1), (1300, 2064, 320, 96, 1), (1300, 2080, 320, 96, 1),
                 (1100, 6160, 1088, 128, 1), (1100, 6176, 1088, 128, 1), (33, 16, 1088, 32, 5), (1100, 528, 3136, 64, 5), (1300, 272, 4160, 96, 6),
                 (200, 6160, 6208, 128, 5)],
        "fp8": [(33, 16, 320, 32, 1), (33, 1056, 320, 32, 1), (900, 4112, 448, 64, 1), (900, 4128, 448, 64, 1), (1300, 4112, 1088, 96, 1), (1300, 4128, 1088, 96, 1),
                (1100, 6160, 1088, 128, 1), (1100, 6176, 1088, 128, 1), (33, 16, 1088, 32, 5), (900, 1040, 4160, 64, 3), (1300, 1040, 6208, 96, 4),
                (200, 6160, 8256, 128, 5)]}


@pytest.mark.parametrize("kind,M,N,K,rows,shares", [(kind, *case) for kind in ROWS for case in ROWS[kind]])
def test_blocks_of_one_byte_rows(gpu, kind, M, N, K, rows, shares):
    import torch
    from pie_amd import ops

    ws = torch.full((6 << 20,), float("nan"), device=gpu) if shares > 1 else None
    assert ops.gemm_rows_plan(kind, M, N, K, 0 if ws is None else ws.numel() * 4) == (rows, shares)
    act, w, sums = exact_problem(gpu, kind, M, N, K, 940 + M + N)
    check_stores(gpu, lambda y, beta, epilogue, rule: ops.gemm_rows_tiled(act, w, y=y, beta=beta, epilogue=epilogue, rule=rule, workspace=ws), sums, 940 + M)


# (format, rows, N, K, rows and columns of a block, shares of K): rows and columns off a block, steps that do not divide by the waves, one share and several
WAVES = [(kind, *case) for kind, cases in {
    "int4b8": [(15, 48, 384, 16, 16, 1), (5, 16, 8320, 16, 16, 5), (17, 4112, 1152, 32, 32, 1), (33, 12304, 1152, 48, 64, 1), (300, 16, 2176, 64, 32, 3), (97, 6160, 1152, 64, 64, 1)],
    "int8": [(15, 48, 192, 16, 16, 1), (17, 528, 4160, 16, 32, 5), (32, 8208, 576, 32, 64, 1), (230, 16, 4160, 48, 32, 5), (65, 12304, 576, 80, 64, 1)],
    "fp8": [(16, 4112, 576, 16, 32, 1), (97, 16, 4160, 32, 16, 5), (33, 12304, 576, 48, 64, 1), (300, 16, 2112, 64, 32, 5)],
    "bf16": [(15, 48, 192, 16, 16, 1), (33, 272, 8256, 16, 32, 6), (97, 2064, 576, 32, 64, 1), (65, 2064, 8256, 80, 64, 6)],
    "bf16 rows": [(15, 48, 192, 16, 16, 1), (97, 16, 4160, 32, 16, 5), (130, 4112, 576, 48, 64, 1), (300, 272, 8256, 80, 32, 6)]}.items() for case in cases]


@pytest.mark.parametrize("kind,M,N,K,rows,cols,shares", WAVES)
def test_blocks_whose_waves_take_the_steps_of_k_in_turn(gpu, kind, M, N, K, rows, cols, shares):
    """And a y on two bytes, with the residual and the gated rules."""
    import torch
    from pie_amd import ops

    kind, tiled = kind.split()[0], not kind.endswith("rows")
    ws = torch.full((4 << 20,), float("nan"), device=gpu) if shares > 1 else None
    act, w, sums = exact_problem(gpu, kind, M, N, K, 1000 + M + N)
    assert ops.gemm_waves_plan(kind, M, N, K, w.group_size, 0 if ws is None else ws.numel() * 4, tiled=tiled) == (rows, cols, shares)
    if kind == "bf16" and tiled:
        w = ops.repack_mfma_tiles(w)

    def call(y, beta, epilogue, rule):
        return ops.gemm_waves_tiled(act, w, y=y, beta=beta, epilogue=epilogue, rule=rule, workspace=ws)

    check_stores(gpu, call, sums, 1000 + M)
    g = torch.Generator(device=gpu).manual_seed(1000 + M)
    y0 = torch.randn(M, N, generator=g, device=gpu).bfloat16()
    bias = torch.randint(-8, 9, (N,), generator=g, device=gpu).float() / 4
    off = lambda cols: torch.empty(M * cols + 1, device=gpu, dtype=torch.bfloat16)[1:].view(M, cols)  # noqa: E731
    assert off(N).data_ptr() % 4 == 2
    assert torch.equal(call(off(N), 0, 0, None), sums.bfloat16())
    assert torch.equal(call(off(N).copy_(y0), 1, 0, None), (sums + y0.float()).bfloat16())
    for rule, add in ((ops.glu(), 0.0), (ops.glu(bias=bias, **RULES), bias)):
        plain = ops.glu(**RULES) if torch.is_tensor(add) else ops.glu()
        assert torch.equal(call(off(N // 2), 0, 1, rule), ops.glu_f32((sums + add).bfloat16().float().contiguous(), plain).bfloat16())


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("height,counts", [(32, [0, 1, 31, 33, 7]), (64, [63, 65, 0, 30]), (96, [95, 97, 1, 100]), (128, [127, 129, 1, 257])])
@pytest.mark.parametrize("N", [288, 272])
def test_blocks_of_routes(gpu, kind, height, counts, N):
    """Every height of a block over whole pairs of column tiles and off one; gathered rows."""
    import torch
    from pie_amd import ops

    E, routes, T, K = len(counts), sum(counts), 70, 320
    assert ops.moe_block_rows(routes, E) == height
    rng = np.random.default_rng(960 + height)
    rows = dev(rng.integers(0, T, routes).astype(np.int32), gpu)
    offs = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), gpu)
    act, w, every = exact_problem(gpu, kind, T, E * N, K, 960 + height)
    sums = torch.cat([every[rows[offs[e]:offs[e + 1]].long(), e * N:(e + 1) * N] for e in range(E)])
    data, scale = w.data.reshape(E, N, K), w.scale.reshape(E, N)
    for offset in (0, 4):
        def run(cols, epilogue):
            y = torch.full((routes * cols + 8,), float("nan"), device=gpu, dtype=torch.bfloat16)[offset:offset + routes * cols].view(routes, cols)
            return ops.moe_grouped_gemm(act, rows, offs, kind, data, scale, N, K, 257, 0, epilogue == 1, y=y, block_rows=0, tiled=True)

        assert torch.equal(run(N, 0), sums.bfloat16())
        assert torch.equal(run(N // 2, 1), ops.glu_f32(sums.bfloat16().float().contiguous(), ops.glu()).bfloat16())


@pytest.mark.parametrize("kind", ["int4b8", "fp8", "bf16"])
def test_sums_that_are_no_numbers(gpu, kind):
    """A NaN is the limit as a gate and minus the limit as a factor; infinities are clamped; both kinds of stores agree."""
    import torch
    from pie_amd import ops

    M, N, K = 257, 288, 512
    act, w, sums = exact_problem(gpu, kind, M, N, K, 980)
    act, sums = act.clone(), sums.clone()
    act[3], act[200, 5], act[130] = float("nan"), float("nan"), 3e38   # (the last: sums past the range of bf16, or of fp32)
    sums[3] = sums[200] = float("nan")
    for rule, gate, up in ((ops.glu(), float("inf"), float("-inf")), (ops.glu(**RULES), 7.0, -7.0)):
        got = []
        for offset in (0, 4):
            y = torch.empty(M * N // 2 + 8, device=gpu, dtype=torch.bfloat16)[offset:offset + M * N // 2].view(M, N // 2)
            got.append(ops.gemm_mfma_tiled(act, w, y=y, epilogue=1, rule=rule).clone())
        assert torch.equal(got[0].isnan(), got[1].isnan()) and torch.equal(got[0].nan_to_num(), got[1].nan_to_num())
        pair = torch.tensor([[gate, up]], device=gpu)
        want = ops.glu_f32(pair, rule).bfloat16()
        assert torch.equal(got[0][3], want.expand(1, N // 2)[0]) and torch.equal(got[0][200], want.expand(1, N // 2)[0])
        rest = [r for r in range(M) if r not in (3, 130, 200)]
        assert torch.equal(got[0][rest], ops.glu_f32(sums[rest].bfloat16().float().contiguous(), rule).bfloat16())
