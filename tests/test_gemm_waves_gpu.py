"""GPU parity: weights in blocks whose waves take the steps of K in turn, against the exact sums in 64 bits and the kernels whose
epilogues they share."""
import numpy as np
import pytest

from gpu_util import bits, dev

WORKSPACE = 32 << 20
# activation rows, N, K -> rows and columns of a block, whether in shares of K (each block that is instantiated; columns off a block, steps that do not divide by
# the waves, fewer steps than waves, rows off a block)
ONE_BYTE = {(5, 16, 576): (16, 16, False), (15, 48, 192): (16, 16, False), (5, 16, 4160): (16, 16, True), (16, 4112, 576): (16, 32, False), (17, 528, 4160): (16, 32, True),
            (5, 8208, 1088): (16, 64, False), (97, 16, 576): (32, 16, False), (97, 16, 4160): (32, 16, True), (17, 4112, 576): (32, 32, False), (32, 8208, 576): (32, 64, False),
            (230, 16, 576): (48, 32, False), (230, 16, 4160): (48, 32, True), (33, 12304, 576): (48, 64, False), (300, 16, 576): (64, 32, False),
            (300, 16, 2112): (64, 32, True), (300, 2064, 576): (64, 64, False), (65, 12304, 576): (80, 64, False), (5, 1024, 64): (16, 16, False)}
INT4 = {(5, 16, 1152): (16, 16, False), (15, 48, 384): (16, 16, False), (5, 16, 8320): (16, 16, True), (16, 4112, 1152): (16, 32, False), (5, 1040, 8320): (16, 32, True),
        (5, 8208, 1152): (16, 64, False), (97, 16, 1152): (32, 16, False), (17, 4112, 1152): (32, 32, False), (161, 144, 4224): (32, 32, True), (32, 8208, 1152): (32, 64, False),
        (230, 16, 1152): (48, 32, False), (230, 16, 3200): (48, 32, True), (33, 12304, 1152): (48, 64, False), (300, 16, 1152): (64, 32, False),
        (300, 16, 2176): (64, 32, True), (97, 6160, 1152): (64, 64, False), (97, 2064, 8320): (64, 64, True), (5, 1024, 128): (16, 16, False)}
BF16 = {(5, 16, 576): (16, 16, False), (15, 48, 192): (16, 16, False), (5, 16, 4160): (16, 16, True), (65, 1040, 576): (16, 32, False), (33, 272, 8256): (16, 32, True),
        (33, 4112, 576): (16, 64, False), (97, 16, 576): (32, 16, False), (97, 16, 4160): (32, 16, True), (97, 1040, 576): (32, 32, False), (97, 2064, 576): (32, 64, False),
        (230, 16, 576): (48, 32, False), (230, 16, 2112): (48, 32, True), (230, 2064, 576): (48, 64, False), (300, 16, 576): (64, 32, False), (300, 16, 2112): (64, 32, True),
        (300, 2064, 576): (64, 64, False), (230, 2064, 1088): (80, 32, False), (230, 4112, 1088): (80, 64, False), (65, 2064, 8256): (80, 64, True), (5, 1024, 64): (16, 16, False)}
BF16_ROWS = {(5, 16, 576): (16, 16, False), (15, 48, 192): (16, 16, False), (5, 16, 4160): (16, 16, True), (65, 1040, 576): (16, 32, False), (17, 528, 8256): (16, 32, True),
             (33, 4112, 576): (16, 64, False), (97, 16, 576): (32, 16, False), (97, 16, 4160): (32, 16, True), (97, 1040, 576): (32, 32, False), (97, 2064, 576): (32, 64, False),
             (17, 2064, 8256): (32, 64, True), (230, 16, 576): (48, 32, False), (230, 16, 2112): (48, 32, True), (130, 4112, 576): (48, 64, False), (300, 16, 576): (64, 32, False),
             (300, 16, 2112): (64, 32, True), (300, 2064, 576): (64, 64, False), (230, 2064, 576): (80, 32, False), (300, 272, 8256): (80, 32, True),
             (230, 4112, 576): (80, 64, False), (65, 2064, 8256): (80, 64, True), (5, 1024, 64): (16, 16, False)}
TABLES = {"int8": ONE_BYTE, "fp8": ONE_BYTE, "int4b8": INT4, "bf16": BF16, "bf16 rows": BF16_ROWS}
CASES = [(kind, *shape) for kind, table in TABLES.items() for shape in table]


def stored(w, kind="bf16"):
    """The weight in the order the kernel reads: the tile-major copy, or as it is."""
    from pie_amd import ops

    return w if kind == "bf16 rows" else ops.repack_mfma_tiles(w)


def weight_and_sums(kind, M, N, K, seed, gpu, group=128, scale_type=None):
    """Activations with a mean (int4 codes' offset then has something to cancel), the weight, exact sums and what fp32 sums of their terms may be off."""
    import torch
    from pie_amd import ops

    g = torch.Generator(device=gpu).manual_seed(seed)
    act = (torch.randn(M, K, generator=g, device=gpu) + 0.25).to(torch.bfloat16)
    x = act.double()
    if kind == "int4b8":
        data = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 8), generator=g, device=gpu, dtype=torch.int32)
        scale = (0.002 + 0.006 * torch.rand(N, K // group, generator=g, device=gpu)).to(torch.bfloat16)
        codes = torch.stack([(data >> (4 * i)) & 0xF for i in range(8)], dim=-1).reshape(N, K).double() - 8.0
        s = scale.double().repeat_interleave(group, dim=1)
        w, size = codes * s, (codes.abs() + 272.0) * s
        view = ops.WeightView("int4b8", data, scale, group, N, K)
    elif kind.startswith("bf16"):
        data = (0.03 * torch.randn(N, K, generator=g, device=gpu)).to(torch.bfloat16)
        w = data.double()
        size = w.abs()
        view = ops.WeightView("bf16", data, None, 0, N, K)
    else:
        scale = (0.0005 + 0.001 * torch.rand(N, generator=g, device=gpu)).to(scale_type or torch.bfloat16)
        if kind == "int8":
            data = torch.randint(-127, 128, (N, K), generator=g, device=gpu, dtype=torch.int8)
            codes = data.double()
        else:
            data = (32 * torch.randn(N, K, generator=g, device=gpu)).to(torch.float8_e4m3fn)
            codes, data = data.double(), data.view(torch.uint8)
        w = codes * scale.double()[:, None]
        size = w.abs()
        view = ops.WeightView(kind, data, scale, 0, N, K)
    return act, view, x @ w.T, K * 2.0 ** -23 * (x.abs() @ size.T)


@pytest.mark.parametrize("kind,M,N,K", CASES, ids=str)
def test_each_block_is_planned_where_it_is_tested(kind, M, N, K):
    from pie_amd import ops

    rows, cols, shared = TABLES[kind][M, N, K]
    kind, tiled = kind.split()[0], not kind.endswith("rows")
    got = ops.gemm_waves_plan(kind, M, N, K, 128, WORKSPACE, tiled=tiled)
    assert got[:2] == (rows, cols) and (got[2] > 1) == shared
    assert ops.gemm_waves_plan(kind, M, N, K, 128, 0, tiled=tiled)[2] == 1   # (no workspace: whole sums)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,N,K", CASES, ids=str)
def test_rows_in_blocks_of_waves(gpu, kind, M, N, K):
    """Plain, onto a residual and as gated pairs, with and without shares of K; bf16 and fp32 row scales."""
    import torch
    from pie_amd import ops

    for scale_type in (torch.bfloat16, torch.float32) if kind in ("int8", "fp8") else (torch.bfloat16,):
        act, w, ref, bound = weight_and_sums(kind, M, N, K, 910 + M, gpu, scale_type=scale_type)
        t = stored(w, kind)
        for work in (None, torch.full((WORKSPACE // 4,), float("nan"), device=gpu)):
            got = ops.gemm_waves_tiled(act, t, workspace=work).double()
            assert torch.isfinite(got).all() and ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
            y0 = torch.randn(M, N, device=gpu).to(torch.bfloat16)
            got = ops.gemm_waves_tiled(act, t, y=y0.clone(), beta=1, workspace=work).double()
            assert ((got - ref - y0.double()).abs() <= 2.0 ** -8 * (ref + y0.double()).abs() + 2 * bound).all()
            pairs = ops.gemm_waves_tiled(act, t, workspace=work)
            assert torch.equal(ops.gemm_waves_tiled(act, t, epilogue=1, workspace=work),
                               ops.swiglu_bf16(torch.cat([pairs[:, 0::2], pairs[:, 1::2]], dim=1).contiguous()))
            top = ref.clamp(min=0)
            got = ops.gemm_waves_tiled(act, t, epilogue=ops.RELU2, workspace=work).double()
            assert ((got - top.square()).abs() <= 2.0 ** -8 * top.square() + 2 * bound * (top + bound)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("group", [256, 1024])
def test_groups_of_several_steps(gpu, group):
    import torch
    from pie_amd import ops

    act, w, ref, bound = weight_and_sums("int4b8", 40, 272, 3072, 930, gpu, group=group)
    got = ops.gemm_waves_tiled(act, ops.repack_mfma_tiles(w)).double()
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
    off = torch.empty(40 * 272 + 1, device=gpu, dtype=torch.bfloat16)[1:].view(40, 272)   # (rows off 8 bytes: value by value)
    from pie_amd._lib import kernels
    import ctypes as C
    t = ops.repack_mfma_tiles(w)
    assert kernels().pie_hip_gemm_waves_tiled(ops.FMT["int4b8"], ops._ptr(act), ops._ptr(t.data), ops._ptr(t.scale), 1, group, ops._ptr(off), 40, 272, 3072, 0, 0, None,
                                              None, C.c_size_t(0), ops._stream()) == 0
    assert torch.equal(off.double(), got)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["int8", "fp8", "int4b8", "bf16", "bf16 rows"])
def test_as_close_to_the_exact_sums_as_the_passes(gpu, kind):
    import torch
    from pie_amd import ops

    act, w, ref, _ = weight_and_sums(kind, 40, 512, 4096, 940, gpu)
    t, ws = stored(w, kind), torch.empty(WORKSPACE // 4, device=gpu)
    err = lambda y: (y.double() - ref).abs().mean()  # noqa: E731
    passes = err(ops.gemm_skinny(act, t))
    assert err(ops.gemm_waves_tiled(act, t)) <= 1.02 * passes and err(ops.gemm_waves_tiled(act, t, workspace=ws)) <= 1.02 * passes


def test_refusals():
    """Groups of half a step, parts of a step, columns off a tile, more rows than were measured, formats without a tile-major copy."""
    from pie_amd import ops

    assert ops.gemm_waves_us("int4b8", 32, 128, 256, 64) > 1e29 and ops.gemm_waves_us("int4b8", 32, 128, 192, 64) > 1e29
    assert ops.gemm_waves_us("int8", 32, 128, 96) > 1e29 and ops.gemm_waves_us("int8", 32, 120, 128) > 1e29
    assert ops.gemm_waves_us("fp8", 513, 128, 128) > 1e29 and ops.gemm_waves_us("fp8", 32, 128, 128, tiled=False) > 1e29
    assert ops.gemm_waves_us("bf16", 32, 128, 96) > 1e29 and ops.gemm_waves_us("bf16", 32, 120, 128, tiled=False) > 1e29
    with pytest.raises(ops.KernelError):
        ops.gemm_waves_plan("int8", 600, 128, 128)


@pytest.mark.parametrize("kind,tiled,rows,tall", [("int4b8", True, 384, 64), ("int8", True, 480, 80), ("fp8", True, 480, 80), ("bf16", True, 480, 80), ("bf16", False, 480, 80)])
def test_the_range_ends_where_it_is_said_to(kind, tiled, rows, tall):
    """The last count of rows and the first that is refused, with and without a workspace, and the last width of one, two and six blocks of rows and the next."""
    from pie_amd import ops

    us = lambda M, N, **kw: ops.gemm_waves_us(kind, M, N, 1024, 128, tiled=tiled, **kw)  # noqa: E731
    for ws in (0, WORKSPACE):
        assert all(us(M, 2048, workspace_bytes=ws) < 1e29 for M in range(1, rows + 1))
        assert us(rows + 1, 2048, workspace_bytes=ws) > 1e29
        with pytest.raises(ops.KernelError):
            ops.gemm_waves_plan(kind, rows + 1, 2048, 1024, 128, ws, tiled=tiled)
        for blocks, M in ((1, 1), (1, tall), (2, 2 * tall), (6, 6 * tall)):
            widest = 1100 // blocks * 64
            assert us(M, widest, workspace_bytes=ws) < 1e29 and us(M, widest + 16, workspace_bytes=ws) > 1e29


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,hq,hk,d,K,shares", [("int4b8", 18, 4, 2, 16, 256, False), ("int4b8", 37, 32, 8, 128, 4096, True), ("int8", 65, 8, 2, 64, 448, False),
                                                     ("int8", 24, 4, 1, 128, 8192, True), ("fp8", 131, 6, 2, 128, 1024, False),
                                                     ("bf16", 77, 32, 8, 64, 2048, False), ("bf16", 19, 4, 2, 64, 8192, True)])
def test_qkv_rope_epilogue_equals_projection_then_rope_kernel(gpu, oracle, kind, M, hq, hk, d, K, shares):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(950 + M)
    x, w, _, _ = weight_and_sums(kind, M, (hq + 2 * hk) * d, K, 950 + M, gpu)
    wt = ops.repack_mfma_tiles(w)
    tab = ops.rope_table(dev(rng.integers(0, 500, M).astype(np.int32), gpu), dev(oracle.rope_inv_freq(d, 10000.0), gpu), d)
    slots = rng.permutation(256)[:M].astype(np.int64)
    slots[1] = -1
    sg = dev(slots, gpu)
    ws = torch.empty(1 << 22, device=gpu) if shares else None
    for pairing, t in ((1, wt), (2, ops.repack_mfma_tiles(ops.pair_qk_rows(w, hq, hk, d)))):
        pools = [torch.full((256, hk, d), 0.5, device=gpu, dtype=torch.bfloat16) for _ in range(4)]
        q1 = ops.qkv_rope_skinny_tiled(x, t, tab, sg, pools[0], pools[1], hq, hk, d, pairing=pairing, waves=True, workspace=ws)
        q2 = ops.qkv_rope_kvwrite(ops.gemm_waves_tiled(x, wt, workspace=ws), pools[2], pools[3], tab, sg, hq, hk, d, pairing == 1)
        assert np.array_equal(bits(q1), bits(q2))
        assert np.array_equal(bits(pools[0]), bits(pools[2])) and np.array_equal(bits(pools[1]), bits(pools[3]))


@pytest.mark.gpu
@pytest.mark.parametrize("kind,M,N,K", [("int8", 5, 2048, 8192), ("fp8", 40, 528, 4160), ("int4b8", 17, 4096, 4096), ("int4b8", 64, 16384, 1024), ("int8", 130, 1024, 2112), ("bf16", 40, 2048, 8192),
                                          ("bf16", 9, 528, 4160)])
def test_shares_that_meet_in_the_norm(gpu, kind, M, N, K):
    import torch
    from pie_amd import ops

    act, w, ref, bound = weight_and_sums(kind, M, N, K, 970 + M, gpu)
    g = torch.Generator(device=gpu).manual_seed(970 + M)
    x0 = torch.randn(M, N, generator=g, device=gpu).to(torch.bfloat16)
    nw = (1 + 0.1 * torch.randn(N, generator=g, device=gpu)).to(torch.bfloat16)
    x, ws = x0.clone(), torch.full((8 * M * N,), float("nan"), device=gpu)
    y, shares = ops.gemm_waves_shares_norm(act, ops.repack_mfma_tiles(w), x, nw, 1e-5, ws)
    assert 2 <= shares <= 8
    total = ref + x0.double()
    assert ((x.double() - total).abs() <= 2.0 ** -8 * total.abs() + bound).all()
    # (the norm's own rounding: two products and a reciprocal root in fp32, the sum of squares of N values in another order)
    want = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-5) * nw.double()
    assert ((y.double() - want).abs() <= (2.0 ** -8 + N * 2.0 ** -24) * want.abs()).all()
