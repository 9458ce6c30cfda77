"""GPU parity: the tiled matrix-core GEMM (prefill / large M) against the CPU oracle in the
reference's large-M evaluation order (int4: dequantise to bf16, then bf16 GEMM with fp32 sums;
int8/fp8/bf16: exact bf16 weights, row scale on the fp32 sum)."""
import numpy as np
import pytest

from gpu_util import bits, dev, ulp_diff
from test_linear_fused_gpu import close_to_oracle, make_weight

pytestmark = pytest.mark.gpu

KINDS = ["int4b8", "int8", "fp8", "bf16"]


def oracle_gemm(oracle, wd, act, y_in=None):
    if wd["kind"] == "int4b8":
        return oracle.gemm_w4a16(act, wd["data"], wd["scale"], wd["G"], mode=1, y_in=y_in)[1]
    if wd["kind"] == "int8":
        return oracle.gemm_w8a16(act, wd["data"], wd["scale"], mode=0, y_in=y_in)[1]
    if wd["kind"] == "fp8":
        return oracle.gemm_fp8(act, wd["data"], wd["scale"], mode=0, y_in=y_in)[1]
    return oracle.gemm_bf16(act, wd["data"], mode=0, y_in=y_in)[1]


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M,N,K", [(128, 256, 256), (200, 200, 1024), (65, 384, 512), (300, 130, 64),
                                   (1, 128, 128)])
def test_gemm_matches_oracle(gpu, oracle, kind, M, N, K):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(600 + M + N)
    wd, mk = make_weight(oracle, rng, kind, N, K, G=64 if K % 128 else 128)
    x = oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    got = bits(ops.gemm_mfma(dev(x, gpu, torch.bfloat16), mk(gpu)))
    ref = oracle_gemm(oracle, wd, x)
    assert got.shape == ref.shape
    assert close_to_oracle(oracle, got, ref)
    assert (ulp_diff(got, ref) <= 1).mean() > 0.98


@pytest.mark.parametrize("kind", KINDS)
def test_gemm_one_hot_rows_are_exact(gpu, oracle, kind):
    """One-hot activations read single dequantised weights: bit-exact, which pins the tile
    indexing, both operand layouts and the in-flight dequantisation."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(610)
    M, N, K = 150, 272, 320
    wd, mk = make_weight(oracle, rng, kind, N, K, G=64)
    ks = rng.integers(0, K, size=M)
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), ks] = 1.0
    xb = oracle.f32_to_bf16(x)
    got = bits(ops.gemm_mfma(dev(xb, gpu, torch.bfloat16), mk(gpu)))
    assert np.array_equal(got, oracle_gemm(oracle, wd, xb))


@pytest.mark.parametrize("kind", ["int4b8", "fp8"])
def test_gemm_beta_and_swiglu(gpu, oracle, kind):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(611)
    M, I, K = 140, 192, 512
    wd, mk = make_weight(oracle, rng, kind, 2 * I, K)
    x = oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    xg = dev(x, gpu, torch.bfloat16)
    w = mk(gpu)
    y0 = oracle.f32_to_bf16(rng.standard_normal((M, 2 * I)).astype(np.float32))
    got = bits(ops.gemm_mfma(xg, w, y=dev(y0, gpu, torch.bfloat16).clone(), beta=1))
    ref = oracle_gemm(oracle, wd, x, y_in=y0)
    assert close_to_oracle(oracle, got, ref) and (ulp_diff(got, ref) <= 1).mean() > 0.98
    perm = np.empty(2 * I, np.int64)
    perm[0::2], perm[1::2] = np.arange(I), np.arange(I) + I
    idx = torch.from_numpy(perm).to(gpu)
    wi = ops.WeightView(w.kind, w.data[idx].contiguous(), w.scale[idx].contiguous(), w.group_size,
                        w.N, w.K)
    fused = bits(ops.gemm_mfma(xg, wi, swiglu=True))
    unfused = bits(ops.swiglu_bf16(ops.gemm_mfma(xg, w)))
    assert fused.shape == (M, I) and np.array_equal(fused, unfused)


def test_gemm_rejects_unsupported_k(gpu, oracle):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(612)
    wd, mk = make_weight(oracle, rng, "bf16", 64, 96)
    with pytest.raises(ops.KernelError):
        ops.gemm_mfma(torch.zeros(8, 96, device=gpu, dtype=torch.bfloat16), mk(gpu))


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M,N,K", [(64, 256, 4096), (33, 130, 2048), (100, 384, 1024), (16, 512, 14336),
                                   (128, 4096, 512)])
def test_gemm_split_k_matches_oracle(gpu, oracle, kind, M, N, K):
    """Decode-batch form: K shares per output tile, fp32 partials summed by the second kernel
    (64-row block tiles up to M = 64, ragged last share when the steps do not divide)."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(630 + M + N)
    wd, mk = make_weight(oracle, rng, kind, N, K)
    x = oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    xg, w = dev(x, gpu, torch.bfloat16), mk(gpu)
    got = bits(ops.gemm_mfma(xg, w, split_k=True))
    ref = oracle_gemm(oracle, wd, x)
    assert close_to_oracle(oracle, got, ref)
    assert (ulp_diff(got, ref) <= 1).mean() > 0.98
    single = bits(ops.gemm_mfma(xg, w))
    assert (ulp_diff(got, single) <= 1).mean() > 0.98


@pytest.mark.parametrize("kind", ["int4b8", "fp8"])
def test_gemm_split_k_beta_swiglu_one_hot(gpu, oracle, kind):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(631)
    M, I, K = 48, 192, 2048
    assert ops.gemm_mfma_workspace_bytes(M, 2 * I, K) > 0
    wd, mk = make_weight(oracle, rng, kind, 2 * I, K)
    w = mk(gpu)
    ks = rng.integers(0, K, size=M)
    x = np.zeros((M, K), np.float32)
    x[np.arange(M), ks] = 1.0
    xb = oracle.f32_to_bf16(x)
    assert np.array_equal(bits(ops.gemm_mfma(dev(xb, gpu, torch.bfloat16), w, split_k=True)),
                          oracle_gemm(oracle, wd, xb))
    x = oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32))
    xg = dev(x, gpu, torch.bfloat16)
    y0 = oracle.f32_to_bf16(rng.standard_normal((M, 2 * I)).astype(np.float32))
    got = bits(ops.gemm_mfma(xg, w, y=dev(y0, gpu, torch.bfloat16).clone(), beta=1, split_k=True))
    ref = oracle_gemm(oracle, wd, x, y_in=y0)
    assert close_to_oracle(oracle, got, ref) and (ulp_diff(got, ref) <= 1).mean() > 0.98
    perm = np.empty(2 * I, np.int64)
    perm[0::2], perm[1::2] = np.arange(I), np.arange(I) + I
    idx = torch.from_numpy(perm).to(gpu)
    wi = ops.WeightView(w.kind, w.data[idx].contiguous(), w.scale[idx].contiguous(), w.group_size,
                        w.N, w.K)
    fused = bits(ops.gemm_mfma(xg, wi, swiglu=True, split_k=True))
    unfused = bits(ops.swiglu_bf16(ops.gemm_mfma(xg, w, split_k=True)))
    assert np.array_equal(fused, unfused)


# the fewest rows, the edges of the 256-row and 128-column blocks, step counts that leave 0 - 2 behind the unrolled loops, many blocks
# (of 128 columns, by the estimates; int8 and fp8 take the fourth in 256)
WIDE = [(129, 16, 256), (255, 144, 320), (257, 272, 448), (300, 16656, 256), (600, 23056, 384)]


def wide_case(oracle, gpu, kind, M, N, K, seed):
    import torch
    from pie_amd import ops

    K = (K + 127) // 128 * 128 if kind == "int4b8" else K
    g = torch.Generator(device=gpu).manual_seed(seed)
    rng = np.random.default_rng(seed)
    _, mk = make_weight(oracle, rng, kind, N, K, G=64 if K % 256 else 128)
    w = mk(gpu)
    return torch.randn(M, K, generator=g, device=gpu).to(torch.bfloat16), w, w if kind == "bf16" else ops.repack_mfma_tiles(w)


def assert_near_exact(got, act, w, ref=None):
    """bf16 rounding of a sum whose fp32 error is bounded by K terms' worth of half-ulps."""
    import torch
    x, wd = act.double(), w.data.reshape(w.N, w.K).double()
    ref = x @ wd.T if ref is None else ref
    assert torch.isfinite(got).all()
    assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + w.K * 2.0 ** -23 * (x.abs() @ wd.abs().T)).all()


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M,N,K", WIDE)
def test_wide_blocks_equal_the_tiles(gpu, oracle, kind, M, N, K):
    """Blocks of 256 rows: the same products summed in the same order as the 128-row tiles (bf16, which takes either by
    its rule: the exact sums)."""
    import torch
    from pie_amd import ops

    act, w, t = wide_case(oracle, gpu, kind, M, N, K, 700 + M)
    got = ops.gemm_mfma_tiled(act, t)
    if kind == "bf16":
        assert_near_exact(got, act, w)
        assert torch.equal(ops.gemm_mfma_tiled(act, w, y=torch.ones_like(got), beta=1),
                           ops.gemm_mfma(act, w, y=torch.ones_like(got), beta=1))
    else:
        assert torch.equal(got, ops.gemm_mfma(act, w))


@pytest.mark.parametrize("kind", KINDS)
def test_wide_epilogues_and_shares(gpu, oracle, kind):
    import torch
    from pie_amd import ops

    act, w, t = wide_case(oracle, gpu, kind, 257, 272, 2048, 720)
    y0 = torch.randn(257, 272, device=gpu).to(torch.bfloat16)
    ws = torch.empty(16 << 20, dtype=torch.uint8, device=gpu)
    plain = ops.gemm_mfma(act, w)
    assert torch.equal(ops.gemm_mfma_tiled(act, t), plain)
    assert torch.equal(ops.gemm_mfma_tiled(act, t, y=y0.clone(), beta=1), ops.gemm_mfma(act, w, y=y0.clone(), beta=1))
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=ops.GELU), ops.gemm_mfma(act, w, swiglu=ops.GELU))
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1), ops.gemm_mfma(act, w, swiglu=True))
    if kind == "bf16":
        bias = torch.randn(272, device=gpu)
        rule = ops.glu(bias, 7.0, 1.702, 1.0)
        assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1, rule=rule), ops.linear_glu("tiled", act, w.data, rule))
    # in shares of K: at most a rounding apart from the sum in one piece (fp32 partials)
    for beta in (0, 1):
        ref = ops.gemm_mfma(act, w, y=y0.clone(), beta=1) if beta else plain
        got = ops.gemm_mfma_tiled(act, t, y=y0.clone() if beta else None, beta=beta, workspace=ws)
        assert (got.float() - ref.float()).abs().max() <= 2.0 ** -7 * float(ref.float().abs().max())
        assert (got == ref).float().mean() > 0.98
    pairs = ops.gemm_mfma_tiled(act, t, workspace=ws)   # (gate, up) columns side by side
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1, workspace=ws),
                       ops.swiglu_bf16(torch.cat([pairs[:, 0::2], pairs[:, 1::2]], dim=1).contiguous()))


# Blocks of 256 columns, in all formats by the estimates: one round, the last block 144 columns wide and the last rows 44; 128 whole
# columns of blocks (three rounds) and a rest of 128-column blocks behind them.  9 and 49 steps of 64 k-values (int4, whose steps are
# pairs: 10 and 50).
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("M,N,K", [(300, 16528, 576), (1500, 32784, 3136)])
def test_wide_blocks_of_256_columns(gpu, kind, M, N, K):
    import torch
    from pie_amd import ops

    g = torch.Generator(device=gpu).manual_seed(730 + M)
    rand = lambda lo, hi, *shape, dtype: torch.randint(lo, hi, shape, generator=g, device=gpu, dtype=dtype)
    K = (K + 127) // 128 * 128 if kind == "int4b8" else K
    if kind == "int4b8":
        w = ops.int4b8_view(rand(-2**31, 2**31 - 1, N, K // 8, dtype=torch.int32), torch.rand(N, K // 128, generator=g, device=gpu).bfloat16(), 128)
    elif kind == "bf16":
        w = ops.WeightView("bf16", torch.randn(N, K, generator=g, device=gpu).bfloat16(), None, 0, N, K)
    else:
        codes = rand(-128, 128, N, K, dtype=torch.int8) if kind == "int8" else rand(0, 0x70, N, K, dtype=torch.uint8)
        w = ops.WeightView(kind, codes, torch.rand(N, generator=g, device=gpu), 0, N, K)
    t = w if kind == "bf16" else ops.repack_mfma_tiles(w)
    act = torch.randn(M, K, generator=g, device=gpu).bfloat16()
    y0 = torch.randn(M, N, generator=g, device=gpu).bfloat16()
    plain = ops.gemm_mfma_tiled(act, t)
    summed = ops.gemm_mfma_tiled(act, t, y=y0.clone(), beta=1)
    if kind == "bf16":
        assert_near_exact(plain, act, w)
        ref = plain.double() + y0.double()   # (the sum is rounded once, with the residual: a step of the plain result's rounding and its own)
        assert ((summed.double() - ref).abs() <= 2.0 ** -8 * (plain.double().abs() + ref.abs())).all()
        bias = torch.randn(N, generator=g, device=gpu)
        rule = ops.glu(bias, 7.0, 1.702, 1.0)
        assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1, rule=rule), ops.linear_glu("tiled", act, w.data, rule))
    else:   # the same products summed in the same order
        assert torch.equal(plain, ops.gemm_mfma(act, w))
        assert torch.equal(summed, ops.gemm_mfma(act, w, y=y0.clone(), beta=1))
        assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=ops.RELU2), ops.gemm_mfma(act, w, swiglu=ops.RELU2))
    pairs = torch.cat([plain[:, 0::2], plain[:, 1::2]], dim=1).contiguous()
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1), ops.swiglu_bf16(pairs))


@pytest.mark.parametrize("kind,M,N,K,G", [
    ("bf16", 256, 128, 192, 0), ("int8", 256, 128, 192, 0), ("fp8", 256, 128, 192, 0),        # K below four steps
    ("int4b8", 256, 128, 128, 128),
    ("bf16", 256, 128, 288, 0), ("int8", 256, 128, 288, 0), ("fp8", 256, 128, 288, 0),        # K off a step
    ("int4b8", 256, 128, 320, 64),
    ("int4b8", 256, 128, 256, 32), ("int4b8", 256, 128, 384, 96), ("int4b8", 40, 128, 256, 64),   # groups
    ("int8", 256, 24, 256, 0), ("fp8", 64, 24, 256, 0), ("int4b8", 256, 24, 256, 128),        # columns without a tile-major copy
])
def test_wide_refusals(gpu, kind, M, N, K, G):
    """Shapes the blocks do not take are refused by the call, not misread (and not by what prepares their weights).  40 rows of
    groups of 64: the columns form does not take them, the blocks do."""
    import torch
    from pie_amd import ops

    act = torch.zeros(M, K, device=gpu, dtype=torch.bfloat16)
    rows, words = -(-N // 256) * 256, K * 2   # (more than any reading of the shape could touch)
    data = torch.zeros(rows * words, device=gpu, dtype=torch.uint8)
    scale = torch.ones(rows * K, device=gpu, dtype=torch.bfloat16)
    w = ops.WeightView(kind, data, None, 0, N, K) if kind == "bf16" else ops.WeightView(kind + "+tiled", data, scale, G, N, K)
    if (M, K, G) == (40, 256, 64):
        assert (ops.gemm_mfma_tiled(act, w) == 0).all()
        return
    with pytest.raises(ops.KernelError):
        ops.gemm_mfma_tiled(act, w)


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (17, 80, 128), (64, 208, 320), (65, 64, 448), (96, 144, 512), (97, 272, 576), (128, 64, 1088)])
def test_columns_of_few_rows(gpu, oracle, kind, M, N, K):
    """Up to 128 rows in blocks of 64 columns, against the exact sums: the edges of the three row counts, columns off a block, one
    step of 64 k-values (the second group of waves has none), odd and even counts, remainders of the four in flight."""
    import torch
    from pie_amd import ops

    act, w, t = wide_case(oracle, gpu, kind, M, N, K, 740 + M)
    codes = w.data.double() if kind == "int8" else w.data.view(torch.float8_e4m3fn).double()
    wd = codes.reshape(N, K) * w.scale.double().reshape(N, 1)
    x = act.double()
    bound = K * 2.0 ** -23 * (x.abs() @ wd.abs().T)
    ref = x @ wd.T
    got = ops.gemm_mfma_tiled(act, t).double()
    assert torch.isfinite(got).all() and ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
    y0 = torch.randn(M, N, device=gpu).to(torch.bfloat16)
    got = ops.gemm_mfma_tiled(act, t, y=y0.clone(), beta=1).double()
    assert ((got - ref - y0.double()).abs() <= 2.0 ** -8 * (ref + y0.double()).abs() + 2 * bound).all()
    pairs = ops.gemm_mfma_tiled(act, t)
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1),
                       ops.swiglu_bf16(torch.cat([pairs[:, 0::2], pairs[:, 1::2]], dim=1).contiguous()))


@pytest.mark.parametrize("M,N,K,G", [(17, 16, 128, 128), (32, 144, 256, 256), (33, 272, 640, 128), (48, 128, 1024, 256), (40, 400, 1152, 128)])
def test_columns_of_few_rows_int4(gpu, oracle, M, N, K, G):
    """17 to 48 rows of int4 weights: the codes' products are summed exactly per group and scaled in fp32, so the exact sums with
    the products' offset of 136 in the bound; columns off a block, one step of 128 k-values, odd counts, groups of two steps."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(760 + M)
    wd, mk = make_weight(oracle, rng, "int4b8", N, K, G=G)
    w = mk(gpu)
    act = torch.randn(M, K, generator=torch.Generator(device=gpu).manual_seed(760 + M), device=gpu).to(torch.bfloat16)
    t = ops.repack_mfma_tiles(w)
    codes = np.stack([(wd["data"] >> (4 * i)) & 0xF for i in range(8)], axis=-1).reshape(N, K).astype(np.float64) - 8.0
    scale = np.repeat(oracle.bf16_to_f32(wd["scale"]).astype(np.float64), G, axis=1)
    wf = torch.from_numpy(codes * scale).to(gpu)
    x = act.double()
    ref = x @ wf.T
    bound = K * 2.0 ** -23 * (x.abs() @ torch.from_numpy((np.abs(codes) + 272.0) * scale).to(gpu).T)
    got = ops.gemm_mfma_tiled(act, t).double()
    assert torch.isfinite(got).all() and ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
    # and what those terms come to: as close to the exact sums as the passes of 16 and 32 rows are
    if K % 512 == 0:
        assert (got - ref).abs().mean() <= 1.02 * (ops.gemm_skinny(act, t).double() - ref).abs().mean()
    pairs = ops.gemm_mfma_tiled(act, t)
    assert torch.equal(ops.gemm_mfma_tiled(act, t, epilogue=1),
                       ops.swiglu_bf16(torch.cat([pairs[:, 0::2], pairs[:, 1::2]], dim=1).contiguous()))


@pytest.mark.parametrize("kind", ["int8", "fp8"])
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (33, 144, 128), (65, 256, 192), (97, 1040, 320), (129, 512, 1088), (200, 5136, 256), (700, 4096, 192), (1300, 8208, 128)])
def test_rows_in_blocks_of_each_height(gpu, oracle, kind, M, N, K):
    """Many rows of one-byte weights against the exact sums: row counts off a block, columns off a block of 128, one step of 64 k-values
    to remainders of those in flight, one to several rounds of blocks, without and with a workspace.  (Each height and shares by the plan: test_gemm_stores_gpu.py.)"""
    import torch
    from pie_amd import ops

    act, w, t = wide_case(oracle, gpu, kind, M, N, K, 780 + M)
    codes = w.data.double() if kind == "int8" else w.data.view(torch.float8_e4m3fn).double()
    wd = codes.reshape(N, K) * w.scale.double().reshape(N, 1)
    x = act.double()
    bound = K * 2.0 ** -23 * (x.abs() @ wd.abs().T)
    ref = x @ wd.T
    for ws in (None, torch.full((4 << 20,), float("nan"), device=gpu)):
        got = ops.gemm_rows_tiled(act, t, workspace=ws)
        assert torch.isfinite(got).all() and ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
        y0 = torch.randn(M, N, device=gpu).to(torch.bfloat16)
        res = ops.gemm_rows_tiled(act, t, y=y0.clone(), beta=1, workspace=ws).double()
        assert ((res - ref - y0.double()).abs() <= 2.0 ** -8 * (ref + y0.double()).abs() + 2 * bound).all()
        assert torch.equal(ops.gemm_rows_tiled(act, t, epilogue=1, workspace=ws),
                           ops.swiglu_bf16(torch.cat([got[:, 0::2], got[:, 1::2]], dim=1).contiguous()))
