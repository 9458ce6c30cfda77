"""GPU parity: int4 weights with fp32 group scales in blocks of up to 64 rows, against the exact sums in 64 bits and the kernels
whose epilogues it shares."""
import numpy as np
import pytest

from gpu_util import bits, dev
from test_linear_fused_gpu import make_weight

pytestmark = pytest.mark.gpu


def groups_case(oracle, gpu, M, N, K, G, seed):
    """Activations with a mean (the codes' offset then has something to cancel), tile-major weights, exact sums and their bound:
    bf16 rounding of the result, fp32 rounding of sums of codes with their offsets."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(seed)
    wd, mk = make_weight(oracle, rng, "int4b8", N, K, G=G)
    act = (torch.randn(M, K, generator=torch.Generator(device=gpu).manual_seed(seed), device=gpu) + 0.25).to(torch.bfloat16)
    codes = np.stack([(wd["data"] >> (4 * i)) & 0xF for i in range(8)], axis=-1).reshape(N, K).astype(np.float64) - 8.0
    scale = np.repeat(oracle.bf16_to_f32(wd["scale"]).astype(np.float64), G, axis=1)
    x = act.double()
    ref = x @ torch.from_numpy(codes * scale).to(gpu).T
    bound = K * 2.0 ** -23 * (x.abs() @ torch.from_numpy((np.abs(codes) + 272.0) * scale).to(gpu).T)
    return act, ops.repack_mfma_tiles(mk(gpu)), ref, bound


@pytest.mark.parametrize("M,N,K,G", [(1, 16, 128, 128), (17, 144, 256, 256), (32, 128, 384, 128), (33, 272, 640, 128), (48, 400, 512, 512),
                                     (49, 112, 768, 256), (64, 256, 1152, 128), (65, 1040, 896, 128), (130, 2064, 1408, 128), (321, 16528, 512, 128)])
def test_blocks_of_group_scaled_rows(gpu, oracle, M, N, K, G):
    """Row counts around each block height, columns off a block of 128, one to eleven steps of 128 k-values (four in flight, their
    remainders), groups of several steps, more blocks than run at once, without and with a workspace: mostly in blocks of 16 rows and without shares.  (Each height and
    shares by the plan: test_gemm_stores_gpu.py.)"""
    import torch
    from pie_amd import ops

    act, t, ref, bound = groups_case(oracle, gpu, M, N, K, G, 810 + M)
    ws = torch.full((1 << 20,), float("nan"), device=gpu)
    for work in (None, ws):
        got = ops.gemm_groups_tiled(act, t, workspace=work).double()
        assert torch.isfinite(got).all() and ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + bound).all()
        y0 = torch.randn(M, N, device=gpu).to(torch.bfloat16)
        got = ops.gemm_groups_tiled(act, t, y=y0.clone(), beta=1, workspace=work).double()
        assert ((got - ref - y0.double()).abs() <= 2.0 ** -8 * (ref + y0.double()).abs() + 2 * bound).all()
        pairs = ops.gemm_groups_tiled(act, t, workspace=work)
        assert torch.equal(ops.gemm_groups_tiled(act, t, epilogue=1, workspace=work),
                           ops.swiglu_bf16(torch.cat([pairs[:, 0::2], pairs[:, 1::2]], dim=1).contiguous()))


def test_shares_are_as_close_to_the_exact_sums_as_the_passes(gpu, oracle):
    import torch
    from pie_amd import ops

    M, N, K = 40, 512, 4096
    act, t, ref, _ = groups_case(oracle, gpu, M, N, K, 128, 830)
    ws = torch.empty(8 * M * N, device=gpu)
    assert ops.gemm_groups_us(M, N, K, 128, ws.numel() * 4) < ops.gemm_groups_us(M, N, K, 128)   # (it does run in shares)
    err = lambda y: (y.double() - ref).abs().mean()  # noqa: E731
    passes = err(ops.gemm_skinny(act, t))
    assert err(ops.gemm_groups_tiled(act, t)) <= 1.02 * passes and err(ops.gemm_groups_tiled(act, t, workspace=ws)) <= 1.02 * passes


def test_refusals(gpu, oracle):
    import torch
    from pie_amd import ops

    for N, K, G in ((128, 256, 64), (64, 192, 64)):   # groups of half a step; not whole steps
        _, mk = make_weight(oracle, np.random.default_rng(840), "int4b8", N, K, G=G)
        assert ops.gemm_groups_us(32, N, K, G) > 1e29
        if K % 128 == 0:
            with pytest.raises(ops.KernelError):
                ops.gemm_groups_tiled(torch.zeros(32, K, device=gpu, dtype=torch.bfloat16), ops.repack_mfma_tiles(mk(gpu)))


@pytest.mark.parametrize("M,hq,hk,d,K,shares", [(18, 4, 2, 16, 256, False), (37, 32, 8, 128, 1024, True), (65, 8, 2, 64, 512, False)])
def test_qkv_rope_epilogue_equals_projection_then_rope_kernel(gpu, oracle, M, hq, hk, d, K, shares):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(850 + M)
    N = (hq + 2 * hk) * d
    _, mk = make_weight(oracle, rng, "int4b8", N, K)
    wt = ops.repack_mfma_tiles(mk(gpu))
    x = dev(oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32)), gpu, torch.bfloat16)
    tab = ops.rope_table(dev(rng.integers(0, 500, M).astype(np.int32), gpu), dev(oracle.rope_inv_freq(d, 10000.0), gpu), d)
    slots = rng.permutation(128)[:M].astype(np.int64)
    slots[1] = -1
    sg = dev(slots, gpu)
    ws = torch.empty(1 << 22, device=gpu) if shares else None
    for pairing, w in ((1, wt), (2, ops.repack_mfma_tiles(ops.pair_qk_rows(mk(gpu), hq, hk, d)))):
        pools = [torch.full((128, hk, d), 0.5, device=gpu, dtype=torch.bfloat16) for _ in range(4)]
        q1 = ops.qkv_rope_skinny_tiled(x, w, tab, sg, pools[0], pools[1], hq, hk, d, pairing=pairing, groups=True, workspace=ws)
        q2 = ops.qkv_rope_kvwrite(ops.gemm_groups_tiled(x, wt, workspace=ws), pools[2], pools[3], tab, sg, hq, hk, d, pairing == 1)
        assert np.array_equal(bits(q1), bits(q2))
        assert np.array_equal(bits(pools[0]), bits(pools[2])) and np.array_equal(bits(pools[1]), bits(pools[3]))


@pytest.mark.parametrize("M,N,K", [(1, 16, 512), (5, 4096, 640), (16, 2064, 1152), (17, 528, 896), (40, 8208, 512), (64, 16384, 384), (130, 1024, 1024)])
def test_shares_that_meet_in_the_norm(gpu, oracle, M, N, K):
    """Projection into the residual and the norm behind it, against the same sums added to the residual and normalised: rows of less
    than a wave, of one and two rounds of the block's threads, shares that do not divide the steps."""
    import torch
    from pie_amd import ops

    act, t, ref, bound = groups_case(oracle, gpu, M, N, K, 128, 870 + M)
    g = torch.Generator(device=gpu).manual_seed(870 + M)
    x0 = torch.randn(M, N, generator=g, device=gpu).to(torch.bfloat16)
    w = (1 + 0.1 * torch.randn(N, generator=g, device=gpu)).to(torch.bfloat16)
    x, ws = x0.clone(), torch.full((8 * M * N,), float("nan"), device=gpu)
    y, shares = ops.gemm_groups_shares_norm(act, t, x, w, 1e-5, ws)
    assert 2 <= shares <= 8
    total = ref + x0.double()
    assert ((x.double() - total).abs() <= 2.0 ** -8 * total.abs() + bound).all()
    # (the norm's own rounding: two products and a reciprocal root in fp32, the sum of squares of N values in another order)
    want = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-5) * w.double()
    assert ((y.double() - want).abs() <= (2.0 ** -8 + N * 2.0 ** -24) * want.abs()).all()


@pytest.mark.parametrize("M,hq,hk,d,K,rows,shares", [(18, 4, 2, 64, 2048, 16, 8), (16, 32, 8, 128, 4096, 16, 4), (30, 32, 8, 128, 2944, 32, 5),
                                                     (37, 16, 4, 128, 4096, 48, 8), (180, 16, 4, 128, 4096, 64, 3)])
def test_qkv_rope_epilogue_of_shares(gpu, oracle, M, hq, hk, d, K, rows, shares):
    """The rotation and the cache's rows behind sums that meet in shares of K, every height of a block."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(890 + M)
    N = (hq + 2 * hk) * d
    ws = torch.full((6 << 20,), float("nan"), device=gpu)
    assert ops.gemm_groups_plan(M, N, K, 128, ws.numel() * 4) == (rows, shares)
    _, mk = make_weight(oracle, rng, "int4b8", N, K)
    wt = ops.repack_mfma_tiles(mk(gpu))
    x = dev(oracle.f32_to_bf16(rng.standard_normal((M, K)).astype(np.float32)), gpu, torch.bfloat16)
    tab = ops.rope_table(dev(rng.integers(0, 500, M).astype(np.int32), gpu), dev(oracle.rope_inv_freq(d, 10000.0), gpu), d)
    slots = rng.permutation(256)[:M].astype(np.int64)
    slots[1] = -1
    sg = dev(slots, gpu)
    for pairing, w in ((1, wt), (2, ops.repack_mfma_tiles(ops.pair_qk_rows(mk(gpu), hq, hk, d)))):
        pools = [torch.full((256, hk, d), 0.5, device=gpu, dtype=torch.bfloat16) for _ in range(4)]
        q1 = ops.qkv_rope_skinny_tiled(x, w, tab, sg, pools[0], pools[1], hq, hk, d, pairing=pairing, groups=True, workspace=ws)
        q2 = ops.qkv_rope_kvwrite(ops.gemm_groups_tiled(x, wt, workspace=ws), pools[2], pools[3], tab, sg, hq, hk, d, pairing == 1)
        assert np.array_equal(bits(q1), bits(q2))
        assert np.array_equal(bits(pools[0]), bits(pools[2])) and np.array_equal(bits(pools[1]), bits(pools[3]))


@pytest.mark.parametrize("M,N,K,rows,shares", [(1, 16, 384, 16, 2), (17, 8208, 384, 32, 2), (33, 8208, 384, 48, 2), (49, 8208, 384, 64, 2)])
def test_shares_that_meet_in_the_norm_by_height(gpu, oracle, M, N, K, rows, shares):
    import torch
    from pie_amd import ops

    ws = torch.full((8 * M * N,), float("nan"), device=gpu)
    assert ops.gemm_groups_plan(M, N, K, 128, ws.numel() * 4, True) == (rows, shares)
    act, t, ref, bound = groups_case(oracle, gpu, M, N, K, 128, 895 + M)
    x0 = torch.randn(M, N, generator=torch.Generator(device=gpu).manual_seed(895), device=gpu).to(torch.bfloat16)
    x = x0.clone()
    y, got = ops.gemm_groups_shares_norm(act, t, x, torch.ones(N, device=gpu, dtype=torch.bfloat16), 1e-5, ws)
    total = ref + x0.double()
    assert got == shares and ((x.double() - total).abs() <= 2.0 ** -8 * total.abs() + bound).all()
    want = x.double() * torch.rsqrt(x.double().square().mean(-1, keepdim=True) + 1e-5)
    assert ((y.double() - want).abs() <= (2.0 ** -8 + N * 2.0 ** -24) * want.abs()).all()
