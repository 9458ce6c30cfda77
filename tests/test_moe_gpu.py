"""GPU parity for the MoE row: routing (softmax, top-k, renormalisation and the expert-sorted
layout), the combine, and the whole expert block at the Qwen3-30B-A3B expert shape against the
oracle's per-route evaluation."""
import numpy as np
import pytest

from gpu_util import bits, dev, ulp_diff
from test_linear_fused_gpu import close_to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,K", [(1, 128, 8), (64, 128, 8), (7, 8, 2), (300, 384, 6), (5, 5, 5),
                                   (2100, 64, 4)])
def test_route_matches_oracle_and_layout_is_a_counting_sort(gpu, oracle, T, E, K):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(500 + T + E)
    logits = oracle.f32_to_bf16(rng.standard_normal((T, E)).astype(np.float32) * 2)
    if T > 6:
        logits[3, :] = logits[3, 0]            # a fully tied row: the first K experts win
        logits[5, 1:4] = logits[5].max()       # tied maxima: lowest indices first
    idx, w, offs, rtok, rpos = (t.cpu().numpy() for t in ops.moe_route(dev(logits, gpu, torch.bfloat16), K))
    oidx, ow = oracle.topk_softmax(logits, K)
    assert np.array_equal(idx, oidx)           # integer outputs: bit-exact
    assert np.allclose(w, ow, rtol=2e-6, atol=1e-9)
    # norm_topk = false: the same routes, the probabilities undivided
    idx_r, w_r = (t.cpu().numpy() for t in ops.moe_route(dev(logits, gpu, torch.bfloat16), K, renormalize=False)[:2])
    _, ow_r = oracle.topk_softmax(logits, K, renorm=False)
    assert np.array_equal(idx_r, oidx) and np.allclose(w_r, ow_r, rtol=2e-6, atol=1e-9)
    # layout: offsets are the exclusive scan of the per-expert route counts
    counts = np.bincount(idx.reshape(-1), minlength=E)
    assert np.array_equal(offs, np.concatenate([[0], np.cumsum(counts)]))
    flat = idx.reshape(-1)
    assert np.array_equal(np.sort(rpos), np.arange(T * K))      # a permutation
    assert np.all(rpos >= offs[flat]) and np.all(rpos < offs[flat + 1])
    assert np.array_equal(rtok[rpos], np.arange(T * K) // K)


@pytest.mark.parametrize("add", [False, True])
def test_combine_is_bit_exact(gpu, oracle, add):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(510)
    T, K, H = 37, 8, 2048
    yr = oracle.f32_to_bf16(rng.standard_normal((T * K, H)).astype(np.float32))
    w = rng.dirichlet(np.ones(K), T).astype(np.float32)
    pos = rng.permutation(T * K).astype(np.int32)
    sorted_y = np.empty_like(yr)
    sorted_y[pos] = yr
    base = oracle.f32_to_bf16(rng.standard_normal((T, H)).astype(np.float32))
    out = dev(base, gpu, torch.bfloat16).clone() if add else None
    got = bits(ops.moe_combine(dev(sorted_y, gpu, torch.bfloat16), dev(pos, gpu), dev(w, gpu), out))
    ref = oracle.moe_combine(yr, w, base if add else None)
    assert np.array_equal(got, ref)


@pytest.mark.parametrize("T,H,E,K", [(64, 2048, 128, 8), (1, 2048, 128, 8), (5, 512, 6, 2), (200, 4096, 64, 6),
                                     (17, 7168, 384, 8)])
def test_norm_route_in_one_launch(gpu, oracle, T, H, E, K):
    """pie_hip_moe_norm_route: the stored normalised rows are pie_hip_rmsnorm's bit for bit, the
    router logits are the oracle's bf16 products up to the order of the fp32 sum, and given the
    logits it stored the routing is the oracle's exactly, laid out as a counting sort."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(530 + T + E)
    x = dev(oracle.f32_to_bf16(rng.standard_normal((T, H)).astype(np.float32) * 3.0), gpu, torch.bfloat16)
    nw = dev(oracle.f32_to_bf16((1.0 + 0.2 * rng.standard_normal(H)).astype(np.float32)), gpu, torch.bfloat16)
    router = oracle.f32_to_bf16(rng.standard_normal((E, H)).astype(np.float32) * (1.0 / np.sqrt(H)))
    for renorm in (True, False):
        xn, lg, idx, w, offs, rtok, rpos = ops.moe_norm_route(x, nw, 1e-6, dev(router, gpu, torch.bfloat16), K,
                                                              renormalize=renorm)
        assert np.array_equal(bits(xn), bits(ops.rmsnorm_bf16(x, nw, 1e-6)))
        want = oracle.gemm_bf16(bits(xn), router, mode=0)[1]
        assert (ulp_diff(bits(lg), want) <= 1).all() and (bits(lg) == want).mean() > 0.97
        oidx, ow = oracle.topk_softmax(bits(lg), K, renorm=renorm)
        idx, w, offs, rtok, rpos = (t.cpu().numpy() for t in (idx, w, offs, rtok, rpos))
        assert np.array_equal(idx, oidx)
        assert np.allclose(w, ow, rtol=2e-6, atol=1e-9)
        counts = np.bincount(idx.reshape(-1), minlength=E)
        assert np.array_equal(offs, np.concatenate([[0], np.cumsum(counts)]))
        flat = idx.reshape(-1)
        assert np.array_equal(np.sort(rpos), np.arange(T * K))
        assert np.all(rpos >= offs[flat]) and np.all(rpos < offs[flat + 1])
        assert np.array_equal(rtok[rpos], np.arange(T * K) // K)
        # the same routing as the two-launch form gives on the same logits
        ref = ops.moe_route(lg, K, renormalize=renorm)
        assert np.array_equal(ref[0].cpu().numpy(), idx) and np.array_equal(ref[1].cpu().numpy(), w)


@pytest.mark.parametrize("T,H,E,K,planes", [(1, 256, 1, 1, 8), (31, 512, 6, 2, 8), (33, 2048, 128, 8, 8), (64, 2304, 130, 8, 8), (257, 2048, 128, 8, 3),
                                            (40, 7168, 384, 8, 8), (2080, 256, 512, 16, 1), (5, 1280, 64, 4, 1),
                                            (16, 2048, 128, 8, 8), (17, 512, 64, 4, 2), (8, 512, 257, 8, 2), (7, 512, 257, 8, 2)])
def test_router_in_shares_of_k(gpu, oracle, T, H, E, K, planes):
    """pie_hip_moe_router_route over tiles of 32 tokens and 128 experts that are full, one over and one short, one to eight shares of K that
    divide its steps or not, a workspace of `planes` shares, and the choice and the sort in one launch and in two: the logits are the oracle's bf16 products up to the order of the fp32 sum (one
    bf16 step where it rounds the other way), and the choice on the logits it stored is pie_hip_moe_route_opt's exactly."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(560 + T + E)
    act = oracle.f32_to_bf16(rng.standard_normal((T, H)).astype(np.float32))
    router = oracle.f32_to_bf16(rng.standard_normal((E, H)).astype(np.float32) * (1.0 / np.sqrt(H)))
    ws = torch.full((planes * T * ((E + 3) // 4 * 4),), float("nan"), device=gpu)
    want = oracle.gemm_bf16(act, router, mode=0)[1]
    for renorm in (True, False):
        lg, idx, w, offs, rtok, rpos = ops.moe_router_route(dev(act, gpu, torch.bfloat16), dev(router, gpu, torch.bfloat16), K, renorm, ws)
        # (sums of a cancelling row differ by more of its own small steps: 2^-20 of the products' magnitude, as float32 sums of K <= 7168 do)
        truth, _, ab = oracle.gemm_bf16(act, router, mode=2, want_abs=True)
        off = np.abs(oracle.bf16_to_f32(bits(lg)).astype(np.float64) - truth)
        assert (off <= 2.0 ** -8 * np.abs(truth) + 2.0 ** -20 * ab + 1e-30).all() and (bits(lg) == want).mean() > 0.97
        ref = ops.moe_route(lg, K, renormalize=renorm)
        assert torch.equal(ref[0], idx) and torch.equal(ref[1], w) and torch.equal(ref[2], offs)
        idx, offs, rtok, rpos = (t.cpu().numpy() for t in (idx, offs, rtok, rpos))
        flat = idx.reshape(-1)
        assert np.array_equal(np.sort(rpos), np.arange(T * K)) and np.array_equal(rtok[rpos], np.arange(T * K) // K)
        assert np.all(rpos >= offs[flat]) and np.all(rpos < offs[flat + 1])
    for bad in ((act[:, :H - 8], router[:, :H - 8], ws), (act, router, ws[:T * E // 2])):
        with pytest.raises(ops.KernelError):
            ops.moe_router_route(dev(np.ascontiguousarray(bad[0]), gpu, torch.bfloat16), dev(np.ascontiguousarray(bad[1]), gpu, torch.bfloat16), K, True, bad[2])


@pytest.mark.parametrize("T,E,K,shared", [(128, 128, 8, 0), (129, 128, 8, 0), (1025, 1, 1, 0), (147, 64, 7, 0), (2048, 128, 8, 0), (2049, 128, 8, 0),
                                          (1024, 512, 16, 0), (5461, 6, 3, 0), (256, 300, 61, 3), (257, 300, 61, 3), (93, 40, 10, 1)])
def test_sort_of_many_routes(gpu, T, E, K, shared):
    """Routes around 1024 (one per thread) and 16384 (sixteen, kept in registers and sorted in LDS), top_k a power of two or not, with shared experts: the
    places are a permutation inside the experts' ranges and each place names its route's token."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(570 + T + E)
    if shared:
        lg = torch.from_numpy(rng.standard_normal((T, E + 1)).astype(np.float32)).to(gpu)
        idx, _, offs, rtok, rpos = ops.moe_route_corrected(lg, torch.zeros(E, device=gpu), K, shared)
    else:
        idx, _, offs, rtok, rpos = ops.moe_route(torch.from_numpy(rng.standard_normal((T, E)).astype(np.float32)).to(gpu, torch.bfloat16), K)
    idx, offs, rtok, rpos = (t.cpu().numpy().reshape(-1) for t in (idx, offs, rtok, rpos))
    R = T * (K + shared)
    assert np.array_equal(offs, np.concatenate([[0], np.cumsum(np.bincount(idx, minlength=E + shared))]))
    assert np.array_equal(np.sort(rpos), np.arange(R)) and np.array_equal(rtok[rpos], np.arange(R) // (K + shared))
    assert np.all(rpos >= offs[idx]) and np.all(rpos < offs[idx + 1])


@pytest.mark.parametrize("T,K,H", [(64, 8, 2048), (3, 2, 512), (130, 6, 8192)])
def test_combine_with_the_next_norm_equals_the_two_launches(gpu, oracle, T, K, H):
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(540 + T)
    y = dev(oracle.f32_to_bf16(rng.standard_normal((T * K, H)).astype(np.float32)), gpu, torch.bfloat16)
    w = dev(rng.dirichlet(np.ones(K), T).astype(np.float32), gpu)
    pos = dev(rng.permutation(T * K).astype(np.int32), gpu)
    base = dev(oracle.f32_to_bf16(rng.standard_normal((T, H)).astype(np.float32)), gpu, torch.bfloat16)
    nw = dev(oracle.f32_to_bf16((1.0 + 0.2 * rng.standard_normal(H)).astype(np.float32)), gpu, torch.bfloat16)
    a = base.clone()
    ops.moe_combine(y, pos, w, a)
    an = ops.rmsnorm_bf16(a, nw, 1e-6)
    b = base.clone()
    bn = ops.moe_combine_norm(y, pos, w, b, nw, 1e-6)
    assert np.array_equal(bits(a), bits(b)) and np.array_equal(bits(an), bits(bn))


def _expert_block(gpu, oracle, seed, T, E, K, tiled, H=2048, Ie=768):
    """norm'd activations -> router -> route -> grouped gate/up (+SwiGLU) -> grouped down ->
    combine, fp8 e4m3 experts with bf16 row scales, against the oracle's per-route evaluation.
    `tiled`: the launches a driver with tile-major weights makes (gate|up in the block-shared
    grouped form, down in the wave-private grouped form over K = Ie), with the driver's
    rows-per-expert hint; otherwise the row-major entry."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(seed)
    x = oracle.f32_to_bf16(rng.standard_normal((T, H)).astype(np.float32))
    router = oracle.f32_to_bf16(rng.standard_normal((E, H)).astype(np.float32) * (1.0 / np.sqrt(H)))

    def fp8_stack(n, k):
        qs, ss = [], []
        for _ in range(E):      # expert by expert: the float copy of a whole stack is gigabytes
            w = oracle.f32_to_bf16(rng.standard_normal((n, k), dtype=np.float32) * 0.02)
            q, s = oracle.quant_fp8_per_channel(w)
            qs.append(q)
            ss.append(oracle.f32_to_bf16(s))
        return np.concatenate(qs), np.concatenate(ss)
    gu_q, gu_s = fp8_stack(2 * Ie, H)      # canonical: per expert gate rows then up rows
    dn_q, dn_s = fp8_stack(H, Ie)

    # ---- oracle: per-route evaluation ----
    logits = oracle.gemm_bf16(x, router, mode=0)[1]
    oidx, ow = oracle.topk_softmax(logits, K)
    yr = np.empty((T * K, H), np.uint16)
    act_ref = np.empty((T * K, Ie), np.uint16)
    for r in range(T * K):
        t, e = r // K, oidx.reshape(-1)[r]
        g = oracle.gemm_fp8(x[t:t + 1], gu_q[e * 2 * Ie:(e + 1) * 2 * Ie],
                            oracle.bf16_to_f32(gu_s[e * 2 * Ie:(e + 1) * 2 * Ie]), mode=0)[1]
        a = oracle.swiglu(g)
        act_ref[r] = a[0]
        yr[r] = oracle.gemm_fp8(a, dn_q[e * H:(e + 1) * H], oracle.bf16_to_f32(dn_s[e * H:(e + 1) * H]),
                                mode=0)[1][0]
    ref = oracle.moe_combine(yr, ow, x)

    # ---- GPU ----
    xg = dev(x, gpu, torch.bfloat16)
    lg = ops.gemm_skinny(xg, ops.WeightView("bf16", dev(router, gpu, torch.bfloat16), None, 0, E, H))
    assert (ulp_diff(bits(lg), logits) <= 1).mean() > 0.99
    idx, w, offs, rtok, rpos = ops.moe_route(lg, K)
    perm = np.empty(2 * Ie, np.int64)
    perm[0::2], perm[1::2] = np.arange(Ie), np.arange(Ie) + Ie
    gu_qi = dev(np.ascontiguousarray(gu_q.reshape(E, 2 * Ie, H)[:, perm]), gpu)
    gu_si = dev(np.ascontiguousarray(gu_s.reshape(E, 2 * Ie)[:, perm]), gpu, torch.bfloat16)
    dn_qg = dev(dn_q.reshape(E, H, Ie), gpu)
    dn_sg = dev(dn_s.reshape(E, H), gpu, torch.bfloat16)
    # the executor's hint (Executor::moe_block): twice the mean routes per expert, at most T
    hint = max(1, min(T, 2 * ((T * K + E - 1) // E))) if tiled else 16
    if tiled:
        # experts stacked along the rows: the tile-major copy keeps expert e at the same stride
        gu_qi = ops.repack_mfma_tiles(ops.WeightView("fp8", gu_qi.reshape(E * 2 * Ie, H), None, 0,
                                                     E * 2 * Ie, H)).data.reshape(E, 2 * Ie, -1)
        dn_qg = ops.repack_mfma_tiles(ops.WeightView("fp8", dn_qg.reshape(E * H, Ie), None, 0,
                                                     E * H, Ie)).data.reshape(E, H, -1)
    h = ops.moe_grouped_gemm(xg, rtok, offs, "fp8", gu_qi, gu_si, 2 * Ie, H, rows_hint=hint, swiglu=True,
                             tiled=tiled)
    y = ops.moe_grouped_gemm(h, None, offs, "fp8", dn_qg, dn_sg, H, Ie, rows_hint=hint, tiled=tiled)
    out = bits(ops.moe_combine(y, rpos, w, xg.clone()))
    same_routes = np.array_equal(idx.cpu().numpy(), oidx)
    assert same_routes, "router near-tie flipped an expert; pick another seed"
    # every stage against the oracle: the SwiGLU'd gate|up rows (route-sorted on the GPU) ...
    pos = rpos.cpu().numpy()
    hb = bits(h)[pos]
    assert close_to_oracle(oracle, hb, act_ref, rel=2.0 ** -6)
    assert (ulp_diff(hb, act_ref) <= 1).mean() > 0.97
    # ... the down projection of each route ...
    yb = bits(y)[pos]
    assert close_to_oracle(oracle, yb, yr, rel=2.0 ** -6)
    assert (ulp_diff(yb, yr) <= 1).mean() > 0.95
    # ... and the combined block
    assert close_to_oracle(oracle, out, ref, rel=2.0 ** -6)
    assert (ulp_diff(out, ref) <= 1).mean() > 0.97
    return dict(xg=xg, rtok=rtok, offs=offs, gu=(gu_qi, gu_si), dn=(dn_qg, dn_sg), hint=hint,
                gu_q=gu_q, gu_s=gu_s, dn_q=dn_q, dn_s=dn_s, oidx=oidx, rpos=pos)


def test_expert_block_at_c5_expert_shape(gpu, oracle):
    """H 2048, expert FFN 768, 32 of the 128 experts, top-4, through the row-major entry."""
    _expert_block(gpu, oracle, 520, T=48, E=32, K=4, tiled=False)


def test_expert_block_at_c5_full_routing_through_the_tile_major_kernels(gpu, oracle):
    """The Qwen3-30B-A3B decode batch as the driver runs it: 64 tokens, 128 experts, top-8,
    H 2048, expert FFN 768, fp8 e4m3 with bf16 row scales, tile-major weights — gate|up through
    the block-shared grouped kernel, down through the wave-private grouped kernel over K = 768
    (six 128-blocks) — every stage against the oracle, then exactness of single weights."""
    import torch
    from pie_amd import ops

    T, E, K, H, Ie = 64, 128, 8, 2048, 768
    st = _expert_block(gpu, oracle, 521, T=T, E=E, K=K, tiled=True)
    # one-hot activation rows reproduce single dequantised weights bit for bit (operand layouts
    # of both grouped kernels): route r of expert e reads a row that is 1 at column c_r
    rng = np.random.default_rng(522)
    offs = st["offs"].cpu().numpy()
    routes = int(offs[-1])
    expert_of = np.repeat(np.arange(E), np.diff(offs))
    # down: K = Ie
    cols = rng.integers(0, Ie, routes)
    a = np.zeros((routes, Ie), np.float32)
    a[np.arange(routes), cols] = 1.0
    y = bits(ops.moe_grouped_gemm(dev(oracle.f32_to_bf16(a), gpu, torch.bfloat16), None, st["offs"], "fp8",
                                  st["dn"][0], st["dn"][1], H, Ie, rows_hint=st["hint"], tiled=True))
    dn_q = st["dn_q"].reshape(E, H, Ie)
    dn_s = oracle.bf16_to_f32(st["dn_s"].reshape(E, H))
    want = oracle.f32_to_bf16(oracle.fp8_decode(dn_q[expert_of, :, cols]) * dn_s[expert_of])
    # (compared as values: a weight code of -0 gives -0 here and +0 from an accumulator that starts at +0)
    assert np.array_equal(oracle.bf16_to_f32(y), oracle.bf16_to_f32(want))
    # gate|up without SwiGLU: K = H, rows gathered by route
    cols = rng.integers(0, H, T)
    a = np.zeros((T, H), np.float32)
    a[np.arange(T), cols] = 1.0
    g = bits(ops.moe_grouped_gemm(dev(oracle.f32_to_bf16(a), gpu, torch.bfloat16), st["rtok"], st["offs"],
                                  "fp8", st["gu"][0], st["gu"][1], 2 * Ie, H, rows_hint=st["hint"],
                                  tiled=True))
    perm = np.empty(2 * Ie, np.int64)
    perm[0::2], perm[1::2] = np.arange(Ie), np.arange(Ie) + Ie
    gu_q = st["gu_q"].reshape(E, 2 * Ie, H)[:, perm]
    gu_s = oracle.bf16_to_f32(st["gu_s"].reshape(E, 2 * Ie)[:, perm])
    tok = st["rtok"].cpu().numpy()
    want = oracle.f32_to_bf16(oracle.fp8_decode(gu_q[expert_of, :, cols[tok]]) * gu_s[expert_of])
    assert np.array_equal(oracle.bf16_to_f32(g), oracle.bf16_to_f32(want))


@pytest.mark.parametrize("fmt,K,G", [("fp8", 768, 0), ("int8", 256, 0), ("int4b8", 512, 128), ("fp8", 256, 0)])
@pytest.mark.parametrize("block_rows", [0, 64, 128, 256])
def test_quantised_experts_in_blocks_of_routes(gpu, oracle, fmt, K, G, block_rows):
    """The tiled grouped GEMM over quantised experts against the row-major passes of 16 rows: experts without routes, with
    one, with a block and one more; columns off the tile, gathered rows, row scales of both types, SwiGLU.  Both sum the
    same exact bf16 products in fp32, in other orders: a sum of K products differs by at most 2 K 2^-24 of the sum of their
    magnitudes, a rounded result by that and half a bf16 step (2^-8) each.  Int4: the passes scale a group's sum in fp32, the
    blocks round every code times its scale to bf16, up to 2^-9 of each product more; the exact sums of either are checked."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(541 + K + block_rows)
    counts = [0, 1, 63, 64, 65, 129, 0, 257, 17]
    E, N, T = len(counts), 144, 96
    routes = sum(counts)
    offs = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), gpu)
    rows = dev(rng.integers(0, T, routes).astype(np.int32), gpu)
    act = dev(oracle.f32_to_bf16(rng.standard_normal((T, K)).astype(np.float32)), gpu, torch.bfloat16)
    if fmt == "int4b8":
        w = dev(rng.integers(-2**31, 2**31, (E, N, K // 8)).astype(np.int32), gpu)
        scale = dev(oracle.f32_to_bf16(rng.uniform(0.005, 0.02, (E, N, K // G)).astype(np.float32)), gpu, torch.bfloat16)
        size = float(8 * 0.02)
    else:
        w = dev(rng.integers(-128, 128, (E, N, K)).astype(np.int8) if fmt == "int8"
                else rng.integers(0, 0x70, (E, N, K)).astype(np.uint8) | (rng.integers(0, 2, (E, N, K)) << 7).astype(np.uint8), gpu)
        scale = dev(rng.uniform(0.001, 0.004, (E, N)).astype(np.float32), gpu)
        if K == 768:
            scale = scale.bfloat16()
        size = 0.004 * (128 if fmt == "int8" else 256)
    bound = K * 4.0 * size * 2 * K * 2.0 ** -24      # |act| < 4 but for one value in 16 000, whose share is far below the slack
    if fmt == "int4b8":
        bound += K * 4.0 * size * 2.0 ** -9
    for swiglu in (False, True):
        args = (act, rows, offs, fmt, w, scale, N, K, 257, G, swiglu)
        want = ops.moe_grouped_gemm(*args).float()
        got = ops.moe_grouped_gemm(*args, block_rows=block_rows).float()
        if swiglu:   # (the gate's rounding moves the result by a step of each factor)
            assert torch.all((got - want).abs() <= 4 * 2.0 ** -8 * want.abs() + 2.0 ** -6 * want.abs().amax())
        else:
            assert torch.all((got - want).abs() <= 2.0 ** -7 * want.abs() + bound)
            if fmt == "int4b8":
                codes = torch.stack([(w >> (4 * i)) & 0xF for i in range(8)], dim=-1).reshape(E, N, K).double() - 8.0
                each = scale.double().repeat_interleave(G, dim=-1)
                x = act.double()[rows.long()]
                # (the passes' codes enter their products as 128 + n, 136 times the activations' sum leaves again)
                for y, weights, offset in ((want, codes * each, 272.0), (got, (codes * each).bfloat16().double(), 0.0)):
                    at = 0
                    for e, n in enumerate(counts):
                        ref = x[at:at + n] @ weights[e].T
                        slack = K * 2.0 ** -23 * (x[at:at + n].abs() @ (weights[e].abs() + offset * each[e]).T)
                        assert torch.all((y[at:at + n].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + slack)
                        at += n
    assert torch.equal(ops.moe_grouped_gemm(act[rows.long()].contiguous(), None, offs, fmt, w, scale, N, K, 257, G, block_rows=block_rows),
                       ops.moe_grouped_gemm(act, rows, offs, fmt, w, scale, N, K, 257, G, block_rows=block_rows))


@pytest.mark.parametrize("fmt", ["fp8", "int8"])
@pytest.mark.parametrize("N,K", [(144, 64), (192, 192), (400, 320), (16, 768), (208, 1088)])
def test_byte_experts_over_tile_major_weights(gpu, oracle, fmt, N, K):
    """Blocks by the routes an expert has (here 64 and 96) over the tile-major copy against blocks of 128 over row-major weights: an expert without routes, with one,
    at the edges of a block, columns off a block, one step of 64 k-values and remainders of those in flight.
    The same exact products in fp32, in another order: the bound of the test above."""
    import torch
    from pie_amd import ops

    rng = np.random.default_rng(560 + N + K)
    counts = [0, 1, 127, 128, 129, 0, 257, 17, 0] + [0] * (4 if K > 1024 else 0)
    E, T, routes = len(counts), 96, sum(counts)
    offs = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), gpu)
    rows = dev(rng.integers(0, T, routes).astype(np.int32), gpu)
    act = dev(oracle.f32_to_bf16(rng.standard_normal((T, K)).astype(np.float32)), gpu, torch.bfloat16)
    w = dev(rng.integers(-128, 128, (E, N, K)).astype(np.int8) if fmt == "int8"
            else rng.integers(0, 0x70, (E, N, K)).astype(np.uint8) | (rng.integers(0, 2, (E, N, K)) << 7).astype(np.uint8), gpu)
    scale = dev(rng.uniform(0.001, 0.004, (E, N)).astype(np.float32), gpu)
    if K == 192:
        scale = scale.bfloat16()
    t = ops.repack_mfma_tiles(ops.WeightView(fmt, w.reshape(E * N, K), scale.reshape(-1), 0, E * N, K)).data.reshape(E, N, K)
    bound = K * 4.0 * 0.004 * (128 if fmt == "int8" else 256) * 2 * K * 2.0 ** -24
    for swiglu in (False, True):
        want = ops.moe_grouped_gemm(act, rows, offs, fmt, w, scale, N, K, 257, 0, swiglu, block_rows=128).float()
        got = ops.moe_grouped_gemm(act, rows, offs, fmt, t, scale, N, K, 257, 0, swiglu, block_rows=0, tiled=True).float()
        if swiglu:
            assert torch.all((got - want).abs() <= 4 * 2.0 ** -8 * want.abs() + 2.0 ** -6 * want.abs().amax())
        else:
            assert torch.all((got - want).abs() <= 2.0 ** -7 * want.abs() + bound)
    assert torch.equal(ops.moe_grouped_gemm(act[rows.long()].contiguous(), None, offs, fmt, t, scale, N, K, 257, 0, block_rows=0, tiled=True),
                       ops.moe_grouped_gemm(act, rows, offs, fmt, t, scale, N, K, 257, 0, block_rows=0, tiled=True))


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
@pytest.mark.parametrize("height,counts", [(32, [0, 1, 31, 32, 33, 64, 0, 7]), (64, [63, 64, 65, 0, 1, 130]), (96, [95, 96, 97, 1, 193, 0]),
                                           (128, [127, 128, 129, 1, 257])])
def test_byte_experts_in_blocks_of_each_height(gpu, oracle, fmt, height, counts):
    """Routes per expert choose a block's rows (32 up to 24 on average, 64 up to 54, 96 up to 84, else 128): experts at a block's edges,
    three steps of 64 k-values and two, columns off a block.  The bound of the test above."""
    import torch
    from pie_amd import ops

    each = sum(counts) / len(counts)
    assert height == (32 if each <= 24 else 64 if each <= 54 else 96 if each <= 84 else 128)
    N, K = 272, 192 if height < 96 else 128
    rng = np.random.default_rng(580 + height)
    E, T, routes = len(counts), 70, sum(counts)
    offs = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), gpu)
    rows = dev(rng.integers(0, T, routes).astype(np.int32), gpu)
    act = dev(oracle.f32_to_bf16(rng.standard_normal((T, K)).astype(np.float32)), gpu, torch.bfloat16)
    w = dev(rng.integers(-128, 128, (E, N, K)).astype(np.int8) if fmt == "int8"
            else rng.integers(0, 0x70, (E, N, K)).astype(np.uint8) | (rng.integers(0, 2, (E, N, K)) << 7).astype(np.uint8), gpu)
    scale = dev(rng.uniform(0.001, 0.004, (E, N)).astype(np.float32), gpu).bfloat16()
    t = ops.repack_mfma_tiles(ops.WeightView(fmt, w.reshape(E * N, K), scale.reshape(-1), 0, E * N, K)).data.reshape(E, N, K)
    bound = K * 4.0 * 0.004 * (128 if fmt == "int8" else 256) * 2 * K * 2.0 ** -24
    want = ops.moe_grouped_gemm(act, rows, offs, fmt, w, scale, N, K, 257, 0, block_rows=128).float()
    got = ops.moe_grouped_gemm(act, rows, offs, fmt, t, scale, N, K, 257, 0, block_rows=0, tiled=True)
    assert torch.all((got.float() - want).abs() <= 2.0 ** -7 * want.abs() + bound)
    assert torch.equal(ops.moe_grouped_gemm(act, rows, offs, fmt, t, scale, N, K, 257, 0, True, block_rows=0, tiled=True),
                       ops.swiglu_bf16(torch.cat([got[:, 0::2], got[:, 1::2]], dim=1).contiguous()))


@pytest.mark.parametrize("fmt", ["int8", "fp8"])
def test_byte_experts_in_blocks_of_128_where_asked(gpu, oracle, fmt):
    """block_rows = 128 with few routes: the same sums as in the smaller blocks the rule takes; other heights are refused."""
    import torch
    from pie_amd import ops

    counts, T, N, K = [0, 1, 31, 33, 7], 40, 160, 192
    rng = np.random.default_rng(599)
    E, routes = len(counts), sum(counts)
    assert ops.moe_block_rows(routes, E) == 32 and ops.moe_block_rows(routes, E, 128) == 128
    offs = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int32), gpu)
    rows = dev(rng.integers(0, T, routes).astype(np.int32), gpu)
    act = dev(oracle.f32_to_bf16(rng.standard_normal((T, K)).astype(np.float32)), gpu, torch.bfloat16)
    w = dev(rng.integers(-128, 128, (E, N, K)).astype(np.int8) if fmt == "int8" else rng.integers(0, 0x70, (E, N, K)).astype(np.uint8), gpu)
    scale = dev(rng.uniform(0.001, 0.004, (E, N)).astype(np.float32), gpu).bfloat16()
    t = ops.repack_mfma_tiles(ops.WeightView(fmt, w.reshape(E * N, K), scale.reshape(-1), 0, E * N, K)).data.reshape(E, N, K)
    call = lambda block_rows: ops.moe_grouped_gemm(act, rows, offs, fmt, t, scale, N, K, 257, 0, block_rows=block_rows, tiled=True)  # noqa: E731
    assert torch.equal(call(128), call(0))
    with pytest.raises(ops.KernelError):
        call(64)


@pytest.mark.parametrize("tokens", [128, 129, 2048, 2049])
def test_sorted_layout_of_prompts(gpu, tokens):
    """A block sorts 1025 to 16384 routes out of its registers, others out of memory: either way each expert's routes are together,
    between its offsets, and name their tokens."""
    import torch
    from pie_amd import ops

    E, K = 128, 8
    logits = torch.randn(tokens, E, generator=torch.Generator(device=gpu).manual_seed(570 + tokens), device=gpu).to(torch.bfloat16)
    idx, _, offs, rtok, rpos = ops.moe_route(logits, K)
    flat, pos = idx.reshape(-1).long(), rpos.reshape(-1).long()
    assert torch.equal(pos.sort().values, torch.arange(tokens * K, device=gpu))
    assert torch.equal(offs.long(), torch.cat([torch.zeros(1, dtype=torch.long, device=gpu), torch.bincount(flat, minlength=E).cumsum(0)]))
    assert torch.all((pos >= offs.long()[flat]) & (pos < offs.long()[flat + 1]))
    assert torch.equal(rtok.long()[pos], torch.arange(tokens * K, device=gpu) // K)
