"""GPU parity: matrix-core prefill attention (tiles of query rows over paged KV) against the CPU
oracle's per-row attention and against the per-row kernel."""
import numpy as np
import pytest

from paged_cases import make_paged_batch

pytestmark = pytest.mark.gpu


def build_rows(b, ctx, chunks, tile_rows):
    """chunks[r] = (first position, count) of request r's query tokens -> row arrays + tiles."""
    row_begin, row_len, tiles = [], [], []
    for r, (p0, n) in enumerate(chunks):
        base = len(row_begin)
        for i in range(n):
            row_begin.append(int(b["page_indptr"][r]))
            row_len.append(min(ctx[r], p0 + i + 1))
        for t0 in range(0, n, tile_rows):
            tiles.append((base + t0, min(tile_rows, n - t0)))
    return (np.array(row_begin, np.int32), np.array(row_len, np.int32),
            np.array([t[0] for t in tiles], np.int32), np.array([t[1] for t in tiles], np.int32))


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hq,hk,d,ps", [(8, 2, 128, 16), (8, 1, 128, 32), (4, 2, 64, 16), (4, 4, 64, 16),
                                        (32, 8, 128, 16), (8, 2, 128, 48)])
def test_tiles_match_oracle_and_row_kernel(gpu, oracle, hq, hk, d, ps, half):
    import torch

    from pie_amd import ops

    rng = np.random.default_rng(60 + hq + d)
    ctx = [200, 75, 33, 1]
    b = make_paged_batch(rng, ctx, hk, d, ps, f32_to_bf16=oracle.f32_to_bf16)
    tr = ops.attn_prefill_tile_rows(hq, hk)
    assert tr == 128 // (hq // hk)
    if half:
        tr //= 2
    # a later chunk of a long prompt, a whole short prompt, a prompt shorter than a tile, one token
    chunks = [(120, 80), (0, 75), (0, 33), (0, 1)]
    row_begin, row_len, tile_start, tile_n = build_rows(b, ctx, chunks, tr)
    rows = len(row_begin)
    q = oracle.f32_to_bf16(rng.standard_normal((rows, hq, d)).astype(np.float32))
    dev = lambda a, dt=None: (lambda t: t.view(dt) if dt is not None else t)(
        torch.from_numpy(np.ascontiguousarray(a)).to(gpu))
    args = (dev(q, torch.bfloat16), dev(b["k_pages"], torch.bfloat16), dev(b["v_pages"], torch.bfloat16),
            dev(b["page_indices"].view(np.int32)), dev(row_begin), dev(row_len))
    o = ops.attention_prefill_tiles(*args, dev(tile_start), dev(tile_n), rows_per_tile=tr)
    torch.cuda.synchronize()
    got_bits = o.view(torch.uint16).cpu().numpy()
    got = oracle.bf16_to_f32(got_bits).astype(np.float64)
    truth, _, _ = oracle.attn_rows_masked(q, b["k_pages"], b["v_pages"], b["page_indices"], row_begin,
                                          row_len, hq, hk, d, ps, [None] * rows)
    # one bf16 rounding of the output + fp32 softmax / accumulation error: the decode kernels' bar
    # (the weights reach the second product as hi + lo bf16 pairs, 16 significant bits)
    tol = 2.0 ** -8 * np.maximum(np.abs(truth), np.abs(got)) + 1e-4
    err = np.abs(got - truth)
    assert np.all(err <= tol), f"worst {np.max(err / tol):.2f}x tol at {np.unravel_index(np.argmax(err / tol), err.shape)}"
    row = ops.attention_rows_paged(*args, int(row_len.max())).view(torch.uint16).cpu().numpy()
    # against the per-row kernel (fp32 weights): the same bar, and mostly the same bf16 value
    # (ulp distances grow without bound for outputs near zero, so they are only counted)
    rowf = oracle.bf16_to_f32(row).astype(np.float64)
    assert np.all(np.abs(got - rowf) <= 2.0 ** -7 * np.maximum(np.abs(rowf), np.abs(got)) + 2e-4)
    ulp = np.abs(got_bits.astype(np.int32) - row.astype(np.int32))
    assert (ulp <= 1).mean() > 0.97


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hq,hk,d,ps", [(8, 2, 128, 16), (4, 4, 64, 48), (8, 1, 64, 16), (32, 8, 128, 64)])
def test_scores_that_outgrow_their_reference(gpu, oracle, hq, hk, d, ps, half):
    """Keys that grow along the context, shrink along it, or jump at its end: what the exponents are relative to has to move at many
    steps, at the first only, or at the last, past contexts of one to several pages and steps that end inside a page.  Against the oracle: a
    bf16 rounding, and weights off by the float32 sums of d products behind them (2^-24 d of the products' magnitude, twice: a weight
    and its sum)."""
    import torch

    from pie_amd import ops

    rng = np.random.default_rng(90 + hq + d + ps)
    ctx = [300, 97, 33, 161]
    b = make_paged_batch(rng, ctx, hk, d, ps, f32_to_bf16=oracle.f32_to_bf16)
    k = oracle.bf16_to_f32(b["k_pages"]).copy()
    grow = [lambda x: 0.2 + 6.0 * x, lambda x: 6.2 - 6.0 * x, lambda x: np.where(x > 0.9, 8.0, 0.1), lambda x: 0.2 + 6.0 * x * x]
    for r, n in enumerate(ctx):
        for j in range(n):
            page = b["page_indices"][int(b["page_indptr"][r]) + j // ps]
            k[page, j % ps] *= grow[r](j / n)
    kb = oracle.f32_to_bf16(k.astype(np.float32)).reshape(b["k_pages"].shape)
    tr = ops.attn_prefill_tile_rows(hq, hk) // (2 if half else 1)
    chunks = [(220, 80), (0, 97), (0, 33), (155, 6)]
    row_begin, row_len, tile_start, tile_n = build_rows(b, ctx, chunks, tr)
    rows = len(row_begin)
    q = oracle.f32_to_bf16(3.0 * rng.standard_normal((rows, hq, d)).astype(np.float32))
    dev = lambda a, dt=None: (lambda t: t.view(dt) if dt is not None else t)(
        torch.from_numpy(np.ascontiguousarray(a)).to(gpu))
    o = ops.attention_prefill_tiles(dev(q, torch.bfloat16), dev(kb, torch.bfloat16), dev(b["v_pages"], torch.bfloat16),
                                    dev(b["page_indices"].view(np.int32)), dev(row_begin), dev(row_len), dev(tile_start), dev(tile_n),
                                    rows_per_tile=tr)
    got = oracle.bf16_to_f32(o.view(torch.uint16).cpu().numpy()).astype(np.float64)
    truth, _, _ = oracle.attn_rows_masked(q, kb, b["v_pages"], b["page_indices"], row_begin, row_len, hq, hk, d, ps, [None] * rows)
    qf, vf = np.abs(oracle.bf16_to_f32(q)), np.abs(oracle.bf16_to_f32(b["v_pages"]))
    mass = (qf.reshape(rows, -1, d) * np.abs(k).max(axis=(0, 1)).max(axis=0)).sum(-1).max() / np.sqrt(d)
    tol = 2.0 ** -8 * np.maximum(np.abs(truth), np.abs(got)) + 2 * d * 2.0 ** -24 * mass * vf.max()
    err = np.abs(got - truth)
    assert np.all(err <= tol), f"worst {np.max(err / tol):.2f}x"
    assert np.sqrt((err ** 2).mean()) <= 2.0 ** -9 * np.sqrt((truth ** 2).mean())


@pytest.mark.parametrize("off_k,off_v", [(4, 0), (0, 4), (4, 4)])
@pytest.mark.parametrize("hq,hk,d,ps", [(8, 2, 128, 16), (4, 4, 64, 48)])
def test_pools_off_a_16_byte_boundary(gpu, oracle, hq, hk, d, ps, off_k, off_v):
    """Pools that begin 8 bytes behind one (which transfers into LDS do not take) give the same bytes."""
    import torch

    from pie_amd import ops

    rng = np.random.default_rng(95 + d)
    ctx = [200, 75, 33, 1]
    b = make_paged_batch(rng, ctx, hk, d, ps, f32_to_bf16=oracle.f32_to_bf16)
    tr = ops.attn_prefill_tile_rows(hq, hk) // 2
    row_begin, row_len, tile_start, tile_n = build_rows(b, ctx, [(120, 80), (0, 75), (0, 33), (0, 1)], tr)
    q = oracle.f32_to_bf16(rng.standard_normal((len(row_begin), hq, d)).astype(np.float32))
    dev = lambda a, dt=None: (lambda t: t.view(dt) if dt is not None else t)(
        torch.from_numpy(np.ascontiguousarray(a)).to(gpu))

    def shifted(t, off):
        flat = torch.zeros(t.numel() + 8, dtype=t.dtype, device=t.device)
        assert flat.data_ptr() % 16 == 0
        flat[off:off + t.numel()] = t.reshape(-1)
        return flat[off:off + t.numel()].view(t.shape)

    qd, k, v = dev(q, torch.bfloat16), dev(b["k_pages"], torch.bfloat16), dev(b["v_pages"], torch.bfloat16)
    rest = (dev(b["page_indices"].view(np.int32)), dev(row_begin), dev(row_len), dev(tile_start), dev(tile_n))
    want = ops.attention_prefill_tiles(qd, k, v, *rest, rows_per_tile=tr)
    got = ops.attention_prefill_tiles(qd, shifted(k, off_k), shifted(v, off_v), *rest, rows_per_tile=tr)
    assert torch.equal(want.view(torch.int16), got.view(torch.int16))


@pytest.mark.parametrize("fmt", ["fp8_e4m3", "int8_per_token_head", "fp8_per_token_head", "fp8_e5m2"])
@pytest.mark.parametrize("hq,hk,d,ps", [(8, 2, 128, 16), (4, 4, 64, 16), (32, 8, 128, 32)])
@pytest.mark.parametrize("half", [False, True])
def test_tiles_over_one_byte_pools_match_the_oracle(gpu, oracle, fmt, hq, hk, d, ps, half):
    """The tile kernel over quantised pools against the oracle's attention over the dequantised
    values float(code) * scale (codes and scales written by the library's quantising write,
    itself bit-exact against the oracle's quantiser), to the bar of the bf16 pools; the per-row
    kernel over the same pools is compared as well."""
    import torch

    from pie_amd import ops

    rng = np.random.default_rng(70 + hq + d)
    ctx = [200, 75, 33, 1]
    b = make_paged_batch(rng, ctx, hk, d, ps, f32_to_bf16=oracle.f32_to_bf16)
    tr = ops.attn_prefill_tile_rows(hq, hk) // (2 if half else 1)
    chunks = [(120, 80), (0, 75), (0, 33), (0, 1)]
    row_begin, row_len, tile_start, tile_n = build_rows(b, ctx, chunks, tr)
    rows = len(row_begin)
    q = oracle.f32_to_bf16(rng.standard_normal((rows, hq, d)).astype(np.float32))
    dev = lambda a, dt=None: (lambda t: t.view(dt) if dt is not None else t)(
        torch.from_numpy(np.ascontiguousarray(a)).to(gpu))
    # quantise the bf16 pools slot by slot with the library's own write kernel
    pages = b["k_pages"].shape[0]
    kp = torch.zeros((pages, ps, hk, d), dtype=torch.uint8, device=gpu)
    vp = torch.zeros_like(kp)
    scaled = fmt not in ("fp8_e4m3", "fp8_e5m2")
    ks = torch.ones((pages, hk, ps), dtype=torch.float32, device=gpu) if scaled else None
    vs = torch.ones((pages, hk, ps), dtype=torch.float32, device=gpu) if scaled else None
    slots = dev(np.arange(pages * ps, dtype=np.int64))
    ops.kv_write_quant(fmt, dev(b["k_pages"], torch.bfloat16).reshape(pages * ps, hk, d),
                       dev(b["v_pages"], torch.bfloat16).reshape(pages * ps, hk, d), slots, kp, vp, ks, vs)
    qd, pi, rb, rl = dev(q, torch.bfloat16), dev(b["page_indices"].view(np.int32)), dev(row_begin), dev(row_len)
    o = ops.attention_prefill_tiles_kvq(fmt, qd, kp, vp, ks, vs, pi, rb, rl, dev(tile_start), dev(tile_n),
                                        rows_per_tile=tr)
    ref = ops.attention_rows_paged_kvq(fmt, qd, kp, vp, ks, vs, pi, rb, rl)[0]
    torch.cuda.synchronize()
    got = oracle.bf16_to_f32(o.view(torch.uint16).cpu().numpy()).astype(np.float64)
    # the oracle: its own quantiser on the same bf16 rows (the codes the GPU wrote, bit for bit),
    # attention in double over float(code) * scale
    deq = {}
    for name in ("k_pages", "v_pages"):
        codes, scales, dq = oracle.kv_quant_rows(b[name].reshape(pages * ps * hk, d), fmt)
        deq[name] = dq.reshape(pages, ps, hk, d)
        pool = (kp if name == "k_pages" else vp).cpu().numpy()
        assert np.array_equal(pool.reshape(-1, d), codes)
    truth, _, _ = oracle.attn_rows_f32kv(q, deq["k_pages"], deq["v_pages"], b["page_indices"], row_begin, row_len,
                                         hq, hk, d, ps, mode=2)
    tol = 2.0 ** -8 * np.maximum(np.abs(truth), np.abs(got)) + 1e-4
    err = np.abs(got - truth)
    assert np.all(err <= tol), f"worst {np.max(err / tol):.2f}x tol"
    want = oracle.bf16_to_f32(ref.view(torch.uint16).cpu().numpy()).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -7 * np.maximum(np.abs(want), np.abs(got)) + 2e-4)


@pytest.mark.parametrize("fmt", ["bf16", "fp8_per_token_head", "int8_per_token_head", "fp8_e5m2"])
@pytest.mark.parametrize("d", [64, 128])
def test_many_tiles_equal_few(gpu, d, fmt):
    """Above 512 blocks a block's waves walk all keys, up to there two groups of them take every other step and meet at the end:
    the same weights and sums in another order, one bf16 rounding each (the bar of the first test, twice).  Extents on and beside
    the steps of 32 keys, tiles of one row; up to four steps, which one group takes alone, and beyond: the second group's last step
    of one key, whole, and missing."""
    import torch
    from pie_amd import ops

    hq, hk, ps = 32, 8, 16
    tr = ops.attn_prefill_tile_rows(hq, hk) // 2
    ctx = [1, 31, 32, 33, 64, 65, 97, 128, 129, 160, 161, 193, 700]
    pages = [-(-c // ps) for c in ctx]
    first = np.concatenate([[0], np.cumsum(pages)])
    row_begin = np.concatenate([np.full(c, f) for c, f in zip(ctx, first)]).astype(np.int32)
    row_len = np.concatenate([np.arange(1, c + 1) for c in ctx]).astype(np.int32)
    tiles, at = [], 0
    for c in ctx:
        tiles += [(at + t, min(tr, c - t)) for t in range(0, c, tr)]
        at += c
    assert len(tiles) * hk > 512
    g = torch.Generator(device=gpu).manual_seed(63 + d)
    rnd = lambda *shape: torch.randn(*shape, generator=g, device=gpu).to(torch.bfloat16)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)
    n = int(first[-1])
    kp, vp = rnd(n, ps, hk, d), rnd(n, ps, hk, d)
    ks = vs = None
    if fmt != "bf16":
        k_rows, v_rows = kp.reshape(-1, hk, d), vp.reshape(-1, hk, d)
        kp, vp = (torch.zeros((n, ps, hk, d), dtype=torch.uint8, device=gpu) for _ in range(2))
        if fmt != "fp8_e5m2":
            ks, vs = (torch.ones((n, hk, ps), dtype=torch.float32, device=gpu) for _ in range(2))
        ops.kv_write_quant(fmt, k_rows, v_rows, torch.arange(n * ps, device=gpu), kp, vp, ks, vs)
    args = (fmt, rnd(at, hq, d), kp, vp, ks, vs, torch.randperm(n, generator=g, device=gpu).int(), dev(row_begin), dev(row_len))
    start, count = (dev(np.array(x, np.int32)) for x in zip(*tiles))
    run = (lambda *tl: ops.attention_prefill_tiles_kvq(*args, *tl, rows_per_tile=tr)) if fmt != "bf16" else \
        (lambda *tl: ops.attention_prefill_tiles(args[1], kp, vp, *args[6:], *tl, rows_per_tile=tr))
    whole = run(start, count).float()
    half = len(tiles) // 2
    assert (len(tiles) - half) * hk <= 512
    parts = torch.zeros_like(whole)
    for sl in (slice(0, half), slice(half, None)):
        o = run(start[sl].contiguous(), count[sl].contiguous()).float()
        for a, m in zip(start[sl].tolist(), count[sl].tolist()):
            parts[a:a + m] = o[a:a + m]
    assert torch.all((whole - parts).abs() <= 2.0 ** -7 * torch.maximum(whole.abs(), parts.abs()) + 2e-4)
