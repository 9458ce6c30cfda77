// Weights times a few to some hundred activation rows: y[M, N] = epilogue( act[M, K] · W[N, K]^T ) over the tile-major copy (bf16 also row-major), the skinny
// GEMM's arithmetic (int8 and fp8 codes scaled by row at the end, an int4 group's code products summed as they are and scaled once, in fp32).
//
// A block is eight waves over the same 16 MT rows and 16 NG columns, and each wave has its own steps of K (64 values, int4 128; wave w the steps w, w + 8, ..): it
// takes its weights straight into registers, brings its rows' values of a step into an LDS region of its own, and waits for nobody until the
// waves' sums meet in LDS at the end.  Two waves to a SIMD: one's transfers, reads and decoding run beside the other's products.
// Why so: these launches are latency.  Blocks whose waves share the activations cross a barrier every step and move a step as slowly as its
// last transfer: 77 rows of 2048 x 2048 int8 took 13.5 us (rings of three to eight steps: the same), passes of 32 rows, which read and decode the weights once
// each, 7.8, this 5.4.  And waves that own columns instead of steps all read the same activations out of LDS: at 64 columns that is 4.6 us
// of LDS time for 77 x 16384 x 2048, a quarter of it here.
// What bounds it: bringing the activations to the CUs (315 KB of 77 rows x 2048 at some 100 bytes a nanosecond, plus as many LDS bytes in and
// out), and with many columns the weights' stream.  Activations by plain loads in the products' layout: 10 - 60 % slower (sixteen rows to a quarter of a
// wave in the address unit); two steps in flight for four waves: the same up to 256 blocks.
// us before / here, weights out of HBM: int8 77 rows of 3072 x 2048 10.6 / 6.1, 16384 x 2048 17.5 / 15.1, 2048 x 8192 15.9 / 12.3; 16 rows of 2048 x 8192 11.2 / 6.1 in shares; 256
// rows of 3072 x 2048 14.4 / 9.3; int4 16 / 64 rows of 4096 x 4096 6.2 / 5.5 and 9.6 / 7.3, 64 of 6144 x 4096 12.7 / 10.4; bf16 77 rows of 3072 x 2048 9.8 / 7.0, 16384 x 2048
// 22.3 / 18.2, 192 of 2048 x 8192 26.2 / 22.3; row-major bf16, as an output head is, 16 / 40 rows of 32000 x 4096 53.2 / 48.8 and 59.1 - 70.0 / 53.4.
#include "gemm_args.hip.h"

#include <algorithm>
#include <cmath>

namespace pie_hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kBlockWaves = 8;

// kSub: products of 32 k-values in a step; kPieces: wave loads of 1 KiB that a tile's weights of a step are
struct WvInt8 {
    static constexpr int kSub = 2, kPieces = 1;
    static constexpr bool kGroups = false, kLds = false;
    static __device__ __forceinline__ bf16x8_t decode(const u32x4_t& r, int s, uint32_t) {
        return __builtin_bit_cast(bf16x8_t, kv_decode_bf16<kKvInt8>(u32x2_t{r[2 * s], r[2 * s + 1]}));
    }
};
struct WvFp8 {
    static constexpr int kSub = 2, kPieces = 1;
    static constexpr bool kGroups = false, kLds = false;
    static __device__ __forceinline__ bf16x8_t decode(const u32x4_t& r, int s, uint32_t) {
        return __builtin_bit_cast(bf16x8_t, kv_decode_bf16<kKvFp8>(u32x2_t{r[2 * s], r[2 * s + 1]}));
    }
};
struct WvInt4 {
    static constexpr int kSub = 4, kPieces = 1;
    static constexpr bool kGroups = true, kLds = false;
    static __device__ __forceinline__ bf16x8_t decode(const u32x4_t& r, int s, uint32_t k128) {   // 128 + n
        const uint32_t v = r[s];
        return __builtin_bit_cast(bf16x8_t, u32x4_t{and_or(v, 0x000F000Fu, k128), and_or(v >> 4, 0x000F000Fu, k128),
                                                    and_or(v >> 8, 0x000F000Fu, k128), and_or(v >> 12, 0x000F000Fu, k128)});
    }
};
struct WvBf16 {
    static constexpr int kSub = 2, kPieces = 2;
    static constexpr bool kGroups = false, kLds = false;
    static __device__ __forceinline__ bf16x8_t decode(const u32x4_t& r, int, uint32_t) { return __builtin_bit_cast(bf16x8_t, r); }
};
// (row-major: sixteen rows to a quarter of a wave would keep the address unit busy, so they come as the activations do, whole lines into the wave's LDS region.
// From the copy the same takes 0.93 at the median of 250 products, 0.78 of 16384 x 2048.)
struct WvBf16Rows {
    static constexpr int kSub = 2, kPieces = 2;
    static constexpr bool kGroups = false, kLds = true;
};

// place of a row's 16-byte granule c: conflict-free for the transfers (whole rows) and for the products' reads
template <int SUB>
__device__ __forceinline__ int swizzle(int row, int c) { return SUB == 4 ? c ^ key_of(row) : c ^ ((row >> 1) & 7); }

template <class F, int MT, int NG>
__global__ __launch_bounds__(64 * kBlockWaves, 1) void gemm_waves_kernel(const GemmArgs a, const Rotation rot, int row_blocks, int per_xcd, int blocks, int per_share) {
    constexpr int SUB = F::kSub, kGranules = 4 * SUB, kRowVecs = MT * 16 * kGranules, kVecs = kRowVecs + (F::kLds ? NG * 16 * kGranules : 0), AC = MT * SUB, WC = F::kLds ? NG * SUB : NG, PC = F::kPieces, KP = kBlockWaves, kTiles = MT * NG;
    constexpr int kOwn = (kTiles + KP - 1) / KP;   // output tiles a wave finishes
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 15, q = lane >> 4;
    // blocks go to the XCDs in turn: each XCD's are neighbours, the row blocks of a column block side by side
    const int block = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (static_cast<int>(blockIdx.x >> 3) >= per_xcd || block >= blocks) return;
    u32x4_t* lds = reinterpret_cast<u32x4_t*>(smem) + wv * kVecs;
    const int m0 = block % row_blocks * (MT * 16), tile0 = block / row_blocks * NG;
    const int N = a.N, K = a.K, M = a.M, T = N / 16, steps = K / (32 * SUB);
    const int first = static_cast<int>(blockIdx.z) * per_share, nk_all = min(per_share, steps - first);
    const int nk = (nk_all - wv + KP - 1) / KP;   // this wave's steps
    auto place = [&](int kt) { return first + wv + KP * kt; };
    const int groups = F::kGroups ? K >> a.g_shift : 0, to_group = F::kGroups ? a.g_shift - 7 : 0;

    uint32_t woff[WC], soff[NG], aoff[AC];
#pragma unroll
    for (int i = 0; i < WC; ++i) {
        if constexpr (F::kLds) {
            const int r = (i * kWave + lane) / kGranules;
            woff[i] = static_cast<uint32_t>(min(tile0 * 16 + r, N - 1)) * (2u * K) + swizzle<SUB>(r, lane & (kGranules - 1)) * 16;
            continue;
        }
        const uint32_t tile = min(tile0 + i, T - 1);
        woff[i] = tile * (steps * (PC * 1024u)) + lane * 16u;
        soff[i] = tile * (groups * 32u) + q * 8u;
    }
#pragma unroll
    for (int u = 0; u < AC; ++u) {
        const int r = (u * kWave + lane) / kGranules;
        aoff[u] = static_cast<uint32_t>(min(m0 + r, M - 1)) * (2u * K) + swizzle<SUB>(r, lane & (kGranules - 1)) * 16;
    }
    u32x4_t raw[NG][PC];
    auto granule = [&](int s) __attribute__((always_inline)) { return PC == 2 ? 4 * s + q : SUB * q + s; };   // of product s of a step
    u32x2_t gs[NG];
    auto load_w = [&](int kt, int i) __attribute__((always_inline)) {
        const int p = place(kt);
        asm volatile("" : "+v"(woff[i]), "+v"(soff[i]));   // (32-bit offsets from scalar bases, not 64-bit sums)
#pragma unroll
        for (int c = 0; c < PC; ++c) raw[i][c] = *reinterpret_cast<const u32x4_t*>(a.w + (static_cast<size_t>(p) * PC + c) * 1024 + woff[i]);
        if constexpr (F::kGroups) gs[i] = *reinterpret_cast<const u32x2_t*>(a.scale + static_cast<size_t>(p >> to_group) * 32 + soff[i]);
    };
    auto issue_a = [&](int kt) __attribute__((always_inline)) {
        const unsigned char* pa = reinterpret_cast<const unsigned char*>(a.act) + static_cast<size_t>(place(kt)) * (64 * SUB);
#pragma unroll
        for (int u = 0; u < AC; ++u) {
            asm volatile("" : "+v"(aoff[u]));
            to_lds(pa + aoff[u], lds + u * kWave);
        }
        PIE_FENCE();
    };
    auto issue = [&](int kt) __attribute__((always_inline)) {
        if constexpr (F::kLds) {
            const unsigned char* pw = a.w + static_cast<size_t>(place(kt)) * (64 * SUB);
#pragma unroll
            for (int i = 0; i < WC; ++i) {
                asm volatile("" : "+v"(woff[i]));
                to_lds(pw + woff[i], lds + kRowVecs + i * kWave);
            }
        } else {
#pragma unroll
            for (int i = 0; i < NG; ++i) load_w(kt, i);
        }
        PIE_FENCE();
        issue_a(kt);
    };
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[MT][NG];
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int n = 0; n < NG; ++n) acc[t][n] = zero;
    if (nk > 0) issue(0);
    // (what the end needs is asked for here: scalar loads left for then would be waited for one after another)
    uint16_t* y = a.y;
    const unsigned char* row_scale = a.scale;
    float* partial = a.partial;
    int beta = a.beta, aligned = a.aligned, bf16_scale = a.scale_is_bf16;
    asm volatile("" : "+s"(y), "+s"(row_scale), "+s"(partial), "+s"(beta), "+s"(aligned), "+s"(bf16_scale));
    const bool add = beta && aligned && !partial;
    uint32_t k128 = 0x43004300u;   // (128.0, 128.0) as a bf16 pair, opaque to the compiler
    asm volatile("" : "+v"(k128));
    const bf16x8_t offset = __builtin_bit_cast(bf16x8_t, u32x4_t{0xC308C308u, 0xC308C308u, 0xC308C308u, 0xC308C308u});   // -136
    for (int kt = 0; kt < nk; ++kt) {
        PIE_WAIT_VM(0);
        asm volatile("" ::: "memory");
        bf16x8_t af[SUB][MT];
#pragma unroll
        for (int s = 0; s < SUB; ++s)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                af[s][t] = __builtin_bit_cast(bf16x8_t, lds[(t * 16 + j) * kGranules + swizzle<SUB>(j, granule(s))]);
        if constexpr (F::kGroups) {
            // (a group's sum starts from -136 times the activations' sums: the codes are multiplied as 128 + n, n of 0 .. 15 for -8 .. 7)
            f32x4_t sx[MT];
#pragma unroll
            for (int s = 0; s < SUB; ++s)
#pragma unroll
                for (int t = 0; t < MT; ++t) sx[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(offset, af[s][t], s ? sx[t] : zero, 0, 0, 0);
            PIE_WAIT_LGKM0();   // (the rows are in registers: the next step's may land)
            PIE_FENCE();
            asm volatile("" ::: "memory");
            if (kt + 1 < nk) issue_a(kt + 1);
#pragma unroll
            for (int n = 0; n < NG; ++n) {
                f32x4_t sum[MT];
#pragma unroll
                for (int s = 0; s < SUB; ++s) {
                    const bf16x8_t bw = F::decode(raw[n][PC == 2 ? s : 0], s, k128);
#pragma unroll
                    for (int t = 0; t < MT; ++t) sum[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw, af[s][t], s ? sum[t] : sx[t], 0, 0, 0);
                }
                const float sc[4] = {bf16_lo(gs[n].x), bf16_hi(gs[n].x), bf16_lo(gs[n].y), bf16_hi(gs[n].y)};
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[t][n][r] = fmaf(sc[r], sum[t][r], acc[t][n][r]);
                load_w(min(kt + 1, nk - 1), n);   // (no branch between the products: behind the last step its own weights once more)
            }
        } else {
            bf16x8_t bw[SUB][NG];
#pragma unroll
            for (int s = 0; s < SUB; ++s)
#pragma unroll
                for (int n = 0; n < NG; ++n) {
                    if constexpr (F::kLds) bw[s][n] = __builtin_bit_cast(bf16x8_t, lds[kRowVecs + (n * 16 + j) * kGranules + swizzle<SUB>(j, granule(s))]);
                    else bw[s][n] = F::decode(raw[n][PC == 2 ? s : 0], s, k128);
                }
            PIE_WAIT_LGKM0();
            PIE_FENCE();
            asm volatile("" ::: "memory");
            if (kt + 1 < nk) issue(kt + 1);
#pragma unroll
            for (int s = 0; s < SUB; ++s)
#pragma unroll
                for (int t = 0; t < MT; ++t)
#pragma unroll
                    for (int n = 0; n < NG; ++n) acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[s][n], af[s][t], acc[t][n], 0, 0, 0);
        }
        PIE_FENCE();
    }
    // what the tiles this wave finishes need, asked for ahead of the meeting: residual, row scales, or slot and angles
    u32x2_t old[kOwn];
    float rs[kOwn][4];
#pragma unroll
    for (int c = 0; c < kOwn; ++c) {
        const int tile = min(c * KP + wv, kTiles - 1), m = min(m0 + tile / NG * 16 + j, M - 1), n = min((tile0 + tile % NG) * 16 + 4 * q, N - 4);
        old[c] = u32x2_t{0, 0};
        if (add) old[c] = *reinterpret_cast<const u32x2_t*>(y + static_cast<size_t>(m) * N + n);
        if constexpr (!F::kGroups && PC == 1) {
            if (bf16_scale) {
#pragma unroll
                for (int r = 0; r < 4; ++r) rs[c][r] = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(row_scale)[n + r]);
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) rs[c][r] = reinterpret_cast<const float*>(row_scale)[n + r];
            }
        }
    }
    PIE_FENCE();
    PIE_MEET();   // (every wave has read its last rows, and no transfer is on its way)
    f32x4_t* meet = reinterpret_cast<f32x4_t*>(smem);   // [wave][tile][lane]
#pragma unroll
    for (int t = 0; t < MT; ++t)
#pragma unroll
        for (int n = 0; n < NG; ++n) meet[(wv * kTiles + t * NG + n) * kWave + lane] = acc[t][n];
    PIE_WAIT_LGKM0();
    PIE_MEET();
    // (lane: row j, columns 4q .. 4q + 3 of a tile)
#pragma unroll
    for (int c = 0; c < kOwn; ++c) {
        const int tile = c * KP + wv;
        if (tile >= kTiles) break;
        f32x4_t sum = meet[tile * kWave + lane];
#pragma unroll
        for (int p = 1; p < KP; ++p) sum += meet[(p * kTiles + tile) * kWave + lane];
        const int m = m0 + tile / NG * 16 + j, n = (tile0 + tile % NG) * 16 + 4 * q;
        if (m >= M || n >= N) continue;
        float v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v[r] = sum[r];
            if constexpr (!F::kGroups && PC == 1) v[r] *= rs[c][r];
        }
        if (partial) {
            *reinterpret_cast<f32x4_t*>(partial + (static_cast<size_t>(blockIdx.z) * M + m) * N + n) = f32x4_t{v[0], v[1], v[2], v[3]};
        } else if (add) {
            const float o[4] = {bf16_lo(old[c].x), bf16_hi(old[c].x), bf16_lo(old[c].y), bf16_hi(old[c].y)};
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += o[r];
            *reinterpret_cast<u32x2_t*>(y + static_cast<size_t>(m) * N + n) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
        } else {
            store4(a, rot, m, n, v);
        }
    }
}

template <class F, int MT, int NG>
int launch(const GemmArgs& a, const Rotation& rot, int shares, hipStream_t stream) {
    constexpr size_t rows_bytes = kBlockWaves * (MT + (F::kLds ? NG : 0)) * F::kSub * 1024, meet_bytes = kBlockWaves * MT * NG * 1024, smem = rows_bytes > meet_bytes ? rows_bytes : meet_bytes;
    static_assert(smem <= 160 * 1024, "");
    constexpr auto kernel = &gemm_waves_kernel<F, MT, NG>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int rows = (a.M + MT * 16 - 1) / (MT * 16), blocks = rows * ((a.N / 16 + NG - 1) / NG), per = (blocks + 7) / 8, steps = a.K / (32 * F::kSub);
    hipLaunchKernelGGL(kernel, dim3(8 * per, 1, shares), dim3(64 * kBlockWaves), smem, stream, a, rot, rows, per, blocks, (steps + shares - 1) / shares);
    return launch_status();
}

struct Plan {
    int row_tiles = 0, tiles = 0, shares = 1;
    double us = 1e30;
};
template <class F, int MT>
int launch(const GemmArgs& a, const Rotation& rot, const Plan& p, hipStream_t stream) {
    if constexpr (MT <= 2)
        if (p.tiles == 1) return launch<F, MT, 1>(a, rot, p.shares, stream);
    return p.tiles == 2 ? launch<F, MT, 2>(a, rot, p.shares, stream) : launch<F, MT, 4>(a, rot, p.shares, stream);
}
template <class F>
int launch(const GemmArgs& a, const Rotation& rot, const Plan& p, hipStream_t stream) {
    switch (p.row_tiles) {
        case 1: return launch<F, 1>(a, rot, p, stream);
        case 2: return launch<F, 2>(a, rot, p, stream);
        case 3: return launch<F, 3>(a, rot, p, stream);
        case 4: return launch<F, 4>(a, rot, p, stream);
        default: break;
    }
    if constexpr (!F::kGroups) return launch<F, 5>(a, rot, p, stream);   // (80 rows of int4 weights do not fit the registers)
    return PIE_HIP_ERR_INVALID;
}

// Rows and columns of a block and shares of K.  A block takes `fixed` and, per step of its waves, `step`, of a full chip `full` more (the activations' way to
// the CUs); blocks past 256 take `again` of that and `start` each round; stores or the shares' sums 0.2 us a MiB.  That and what the weights take at 6 TB/s (int4
// and row-major bf16 5.5) add up as cubes: either alone where the other is short, a quarter more where they are equal.
// Shares that meet in a kernel of their own (`norm`: in the norm's) cost what gemm_groups_mfma.hip's do.  Fitted to 20000 launches of 720 products (5 - 480 rows, int4 - 384; 15 matrices
// of 1024 - 28672 x 1024 - 14336, weights out of HBM and rows that a kernel has just written): 7 - 9 % rms, and the plan taken is within 0.5 % of the fastest on
// average (the worst 19 %: 160 int8 rows of 2048 x 8192 in four shares 20.7 us, in whole rows 17.4).  Bf16, both orders, over 17 matrices up to 32000 x 4096: 8 - 10 % rms, 0.5 %
// over the fastest on average (the worst 16 %).
struct Cost {
    float fixed, step, full, again, start;
};
constexpr Cost kOneByte[5][3] = {{{1.00f, 0.61f, 0.00f, 0.44f, 0.29f}, {1.13f, 0.66f, 0.06f, 0.55f, 0.37f}, {1.67f, 0.76f, 0.18f, 0.74f, 0.37f}},
                                 {{1.24f, 0.61f, 0.13f, 0.68f, 0.25f}, {1.69f, 0.66f, 0.20f, 0.76f, 0.23f}, {2.33f, 0.87f, 0.34f, 0.71f, 0.54f}},
                                 {{1.50f, 0.68f, 0.22f, 0.72f, 0.42f}, {2.00f, 0.82f, 0.24f, 0.77f, 0.44f}, {3.34f, 1.07f, 0.37f, 0.71f, 3.75f}},
                                 {{1.75f, 0.87f, 0.23f, 0.74f, 0.44f}, {2.40f, 0.99f, 0.27f, 0.76f, 0.53f}, {3.81f, 1.25f, 0.45f, 0.72f, 3.89f}},
                                 {{2.13f, 0.97f, 0.29f, 0.74f, 0.44f}, {3.22f, 1.18f, 0.27f, 0.75f, 2.94f}, {4.65f, 1.49f, 0.42f, 0.78f, 4.22f}}};
constexpr Cost kInt4[4][3] = {{{1.25f, 0.83f, 0.00f, 0.61f, 0.42f}, {1.69f, 0.89f, 0.07f, 0.85f, 0.22f}, {2.28f, 1.16f, 0.15f, 0.84f, 0.31f}},
                              {{1.63f, 1.05f, 0.08f, 0.74f, 0.67f}, {2.08f, 1.11f, 0.21f, 0.82f, 0.34f}, {2.83f, 1.49f, 0.37f, 0.82f, 2.24f}},
                              {{2.04f, 1.26f, 0.26f, 0.75f, 2.41f}, {2.48f, 1.42f, 0.35f, 0.78f, 2.33f}, {3.69f, 1.95f, 0.39f, 0.85f, 2.64f}},
                              {{2.24f, 1.63f, 0.36f, 0.72f, 2.53f}, {2.88f, 1.84f, 0.39f, 0.78f, 2.58f}, {4.22f, 2.55f, 0.44f, 0.83f, 3.04f}}};
constexpr Cost kBf16[5][3] = {{{1.00f, 0.58f, 0.00f, 0.66f, 0.00f}, {1.06f, 0.64f, 0.14f, 0.72f, 0.00f}, {1.31f, 1.08f, 0.12f, 0.72f, 0.00f}},
                              {{1.60f, 0.59f, 0.12f, 0.81f, 0.00f}, {1.78f, 0.79f, 0.15f, 0.80f, 0.00f}, {2.16f, 1.23f, 0.22f, 0.78f, 2.04f}},
                              {{}, {2.18f, 0.97f, 0.17f, 0.82f, 0.06f}, {2.89f, 1.51f, 0.26f, 0.81f, 2.61f}},
                              {{}, {2.54f, 1.13f, 0.26f, 0.77f, 0.18f}, {3.47f, 1.65f, 0.39f, 0.79f, 2.93f}},
                              {{}, {3.18f, 1.38f, 0.24f, 0.77f, 2.25f}, {4.03f, 1.87f, 0.37f, 0.80f, 3.36f}}};
constexpr Cost kBf16Rows[5][3] = {{{1.00f, 0.56f, 0.00f, 0.91f, 0.00f}, {1.00f, 0.67f, 0.21f, 0.90f, 0.00f}, {1.00f, 1.25f, 0.24f, 0.80f, 0.00f}},
                                  {{1.35f, 0.58f, 0.22f, 0.89f, 0.00f}, {1.46f, 0.87f, 0.24f, 0.88f, 0.03f}, {1.85f, 1.37f, 0.39f, 0.78f, 2.31f}},
                                  {{}, {1.91f, 1.07f, 0.27f, 0.83f, 0.18f}, {2.63f, 1.62f, 0.41f, 0.74f, 3.28f}},
                                  {{}, {2.33f, 1.18f, 0.40f, 0.87f, 1.61f}, {3.24f, 1.73f, 0.65f, 0.72f, 3.54f}},
                                  {{}, {2.87f, 1.46f, 0.33f, 0.82f, 2.44f}, {3.90f, 1.99f, 0.50f, 0.77f, 3.85f}}};
// What was measured, and is taken: six blocks of rows, and 1100 blocks in all (70400 columns of up to 80 rows, int4 64: an output head of 128256 is past that).
constexpr int kRowBlocks = 6, kBlocks = 1100;
constexpr int most_rows(bool int4) { return kRowBlocks * (int4 ? 64 : 80); }
enum class Form { Int4, OneByte, Bf16, Bf16Rows };
Form form_of(int format, bool tiled) {
    return format == PIE_HIP_FMT_INT4B8 ? Form::Int4 : format != PIE_HIP_FMT_BF16 ? Form::OneByte : tiled ? Form::Bf16 : Form::Bf16Rows;
}
Plan find_plan(Form form, int M, int N, int K, size_t ws_bytes, bool norm) {
    const bool int4 = form == Form::Int4;
    const Cost(*costs)[3] = int4 ? kInt4 : form == Form::OneByte ? kOneByte : form == Form::Bf16 ? kBf16 : kBf16Rows;
    const int steps = K / (int4 ? 128 : 64);
    const double stream_us = 2.6 + 1e-6 * N * K * (int4 ? 0.516 / 5.5 : form == Form::OneByte ? 1.0 / 6.0 : form == Form::Bf16 ? 2.0 / 6.0 : 2.0 / 5.5);
    Plan best;
    for (int mt = 1; mt <= (int4 ? 4 : 5); ++mt) {
        const int rows = (M + mt * 16 - 1) / (mt * 16);
        if (rows > kRowBlocks || (rows > 1 && mt > 1 && rows * mt * 16 > 1.3 * M + 16)) continue;
        for (int n = mt <= 2 ? 0 : 1; n < 3; ++n) {   // (16 columns of 48 and more rows are next to never the fastest)
            const Cost& c = costs[mt - 1][n];
            const int tiles = rows * ((N / 16 + (1 << n) - 1) >> n);
            for (int s = norm ? 2 : 1; s <= 8; ++s) {
                const int per = (steps + s - 1) / s, blocks = tiles * s;
                const double bytes = 4.0 * s * M * N;
                if (blocks > (s > 1 ? 520 : kBlocks)) break;
                if (s > 1 && (per < 4 || bytes > static_cast<double>(ws_bytes))) break;
                if ((s - 1) * per >= steps) continue;   // (the last share would be empty)
                const int turns = (per + kBlockWaves - 1) / kBlockWaves, again = (blocks + 255) / 256 - 1;
                const double step = c.step + c.full * std::min(1.0, blocks / 256.0);
                const double own = c.fixed + turns * step + again * c.again * (turns * step + c.start) + 0.2e-6 * (s > 1 ? bytes : 2.0 * M * N);
                double us = std::cbrt(own * own * own + stream_us * stream_us * stream_us);
                if (norm) us += 0.1 * s + bytes / 4e6;
                else if (s > 1) us += 3.0 + bytes / 3.2e6;
                if (us < best.us) best = {mt, 1 << n, s, us};
            }
        }
    }
    return best;
}
bool fits(int format, int M, int N, int K, int group_size) {
    if (format == PIE_HIP_FMT_INT4B8) {
        if (group_size < 128 || (group_size & (group_size - 1)) != 0 || K % group_size != 0) return false;
    } else if (format != PIE_HIP_FMT_INT8 && format != PIE_HIP_FMT_FP8 && format != PIE_HIP_FMT_BF16) {
        return false;
    }
    return M > 0 && M <= most_rows(format == PIE_HIP_FMT_INT4B8) && N > 0 && N % 16 == 0 && K > 0 && K % (format == PIE_HIP_FMT_INT4B8 ? 128 : 64) == 0 && (format == PIE_HIP_FMT_BF16 ? 2ll : 1ll) * N * K <= 0xFFFFFFFFll &&
           2ll * M * K <= 0xFFFFFFFFll;
}
// (the same few questions are asked for every layer of a pass: the last answers are kept, per thread)
Plan plan_of(Form form, int M, int N, int K, size_t ws_bytes, bool norm) {
    struct Asked {
        int form = -1, M, N, K, norm;
        size_t ws_bytes;
        Plan plan;
    };
    thread_local Asked asked[16];
    thread_local unsigned next = 0;
    for (const Asked& q : asked)
        if (q.form == static_cast<int>(form) && q.M == M && q.N == N && q.K == K && q.norm == static_cast<int>(norm) && q.ws_bytes == ws_bytes) return q.plan;
    Asked& q = asked[next++ % 16];
    q.form = static_cast<int>(form), q.M = M, q.N = N, q.K = K, q.norm = norm, q.ws_bytes = ws_bytes;
    return q.plan = find_plan(form, M, N, K, ws_bytes, norm);
}
// (`shares`: the sums stay in the workspace, in that many shares)
int run(int format, GemmArgs a, const Rotation& rot, int group_size, void* ws, size_t ws_bytes, hipStream_t stream, int* shares = nullptr, bool tiled = true) {
    if (!fits(format, a.M, a.N, a.K, group_size) || reinterpret_cast<uintptr_t>(a.act) % 16 || reinterpret_cast<uintptr_t>(a.w) % 16 ||
        (format == PIE_HIP_FMT_INT4B8 && reinterpret_cast<uintptr_t>(a.scale) % 8))
        return PIE_HIP_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(ws) % 16) ws = nullptr;
    const Form form = form_of(format, tiled);
    const Plan p = plan_of(form, a.M, a.N, a.K, ws ? ws_bytes : 0, shares != nullptr);
    if (p.row_tiles == 0) return PIE_HIP_ERR_UNSUPPORTED;
    if (format == PIE_HIP_FMT_INT4B8) a.g_shift = __builtin_ctz(static_cast<unsigned>(group_size));
    a.aligned = reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
    a.partial = p.shares > 1 ? static_cast<float*>(ws) : nullptr;
    const int st = form == Form::Int4               ? launch<WvInt4>(a, rot, p, stream)
                   : form == Form::Bf16             ? launch<WvBf16>(a, rot, p, stream)
                   : form == Form::Bf16Rows         ? launch<WvBf16Rows>(a, rot, p, stream)
                   : format == PIE_HIP_FMT_FP8      ? launch<WvFp8>(a, rot, p, stream)
                                                    : launch<WvInt8>(a, rot, p, stream);
    if (shares) *shares = p.shares;
    if (st != PIE_HIP_OK || p.shares == 1 || shares) return st;
    return launch_shares_reduce(a, rot, p.shares, stream);
}
bool known(int format, const void* scale) {
    return format == PIE_HIP_FMT_BF16 || ((format == PIE_HIP_FMT_INT4B8 || format == PIE_HIP_FMT_INT8 || format == PIE_HIP_FMT_FP8) && scale);
}

}  // namespace
}  // namespace pie_hip

extern "C" float pie_hip_gemm_waves_us(int format, int tiled, int M, int N, int K, int group_size, size_t workspace_bytes, int norm) {
    using namespace pie_hip;
    return static_cast<float>(fits(format, M, N, K, group_size) && (tiled || format == PIE_HIP_FMT_BF16) ? plan_of(form_of(format, tiled != 0), M, N, K, workspace_bytes, norm != 0).us : 1e30);
}

extern "C" int pie_hip_gemm_waves_plan(int format, int tiled, int M, int N, int K, int group_size, size_t workspace_bytes, int norm, int* block_rows, int* block_columns, int* shares) {
    using namespace pie_hip;
    if (!block_rows || !block_columns || !shares) return PIE_HIP_ERR_INVALID;
    const Plan p = fits(format, M, N, K, group_size) && (tiled || format == PIE_HIP_FMT_BF16) ? plan_of(form_of(format, tiled != 0), M, N, K, workspace_bytes, norm != 0) : Plan{};
    if (p.row_tiles == 0) return PIE_HIP_ERR_UNSUPPORTED;
    *block_rows = p.row_tiles * 16;
    *block_columns = p.tiles * 16;
    *shares = p.shares;
    return PIE_HIP_OK;
}

namespace pie_hip {
namespace {
int product(int format, bool tiled, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16, int group_size, uint16_t* y_bf16, int M, int N, int K,
            int beta, int epilogue, const PieHipGlu* glu, void* workspace, size_t workspace_bytes, void* stream) {
    if (!glu_ok(glu, epilogue)) return PIE_HIP_ERR_INVALID;
    if (!known(format, scale) || !act_bf16 || !weight || !y_bf16 || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
    const int pointwise = pointwise_code(epilogue), swiglu = epilogue == PIE_HIP_EPI_SWIGLU ? 1 : 0;
    if ((swiglu && N % 2 != 0) || ((swiglu || pointwise) && beta)) return PIE_HIP_ERR_INVALID;
    GemmArgs a{};
    a.act = act_bf16;
    a.w = static_cast<const unsigned char*>(weight);
    a.scale = static_cast<const unsigned char*>(scale);
    a.y = y_bf16;
    a.M = M;
    a.N = N;
    a.K = K;
    a.beta = beta;
    a.swiglu = swiglu;
    a.pointwise = pointwise;
    if (glu) a.glu = *glu;
    a.scale_is_bf16 = scale_is_bf16;
    return run(format, a, Rotation{}, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream), nullptr, tiled);
}
}  // namespace
}  // namespace pie_hip

extern "C" int pie_hip_gemm_waves_tiled(int format, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16, int group_size, uint16_t* y_bf16,
                                        int M, int N, int K, int beta, int epilogue, const PieHipGlu* glu, void* workspace, size_t workspace_bytes, void* stream) {
    return pie_hip::product(format, true, act_bf16, weight, scale, scale_is_bf16, group_size, y_bf16, M, N, K, beta, epilogue, glu, workspace, workspace_bytes, stream);
}

extern "C" int pie_hip_gemm_waves_bf16(const uint16_t* act_bf16, const void* weight, uint16_t* y_bf16, int M, int N, int K, int beta, int epilogue, const PieHipGlu* glu,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    return pie_hip::product(PIE_HIP_FMT_BF16, false, act_bf16, weight, nullptr, 0, 0, y_bf16, M, N, K, beta, epilogue, glu, workspace, workspace_bytes, stream);
}

extern "C" int pie_hip_gemm_waves_shares(int format, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16, int group_size, int M, int N, int K,
                                         void* workspace, size_t workspace_bytes, int* shares, void* stream) {
    using namespace pie_hip;
    if (!known(format, scale) || !act_bf16 || !weight || !workspace || !shares || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
    GemmArgs a{};
    a.act = act_bf16;
    a.w = static_cast<const unsigned char*>(weight);
    a.scale = static_cast<const unsigned char*>(scale);
    a.M = M;
    a.N = N;
    a.K = K;
    a.scale_is_bf16 = scale_is_bf16;
    return run(format, a, Rotation{}, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream), shares);
}

extern "C" int pie_hip_qkv_rope_waves_tiled(int format, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16, int group_size, int M, int K,
                                            const float* rope_table, const int64_t* kv_slots, uint16_t* q_out, uint16_t* k_pages, uint16_t* v_pages, int num_q_heads,
                                            int num_kv_heads, int head_dim, int pairing, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace pie_hip;
    if (!known(format, scale) || !act_bf16 || !weight || !rope_table || !kv_slots || !q_out || !k_pages || !v_pages || M <= 0 || K <= 0 || num_q_heads <= 0 ||
        num_kv_heads <= 0 || head_dim <= 0 || (pairing != PIE_HIP_ROPE_ADJACENT && pairing != PIE_HIP_ROPE_HALF_PAIRED_ROWS))
        return PIE_HIP_ERR_INVALID;
    // (outputs leave in 8-byte stores)
    if ((head_dim & (head_dim - 1)) != 0 || head_dim % 16 != 0 ||
        (reinterpret_cast<uintptr_t>(q_out) | reinterpret_cast<uintptr_t>(k_pages) | reinterpret_cast<uintptr_t>(v_pages)) % 8)
        return PIE_HIP_ERR_UNSUPPORTED;
    GemmArgs a{};
    a.act = act_bf16;
    a.w = static_cast<const unsigned char*>(weight);
    a.scale = static_cast<const unsigned char*>(scale);
    a.y = q_out;
    a.M = M;
    a.N = (num_q_heads + 2 * num_kv_heads) * head_dim;
    a.K = K;
    a.scale_is_bf16 = scale_is_bf16;
    Rotation r;
    r.table = rope_table;
    r.slots = kv_slots;
    r.k_pages = k_pages;
    r.v_pages = v_pages;
    r.hq = num_q_heads;
    r.hk = num_kv_heads;
    r.d = head_dim;
    r.half_out = pairing == PIE_HIP_ROPE_HALF_PAIRED_ROWS;
    return run(format, a, r, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
