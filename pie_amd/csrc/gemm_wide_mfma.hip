// Tiled weight-only GEMM for prompts: y[M, N] = epilogue( act[M, K] · W[N, K]^T ), the same contract and rounding as
// the kernel of gemm_mfma.hip, in blocks of 256 rows x 256 (or 128) columns.
//
// The tiles of gemm_mfma.hip (four waves to a SIMD pair, each reading operands, decoding and multiplying in turn) kept the
// matrix pipe busy for less than half the time: a wave issues a vector instruction every eight cycles, the decoding of
// int4 weights takes as many of those as half the MFMAs' time, and every step ended in a wait for all transfers.  Here:
//   - eight waves, two to a SIMD, the second four one barrier behind the first: one wave's operand reads and transfers run
//     beside the other's MFMAs; a wave's tile of 128 x 64 needs 24 reads of 16 bytes per 64 MFMAs;
//   - the weights are the MFMAs' first operand, so that a lane ends with four neighbouring columns, and
//     stores 16 bytes with its neighbour's (store_pair: 1.8 % of an 8b prompt of 2048 tokens; the figures below are from before it);
//   - weights are decoded between the MFMAs, one vector per phase, from the tile-major copy;
//   - transfers into LDS run one to two steps ahead and no wait drains them;
//   - a chiplet's blocks are neighbours (the row blocks of a column block share its weights in one L2).
// What bounds it now: at 256 columns the matrix pipe and the decoding that shares its issue slots (int4: 1.4 us a step of 64
// k-values for a block alone, 1.6 with the chip full, where the MFMAs take 0.9 at 2.4 GHz), at 128 the LDS reads.
// Before / after, us (int4, fp8, bf16):
//   2048 x 28672 x 4096   546 / 436,  519 / 425,  476 / 410      2048 x 4096 x 14336   245 / 214,  231 / 201,  202 / 190
//   1024 x 28672 x 4096   302 / 229,  275 / 224,  295 / 206       489 x 4096 x 14336    84 /  71,   93 /  68,   97 /  64
//   1319 x 16384 x 2048   125 / 110,  119 / 109,  114 /  98      1024 x 6144 x 4096     71 /  61,   70 /  59,   60 /  53
// (the fourth in K shares; int4 and fp8 there against the skinny GEMM, which the driver's int4 prompts of such shapes keep:
// these blocks round an int4 code times its scale to bf16, the skinny GEMM scales a group's sum in fp32).
#include "gemm_args.hip.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace pie_hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));

constexpr int kRows = 256, kStepK = 64, kWaves = 8;
constexpr int kActVecs = kRows * kStepK / 8;   // 16-byte vectors of an activation stage

// ---- what a thread stages of a step's weights: V (32 or 16) of them, loaded from the tile-major copy (blocks of 1 KiB, 16 rows
// by 64 bytes, lane 16 q + j its bytes 16 q .. 16 q + 15 of row j), as V / 8 16-byte vectors of bf16; wave w takes the
// tiles of 16 rows from w V / 16 on.  (Row-major, a wave's load touches 32 rows' cache lines for 32 bytes each and took
// the address unit longer than the MFMAs of a phase.) -----------------------------------------------------------------
template <int V>
struct WInt4T {   // a block is 128 values deep, a step half of it
    static constexpr bool kDirect = false, kRowScale = false;
    static constexpr int kLoads = 2, kDepth = 128;
    struct Raw {
        uint32_t v[V / 8];
        uint16_t gs;
    };
    static __device__ __forceinline__ int tile(int wv, int lane, int) { return V == 32 ? 2 * wv + (lane >> 5) : wv; }
    static __device__ __forceinline__ int granule(int lane, int v) { return V == 32 ? ((lane >> 4) & 1) * 4 + v : (lane >> 4) * 2 + v; }
    // bytes of the thread's first value in a step's half block, of its row's first scale
    static __device__ __forceinline__ uint32_t offset(int lane) {
        return V == 32 ? (lane & 31) * 16 : ((lane >> 5) * 16 + (lane & 15)) * 16 + ((lane >> 4) & 1) * 8;
    }
    static __device__ __forceinline__ Raw load(const GemmArgs& a, const uint32_t* first, uint32_t scales, int k) {
        Raw r;
        const unsigned char* p = a.w + static_cast<size_t>(k >> 7) * 1024 + ((k >> 6) & 1) * 512 + first[0];
        if constexpr (V == 32) {
            const u32x4_t t = *reinterpret_cast<const u32x4_t*>(p);
            r.v[0] = t.x; r.v[1] = t.y; r.v[2] = t.z; r.v[3] = t.w;
        } else {
            const u32x2_t t = *reinterpret_cast<const u32x2_t*>(p);
            r.v[0] = t.x; r.v[1] = t.y;
        }
        r.gs = *reinterpret_cast<const uint16_t*>(a.scale + static_cast<size_t>(k >> a.g_shift) * 32 + scales);
        return r;
    }
    // (nibble - 8) * scale: the even nibbles become the fp16 pairs 1024 + n, the odd ones (where they are) 1024 + 16 n, and
    // one mixed-precision fma takes a half straight to the fp32 product.  Exact in fp32, so one rounding to bf16.  (A word's
    // pairs are its codes in order, see pie_hip_repack_mfma_tiles_int4.)
    static __device__ __forceinline__ u32x4_t decode(const Raw& r, int s, uint32_t k1024) {
        const float gs = bf16_bits_to_f32(r.gs);
        const float scale[2] = {gs, 0.0625f * gs}, off[2] = {-1032.f * gs, -72.f * gs};
        u32x4_t o;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f16x2_t pr = __builtin_bit_cast(f16x2_t, and_or(j < 2 ? r.v[s] : r.v[s] >> 8, j & 1 ? 0x00F000F0u : 0x000F000Fu, k1024));
            o[j] = pack_bf16x2(fmaf(static_cast<float>(pr.x), scale[j & 1], off[j & 1]), fmaf(static_cast<float>(pr.y), scale[j & 1], off[j & 1]));
        }
        return o;
    }
};
template <int V, int KVF>
struct WByteT {   // a block is a step deep
    static constexpr bool kDirect = false, kRowScale = true;
    static constexpr int kLoads = V / 16, kDepth = 64;
    struct Raw {
        u32x4_t v[V / 16];
    };
    static __device__ __forceinline__ int tile(int wv, int, int v) { return V == 32 ? 2 * wv + (v >> 1) : wv; }
    static __device__ __forceinline__ int granule(int lane, int v) { return (lane >> 4) * 2 + (v & 1); }
    static __device__ __forceinline__ uint32_t offset(int lane) { return lane * 16; }
    static __device__ __forceinline__ Raw load(const GemmArgs& a, const uint32_t* first, uint32_t, int k) {
        Raw r;
#pragma unroll
        for (int i = 0; i < V / 16; ++i) r.v[i] = *reinterpret_cast<const u32x4_t*>(a.w + static_cast<size_t>(k >> 6) * 1024 + first[i]);
        return r;
    }
    static __device__ __forceinline__ u32x4_t decode(const Raw& r, int s, uint32_t) {
        return kv_decode_bf16<KVF>(u32x2_t{r.v[s >> 1][2 * (s & 1)], r.v[s >> 1][2 * (s & 1) + 1]});
    }
};
struct WBf16T {   // row-major, moved without registers
    static constexpr bool kDirect = true, kRowScale = false;
    static constexpr int kLoads = 0, kDepth = 64;
    struct Raw {};
    static __device__ __forceinline__ int tile(int, int, int) { return 0; }
    static __device__ __forceinline__ int granule(int, int) { return 0; }
    static __device__ __forceinline__ uint32_t offset(int) { return 0; }
    static __device__ __forceinline__ Raw load(const GemmArgs&, const uint32_t*, uint32_t, int) { return {}; }
    static __device__ __forceinline__ u32x4_t decode(const Raw&, int, uint32_t) { return u32x4_t{0u, 0u, 0u, 0u}; }
};
struct WInt4 {
    template <int V> using Staged = WInt4T<V>;
};
struct WFp8 {
    template <int V> using Staged = WByteT<V, kKvFp8>;
};
struct WInt8 {
    template <int V> using Staged = WByteT<V, kKvInt8>;
};
struct WBf16 {
    template <int V> using Staged = WBf16T;
};

// position of granule g of tile row r (in 16-byte vectors)
__device__ __forceinline__ int swz(int r, int g) { return r * 8 + (g ^ ((r >> 1) & 7)); }

template <class FMT, int COLS>
struct Wide {
    static constexpr int kVals = COLS / 8;          // weights a thread stages per step
    using F = typename FMT::template Staged<kVals>;
    static constexpr int kAH = COLS / 128;          // halves of 64 rows of a wave's tile: 128 x 64 or 64 x 64 outputs
    static constexpr int kWn = COLS / 64;           // waves along the columns
    static constexpr int kStages = COLS == 256 ? 2 : 3;
    static constexpr int kColVecs = COLS * kStepK / 8;
    static constexpr int kColStages = kStages;
    static constexpr size_t kSmem = (static_cast<size_t>(kStages) * kActVecs + static_cast<size_t>(kColStages) * kColVecs) * 16;
};

template <class FMT, int COLS>
__global__ __launch_bounds__(kWaves* kWave, 2) void gemm_wide_kernel(const GemmArgs a, int first_col, int row_blocks, int per_xcd, int tiles) {
    using W = Wide<FMT, COLS>;
    using F = typename W::F;
    constexpr int AH = W::kAH, S = W::kStages;
    extern __shared__ __align__(16) unsigned char smem[];
    u32x4_t* lds_a = reinterpret_cast<u32x4_t*>(smem);
    u32x4_t* lds_b = lds_a + S * kActVecs;
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 15, q = lane >> 4;
    const int wm = wv / W::kWn, wn = wv % W::kWn;
    // blocks go to the XCDs in turn: each XCD's are neighbours, the row blocks of a column block side by side
    const int tile = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (tile >= tiles) return;
    const int m0 = tile % row_blocks * kRows, n0 = first_col + tile / row_blocks * COLS;
    const int M = a.M, N = a.N, K = a.K;
    const int nk_all = K / kStepK;
    const int per_split = (nk_all + static_cast<int>(gridDim.z) - 1) / static_cast<int>(gridDim.z);
    const int kbeg = blockIdx.z * per_split;
    const int nk = min(per_split, nk_all - kbeg);

    // direct transfers: a chunk (1 KiB) is eight tile rows; lane p lands at position p of it, which holds granule
    // (p % 8) ^ key(row).  With 256 columns a tile's rows move in halves, those that a wave's phases read together: activations
    // 0 - 63 and 64 - 127 of either half of the waves, columns 0 - 31 and 32 - 63 of every wave's 64.
    constexpr int AC = 4, BC = F::kDirect ? COLS / 64 : 0;   // chunks per wave
    uint32_t aoff[4], boff[4];   // bytes (the launcher checked that they fit); half h, chunk u at 2h + u
    int arow[4], brow[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        arow[u] = AH == 2 ? (u & 1) * 128 + (u >> 1) * 64 + wv * 8 : (u * kWaves + wv) * 8;
        brow[u] = AH == 2 ? ((u & 1) * 2 + (wv >> 2)) * 64 + (u >> 1) * 32 + (wv & 3) * 8 : (u * kWaves + wv) * 8;
        const int ar = arow[u] + (lane >> 3), br = brow[u] + (lane >> 3);
        aoff[u] = static_cast<uint32_t>(min(m0 + ar, M - 1)) * (2u * K) + ((lane & 7) ^ ((ar >> 1) & 7)) * 16;
        if (u < BC) boff[u] = static_cast<uint32_t>(min(n0 + br, N - 1)) * (2u * K) + ((lane & 7) ^ ((br >> 1) & 7)) * 16;
    }
    // chunks [u0, u1) of step kt's activations (bf16 weights)
    auto issue_a = [&](int kt, int stage, int u0, int u1) {
        const unsigned char* p = reinterpret_cast<const unsigned char*>(a.act) + static_cast<size_t>(kbeg + min(kt, nk - 1)) * (kStepK * 2);
#pragma unroll
        for (int u = u0; u < u1; ++u)
            __builtin_amdgcn_global_load_lds(p + aoff[u], PIE_LDS_PTR(lds_a + stage * kActVecs + arow[u] * 8), 16, 0, 0);
    };
    auto issue_b = [&](int kt, int stage, int u0, int u1) {
        const unsigned char* p = a.w + static_cast<size_t>(kbeg + min(kt, nk - 1)) * (kStepK * 2);
#pragma unroll
        for (int u = u0; u < u1 && u < BC; ++u)
            __builtin_amdgcn_global_load_lds(p + boff[u], PIE_LDS_PTR(lds_b + stage * W::kColVecs + brow[u] * 8), 16, 0, 0);
    };
    // quantised weights: the thread's tiles (at most two) in bytes of the first block, its rows' scales
    constexpr int VPT = W::kVals / 8;   // 16-byte vectors of bf16
    uint32_t w_first[2], s_first = 0;
    if constexpr (!F::kDirect) {
        const int last = (N + 15) / 16 - 1;
#pragma unroll
        for (int i = 0; i < 2; ++i)
            w_first[i] = static_cast<uint32_t>(min(n0 / 16 + F::tile(wv, lane, 2 * i), last)) * (K / F::kDepth * 1024u) + F::offset(lane);
        s_first = (static_cast<uint32_t>(min(n0 / 16 + F::tile(wv, lane, 0), last)) * (K >> a.g_shift) * 16u + j) * 2u;
    }
    auto load_w = [&](int kt) { return F::load(a, w_first, s_first, (kbeg + min(kt, nk - 1)) * kStepK); };

    uint32_t magic = 0x64006400u;   // (1024, 1024) as an fp16 pair, opaque to the compiler
    asm volatile("" : "+v"(magic));
    auto store_w = [&](const typename F::Raw& r, int stage, int v) {
        if constexpr (!F::kDirect) lds_b[stage * W::kColVecs + swz(F::tile(wv, lane, v) * 16 + j, F::granule(lane, v))] = F::decode(r, v, magic);
    };

    f32x4_t acc[4 * AH][4];
#pragma unroll
    for (int t = 0; t < 4 * AH; ++t)
#pragma unroll
        for (int n = 0; n < 4; ++n) acc[t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    // quantised weights: registers hold S steps, which are decoded one vector per phase
    typename F::Raw rr[S];
#pragma unroll
    for (int i = 0; i < S; ++i) rr[i] = load_w(i);
    PIE_FENCE();
    issue_a(0, 0, 0, 4);
    issue_b(0, 0, 0, 4);
    issue_a(1, 1, 0, AH == 2 ? 2 : 4);   // (in steady state a step's transfers begin in the second step before it)
    issue_b(1, 1, 0, 4);
    PIE_FENCE();
#pragma unroll
    for (int v = 0; v < VPT; ++v) store_w(rr[0], 0, v);
    PIE_FENCE();
    rr[0] = load_w(S);
    store_w(rr[1], 1, 0);
    if constexpr (F::kDirect) PIE_WAIT_VM(AC / AH + BC);
    else PIE_WAIT_VM(0);
    PIE_WAIT_LGKM0();
    PIE_MEET();
    if (wv >= kWaves / 2) PIE_MEET();

    bf16x8_t af[2][4], bf[2][2][2];   // [k half][row tile], [column half][k half][column tile]
    const int key = j >> 1;
    // (the operands of a phase's first eight MFMAs first: they start when those have arrived)
    auto read_ab = [&](int a_stage, int a_half, int b_stage, int b_half) {   // a half of -1: not read
        const u32x4_t* A = lds_a + a_stage * kActVecs + (wm * 64 * AH + max(a_half, 0) * 64 + j) * 8;
        const u32x4_t* B = lds_b + b_stage * W::kColVecs + (wn * 64 + max(b_half, 0) * 32 + j) * 8;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int at = (ks * 4 + q) ^ key;
            if (b_half >= 0) {
#pragma unroll
                for (int t = 0; t < 2; ++t) bf[b_half][ks][t] = __builtin_bit_cast(bf16x8_t, B[t * 128 + at]);
            }
            if (a_half >= 0) {
#pragma unroll
                for (int t = 0; t < 4; ++t) af[ks][t] = __builtin_bit_cast(bf16x8_t, A[t * 128 + at]);
            }
            PIE_FENCE();
        }
    };
    // A phase's MFMAs.  Between them the wave decodes one vector of the weights `r` into the tile `w_stage`: a wave issues a
    // vector instruction every eight cycles and an MFMA keeps the matrix pipe for sixteen, so one decode instruction behind
    // each is free, while in the memory part the same instructions outlast the other wave's MFMAs.
    auto multiply = [&](int ah, int bh, const typename F::Raw& r, int w_stage, int v) {
        PIE_MEET();
        __builtin_amdgcn_s_setprio(1);
        store_w(r, w_stage, v);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int n = 0; n < 2; ++n)
                    acc[ah * 4 + t][bh * 2 + n] =
                        __builtin_amdgcn_mfma_f32_16x16x32_bf16(bf[bh][ks][n], af[ks][t], acc[ah * 4 + t][bh * 2 + n], 0, 0, 0);
        if constexpr (!F::kDirect) {
#pragma unroll
            for (int u = 0; u < 16; ++u) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
        }
        __builtin_amdgcn_s_setprio(0);
        PIE_MEET();
    };
    // One step of 64 k-values; `stage` = kt % S.  A step is 2 AH phases, each a memory part (operand reads, loads ahead) and
    // 16 MFMAs, with a barrier behind either; the waves of the second half are one barrier behind, so that on every SIMD one
    // wave's memory part runs beside the other's MFMAs.
    // What a phase reads is overwritten no earlier than two phases later, when the waves behind have waited for their reads
    // too, and what it reads was waited for by all waves a phase before; every wait leaves the transfers issued
    // since in flight.  A step's weights are decoded from the last phase of the second step before it on.
    constexpr int HA = 2, HB = F::kDirect ? 2 : 0, L = F::kLoads;   // vector-memory operations of a half tile, of the weights
    auto step = [&](auto slot, int kt) {
        constexpr int stage = decltype(slot)::value, next = (stage + 1) % S, after = (stage + 2) % S;
        if constexpr (AH == 2) {
            read_ab(stage, 0, stage, 0);
            issue_a(kt + 1, next, 2, 4);
            if constexpr (F::kDirect) PIE_WAIT_VM(2 * HA + 3 * HB);   // this step's second column half has landed
            multiply(0, 0, rr[next], next, 1);
            read_ab(0, -1, stage, 1);
            PIE_WAIT_VM(2 * HA + 2 * HB + L);                         // and its second half of the rows
            multiply(0, 1, rr[next], next, 2);
            read_ab(stage, 1, 0, -1);
            issue_a(kt + 2, stage, 0, 2);
            issue_b(kt + 2, stage, 0, 2);
            multiply(1, 1, rr[next], next, 3);
            issue_b(kt + 2, stage, 2, 4);
            PIE_WAIT_VM(2 * HA + 3 * HB);                             // step kt + 1's first halves, step kt + 2's weights
            rr[next] = load_w(kt + 3);
            PIE_WAIT_LGKM0();
            multiply(1, 0, rr[stage], stage, 0);
        } else {
            read_ab(stage, 0, stage, 0);
            issue_a(kt + 2, after, 0, 4);   // (last read in step kt - 1)
            issue_b(kt + 2, after, 0, 4);
            multiply(0, 0, rr[next], next, 1);
            read_ab(0, -1, stage, 1);
            PIE_WAIT_VM(AC + BC + L);   // step kt + 1's transfers
            rr[next] = load_w(kt + 4);
            PIE_WAIT_LGKM0();
            multiply(0, 1, rr[after], after, 0);
        }
    };
    int kt = 0;
    for (; kt + S <= nk; kt += S) {
        step(std::integral_constant<int, 0>{}, kt);
        step(std::integral_constant<int, 1>{}, kt + 1);
        if constexpr (S == 3) step(std::integral_constant<int, 2>{}, kt + 2);
    }
    if (kt < nk) step(std::integral_constant<int, 0>{}, kt);
    if (S == 3 && kt + 1 < nk) step(std::integral_constant<int, 1>{}, kt + 1);
    if (wv < kWaves / 2) PIE_MEET();
    __builtin_amdgcn_s_waitcnt(0x0070);   // (transfers past the last step land before the block ends)

    // ---- epilogue: a lane holds four neighbouring columns of one row per tile ----
    float rs[4][4];   // (all asked for at once)
    if constexpr (F::kRowScale) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int c = min(n0 + wn * 64 + nt * 16 + 4 * q + r, N - 1);
                rs[nt][r] = a.scale_is_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(a.scale)[c]) : reinterpret_cast<const float*>(a.scale)[c];
            }
        PIE_FENCE();
    }
    auto value = [&](int t, int nt, int r) __attribute__((always_inline)) { return F::kRowScale ? acc[t][nt][r] * rs[nt][r] : acc[t][nt][r]; };
    const int row0 = m0 + wm * 64 * AH + j, col0 = n0 + wn * 64 + 4 * q;
    if (a.partial) {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int n = col0 + nt * 16;
            if (n >= N) continue;
#pragma unroll
            for (int t = 0; t < 4 * AH; ++t) {
                const int m = row0 + t * 16;
                if (m >= M) continue;
                float* p = a.partial + (static_cast<size_t>(blockIdx.z) * M + m) * N + n;
                if (N % 4 == 0) *reinterpret_cast<f32x4_t*>(p) = f32x4_t{value(t, nt, 0), value(t, nt, 1), value(t, nt, 2), value(t, nt, 3)};
                else
                    for (int r = 0; r < 4 && n + r < N; ++r) p[r] = value(t, nt, r);
            }
        }
    } else if (a.lines) {
        by_output(a, [&](auto out) __attribute__((always_inline)) {
#pragma unroll
            for (int nt = 0; nt < 4; nt += 2) {
                const int n = col0 + nt * 16;
                if (n >= N) continue;
                int row_step;
                uint16_t* to = pair_place<decltype(out)::value>(a, row0, n, q, row_step);
#pragma unroll
                for (int t = 0; t < 4 * AH; ++t, to += row_step) {
                    if (row0 + t * 16 >= M) break;   // (no later row is one either)
                    float v[2][4];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[i][r] = value(t, nt + i, r);
                    store_pair<decltype(out)::value>(a, to, n, v[0], v[1]);
                }
            }
        });
    } else {
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) {
            const int n = col0 + nt * 16;
            if (n >= N) continue;
#pragma unroll
            for (int t = 0; t < 4 * AH; ++t) {
                const int m = row0 + t * 16;
                if (m >= M) continue;
                float v[4] = {value(t, nt, 0), value(t, nt, 1), value(t, nt, 2), value(t, nt, 3)};
                wide_store(a, m, n, v);
            }
        }
    }
}

// ---- experts: the rows of a problem gathered by route, one-byte weights, blocks of 32 to 128 rows x 64 NG columns --------
// A hundred rows per expert make an expert's weights as many bytes as its products are time, and each is wanted by one
// block only.  So weights do not pass through LDS: a wave owns 16 NG columns for all rows of the block, the tile-major copy gives it
// the MFMAs' operand by plain loads, three or four steps ahead in registers, each decoded once.  The activations are shared in LDS,
// as far ahead.  Two or three blocks of four waves to a CU, independent of one another: one's prologue, waits and stores run
// beside the other's MFMAs.  A row block's column blocks stay on one chiplet and share its activations there.
// Bound by the weights up to 50 routes per expert (5.8 TB/s at four), above by the products too: 128 fp8 experts of 1536 x 2048 at 82 routes 111 us
// (402 MB; the tiles through LDS 147), of 2048 x 768 74 (84 through LDS).
// The same for one matrix and up to 128 rows (64 columns per block, two groups of waves that take the steps in turn and meet at the
// end: a block is alone on its CU, and one wave per SIMD waits out every step's chain): 77 rows of 16384 x 2048 int8 16.7 us, fp8
// 16.4 (128 x 128 tiles 27 and 26, passes of 32 rows 26 and 24; one group 18.4 and 17.7), 40 rows 13.7 and 11.3 (18.5 and 16.6).
// RT row tiles of 16, NG column tiles per wave, S steps of 64 k-values in flight (LDS stages and weight registers).
// Whole: one block has all rows; Experts: rows gathered by route; Rows: blocks of a matrix of many rows, in shares of K (blockIdx.z) where
// they are few.
enum class Form { Whole, Experts, Rows };
// (Blocks of 32 rows run six to a CU, up to 80 registers: 64 tokens of the mixture 9.34 ms, with five 9.54.)
template <int KVF, int RT, int NG, int S, Form FORM, int KP = 1>
__global__ __launch_bounds__(256 * KP, S == 3 ? (RT == 2 ? 6 : 3) : 2) void gemm_columns_kernel(GemmArgs a, int col_blocks, int row_blocks, int per_share) {
    constexpr bool EXPERTS = FORM == Form::Experts;
    constexpr int kRowsB = RT * 16, kVecs = kRowsB * kStepK / 8, HT = RT / 2, AC = RT / 2;   // a half's row tiles; chunks of eight rows per wave
    extern __shared__ __align__(16) unsigned char smem[];
    const int part = KP == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / 256);
    u32x4_t* lds = reinterpret_cast<u32x4_t*>(smem) + part * S * kVecs;
    const int tid = threadIdx.x & 255, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 15, q = lane >> 4;
    // (Rows: each XCD's blocks are neighbours, the row blocks of a column block side by side)
    const int at = EXPERTS            ? static_cast<int>(blockIdx.x >> 3)
                   : FORM == Form::Rows ? static_cast<int>((blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3))
                                        : static_cast<int>(blockIdx.x);
    if (FORM == Form::Rows && at >= row_blocks * col_blocks) return;
    int problem = 0, m0 = FORM == Form::Rows ? at % row_blocks * kRowsB : 0, M = a.M;
    if constexpr (EXPERTS)
        if (!grouped_place(a.offsets, a.problems, kRowsB, at / col_blocks * 8 + static_cast<int>(blockIdx.x & 7), lane, problem, m0, M)) return;
    const int N = a.N, K = a.K, nk_matrix = K / kStepK, T = (N + 15) / 16;
    const int first = FORM == Form::Rows ? static_cast<int>(blockIdx.z) * per_share : 0;
    const int nk_all = FORM == Form::Rows ? min(per_share, nk_matrix - first) : nk_matrix;
    const int nk = (nk_all - part + KP - 1) / KP;   // this group's steps: part, part + KP, ..
    auto place = [&](int kt) { return first + min(part + KP * min(kt, max(nk, 1) - 1), nk_all - 1); };   // (past them, or without any: a step again)
    const int tile0 = ((FORM == Form::Rows ? at / row_blocks : at % col_blocks) * 4 + wv) * NG;
    const unsigned char* w = a.w + static_cast<size_t>(problem) * a.w_stride;
    const unsigned char* scale = a.scale + static_cast<size_t>(problem) * a.scale_stride;

    // the weights first: they depend on the problem alone, the activations on the routes' rows too
    uint32_t woff[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) woff[i] = static_cast<uint32_t>(min(tile0 + i, T - 1)) * (nk_matrix * 1024u) + lane * 16u;
    u32x4_t raw[S][NG];
    auto load_w = [&](int kt, int slot) __attribute__((always_inline)) {
        const unsigned char* pw = w + static_cast<size_t>(place(kt)) * 1024;
#pragma unroll
        for (int i = 0; i < NG; ++i) raw[slot][i] = *reinterpret_cast<const u32x4_t*>(pw + woff[i]);
        PIE_FENCE();
    };
    const unsigned char* aptr[AC];
    int arow[AC];
#pragma unroll
    for (int u = 0; u < AC; ++u) {
        arow[u] = min(m0 + (u * 4 + wv) * 8 + (lane >> 3), M - 1);
        if (EXPERTS && a.act_rows) arow[u] = a.act_rows[arow[u]];
    }
    PIE_FENCE();
#pragma unroll
    for (int i = 0; i < S; ++i) load_w(i, i);
#pragma unroll
    for (int u = 0; u < AC; ++u)
        aptr[u] = reinterpret_cast<const unsigned char*>(a.act) + static_cast<size_t>(arow[u]) * (2u * K) +
                  ((lane & 7) ^ ((((u * 4 + wv) * 8 + (lane >> 3)) >> 1) & 7)) * 16;
    auto issue_a = [&](int kt, int stage) __attribute__((always_inline)) {
        const size_t k = static_cast<size_t>(place(kt)) * (kStepK * 2);
#pragma unroll
        for (int u = 0; u < AC; ++u) to_lds(aptr[u] + k, lds + stage * kVecs + (u * 4 + wv) * 64);
        PIE_FENCE();
    };
    bf16x8_t af[2][HT], bw[2][NG];   // [phase & 1][row tile], [k half][column tile]
    const int key = j >> 1;
    auto read_a = [&](int stage, int s, int rh, int to) __attribute__((always_inline)) {
        const u32x4_t* A = lds + stage * kVecs + (rh * HT * 16 + j) * 8 + ((2 * q + s) ^ key);
#pragma unroll
        for (int t = 0; t < HT; ++t) af[to][t] = __builtin_bit_cast(bf16x8_t, A[t * 128]);
    };
    auto decode = [&](const u32x4_t& r, int s) __attribute__((always_inline)) {
        return __builtin_bit_cast(bf16x8_t, kv_decode_bf16<KVF>(u32x2_t{r[2 * s], r[2 * s + 1]}));
    };
    f32x4_t acc[RT][NG];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int n = 0; n < NG; ++n) acc[t][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};

#pragma unroll
    for (int i = 0; i < S; ++i) issue_a(i, i);
    constexpr int kOps = AC + NG;
    PIE_WAIT_VM((S - 1) * AC);
    PIE_MEET();
    read_a(0, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < NG; ++i) bw[0][i] = decode(raw[0][i], 0);
    auto mfmas = [&](int s, int rh) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < HT; ++t)
#pragma unroll
            for (int n = 0; n < NG; ++n)
                acc[rh * HT + t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[s][n], af[rh][t], acc[rh * HT + t][n], 0, 0, 0);
    };
    auto order = [&]() __attribute__((always_inline)) {   // the reads ahead between the first MFMAs, the decoding between all
#pragma unroll
        for (int u = 0; u < HT * NG; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (u < HT) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, 1, 0);
        }
        PIE_FENCE();
    };
    auto step = [&](auto slot, int kt) __attribute__((always_inline)) {
        constexpr int cur = decltype(slot)::value, next = (cur + 1) % S;
        PIE_FENCE();
        read_a(cur, 0, 1, 1);
#pragma unroll
        for (int i = 0; i < NG / 2; ++i) bw[1][i] = decode(raw[cur][i], 1);
        mfmas(0, 0);
        order();
        read_a(cur, 1, 0, 0);
#pragma unroll
        for (int i = NG / 2; i < NG; ++i) bw[1][i] = decode(raw[cur][i], 1);
        mfmas(0, 1);
        order();
        // step kt + 1 has come
        if (kt < S - 2) PIE_WAIT_VM((S - 2) * AC);   // (of the first S the weights left first)
        else PIE_WAIT_VM((S - 2) * kOps);
        read_a(cur, 1, 1, 1);
#pragma unroll
        for (int i = 0; i < NG / 2; ++i) bw[0][i] = decode(raw[next][i], 0);
        mfmas(1, 0);
        order();
        PIE_WAIT_LGKM0();
        PIE_MEET();
        read_a(next, 0, 0, 0);
        PIE_FENCE();
        issue_a(kt + S, cur);
        load_w(kt + S, cur);
#pragma unroll
        for (int i = NG / 2; i < NG; ++i) bw[0][i] = decode(raw[next][i], 0);
        mfmas(1, 1);
        order();
    };
    // (a group a step short of the others meets them all the same)
    const int rounds = (nk_all + KP - 1) / KP;
    auto steps = [&](int kt, auto whole) __attribute__((always_inline)) {
        auto one = [&](auto slot) __attribute__((always_inline)) {
            constexpr int i = decltype(slot)::value;
            if (decltype(whole)::value || kt + i < nk) step(slot, kt + i);
            else if (KP > 1 && kt + i < rounds) PIE_MEET();
        };
        one(std::integral_constant<int, 0>{});
        one(std::integral_constant<int, 1>{});
        one(std::integral_constant<int, 2>{});
        if constexpr (S > 3) one(std::integral_constant<int, 3>{});
    };
    static_assert(S == 3 || S == 4, "steps() is unrolled by hand");
    int kt = 0;
    for (; kt + S <= nk_all / KP; kt += S) steps(kt, std::true_type{});
    if (kt < rounds) steps(kt, std::false_type{});
    __builtin_amdgcn_s_waitcnt(0x0070);   // (transfers past the last step land before the block ends)
    if constexpr (KP > 1) {   // the groups' sums meet in the activations' place
        static_assert(NG == 1 && KP == 2 && RT * 256 <= S * kVecs, "");
        __syncthreads();
        f32x4_t* meet = reinterpret_cast<f32x4_t*>(smem);
        if (part > 0) {
#pragma unroll
            for (int t = 0; t < RT; ++t) meet[t * 256 + tid] = acc[t][0];
        }
        __syncthreads();
        if (part > 0) return;
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t][0] += meet[t * 256 + tid];
    }

    // (a decode batch's few rows: nothing to gain, registers to lose; 128 routes of int8 experts: one register more than three blocks to a CU leave)
    if constexpr (NG == 2 && !(EXPERTS && (RT == 2 || (RT == 8 && KVF == kKvInt8))))
        if (a.lines && !(FORM == Form::Rows && a.partial)) {
            const int n = tile0 * 16 + 4 * q;
            if (n >= N) return;
            float rs[2][4];
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    rs[i][r] = a.scale_is_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(scale)[n + 16 * i + r])
                                               : reinterpret_cast<const float*>(scale)[n + 16 * i + r];
            by_output(a, [&](auto out) __attribute__((always_inline)) {
                int row_step;
                uint16_t* to = pair_place<decltype(out)::value>(a, m0 + j, n, q, row_step);
#pragma unroll
                for (int t = 0; t < RT; ++t, to += row_step) {
                    if (m0 + t * 16 + j >= M) break;   // (no later row is one either)
                    float v[2][4];
#pragma unroll
                    for (int i = 0; i < 2; ++i)
#pragma unroll
                        for (int r = 0; r < 4; ++r) v[i][r] = acc[t][i][r] * rs[i][r];
                    store_pair<decltype(out)::value>(a, to, n, v[0], v[1]);
                }
            });
            return;
        }
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int n = (tile0 + i) * 16 + 4 * q;
        if (n >= N) continue;
        float rs[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int c = min(n + r, N - 1);
            rs[r] = a.scale_is_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(scale)[c]) : reinterpret_cast<const float*>(scale)[c];
        }
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int m = m0 + t * 16 + j;
            if (m >= M) continue;
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = acc[t][i][r] * rs[r];
            if (FORM == Form::Rows && a.partial) *reinterpret_cast<f32x4_t*>(a.partial + (static_cast<size_t>(blockIdx.z) * M + m) * N + n) = f32x4_t{v[0], v[1], v[2], v[3]};
            else wide_store(a, m, n, v);
        }
    }
}

// Sums the K shares' partials of four columns and applies the epilogue the kernel would have applied.
__global__ __launch_bounds__(256) void wide_reduce_kernel(const GemmArgs a, int splits) {
    const int N = a.N, quads = (N + 3) / 4;
    const size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= static_cast<size_t>(a.M) * quads) return;
    const int m = static_cast<int>(idx / quads), n = static_cast<int>(idx % quads) * 4;
    const size_t plane = static_cast<size_t>(a.M) * N;
    const float* p = a.partial + static_cast<size_t>(m) * N + n;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
    for (int z = 0; z < splits; ++z) {
        if (N % 4 == 0) {
            const f32x4_t t = *reinterpret_cast<const f32x4_t*>(p + z * plane);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] += t[r];
        } else {
            for (int r = 0; r < 4 && n + r < N; ++r) v[r] += p[z * plane + r];
        }
    }
    wide_store(a, m, n, v);
}

template <class F, int COLS>
int launch(const GemmArgs& a, int first_col, int col_blocks, int splits, hipStream_t stream) {
    using W = Wide<F, COLS>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wide_kernel<F, COLS>),
                                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(W::kSmem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int rows = (a.M + kRows - 1) / kRows;
    const int tiles = rows * col_blocks, per = (tiles + 7) / 8;
    hipLaunchKernelGGL((gemm_wide_kernel<F, COLS>), dim3(8 * per, 1, splits), dim3(kWaves * kWave), W::kSmem, stream, a, first_col,
                       rows, per, tiles);
    return launch_status();
}

// What a launch takes, in microseconds: a round of up to one block per CU is `fixed` and, per step of 64 k-values, `step` for
// a few blocks; `fixed_full` and `step_full` more when all 256 CUs have one (shared caches, stores, power), most of it only
// when nearly all have.  Fitted to 160 - 4096 rows of 4096 x 14336, 28672 x 4096, 16384 x 2048 and 4096 x 4096 (within 7 %), before the blocks stored 16
// bytes a lane.  Over 50 matrices of 129 - 2048 rows with these stores and each call's weights out of HBM: int8 and fp8 within 6 % at the median from K of 2048 on and up
// to a fifth low at 1024, int4 at most 11 % high.  Bf16 with these stores and short K, us by 256 rows of 8 waves / blocks of 128 columns / of 256: 2011 x 8192 x 512 37.0 /
// 29.9 / 25.7, x 256 29.8 / 22.2 / 20.0, x 1024 50.4 / 44.4 / 36.0, 500 x 16384 x 256 17.4 / 13.3 / 18.2, 2011 x 4096 x 1024 26.8 / 22.6 / 30.4, 1000 x 2048 x 1024 14.4 / 18.3 /
// 26.9 (blocks of 128 rows): within 9 %, and which is faster by all 17 shapes of the test.  (Int4 stays so: lower figures would take rows from the blocks that scale groups in fp32.)
struct Rate {
    double fixed, step, fixed_full, step_full;
};
struct Rates {
    Rate wide256, wide128;
    double few, many, round, tall;   // the kernel of gemm_mfma.hip, per step: up to 256 blocks of 128 rows (few + many per
                                     // 256), each 256 of more, each 256 blocks of 256 rows
};
constexpr Rates kRates[] = {
    /* int4 */ {{14.0, 1.36, 8.0, 0.26}, {6.0, 0.76, 1.0, 0.15}, 0.57, 0.20, 0.64, 1.14},
    /* int8 */ {{14.0, 1.31, 10.0, 0.22}, {7.0, 0.72, 2.0, 0.12}, 0.54, 0.20, 0.62, 1.10},
    /* fp8 */ {{14.0, 1.31, 10.0, 0.20}, {7.0, 0.71, 2.0, 0.12}, 0.47, 0.17, 0.58, 1.08},
    /* bf16 */ {{9.0, 0.90, 2.8, 0.43}, {6.0, 0.62, 1.0, 0.19}, 0.36, 0.21, 0.57, 0.93},
};
double launch_us(const Rate& r, long long blocks, int steps) {
    const long long rounds = blocks / 256;
    const double fill = static_cast<double>(blocks % 256) / 256.0, cube = fill * fill * fill;
    return 3.0 + rounds * (r.fixed + r.fixed_full + steps * (r.step + r.step_full)) +
           (fill > 0.0 ? r.fixed + cube * r.fixed_full + steps * (r.step + cube * r.step_full) : 0.0);
}

// How the wide form runs a shape: `first` blocks of 256 columns and the rest in blocks of 128, in `splits` shares of K.
// Whole rounds of the larger block are the fastest; what is left over may fill the machine better in smaller ones (2048 rows of
// 28672 columns: 896 blocks of 256 are 3.5 rounds, 457 us int4; 768 of them and 256 of 128 columns 437).  Few blocks over a long K run in shares that fill
// one round, whose fp32 sums a second kernel adds in the order of K (160 rows of 4096 x 14336 int4: 32 blocks 175 us, in eight
// shares 42).
struct Plan {
    int first = 0, splits = 1;
    double us = 1e30;
};
Plan plan_of(const Rates& r, int M, int N, int K, size_t ws_bytes) {
    const int rows = (M + kRows - 1) / kRows, steps = K / kStepK, c256 = (N + 255) / 256;
    auto rest_of = [&](int first) { return (std::max(0, N - first * 256) + 127) / 128; };
    Plan best;
    const int whole = static_cast<int>(static_cast<long long>(rows) * c256 / 256 * 256 / rows);
    for (int first : {0, whole, c256}) {
        double us = 0.0;
        if (first) us += launch_us(r.wide256, static_cast<long long>(rows) * first, steps);
        if (rest_of(first)) us += launch_us(r.wide128, static_cast<long long>(rows) * rest_of(first), steps);
        if (us < best.us) best = {first, 1, us};
    }
    const long long blocks = static_cast<long long>(rows) * rest_of(0);
    for (int s = 2; s <= 8 && blocks * s <= 256 && steps / s >= 8; ++s) {
        if (static_cast<long long>((steps + s - 1) / s) * (s - 1) + 4 > steps) continue;   // (the last share would be next to nothing)
        const size_t bytes = static_cast<size_t>(s) * M * N * sizeof(float);
        if (bytes > ws_bytes) break;
        const double us = launch_us(r.wide128, blocks * s, (steps + s - 1) / s) + 3.0 + (0.9 * bytes + 2.0 * M * N) / 4e6;
        if (us < best.us) best = {0, s, us};
    }
    return best;
}
// Most bytes the shares of any number of rows from 129 to `most_rows` can take: blocks * shares <= 256 bounds them by 32 MiB.
size_t shares_bytes(int most_rows, int N, int K) {
    const int steps = K / kStepK, cols = (N + 127) / 128;
    size_t bytes = 0;
    for (int rows = 1; most_rows > 128 && rows <= (most_rows + kRows - 1) / kRows && rows * cols <= 128; ++rows) {
        const int s = std::min({8, 256 / (rows * cols), steps / 8});
        if (s > 1) bytes = std::max(bytes, static_cast<size_t>(s) * std::min(most_rows, rows * kRows) * N * sizeof(float));
    }
    return bytes;
}
template <int KVF, int RT>
int launch_experts(const GemmArgs& a, int routes, hipStream_t stream) {
    constexpr int NG = 2, S = 3;   // three blocks of 128 columns to a CU: one's prologue, waits and stores run beside the others' products
    constexpr size_t smem = S * static_cast<size_t>(RT * 16) * kStepK * 2;
    constexpr auto kernel = &gemm_columns_kernel<KVF, RT, NG, S, Form::Experts>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int cols = (a.N + 64 * NG - 1) / (64 * NG);
    const long long rows = routes / (RT * 16) + std::min(routes, a.problems);   // (no cut of the routes into problems makes more)
    const long long blocks = (rows + 7) / 8 * 8 * cols;
    if (blocks > 0x7FFFFFFF) return PIE_HIP_ERR_UNSUPPORTED;
    hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), smem, stream, a, cols, 0, 0);
    return launch_status();
}
// A block's rows by the routes an expert has on average, so that most experts are one block and few of its rows are none's.  128 fp8
// experts of 1536 x 2048, us in blocks of 32 / 64 / 96 / 128 rows: 4 routes each 69 / 76 / 81 / 100, 20 78 / 80 / 87 / 104, 44 122 / 86 / 94 / 118, 62 - / 112 / 97 /
// 114, 78 - / 137 / 110 / 117, 94 - / 143 / 132 / 127; of 2048 x 768 41 / 44 / 60 / 60, 46 / 49 / 62 / 64, 66 / 55 / 65 / 69, - / 73 / 70 / 75, - / 89 / 73 / 77, - / 91 / 95 / 82.
int expert_rows(int routes, int experts) {
    const double each = static_cast<double>(routes) / experts;
    return each <= 24 ? 32 : each <= 54 ? 64 : each <= 84 ? 96 : 128;
}
template <int KVF>
int launch_experts(const GemmArgs& a, int routes, int block_rows, hipStream_t stream) {
    switch (block_rows ? block_rows : expert_rows(routes, a.problems)) {
        case 32: return launch_experts<KVF, 2>(a, routes, stream);
        case 64: return launch_experts<KVF, 4>(a, routes, stream);
        case 96: return launch_experts<KVF, 6>(a, routes, stream);
        default: return launch_experts<KVF, 8>(a, routes, stream);
    }
}
template <int KVF, int RT>
int launch_rows(const GemmArgs& a, int shares, hipStream_t stream) {
    constexpr int NG = 2, S = 3;
    constexpr size_t smem = S * static_cast<size_t>(RT * 16) * kStepK * 2;
    constexpr auto kernel = &gemm_columns_kernel<KVF, RT, NG, S, Form::Rows>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int rows = (a.M + RT * 16 - 1) / (RT * 16), cols = (a.N + 64 * NG - 1) / (64 * NG), steps = a.K / kStepK;
    hipLaunchKernelGGL(kernel, dim3((rows * cols + 7) / 8 * 8, 1, shares), dim3(256), smem, stream, a, cols, rows, (steps + shares - 1) / shares);
    return launch_status();
}
template <int KVF, int RT>
int launch_columns(const GemmArgs& a, hipStream_t stream) {
    constexpr int S = 4, KP = 2;
    constexpr size_t smem = KP * S * static_cast<size_t>(RT * 16) * kStepK * 2;
    constexpr auto kernel = &gemm_columns_kernel<KVF, RT, 1, S, Form::Whole, KP>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int cols = (a.N + 63) / 64;
    hipLaunchKernelGGL(kernel, dim3(cols), dim3(256 * KP), smem, stream, a, cols, 1, 0);
    return launch_status();
}
template <int KVF>
int launch_columns(const GemmArgs& a, hipStream_t stream) {
    return a.M <= 64 ? launch_columns<KVF, 4>(a, stream) : a.M <= 96 ? launch_columns<KVF, 6>(a, stream) : launch_columns<KVF, 8>(a, stream);
}
bool fits(int format, int M, int N, int K, int group_size) {
    if (K % (format == PIE_HIP_FMT_INT4B8 ? 128 : 64) != 0 || K < 4 * kStepK) return false;
    if (format == PIE_HIP_FMT_INT4B8 && (group_size < 64 || (group_size & (group_size - 1)) != 0 || K % group_size != 0)) return false;
    return 2ll * M * K <= 0xFFFFFFFFll && 2ll * (N + 15) * K <= 0xFFFFFFFFll && (M + 255ll) / 256 * ((N + 127ll) / 128) < 0x0FFFFFFF;
}

// up to 128 rows of one-byte weights, 17 to 48 of int4 ones (those in gemm_groups_mfma.hip)
bool columns_fit(int format, int M, int N, int K, int group_size) {
    if (N % 16 != 0 || static_cast<long long>(N) * K > 0xFFFFFFFFll) return false;
    if (format == PIE_HIP_FMT_INT4B8)
        return M > 16 && M <= 48 && gemm_groups_us(M, N, K, group_size, 0) < 1e30;
    return M <= 128 && (format == PIE_HIP_FMT_FP8 || format == PIE_HIP_FMT_INT8) && K % kStepK == 0;
}
// A round of blocks (one to a CU, two with 64 rows' LDS) takes 4 to 5.5 us and, a step, 0.19 - 0.35 for a few blocks and 0.08 - 0.13 more when all CUs have
// one, or what the weights take at 6 TB/s (measured at 17 - 128 rows of 15 matrices of 1024 - 28672 x 1024 - 14336, weights out of HBM: 9 % rms).
double columns_us(int format, int M, int N, int K, int group_size, size_t ws_bytes) {
    if (format == PIE_HIP_FMT_INT4B8) return gemm_groups_us(M, N, K, group_size, ws_bytes);
    const int size = M <= 64 ? 0 : M <= 96 ? 1 : 2, fp8 = format == PIE_HIP_FMT_FP8;
    constexpr double kFixed[3] = {3.8, 4.6, 5.5}, kStepUs[2][3] = {{0.23, 0.30, 0.35}, {0.19, 0.28, 0.34}}, kFull[2][3] = {{0.10, 0.12, 0.12}, {0.08, 0.13, 0.13}};
    const long long blocks = (N + 63) / 64, slots = size == 0 ? 512 : 256;
    const double crowd = size == 0 && blocks > 256 ? (fp8 ? 1.8 : 1.42) : 1.0, step = (kStepUs[fp8][size] + kFull[fp8][size] * std::min(1.0, blocks / 256.0)) * crowd;
    return std::max(kFixed[size] + static_cast<double>((blocks + slots - 1) / slots) * (K / kStepK) * step, 2.6 + 1e-6 * N * K / 6.0);
}

// ---- one-byte weights and many rows in blocks of 32 to 128 rows x 128 columns ---------------------------------------------------
// (The blocks of 256 rows pass the decoded weights through LDS, in rounds of one block to a CU, and pad their rows.  Three small blocks to a CU
// fill the machine from some hundred rows on and hide one another's prologue and stores.  Weights from HBM, us there / here, fp8: 400 / 1300 / 2048
// rows of 5120 x 2048 30.9 / 17.0, 37.3 / 33.8 and 60.2 / 46.9; 320 / 512 rows of 28672 x 4096 109 / 84 and 114 / 112; int8: 400 of 2048 x 4096 26.1 / 20.5.)
// Blocks that share a CU with c - 1 others take `fixed` and `step` of the c-th column (four: more in proportion), where only some CUs have the c-th up to an
// eighth less.  A block alone waits for its weights from HBM at every step, three of which are in flight: 0.33 - 0.54 us a step whatever the
// rows, which is why a long K of few blocks pays for shares.  Shares' sums meet in a second kernel, 3 us and their bytes at 3.6 TB/s.  Measured over 50
// matrices of 1024 - 28672 x 1024 - 14336 and 129 - 2048 rows, each call's weights out of HBM: 6 % rms, the faster of both kernels missed by 1 % on
// average.
struct RowsPlan {
    int row_tiles = 0, shares = 1;
    double us = 1e30;
};
struct Round {
    double fixed, step;
};
constexpr Round kRowRounds[2][4][4] = {{{{3.8, 0.325}, {4.6, 0.364}, {5.0, 0.490}, {5.6, 0.705}},
                                     {{4.4, 0.463}, {5.9, 0.529}, {7.9, 0.735}, {8.6, 0.959}},
                                     {{5.6, 0.481}, {8.4, 0.647}, {10.0, 0.952}, {12.2, 1.275}},
                                     {{7.1, 0.538}, {9.8, 0.830}, {11.4, 1.220}, {14.5, 1.611}}},
                                    {{{3.5, 0.430}, {4.4, 0.466}, {5.9, 0.585}, {6.3, 0.751}},
                                     {{4.6, 0.468}, {6.3, 0.571}, {7.8, 0.813}, {8.7, 1.050}},
                                     {{5.7, 0.512}, {8.0, 0.716}, {10.0, 1.026}, {11.7, 1.398}},
                                     {{7.1, 0.586}, {9.8, 0.889}, {11.6, 1.295}, {14.1, 1.731}}}};
// Microseconds of `n` blocks of 16 `row_tiles` rows, `per` steps each, over a matrix of `mb` million weights.
double row_blocks_us(int format, int row_tiles, long long n, int per, double mb) {
    const int c = static_cast<int>(std::min(4ll, (n + 255) / 256));
    const Round& r = kRowRounds[format == PIE_HIP_FMT_INT8][row_tiles / 2 - 1][c - 1];
    const double us = r.fixed + r.step * per;
    // (32 rows of fp8, three to a CU: a fifth less where only some CUs have the third, and a part that goes with the matrix, which each chiplet reads
    // for few rows.  1237 x 2048 x 4096 takes 34.5 us: priced at 33.2, at 37.2 by the others' rule, where 64 rows take 38.1.)
    const bool thin = row_tiles == 2 && c == 3 && format == PIE_HIP_FMT_FP8;
    const double less = c == 1 ? 0.04 : thin ? 0.19 : 0.13;
    return (n > 1024 ? us * static_cast<double>(n) / 1024.0 : us * (1.0 - less * (c - n / 256.0))) + (thin ? 0.09 * mb : 0.0);
}
RowsPlan rows_plan(int format, int M, int N, int K, size_t ws_bytes) {
    const int steps = K / kStepK;
    RowsPlan best;
    for (int half = 1; half <= 4; ++half) {
        const long long tiles = (M + half * 32ll - 1) / (half * 32) * ((N + 127) / 128);
        for (int s = 1; s <= 6; ++s) {
            const int per = (steps + s - 1) / s;
            const size_t bytes = static_cast<size_t>(s) * M * N * sizeof(float);
            if (s > 1 && (per < 4 || bytes > ws_bytes || tiles * (s - 1) >= 768)) break;
            if ((s - 1) * per >= steps) continue;   // (the last share would be empty)
            double us = row_blocks_us(format, half * 2, tiles * s, per, 1e-6 * N * K);
            if (s > 1) us += 3.0 + static_cast<double>(bytes) / 3.6e6;
            if (us < best.us) best = {half * 2, s, us};
        }
    }
    return best;
}
bool rows_fit(int format, int M, int N, int K) {
    return (format == PIE_HIP_FMT_FP8 || format == PIE_HIP_FMT_INT8) && M > 0 && N > 0 && N % 16 == 0 && K > 0 && K % kStepK == 0 &&
           static_cast<long long>(N) * K <= 0xFFFFFFFFll && (M + 31ll) / 32 * ((N + 127ll) / 128) < 0x0FFFFFFF;
}
// Microseconds of a grouped product over tile-major one-byte experts with fewer than 16 routes each, in passes of 16 routes or in blocks of 32.  The
// passes split K over a block's waves and spread an expert over the chip.  The blocks of an expert stay on one chiplet, which reads 0.9 TB/s: fewer experts
// than chiplets leave the others idle, and few columns wait for HBM at every step of K.  Both products of 8 fp8 experts of 28672 x 4096 and 4096 x 14336 with two routes each, passes /
// blocks of 1, 2, 4 and 16 tokens: 76 / 151, 143 / 192, 162 / 219 and 243 / 248 us; of 128 of 1536 x 2048 and 2048 x 768 with eight: 21 / 18, 24 / 21, 39 / 31 and 83 / 75.
// Fitted to both products of 14 mixtures of 8 to 256 experts: the faster of both ways missed by 1 % on average.
double few_routes_us(int format, int routes, int experts, int N, int K, bool swiglu, bool blocks) {
    const double each = static_cast<double>(routes) / experts, touched = experts * (1.0 - std::exp(-each)), mb = 1e-6 * N * K;
    if (blocks) {
        const long long per_chiplet = static_cast<long long>(std::ceil(touched / 8.0 - 1e-9));
        return std::max({row_blocks_us(format, 2, per_chiplet * 8 * ((N + 127) / 128), K / kStepK, 0.0), 4.0 + touched * mb / 6.05, 4.0 + per_chiplet * mb / 0.9});
    }
    // (gathered rows and the gate's epilogue: 2.5 us from a second chunk of K on)
    const double gate = swiglu ? std::min(1.0, std::max(0.0, K / 1000.0 - 1.0)) : 0.0;
    return format == PIE_HIP_FMT_INT8 ? 5.0 + touched * mb / 5.93 + 0.00060 * K + 0.085 * each + 2.7 * gate
                                      : 4.3 + touched * mb / 5.91 + 0.00046 * K + 0.106 * each + 2.4 * gate;
}
template <int KVF>
int launch_rows(const GemmArgs& a, const RowsPlan& p, hipStream_t stream) {
    return p.row_tiles == 2   ? launch_rows<KVF, 2>(a, p.shares, stream)
           : p.row_tiles == 4 ? launch_rows<KVF, 4>(a, p.shares, stream)
           : p.row_tiles == 6 ? launch_rows<KVF, 6>(a, p.shares, stream)
                              : launch_rows<KVF, 8>(a, p.shares, stream);
}

template <class F>
int run(GemmArgs a, const Plan& p, float* ws, hipStream_t stream) {
    int st = PIE_HIP_OK;
    a.aligned = reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
    a.lines = stores_lines(a.y, a.N);
    if (p.splits > 1) a.partial = ws;
    if (p.first) st = launch<F, 256>(a, 0, p.first, 1, stream);
    const int rest = (std::max(0, a.N - p.first * 256) + 127) / 128;
    if (st == PIE_HIP_OK && rest) st = launch<F, 128>(a, p.first * 256, rest, p.splits, stream);
    if (st != PIE_HIP_OK || p.splits == 1) return st;
    const size_t quads = static_cast<size_t>(a.M) * ((a.N + 3) / 4);
    hipLaunchKernelGGL(wide_reduce_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, stream, a, p.splits);
    return launch_status();
}

}  // namespace

double gemm_wide_us(int format, int M, int N, int K, int group_size, size_t ws_bytes) {
    if (columns_fit(format, M, N, K, group_size)) return columns_us(format, M, N, K, group_size, ws_bytes);
    return fits(format, M, N, K, group_size) ? plan_of(kRates[format], M, N, K, ws_bytes).us : 1e30;
}
// (the choice between its two heights is launch_gemm's)
double gemm_tiles_us(int format, int M, int N, int K) {
    const Rates& r = kRates[format];
    const long long cols = (N + 127) / 128, low = cols * ((M + 127) / 128), high = cols * ((M + 255) / 256);
    const long long low_rounds = (low + 255) / 256, high_rounds = (high + 255) / 256;
    const double steps = K / kStepK;
    // (bf16: a round of either height starts and stores for a while, which at a short K is most of it; where few blocks run it is up to a fifth high: 500 x 2048 x
    // 256 10.6 for 8.9, 1000 x 4096 x 512 13.6 for 12.0, 200 x 4096 x 4096 35.4 for 37.4)
    const bool tall = 1.85 * static_cast<double>(high_rounds) < static_cast<double>(low_rounds);
    if (format == PIE_HIP_FMT_BF16) {
        if (tall) return 3.0 + high_rounds * (9.8 + steps * r.tall);
        return 3.5 + 5.5 * static_cast<double>(low_rounds) + steps * (low <= 256 ? r.few + r.many * static_cast<double>(low) / 256.0 : r.round * static_cast<double>(low_rounds));
    }
    if (tall) return high_rounds * (5.0 + steps * r.tall);
    return 7.0 + steps * (low <= 256 ? r.few + r.many * static_cast<double>(low) / 256.0 : r.round * static_cast<double>(low_rounds));
}

int launch_gemm_wide(int format, const GemmArgs& a, int group_size, void* ws, size_t ws_bytes, hipStream_t stream) {
    if (format == PIE_HIP_FMT_INT4B8 && columns_fit(format, a.M, a.N, a.K, group_size)) {
        const int st = launch_gemm_groups(a, group_size, ws, ws_bytes, stream);
        if (st != PIE_HIP_ERR_UNSUPPORTED) return st;
    } else if (columns_fit(format, a.M, a.N, a.K, group_size) && reinterpret_cast<uintptr_t>(a.act) % 16 == 0 && reinterpret_cast<uintptr_t>(a.w) % 16 == 0) {
        GemmArgs b = a;
        b.aligned = reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
        return format == PIE_HIP_FMT_FP8 ? launch_columns<kKvFp8>(b, stream) : launch_columns<kKvInt8>(b, stream);
    }
    if (!fits(format, a.M, a.N, a.K, group_size) || reinterpret_cast<uintptr_t>(a.act) % 16 || reinterpret_cast<uintptr_t>(a.w) % 16)
        return PIE_HIP_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(ws) % 16) ws = nullptr;
    const Plan p = plan_of(kRates[format], a.M, a.N, a.K, ws ? ws_bytes : 0);
    switch (format) {
        case PIE_HIP_FMT_INT4B8: return run<WInt4>(a, p, static_cast<float*>(ws), stream);
        case PIE_HIP_FMT_INT8: return run<WInt8>(a, p, static_cast<float*>(ws), stream);
        case PIE_HIP_FMT_FP8: return run<WFp8>(a, p, static_cast<float*>(ws), stream);
        case PIE_HIP_FMT_BF16: return run<WBf16>(a, p, static_cast<float*>(ws), stream);
        default: return PIE_HIP_ERR_INVALID;
    }
}

int launch_gemm_experts(int format, const GemmArgs& a, int routes, int block_rows, hipStream_t stream) {
    GemmArgs b = a;
    b.aligned = reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
    b.lines = stores_lines(a.y, a.N);
    if (a.K % kStepK != 0 || a.N % 16 != 0 || static_cast<long long>(a.N) * a.K > 0xFFFFFFFFll ||
        reinterpret_cast<uintptr_t>(a.act) % 16 || reinterpret_cast<uintptr_t>(a.w) % 16 || a.w_stride % 16)
        return PIE_HIP_ERR_UNSUPPORTED;
    if (format == PIE_HIP_FMT_FP8) return launch_experts<kKvFp8>(b, routes, block_rows, stream);
    if (format == PIE_HIP_FMT_INT8) return launch_experts<kKvInt8>(b, routes, block_rows, stream);
    return PIE_HIP_ERR_UNSUPPORTED;
}

}  // namespace pie_hip

extern "C" int pie_hip_moe_block_rows(int num_routes, int num_experts, int block_rows) {
    if (num_routes <= 0 || num_experts <= 0 || (block_rows != 0 && block_rows != 128)) return 0;
    return block_rows ? block_rows : pie_hip::expert_rows(num_routes, num_experts);
}

extern "C" float pie_hip_moe_few_routes_us(int format, int num_routes, int num_experts, int N, int K, int swiglu, int in_blocks) {
    if ((format != PIE_HIP_FMT_FP8 && format != PIE_HIP_FMT_INT8) || num_routes <= 0 || num_experts <= 0 || N <= 0 || K <= 0) return 1e30f;
    return static_cast<float>(pie_hip::few_routes_us(format, num_routes, num_experts, N, K, swiglu != 0, in_blocks != 0));
}

extern "C" float pie_hip_gemm_rows_us(int format, int M, int N, int K, size_t workspace_bytes) {
    return pie_hip::rows_fit(format, M, N, K) ? static_cast<float>(pie_hip::rows_plan(format, M, N, K, workspace_bytes).us) : 1e30f;
}

extern "C" int pie_hip_gemm_rows_plan(int format, int M, int N, int K, size_t workspace_bytes, int* block_rows, int* shares) {
    if (!block_rows || !shares) return PIE_HIP_ERR_INVALID;
    if (!pie_hip::rows_fit(format, M, N, K)) return PIE_HIP_ERR_UNSUPPORTED;
    const pie_hip::RowsPlan p = pie_hip::rows_plan(format, M, N, K, workspace_bytes);
    *block_rows = p.row_tiles * 16;
    *shares = p.shares;
    return PIE_HIP_OK;
}

extern "C" int pie_hip_gemm_rows_tiled(int format, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16,
                                       uint16_t* y_bf16, int M, int N, int K, int beta, int epilogue, const PieHipGlu* glu,
                                       void* workspace, size_t workspace_bytes, void* stream) {
    using namespace pie_hip;
    if (!glu_ok(glu, epilogue)) return PIE_HIP_ERR_INVALID;
    if (!act_bf16 || !weight || !scale || !y_bf16 || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
    const int pointwise = pointwise_code(epilogue), swiglu = epilogue == PIE_HIP_EPI_SWIGLU ? 1 : 0;
    if ((swiglu && N % 2 != 0) || ((swiglu || pointwise) && beta)) return PIE_HIP_ERR_INVALID;
    if (!rows_fit(format, M, N, K) || reinterpret_cast<uintptr_t>(act_bf16) % 16 || reinterpret_cast<uintptr_t>(weight) % 16) return PIE_HIP_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(workspace) % 16) workspace = nullptr;
    const RowsPlan p = rows_plan(format, M, N, K, workspace ? workspace_bytes : 0);
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
    a.aligned = reinterpret_cast<uintptr_t>(y_bf16) % 8 == 0;
    a.lines = stores_lines(y_bf16, N);
    a.partial = p.shares > 1 ? static_cast<float*>(workspace) : nullptr;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int st = format == PIE_HIP_FMT_FP8 ? launch_rows<kKvFp8>(a, p, s) : launch_rows<kKvInt8>(a, p, s);
    if (st != PIE_HIP_OK || p.shares == 1) return st;
    const size_t quads = static_cast<size_t>(M) * (N / 4);
    hipLaunchKernelGGL(wide_reduce_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, s, a, p.shares);
    return launch_status();
}

extern "C" float pie_hip_gemm_mfma_us(int format, int M, int N, int K, int group_size, int tiled, size_t workspace_bytes) {
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || M <= 0 || N <= 0 || K <= 0) return 1e30f;
    const double tiles = M > 128 ? pie_hip::gemm_tiles_us(format, M, N, K) : 1e30;
    if (M <= 128 && !(tiled && pie_hip::columns_fit(format, M, N, K, group_size))) return 1e30f;
    const double wide = tiled || format == PIE_HIP_FMT_BF16 ? pie_hip::gemm_wide_us(format, M, N, K, group_size, workspace_bytes) : 1e30;
    return static_cast<float>(std::min(tiles, wide));
}

extern "C" int pie_hip_gemm_bf16_wide(int M, int N, int K, size_t workspace_bytes) {
    using namespace pie_hip;
    return M > 128 && N > 0 && K > 0 && gemm_wide_us(PIE_HIP_FMT_BF16, M, N, K, 0, workspace_bytes) < gemm_tiles_us(PIE_HIP_FMT_BF16, M, N, K) ? 1 : 0;
}

extern "C" size_t pie_hip_gemm_mfma_tiled_workspace_bytes(int most_rows, int N, int K) {
    return N > 0 && K > 0 ? pie_hip::shares_bytes(most_rows, N, K) : 0;
}

extern "C" int pie_hip_gemm_mfma_tiled(int format, const uint16_t* act_bf16, const void* weight, const void* scale, int scale_is_bf16,
                                       int group_size, uint16_t* y_bf16, int M, int N, int K, int beta, int epilogue,
                                       const PieHipGlu* glu, void* workspace, size_t workspace_bytes, void* stream) {
    using namespace pie_hip;
    if (!glu_ok(glu, epilogue)) return PIE_HIP_ERR_INVALID;
    if (!act_bf16 || !weight || !y_bf16 || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || (format != PIE_HIP_FMT_BF16 && !scale)) return PIE_HIP_ERR_INVALID;
    const int pointwise = pointwise_code(epilogue), swiglu = epilogue == PIE_HIP_EPI_SWIGLU ? 1 : 0;
    if ((swiglu && N % 2 != 0) || ((swiglu || pointwise) && beta)) return PIE_HIP_ERR_INVALID;
    if (format != PIE_HIP_FMT_BF16 && N % 16 != 0) return PIE_HIP_ERR_UNSUPPORTED;   // (there is no tile-major copy)
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
    if (format == PIE_HIP_FMT_INT4B8 && group_size > 0) a.g_shift = __builtin_ctz(static_cast<unsigned>(group_size));
    return launch_gemm_wide(format, a, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
