// Int4 weights times two and more activation rows with the group scales kept in fp32: y[M, N] = epilogue( act[M, K] · W[N, K]^T ),
// the skinny GEMM's arithmetic (a group's code products are summed as they are and scaled once, in fp32) in blocks of 16 to 64
// rows x 128 columns, two blocks of four waves to a CU.
//
// The skinny GEMM's passes of 32 rows read and decode the weights once each, stage their rows per wave, and their number costs in
// powers of two.  Here a wave owns 32 columns for all rows of the block: the tile-major copy gives it the MFMAs' operand by plain
// loads, four steps of 128 k-values ahead in registers, decoded once per 64 rows; the block's waves share the activations in LDS.
// The codes enter the products as 128 + n; a product of -136 against the activations is the accumulator they start from.  A
// step is three phases of 4 RT products, so that there is something to do beside each: the sums' phase decodes the first
// column tile and scales the last step's second, the first tile's decodes the second, the second's scales the first and reads
// the next step's activations.
// What bounds it: issue.  A SIMD that multiplies issues a vector instruction every five cycles whoever's it is, and a product of
// 16 x 16 x 32 takes eight of them: 48 products, 140 vector instructions and 16 LDS reads a step of two blocks are 1.1 us of 64
// rows, the matrix pipe alone 0.7.  (Two halves of a step with their reads spread over it: the same.  Products of 32 x 32 x 16 and
// sums made by a kernel before: the chip lowers its clock to 1.8 GHz, 99 us against 107 at 321 x 28672 x 4096, slower at
// all other shapes.  A second group of waves per block taking every other step: the same or slower.)
// Skinny GEMM / here, us: 321 x 4096 x 14336 69 / 58, x 6144 x 4096 70 / 32, x 4096 x 4096 26 / 21; 96 x 28672 x 4096 50 / 35;
// 64 x 4096 x 14336 22 / 20; 48 x 28672 x 4096 31 / 24.
#include "gemm_args.hip.h"

#include <algorithm>
#include <type_traits>

namespace pie_hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

constexpr int kStep = 128, kStages = 4, kTiles = 2;   // k-values of a step; steps in flight; column tiles of a wave
constexpr int kCols = 4 * kTiles * 16;                // columns of a block

template <int RT>
__global__ __launch_bounds__(256, 2) void gemm_groups_kernel(const GemmArgs a, const Rotation rot, int row_blocks, int per_xcd, int blocks, int per_share) {
    constexpr int S = kStages, NG = kTiles, kVecs = RT * 16 * (kStep / 8), kOps = RT + 2 * NG;
    static_assert(RT >= 1 && RT <= 4 && NG == 2, "a quarter of a phase scales one row tile; two tiles' sums");
    extern __shared__ __align__(16) unsigned char smem[];
    u32x4_t* lds = reinterpret_cast<u32x4_t*>(smem);
    const int tid = threadIdx.x, lane = tid & (kWave - 1);
    const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
    const int j = lane & 15, q = lane >> 4;
    // blocks go to the XCDs in turn: each XCD's are neighbours, the row blocks of a column block side by side
    const int block = static_cast<int>(blockIdx.x & 7) * per_xcd + static_cast<int>(blockIdx.x >> 3);
    if (block >= blocks) return;
    const int m0 = block % row_blocks * (RT * 16), tile0 = (block / row_blocks * 4 + wv) * NG;
    const int N = a.N, K = a.K, M = a.M, T = N / 16, nb = K / kStep;
    const int first = static_cast<int>(blockIdx.z) * per_share, nk = min(per_share, nb - first);   // this share's steps
    auto place = [&](int kt) { return first + min(kt, nk - 1); };   // (past them: the last one again)
    const int groups = K >> a.g_shift, to_group = a.g_shift - 7;

    uint32_t woff[NG], soff[NG];
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const uint32_t tile = min(tile0 + i, T - 1);
        woff[i] = tile * (nb * 1024u) + lane * 16u;
        soff[i] = tile * (groups * 32u) + q * 8u;
    }
    u32x4_t raw[S][NG];
    u32x2_t gs[S][NG];
    auto load_w = [&](int kt, int slot) __attribute__((always_inline)) {
        const int b = place(kt);
        const unsigned char* pw = a.w + static_cast<size_t>(b) * 1024;
        const unsigned char* ps = a.scale + static_cast<size_t>(b >> to_group) * 32;
#pragma unroll
        for (int i = 0; i < NG; ++i) {
            asm volatile("" : "+v"(woff[i]), "+v"(soff[i]));   // (32-bit offsets from scalar bases, not 64-bit sums)
            raw[slot][i] = *reinterpret_cast<const u32x4_t*>(pw + woff[i]);
            gs[slot][i] = *reinterpret_cast<const u32x2_t*>(ps + soff[i]);
        }
        PIE_FENCE();
    };
    uint32_t aoff[RT];
#pragma unroll
    for (int u = 0; u < RT; ++u) {
        const int r = (u * 4 + wv) * 4 + (lane >> 4);
        aoff[u] = static_cast<uint32_t>(min(m0 + r, M - 1)) * (2u * K) + ((lane & 15) ^ key_of(r)) * 16;
    }
    auto issue_a = [&](int kt, int stage) __attribute__((always_inline)) {
        const unsigned char* pa = reinterpret_cast<const unsigned char*>(a.act) + static_cast<size_t>(place(kt)) * (kStep * 2);
#pragma unroll
        for (int u = 0; u < RT; ++u) {
            asm volatile("" : "+v"(aoff[u]));
            to_lds(pa + aoff[u], lds + stage * kVecs + (u * 4 + wv) * 64);
        }
        PIE_FENCE();
    };
    const int key = key_of(j);
    bf16x8_t af[RT][4], bw[2][4];
    auto read_a = [&](int stage, int s) __attribute__((always_inline)) {
        const u32x4_t* A = lds + stage * kVecs + j * 16 + ((4 * q + s) ^ key);
#pragma unroll
        for (int t = 0; t < RT; ++t) af[t][s] = __builtin_bit_cast(bf16x8_t, A[t * 256]);
    };
    uint32_t k128 = 0x43004300u;   // (128.0, 128.0) as a bf16 pair, opaque to the compiler
    asm volatile("" : "+v"(k128));
    auto decode = [&](const u32x4_t& r, int s) __attribute__((always_inline)) {
        const uint32_t v = r[s];
        return __builtin_bit_cast(bf16x8_t, u32x4_t{and_or(v, 0x000F000Fu, k128), and_or(v >> 4, 0x000F000Fu, k128),
                                                    and_or(v >> 8, 0x000F000Fu, k128), and_or(v >> 12, 0x000F000Fu, k128)});
    };
    const bf16x8_t offset = __builtin_bit_cast(bf16x8_t, u32x4_t{0xC308C308u, 0xC308C308u, 0xC308C308u, 0xC308C308u});   // -136
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t acc[RT][NG], sum[NG][RT], sx[RT];
    float sc[NG][4];
#pragma unroll
    for (int t = 0; t < RT; ++t)
#pragma unroll
        for (int i = 0; i < NG; ++i) acc[t][i] = sum[i][t] = zero;
#pragma unroll
    for (int i = 0; i < NG; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) sc[i][r] = 0.f;

    // (lane: row j, columns 4q .. 4q + 3 of a tile)
    auto scale = [&](int i, int t) __attribute__((always_inline)) {
        if (t < RT)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[t][i][r] = fmaf(sc[i][r], sum[i][t][r], acc[t][i][r]);
    };
    auto unpack = [&](int i, const u32x2_t& g) __attribute__((always_inline)) {
        sc[i][0] = bf16_lo(g.x);
        sc[i][1] = bf16_hi(g.x);
        sc[i][2] = bf16_lo(g.y);
        sc[i][3] = bf16_hi(g.y);
    };
    auto spread = [&](auto vector, auto reads) __attribute__((always_inline)) {   // a quarter's products, vector instructions between
#pragma unroll
        for (int u = 0; u < RT; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, (decltype(vector)::value + RT - 1) / RT, 0);
        }
        if (decltype(reads)::value) __builtin_amdgcn_sched_group_barrier(0x100, RT, 0);
        PIE_FENCE();
    };

#pragma unroll
    for (int i = 0; i < S; ++i) {
        issue_a(i, i);
        load_w(i, i);
    }
    PIE_WAIT_VM((S - 1) * kOps);
    PIE_MEET();
#pragma unroll
    for (int s = 0; s < 4; ++s) read_a(0, s);
    auto step = [&](auto slot, int kt) __attribute__((always_inline)) {
        constexpr int cur = decltype(slot)::value, next = (cur + 1) % S;
        // -136 times the activations' sums; the step before's second tile is scaled, the first one decoded
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int t = 0; t < RT; ++t) sx[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(offset, af[t][s], s ? sx[t] : zero, 0, 0, 0);
            bw[0][s] = decode(raw[cur][0], s);
            scale(1, s);
            spread(std::integral_constant<int, 11>{}, std::false_type{});
        }
        unpack(0, gs[cur][0]);
        unpack(1, gs[cur][1]);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int t = 0; t < RT; ++t) sum[0][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[0][s], af[t][s], s ? sum[0][t] : sx[t], 0, 0, 0);
            bw[1][s] = decode(raw[cur][1], s);
            spread(std::integral_constant<int, 9>{}, std::false_type{});
        }
        PIE_WAIT_VM((S - 2) * kOps);   // step kt + 1 has come
        PIE_MEET();                    // and everybody has read step kt
        issue_a(kt + S, cur);
        load_w(kt + S, cur);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
#pragma unroll
            for (int t = 0; t < RT; ++t) sum[1][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bw[1][s], af[t][s], s ? sum[1][t] : sx[t], 0, 0, 0);
            scale(0, s);
            read_a(next, s);
            spread(std::integral_constant<int, 4>{}, std::true_type{});
        }
    };
    int kt = 0;
    for (; kt + S <= nk; kt += S) {
        step(std::integral_constant<int, 0>{}, kt);
        step(std::integral_constant<int, 1>{}, kt + 1);
        step(std::integral_constant<int, 2>{}, kt + 2);
        step(std::integral_constant<int, 3>{}, kt + 3);
    }
    if (kt < nk) step(std::integral_constant<int, 0>{}, kt);
    if (kt + 1 < nk) step(std::integral_constant<int, 1>{}, kt + 1);
    if (kt + 2 < nk) step(std::integral_constant<int, 2>{}, kt + 2);
#pragma unroll
    for (int t = 0; t < RT; ++t) scale(1, t);
    __builtin_amdgcn_s_waitcnt(0x0070);   // (transfers past the last step land before the block ends)
    if (a.lines && !a.partial && !rot.table) {
        const int n = tile0 * 16 + 4 * q;
        if (n >= N) return;
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
                    for (int r = 0; r < 4; ++r) v[i][r] = acc[t][i][r];
                store_pair<decltype(out)::value>(a, to, n, v[0], v[1]);
            }
        });
        return;
    }
#pragma unroll
    for (int i = 0; i < NG; ++i) {
        const int n = (tile0 + i) * 16 + 4 * q;
        if (n >= N) continue;
#pragma unroll
        for (int t = 0; t < RT; ++t) {
            const int m = m0 + t * 16 + j;
            if (m >= M) continue;
            float v[4] = {acc[t][i][0], acc[t][i][1], acc[t][i][2], acc[t][i][3]};
            if (a.partial) *reinterpret_cast<f32x4_t*>(a.partial + (static_cast<size_t>(blockIdx.z) * M + m) * N + n) = acc[t][i];
            else store4(a, rot, m, n, v);
        }
    }
}

// The shares' sums in the order of K, and the epilogue.
__global__ __launch_bounds__(256) void shares_reduce_kernel(const GemmArgs a, const Rotation rot, int shares) {
    const int quads = a.N / 4;
    const size_t idx = static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x;
    if (idx >= static_cast<size_t>(a.M) * quads) return;
    const int m = static_cast<int>(idx / quads), n = static_cast<int>(idx % quads) * 4;
    const size_t plane = static_cast<size_t>(a.M) * a.N;
    const float* p = a.partial + static_cast<size_t>(m) * a.N + n;
    f32x4_t sum = *reinterpret_cast<const f32x4_t*>(p);
    for (int z = 1; z < shares; ++z) sum += *reinterpret_cast<const f32x4_t*>(p + z * plane);
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    store4(a, rot, m, n, v);
}

}  // namespace
int launch_shares_reduce(const GemmArgs& a, const Rotation& rot, int shares, hipStream_t stream) {
    const size_t quads = static_cast<size_t>(a.M) * (a.N / 4);
    hipLaunchKernelGGL(shares_reduce_kernel, dim3(static_cast<unsigned>((quads + 255) / 256)), dim3(256), 0, stream, a, rot, shares);
    return launch_status();
}
namespace {

template <int RT>
int launch(const GemmArgs& a, const Rotation& rot, int shares, hipStream_t stream) {
    constexpr size_t smem = kStages * static_cast<size_t>(RT * 16) * kStep * 2;
    constexpr auto kernel = &gemm_groups_kernel<RT>;
    static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
    if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
    const int rows = (a.M + RT * 16 - 1) / (RT * 16), blocks = rows * ((a.N + kCols - 1) / kCols), per = (blocks + 7) / 8;
    const int steps = a.K / kStep;
    hipLaunchKernelGGL(kernel, dim3(8 * per, 1, shares), dim3(256), smem, stream, a, rot, rows, per, blocks, (steps + shares - 1) / shares);
    return launch_status();
}

// Rows per block and shares of K.  A block alone on its CU takes 3.7 us and `alone` a step, or what its weights take at 6.3 TB/s; two to a
// CU take 2 us more and `pair`; rounds of 512 blocks take 2 us and their steps each, what is left over a sixth of one.
// The shares' sums meet in a second kernel: 3 us and their bytes at 3.2 TB/s, or (`norm`) 0.1 us a share and their bytes at 4 TB/s on top of the norm
// that would run anyway.  Fitted to 5 - 800 rows of 28672 x 4096, 6144 x 4096, 4096 x 4096 and 4096 x 14336: the plan taken is within 8 % of the fastest of all.
struct Plan {
    int row_tiles = 0, shares = 1;
    double us = 1e30;
};
Plan plan_of(int M, int N, int K, size_t ws_bytes, bool norm) {
    constexpr double kAlone[] = {0.28, 0.44, 0.60, 0.80}, kPair[] = {0.55, 0.715, 0.92, 1.19};
    const int steps = K / kStep;
    Plan best;
    for (int rt = 1; rt <= 4; ++rt) {
        const long long tiles = (M + rt * 16ll - 1) / (rt * 16) * ((N + kCols - 1) / kCols);
        for (int s = norm ? 2 : 1; s <= 8; ++s) {
            const int per = (steps + s - 1) / s;
            const size_t bytes = static_cast<size_t>(s) * M * N * sizeof(float);
            if (s > 1 && (per < 2 || bytes > ws_bytes || tiles * (s - 1) >= 512)) break;
            if ((s - 1) * per >= steps) continue;   // (the last share would be empty)
            const double n = static_cast<double>(tiles) * s, alone = kAlone[rt - 1], pair = kPair[rt - 1];
            double us;
            if (n <= 256) us = 3.7 + per * std::max(alone, n * 8448 / 6.3e6);
            else if (n <= 512) us = 5.7 + per * (alone + (pair - alone) * (0.3 + 0.7 * (n - 256) / 256));
            else us = 2.0 + (n / 512 + 1.0 / 6.0) * (2.0 + per * pair);
            if (norm) us += 0.1 * s + static_cast<double>(bytes) / 4e6;
            else if (s > 1) us += 3.0 + static_cast<double>(bytes) / 3.2e6;
            if (us < best.us) best = {rt, s, us};
        }
    }
    return best;
}
bool fits(int M, int N, int K, int group_size) {
    return M > 0 && N % 16 == 0 && K % kStep == 0 && group_size >= kStep && (group_size & (group_size - 1)) == 0 && K % group_size == 0 &&
           static_cast<long long>(N) * K <= 0xFFFFFFFFll && 2ll * M * K <= 0xFFFFFFFFll && (M + 31ll) / 32 * ((N + kCols - 1ll) / kCols) < 0x0FFFFFFF;
}
// (`shares`: the sums stay in the workspace, in that many shares)
int run(GemmArgs a, const Rotation& rot, int group_size, void* ws, size_t ws_bytes, hipStream_t stream, int* shares = nullptr) {
    if (!fits(a.M, a.N, a.K, group_size) || reinterpret_cast<uintptr_t>(a.act) % 16 || reinterpret_cast<uintptr_t>(a.w) % 16 ||
        reinterpret_cast<uintptr_t>(a.scale) % 8)
        return PIE_HIP_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(ws) % 16) ws = nullptr;
    const Plan p = plan_of(a.M, a.N, a.K, ws ? ws_bytes : 0, shares != nullptr);
    if (p.row_tiles == 0) return PIE_HIP_ERR_UNSUPPORTED;
    a.g_shift = __builtin_ctz(static_cast<unsigned>(group_size));
    a.aligned = reinterpret_cast<uintptr_t>(a.y) % 8 == 0;
    a.lines = stores_lines(a.y, a.N);
    a.partial = p.shares > 1 ? static_cast<float*>(ws) : nullptr;
    const int st = p.row_tiles == 1   ? launch<1>(a, rot, p.shares, stream)
                   : p.row_tiles == 2 ? launch<2>(a, rot, p.shares, stream)
                   : p.row_tiles == 3 ? launch<3>(a, rot, p.shares, stream)
                                      : launch<4>(a, rot, p.shares, stream);
    if (shares) *shares = p.shares;
    if (st != PIE_HIP_OK || p.shares == 1 || shares) return st;
    return launch_shares_reduce(a, rot, p.shares, stream);
}

}  // namespace

int launch_gemm_groups(const GemmArgs& a, int group_size, void* ws, size_t ws_bytes, hipStream_t stream) {
    return run(a, Rotation{}, group_size, ws, ws_bytes, stream);
}
double gemm_groups_us(int M, int N, int K, int group_size, size_t ws_bytes) {
    return fits(M, N, K, group_size) ? plan_of(M, N, K, ws_bytes, false).us : 1e30;
}

}  // namespace pie_hip

extern "C" float pie_hip_gemm_groups_us(int M, int N, int K, int group_size, size_t workspace_bytes) {
    return static_cast<float>(pie_hip::gemm_groups_us(M, N, K, group_size, workspace_bytes));
}

extern "C" int pie_hip_gemm_groups_plan(int M, int N, int K, int group_size, size_t workspace_bytes, int norm, int* block_rows, int* shares) {
    using namespace pie_hip;
    if (!block_rows || !shares) return PIE_HIP_ERR_INVALID;
    const Plan p = fits(M, N, K, group_size) ? plan_of(M, N, K, workspace_bytes, norm != 0) : Plan{};
    if (p.row_tiles == 0) return PIE_HIP_ERR_UNSUPPORTED;
    *block_rows = p.row_tiles * 16;
    *shares = p.shares;
    return PIE_HIP_OK;
}

extern "C" float pie_hip_gemm_groups_shares_us(int M, int N, int K, int group_size, size_t workspace_bytes) {
    using namespace pie_hip;
    return static_cast<float>(fits(M, N, K, group_size) ? plan_of(M, N, K, workspace_bytes, true).us : 1e30);
}

extern "C" int pie_hip_gemm_groups_shares(const uint16_t* act_bf16, const void* weight, const void* scale, int group_size, int M, int N, int K,
                                          void* workspace, size_t workspace_bytes, int* shares, void* stream) {
    using namespace pie_hip;
    if (!act_bf16 || !weight || !scale || !workspace || !shares || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
    GemmArgs a{};
    a.act = act_bf16;
    a.w = static_cast<const unsigned char*>(weight);
    a.scale = static_cast<const unsigned char*>(scale);
    a.M = M;
    a.N = N;
    a.K = K;
    return run(a, Rotation{}, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream), shares);
}

extern "C" int pie_hip_gemm_groups_tiled(const uint16_t* act_bf16, const void* weight, const void* scale, int group_size, uint16_t* y_bf16,
                                         int M, int N, int K, int beta, int epilogue, const PieHipGlu* glu, void* workspace,
                                         size_t workspace_bytes, void* stream) {
    using namespace pie_hip;
    if (!glu_ok(glu, epilogue)) return PIE_HIP_ERR_INVALID;
    if (!act_bf16 || !weight || !scale || !y_bf16 || M <= 0 || N <= 0 || K <= 0) return PIE_HIP_ERR_INVALID;
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
    return launch_gemm_groups(a, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}

extern "C" int pie_hip_qkv_rope_groups_tiled(const uint16_t* act_bf16, const void* weight, const void* scale, int group_size, int M, int K,
                                             const float* rope_table, const int64_t* kv_slots, uint16_t* q_out, uint16_t* k_pages,
                                             uint16_t* v_pages, int num_q_heads, int num_kv_heads, int head_dim, int pairing,
                                             void* workspace, size_t workspace_bytes, void* stream) {
    using namespace pie_hip;
    if (!act_bf16 || !weight || !scale || !rope_table || !kv_slots || !q_out || !k_pages || !v_pages || M <= 0 || K <= 0 || num_q_heads <= 0 ||
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
    Rotation r;
    r.table = rope_table;
    r.slots = kv_slots;
    r.k_pages = k_pages;
    r.v_pages = v_pages;
    r.hq = num_q_heads;
    r.hk = num_kv_heads;
    r.d = head_dim;
    r.half_out = pairing == PIE_HIP_ROPE_HALF_PAIRED_ROWS;
    return run(a, r, group_size, workspace, workspace_bytes, static_cast<hipStream_t>(stream));
}
