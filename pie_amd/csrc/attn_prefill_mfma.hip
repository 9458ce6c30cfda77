// Prefill attention over paged KV on the matrix cores (gfx950, v_mfma_f32_16x16x32_bf16).
//
//   o[row, h, :] = softmax_j( q[row, h, :] . K[j, kvh, :] * scale ) . V[j, kvh, :],  j < row_kv_len[row]
// for tiles of consecutive query rows that share one page list (the tokens of one prefill
// chunk): same result contract as pie_hip_attn_rows_paged, i.e. the causal prefill branch of
// the reference's paged kernel (driver/cuda/src/ops/attention_naive_paged.cu:148-317) and of
// build_request_flash_attn (driver/portable/src/graph_common.cpp:347-396).
//
// One block (4 waves) = one tile x one kv head = 128 (token, q head) rows, 32 per wave as two
// 16-row MFMA tiles.  Keys advance 32 at a time:
//   S^T[key, query]  = K . Q^T     A = K fragment from LDS (row = key, k = d),  B = Q fragment kept
//                                  in registers (col = query, k = d)
//   O^T[d, query]   += V^T . P^T   A = V^T fragment from LDS (row = d, k = key), B = P in registers
// Both products put the query on the lane%16 axis, so the online-softmax state (max, sum,
// rescale) is per lane and the probabilities leave the first product already in the register
// layout the second one consumes — with the 32 keys of a step in the order
// [4g..4g+3, 16+4g..16+4g+3] per 16-lane group g, which is the order V^T is laid out in LDS.
// The next step's K/V are requested before the current step is multiplied: bf16 rows go straight into LDS as they are stored and V^T is read
// transposed, one-byte rows are decoded on the way.  Probabilities enter the second product as a hi + lo pair of bf16 values
// (fp32 accumulators), and the normaliser sums the unrounded values.
#include "gemm_args.hip.h"

#include <cstddef>
#include <type_traits>

namespace pie_hip {
namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

constexpr int kTileWaves = 4;
constexpr int kTileThreads = kTileWaves * kWave;
constexpr int kStepKeys = 32;
constexpr int kBlockRows = 128;           // (token, head) rows per block

// LDS places, in elements.  An operand read takes 16 bytes per lane, and the lanes served together are 0 - 3, 12 - 15, 20 - 23 and
// 24 - 27 (and so on): quarters of two neighbouring granules' rows, which have to fall into 16 different granules of the
// banks.  K rows are padded by a granule, and rows 4 - 11 of 16 swap neighbouring granules.
template <int D>
__device__ __forceinline__ int k_at(int key, int c) { return key * (D + 8) + (c ^ ((key + 4) >> 3 & 1)) * 8; }
// V^T rows are 64 bytes whose four granules change places by (row / 4) % 4 -> 0, 2, 3, 1; every 16 rows are padded by one, so that
// the rows that neighbouring threads write differ too.
__device__ __forceinline__ int vt_at(int row, int slot) {
    const int r = row >> 2;
    return row * kStepKeys + (row >> 4) * 8 + ((((slot >> 3) ^ (r & 1) << 1 ^ (r & 2) ^ (r & 2) >> 1) & 3) << 3 | (slot & 7));
}

// two buffers: a step's tiles are written while the previous step's are read, one barrier per step
template <int D, bool Q8>
struct TileLds {
    alignas(16) uint16_t ks[2][kStepKeys * (D + 8)];
    alignas(16) uint16_t vt[2][D * kStepKeys + D / 16 * 8];
    alignas(16) float sc[2][Q8 ? 2 * kStepKeys : 4];   // K | V scales of a step
};
// bf16 pools: a step's rows as they are stored, moved without registers.  A transfer of a wave fills 1 KiB in the order of its lanes (4 rows of 128 values, 8 of 64),
// so rows have no padding; a row's 16-byte pieces change places instead, K's by the row (the sixteen rows an operand read takes find
// different banks), V's in pairs by the row (the eight rows of 32 bytes that half a wave's transposing read takes).
constexpr int kRawStages = 2;
template <int D>
struct RawLds {
    alignas(256) uint16_t k[kRawStages][kStepKeys * D];
    alignas(256) uint16_t v[kRawStages][kStepKeys * D];
};
template <int D>
__device__ __forceinline__ int raw_k(int key, int piece) { return piece ^ (key / (128 / D) & (D / 8 - 1)); }
template <int D>
__device__ __forceinline__ int raw_v(int key, int piece) { return piece ^ (key / (128 / D) & (D / 16 - 1)) << 1; }
// Four operands of V^T, rows 4 g .. and 16 + 4 g .. of the lane's group out of stored rows: two transposing reads each, `AT` and `HIGH` bytes behind their
// addresses.  (In one block with their wait: the compiler takes the builtin's read to depend on every transfer into LDS and waits for the next step's, too.)
template <int AT, int HIGH>
__device__ __forceinline__ void read_transposed(uint32_t a0, uint32_t a1, uint32_t a2, uint32_t a3, bf16x8_t* out) {
    u32x2_t r[8];
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8 offset:%12\n\t"
        "ds_read_b64_tr_b16 %1, %8 offset:%13\n\t"
        "ds_read_b64_tr_b16 %2, %9 offset:%12\n\t"
        "ds_read_b64_tr_b16 %3, %9 offset:%13\n\t"
        "ds_read_b64_tr_b16 %4, %10 offset:%12\n\t"
        "ds_read_b64_tr_b16 %5, %10 offset:%13\n\t"
        "ds_read_b64_tr_b16 %6, %11 offset:%12\n\t"
        "ds_read_b64_tr_b16 %7, %11 offset:%13\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
        : "v"(a0), "v"(a1), "v"(a2), "v"(a3), "n"(AT), "n"(HIGH)
        : "memory");
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = __builtin_bit_cast(bf16x8_t, u32x4_t{r[2 * i].x, r[2 * i].y, r[2 * i + 1].x, r[2 * i + 1].y});
}
template <int D, bool Q8>
constexpr size_t kTileBytes = Q8 ? sizeof(TileLds<D, Q8>) : sizeof(RawLds<D>);
// ... or a group's accumulators, maxima and sums at the end
template <int D, bool Q8>
constexpr size_t kGroupBytes = kTileBytes<D, Q8> > (D / 16 + 1) * kTileThreads * 16 ? kTileBytes<D, Q8> : (D / 16 + 1) * kTileThreads * 16;

// slot of key kappa (0..31) inside a V^T row
__device__ __forceinline__ int vt_slot(int kappa) {
    return kappa < 16 ? 8 * (kappa >> 2) + (kappa & 3) : 8 * ((kappa - 16) >> 2) + 4 + (kappa & 3);
}

// QT: 16-row MFMA tiles per wave (2: 128 rows per block, K/V fragments read once per two tiles;
// 1: 64 rows per block, twice the blocks for small batches).
// KVF: one-byte pools (the codes become bf16 — exactly — on the way into the LDS tiles, one
// 16-code piece per thread and matrix; the step's per-(token, kv head) scales sit in LDS and
// multiply the scores (K) and the probabilities (V): float(code) * scale as in the row kernels).
// KP: groups of four waves that take a tile's steps in turn and meet at the end (in LDS, in fp32).  A block alone on its
// CU is one wave per SIMD, which waits out every step's chain of products, exponentials and barrier: 1.25 us for 32 keys.
// Up to 512 blocks of one 16-row tile per wave run in two groups: 358 rows behind 300 keys (32 heads over 8 of 128, 184
// blocks) 25 -> 20 us, 128 behind 2000 67 -> 48, a prompt of 489 20.5 -> 17, of 1024 40 -> 34.  (Four groups: 20, 41, 18; at
// 128 registers they spill.)
// What bounds it: instructions.  A wave issues one in four to five cycles, and the 24 products of a step (384 cycles) cover those beside them in part only.  bf16
// rows used to pass through registers, where V was transposed by packing pairs, and each step took the maximum over a query's lanes and mostly
// rescaled the accumulators: 158 vector instructions a step, now about 80 (places found by scalars, see issue; kSlack).  us before / after, 32 heads over 8 of
// 128: 489 rows 16.0 / 12.9, 1024 34.5 / 24.4, 2048 86 / 67, 4096 278 / 207 (in 128-row tiles 270 / 199), 8192 978 / 737, 128 behind 2000 46 / 34; three
// prompts of 412 with 32 heads over 4 20.5 / 17.3; 2048 rows of 32 heads over 8 of 64 57 / 43.  (Page ids kept in the lanes, three stages, tiles dealt long and
// short in turn: the same.)
template <int D, int GQA, int QT, int KVF = kKvBf16, int KP = 1>
__global__ __launch_bounds__(kTileThreads* KP, 2) void attn_prefill_tile_kernel(
    const uint16_t* __restrict__ q, const void* __restrict__ k_pages_raw,
    const void* __restrict__ v_pages_raw, const float* __restrict__ k_scales,
    const float* __restrict__ v_scales, uint16_t* __restrict__ o,
    const uint32_t* __restrict__ page_indices, const uint32_t* __restrict__ row_begin,
    const int32_t* __restrict__ row_len, const int32_t* __restrict__ tile_start,
    const int32_t* __restrict__ tile_rows, int hq, int hk, int ps, float scale_log2e) {
    constexpr int TQ = 32 * QT * kTileWaves / (2 * GQA);   // query tokens per tile: 64 QT / GQA
    constexpr int KS = D / 32;             // k steps of the first product
    constexpr int DT = D / 16;             // d tiles of the second product
    constexpr int LPR = D / 8;             // 16-byte pieces per K/V row
    constexpr bool Q8 = KVF != kKvBf16;
    constexpr int LPRQ = D / 16;           // 16-code pieces per one-byte row
    static_assert(kStepKeys * LPRQ <= kTileThreads, "one-byte pieces fit one per thread");
    const unsigned char* k_bytes = static_cast<const unsigned char*>(k_pages_raw);
    const unsigned char* v_bytes = static_cast<const unsigned char*>(v_pages_raw);
    // two LDS buffers: a step's tiles are written while the previous step's are read, one
    // barrier per step
    static_assert(KP == 1 || QT == 1, "the groups' results meet in the tiles' place");
    using L = TileLds<D, Q8>;
    extern __shared__ __align__(16) unsigned char smem[];

    // Blocks start in the order of their linear index: tile-major, the kv heads of a tile side by
    // side.  A caller that lists its tiles longest first therefore gets the long causal tiles
    // started first and the short ones handed to the slots that free up — the longest-first rule,
    // which for a causal prompt of more tiles than slots comes within a step of an even split
    // (measured, 32 q / 8 kv heads of 128: 3072 tokens 242 -> 169 us, 4096 tokens 355 -> 278, 8192
    // tokens 1072 -> 934).
    const int lin = blockIdx.y * gridDim.x + blockIdx.x;
    const int tile = lin / hk;
    const int kvh = lin - tile * hk;
    const int part = KP == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kTileThreads);
    const int tid = threadIdx.x & (kTileThreads - 1), lane = tid & (kWave - 1), wv = tid / kWave;
    const int l16 = lane & 15, g = lane >> 4;
    const int s0 = tile_start[tile], n_rows = tile_rows[tile];
    const uint32_t pg_lo = row_begin[s0];
    L& lds = *reinterpret_cast<L*>(smem + part * kGroupBytes<D, Q8>);
    RawLds<D>& raw = *reinterpret_cast<RawLds<D>*>(smem + part * kGroupBytes<D, Q8>);

    // (every wave finds the longest extent for itself: no barrier between the loads that lead to the first keys)
    int longest = row_len[s0 + min(lane, max(n_rows, 1) - 1)];
    if constexpr (TQ > kWave) longest = max(longest, row_len[s0 + min(lane + kWave, max(n_rows, 1) - 1)]);
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) longest = max(longest, __shfl_xor(longest, sh, kWave));
    const int kmax = max(0, __builtin_amdgcn_readfirstlane(longest));
    // this lane's two query rows (one per 16-row tile of the wave)
    int my_len[QT];
    bf16x8_t qf[QT][KS];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        const int m = wv * 16 * QT + qt * 16 + l16;
        const int h = m / TQ, t = m % TQ;
        const bool valid = t < n_rows;
        const int row = s0 + (valid ? t : 0);
        my_len[qt] = valid ? row_len[row] : 0;
        const uint16_t* qp = q + (static_cast<size_t>(row) * hq + kvh * GQA + h) * D + 8 * g;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            u32x4_t v = *reinterpret_cast<const u32x4_t*>(qp + 32 * ks);
            if (!valid) v = u32x4_t{0u, 0u, 0u, 0u};
            qf[qt][ks] = __builtin_bit_cast(bf16x8_t, v);
        }
    }

    // the shortest causal extent among this wave's rows: steps below it need no masking
    int min_len_v = my_len[0];
#pragma unroll
    for (int qt = 1; qt < QT; ++qt) min_len_v = min(min_len_v, my_len[qt]);
#pragma unroll
    for (int sh = 1; sh < kWave; sh <<= 1) min_len_v = min(min_len_v, __shfl_xor(min_len_v, sh, kWave));
    const int min_len = __builtin_amdgcn_readfirstlane(min_len_v);

    constexpr int PF = 2;   // one-byte pools: steps of K/V in flight
    // from a group's step to its next: up to four steps the first group takes all (the meeting costs what sharing them saves, 128
    // keys 8.1 us alone and 8.3 shared)
    const bool shared = KP > 1 && kmax > 4 * kStepKeys;
    const int advance = shared ? kStepKeys * KP : kStepKeys;
    u32x4_t kreg[PF], vreg[PF];
    float sreg[PF];   // one-byte pools: thread t < 32 holds the K scale of key t, t < 64 V's
    // one-byte pools: thread -> (key, 16-code piece); threads past the tile idle (neighbouring threads take neighbouring pieces of a row: with
    // neighbouring keys a wave's load touched 16 rows' lines for 64 bytes each, which kept the address unit busy for longer than the products took)
    const int own_key = tid / LPRQ, own_piece = tid % LPRQ;
    // bf16 pools: a wave's transfer u moves keys own_first + u * 16 .., a lane the piece that belongs where it lands
    constexpr int MOVES = kStepKeys * LPR / kTileThreads, MKEYS = kWave / LPR;   // transfers per wave and matrix; keys of one
    const int wave = __builtin_amdgcn_readfirstlane(wv), raw_key = wave * MKEYS + lane / LPR;
    const uint32_t row_bytes = static_cast<uint32_t>(hk) * D * 2;
    uint32_t k_off = (raw_key & 15) * row_bytes + raw_k<D>(raw_key, lane % LPR) * 16, v_off = (raw_key & 15) * row_bytes + raw_v<D>(raw_key, lane % LPR) * 16;
    const int ps_shift = (ps & (ps - 1)) == 0 ? __builtin_ctz(static_cast<unsigned>(ps)) : -1;
    const uint32_t page_bytes = static_cast<uint32_t>(ps) * row_bytes;
    const bool aligned = (reinterpret_cast<uintptr_t>(k_bytes) | reinterpret_cast<uintptr_t>(v_bytes)) % 16 == 0;
    const unsigned char *k_head = k_bytes + kvh * (D * 2), *v_head = v_bytes + kvh * (D * 2);
    // a 32-key step touches at most two pages (page_size % 16 == 0): their ids come through
    // scalar loads, so the vector-memory queue holds K/V loads only, in step order
    auto issue = [&](int slot, int j0) {
        const int ja = min(j0, kmax - 1), jb = min(j0 + kStepKeys - 1, kmax - 1);
        // (the step's first page by one scalar division; a key is in it or in the next one — no
        // division per lane, which was a fifth of the step's instructions)
        const int page_a = ps_shift >= 0 ? ja >> ps_shift : ja / ps;
        const int pa_end = (page_a + 1) * ps;
        const uint32_t pid_a = __builtin_amdgcn_readfirstlane(page_indices[pg_lo + page_a]);
        const uint32_t pid_b = __builtin_amdgcn_readfirstlane(page_indices[pg_lo + page_a + (jb >= pa_end ? 1 : 0)]);
        auto token_head = [&](int key) {
            const int j = min(j0 + key, kmax - 1);
            const bool in_a = j < pa_end;
            return (static_cast<size_t>(in_a ? pid_a : pid_b) * ps + (j - (in_a ? pa_end - ps : pa_end))) * hk + kvh;
        };
        auto token_sc = [&](int key) {   // the key's place in a scale pool
            const int j = min(j0 + key, kmax - 1);
            const bool in_a = j < pa_end;
            return kv_scale_index(in_a ? pid_a : pid_b, j - (in_a ? pa_end - ps : pa_end), kvh, hk, ps);
        };
        if constexpr (Q8) {
            if (own_key < kStepKeys) {
                const size_t off = token_head(own_key) * D + own_piece * 16;
                kreg[slot] = *reinterpret_cast<const u32x4_t*>(k_bytes + off);
                vreg[slot] = *reinterpret_cast<const u32x4_t*>(v_bytes + off);
            }
            if (tid < 2 * kStepKeys) {
                const float* sp = tid < kStepKeys ? k_scales : v_scales;
                sreg[slot] = sp ? sp[token_sc(tid % kStepKeys)] : 1.f;
            }
        } else {
            u32x4_t* kl = reinterpret_cast<u32x4_t*>(raw.k[slot]) + wave * kWave;
            u32x4_t* vl = reinterpret_cast<u32x4_t*>(raw.v[slot]) + wave * kWave;
            auto move_all = [&](auto direct) __attribute__((always_inline)) {
                auto move = [&](const unsigned char* from, u32x4_t* to) __attribute__((always_inline)) {
                    if constexpr (decltype(direct)::value) to_lds(from, to);
                    else to[lane] = *reinterpret_cast<const u32x4_t*>(from);
                };
                if (j0 + kStepKeys <= kmax) {
                    // a whole step: sixteen keys are in one page, and scalars find where; a lane adds its own offset
                    asm volatile("" : "+v"(k_off), "+v"(v_off));   // (32-bit offsets from scalar bases, not 64-bit sums)
#pragma unroll
                    for (int u = 0; u < MOVES; ++u) {
                        const int key = D == 128 ? 16 * u : wave * MKEYS / 16 * 16;   // 0 or 16
                        const bool in_b = key && pa_end - j0 == 16;
                        const size_t at = static_cast<uint64_t>(in_b ? pid_b : pid_a) * page_bytes + (in_b ? 0u : static_cast<uint32_t>(j0 + key - pa_end + ps) * row_bytes);
                        move(k_head + at + k_off, kl + u * kTileThreads);
                        move(v_head + at + v_off, vl + u * kTileThreads);
                    }
                } else {
#pragma unroll
                    for (int u = 0; u < MOVES; ++u) {
                        const int key = u * (kTileWaves * MKEYS) + raw_key;
                        const size_t at = token_head(key) * (D * 2);
                        move(k_bytes + at + raw_k<D>(key, lane % LPR) * 16, kl + u * kTileThreads);
                        move(v_bytes + at + raw_v<D>(key, lane % LPR) * 16, vl + u * kTileThreads);
                    }
                }
            };
            // (pools off a 16-byte boundary pass through registers)
            if (aligned) move_all(std::true_type{});
            else move_all(std::false_type{});
        }
    };
    auto stage = [&](int slot) {   // one-byte pools: register slot = LDS buffer
        if constexpr (Q8) {
            uint16_t* Ks = lds.ks[slot];
            uint16_t* Vt = lds.vt[slot];
            float* s_sc = lds.sc[slot];
            if (own_key < kStepKeys) {
                const u32x4_t kw = kreg[slot], vw = vreg[slot];
                *reinterpret_cast<u32x4_t*>(&Ks[k_at<D>(own_key, 2 * own_piece)]) = kv_decode_bf16<KVF>(u32x2_t{kw.x, kw.y});
                *reinterpret_cast<u32x4_t*>(&Ks[k_at<D>(own_key, 2 * own_piece + 1)]) = kv_decode_bf16<KVF>(u32x2_t{kw.z, kw.w});
                const int col = vt_slot(own_key);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    float f[8];
                    kv_decode_f32<KVF>(u32x2_t{vw[2 * h], vw[2 * h + 1]}, f);
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        Vt[vt_at(own_piece * 16 + 8 * h + e, col)] = static_cast<uint16_t>(__float_as_uint(f[e]) >> 16);
                }
            }
            if (tid < 2 * kStepKeys) s_sc[tid] = sreg[slot];
        }
    };

    f32x4_t acc[QT][DT];
    constexpr float kSlack = 8.f;
    float mx[QT], limit[QT], off[QT], lsum[QT];
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        mx[qt] = limit[qt] = -INFINITY;
        off[qt] = 0.f;
        lsum[qt] = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) acc[qt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    }

    // bf16 pools: the lane's places in a stage, for K's step ks and V's tile dt the places with those bits of the piece flipped
    const int k_place = l16 * D + raw_k<D>(l16, g) * 8;
    const int v_row = 4 * g + (l16 >> 2), v_place = v_row * D + raw_v<D>(v_row, (l16 & 3) >> 1) * 8 + (l16 & 1) * 4;
    const uint32_t raw_at = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(PIE_LDS_PTR(&raw)));
    uint32_t v_at[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) v_at[dt] = raw_at + 2 * (v_place ^ dt * 16);
    // Step j reads buffer j % 2.  On entry its tiles are there and the block has met.  One-byte pools: the
    // step first stages step j + 1 from the other register slot into the other buffer (whose
    // readers passed the last barrier), then refills that slot with step j + 3.
    auto step = [&](auto slot_tag, int j0) {
        constexpr int slot = decltype(slot_tag)::value;
        const uint16_t* Ks = Q8 ? lds.ks[slot] : raw.k[slot];
        const uint16_t* Vt = Q8 ? lds.vt[slot] : raw.v[slot];
        const float* s_sc = lds.sc[slot];
        if constexpr (Q8) {
            if (j0 + advance < kmax) stage(slot ^ 1);
            if (j0 + 3 * advance < kmax) issue(slot ^ 1, j0 + 3 * advance);   // (slot ^ 1 held step j + 1)
        }
        // (one-byte pools) the scales of this lane's keys 16nt + 4g + r
        f32x4_t ksc[2], vsc[2];
        if constexpr (Q8) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                ksc[nt] = *reinterpret_cast<const f32x4_t*>(&s_sc[16 * nt + 4 * g]);
                vsc[nt] = *reinterpret_cast<const f32x4_t*>(&s_sc[kStepKeys + 16 * nt + 4 * g]);
            }
        }
        // S^T = K . Q^T for both query tiles
        f32x4_t st[QT][2];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) st[qt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                const bf16x8_t kf = __builtin_bit_cast(
                    bf16x8_t, *reinterpret_cast<const u32x4_t*>(&Ks[Q8 ? k_at<D>(16 * nt + l16, 4 * ks + g) : (k_place ^ ks * 32) + 16 * nt * D]));
#pragma unroll
                for (int qt = 0; qt < QT; ++qt)
                    st[qt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf, qf[qt][ks], st[qt][nt], 0, 0, 0);
            }
        }
        // bf16 pools: V^T out of the stored rows, four tiles at a time, the first beside the products above
        [[maybe_unused]] bf16x8_t vraw[4];
        auto v_read = [&](auto first_tag) {
            constexpr int d0 = decltype(first_tag)::value, at = offsetof(RawLds<D>, v) + slot * sizeof(raw.v[0]);
            read_transposed<at, at + 16 * D * 2>(v_at[d0], v_at[d0 + 1], v_at[d0 + 2], v_at[d0 + 3], vraw);
        };
        if constexpr (!Q8) v_read(std::integral_constant<int, 0>{});
        // online softmax per query (= per lane%16); the 8 keys of this lane: 16nt + 4g + r.
        // bf16 pools keep a maximum in raw score units and fold the softmax scale into
        // the exponent's fma; steps wholly inside every row's causal extent skip the masking
        // (a wave-uniform branch); exponentials are the bare v_exp_f32 (arguments <= kSlack).
        bf16x8_t pf_hi[QT], pf_lo[QT];
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
            for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if constexpr (Q8) st[qt][nt][r] *= scale_log2e * ksc[nt][r];
        if (j0 + kStepKeys > min_len) {
#pragma unroll
            for (int qt = 0; qt < QT; ++qt)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int r = 0; r < 4; ++r) st[qt][nt][r] = j0 + 16 * nt + 4 * g + r < my_len[qt] ? st[qt][nt][r] : -INFINITY;
        }
        const float c = Q8 ? 1.f : scale_log2e;   // (one-byte pools: already in the scores)
        // What the exponents are relative to moves only when a score is 2^kSlack over it: weights up to that are as exact in
        // floating point, and most steps need neither the maximum over the lanes of a query nor the accumulators' rescale.
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            float top = st[qt][0][0];
#pragma unroll
            for (int e = 1; e < 8; ++e) top = fmaxf(top, st[qt][e >> 2][e & 3]);
            if (__any(top > limit[qt])) {
                const float m_new = rows_max(fmaxf(mx[qt], top));
                off[qt] = m_new == -INFINITY ? 0.f : -m_new * c;
                const float alpha = __builtin_amdgcn_exp2f(fmaf(mx[qt], c, off[qt]));
                mx[qt] = m_new;
                limit[qt] = m_new + kSlack / c;
                lsum[qt] *= alpha;
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) acc[qt][dt] *= alpha;
            }
        }
#pragma unroll
        for (int qt = 0; qt < QT; ++qt) {
            // The weights reach the second product as hi + lo with both parts bf16 (hi by
            // truncation, lo = bf16(p - hi)): 16 significant bits, so P . V keeps the accuracy
            // of fp32 weights (the reference multiplies fp32 probabilities,
            // driver/cuda/src/ops/attention_naive_paged.cu:148-317), and the normaliser sums
            // the unrounded values, as the decode kernel does.
            float sum = 0.f;
            uint32_t hi[4], lo[4];
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                float p0 = __builtin_amdgcn_exp2f(fmaf(st[qt][e >> 2][e & 3], c, off[qt]));
                float p1 = __builtin_amdgcn_exp2f(fmaf(st[qt][e >> 2][(e & 3) + 1], c, off[qt]));
                sum += p0 + p1;
                if constexpr (Q8) {   // V = float(code) * scale: the scale rides on the weight
                    p0 *= vsc[e >> 2][e & 3];
                    p1 *= vsc[e >> 2][(e & 3) + 1];
                }
                const uint32_t u0 = __float_as_uint(p0), u1 = __float_as_uint(p1);
                hi[e >> 1] = __builtin_amdgcn_perm(u1, u0, 0x07060302u);
                lo[e >> 1] = pack_bf16x2(p0 - __uint_as_float(u0 & 0xFFFF0000u),
                                         p1 - __uint_as_float(u1 & 0xFFFF0000u));
            }
            pf_hi[qt] = __builtin_bit_cast(bf16x8_t, u32x4_t{hi[0], hi[1], hi[2], hi[3]});
            pf_lo[qt] = __builtin_bit_cast(bf16x8_t, u32x4_t{lo[0], lo[1], lo[2], lo[3]});
            lsum[qt] += sum;
        }
        // O^T += V^T . P^T
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            bf16x8_t vf;
            if constexpr (Q8) {
                vf = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const u32x4_t*>(&Vt[vt_at(16 * dt + l16, 8 * g)]));
            } else {
                if constexpr (DT > 4)
                    if (dt == 4) v_read(std::integral_constant<int, DT - 4>{});
                vf = vraw[dt & 3];
            }
#pragma unroll
            for (int qt = 0; qt < QT; ++qt) {
                acc[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf_hi[qt], acc[qt][dt], 0, 0, 0);
                acc[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf_lo[qt], acc[qt][dt], 0, 0, 0);
            }
        }
    };

    const int first = KP == 1 || shared || part == 0 ? part * kStepKeys : kmax;
    if constexpr (Q8) {
        if (first < kmax) issue(0, first);
        if (first + advance < kmax) issue(1, first + advance);
        if (first < kmax) stage(0);
        if (first + 2 * advance < kmax) issue(0, first + 2 * advance);
        __syncthreads();
        for (int j0 = 0; j0 < kmax; j0 += PF * advance) {   // unrolled by PF: compile-time register slots
            if (KP == 1 || first + j0 < kmax) step(std::integral_constant<int, 0>{}, first + j0);
            __syncthreads();   // step j + 1 is staged, step j read
            if (j0 + advance < kmax) {
                if (KP == 1 || first + j0 + advance < kmax) step(std::integral_constant<int, 1>{}, first + j0 + advance);
                __syncthreads();
            }
        }
    } else {
        // one barrier a step: behind it everybody's transfers of the step have landed and the stage of the step before is free
        if (first < kmax) issue(0, first);
        auto turn = [&](auto slot_tag, int j0) {
            constexpr int slot = decltype(slot_tag)::value;
            __builtin_amdgcn_s_waitcnt(0x0070);   // (LDS writes too: pools off a 16-byte boundary)
            PIE_MEET();
            if (first + j0 + advance < kmax) issue(slot ^ 1, first + j0 + advance);
            if (KP == 1 || first + j0 < kmax) step(slot_tag, first + j0);
        };
        for (int j0 = 0; j0 < kmax; j0 += 2 * advance) {
            turn(std::integral_constant<int, 0>{}, j0);
            if (j0 + advance < kmax) turn(std::integral_constant<int, 1>{}, j0 + advance);
        }
        __syncthreads();
    }
    if constexpr (KP > 1) {
        // the other groups' accumulators, maxima and sums in their tiles' place; the first group adds them up
        if (!shared && part > 0) return;
        if (part > 0) {
            f32x4_t* mine = reinterpret_cast<f32x4_t*>(&lds);
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) mine[dt * kTileThreads + tid] = acc[0][dt];
            mine[DT * kTileThreads + tid] = f32x4_t{mx[0], lsum[0], 0.f, 0.f};
        }
        if (shared) __syncthreads();
        if (part > 0) return;
        const float c = Q8 ? 1.f : scale_log2e;
#pragma unroll
        for (int other = 1; other < KP && shared; ++other) {
            const f32x4_t* its = reinterpret_cast<const f32x4_t*>(smem + other * kGroupBytes<D, Q8>);
            const f32x4_t st = its[DT * kTileThreads + tid];
            const float m_new = fmaxf(mx[0], st[0]), safe = m_new == -INFINITY ? 0.f : m_new;
            const float wa = __builtin_amdgcn_exp2f((mx[0] - safe) * c), wb = __builtin_amdgcn_exp2f((st[0] - safe) * c);
            mx[0] = m_new;
            lsum[0] = lsum[0] * wa + st[1] * wb;
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[0][dt] = acc[0][dt] * wa + its[dt * kTileThreads + tid] * wb;
        }
    }

    // normalise and store: this lane holds, for its query, d = 16 dt + 4 g + r
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
        float l = lsum[qt];
        l += __shfl_xor(l, 16, kWave);
        l += __shfl_xor(l, 32, kWave);
        const int m = wv * 16 * QT + qt * 16 + l16;
        if (m % TQ >= n_rows) continue;
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        uint16_t* op = o + (static_cast<size_t>(s0 + m % TQ) * hq + kvh * GQA + m / TQ) * D + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
            const f32x4_t a = acc[qt][dt];
            const u32x2_t w = {pack_bf16x2(a[0] * inv, a[1] * inv), pack_bf16x2(a[2] * inv, a[3] * inv)};
            *reinterpret_cast<u32x2_t*>(op + 16 * dt) = w;
        }
    }
}

template <int D, int GQA, int QT>
int launch_tiles(int kv_format, const uint16_t* q, const void* k_pages, const void* v_pages,
                 const float* k_scales, const float* v_scales, uint16_t* o,
                 const uint32_t* page_indices, const uint32_t* row_begin, const int32_t* row_len,
                 const int32_t* tile_start, const int32_t* tile_rows, int num_tiles, int hq, int hk,
                 int ps, float scale, hipStream_t stream) {
    const float sl = scale * 1.4426950408889634f;
    auto run = [&](auto format, auto groups) {
        constexpr int KVF = decltype(format)::value, KP = decltype(groups)::value;
        constexpr size_t smem = KP * kGroupBytes<D, KVF != kKvBf16>;
        static const hipError_t attr = hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_prefill_tile_kernel<D, GQA, QT, KVF, KP>),
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(smem));
        if (attr != hipSuccess) return PIE_HIP_ERR_LAUNCH;
        hipLaunchKernelGGL((attn_prefill_tile_kernel<D, GQA, QT, KVF, KP>), dim3(num_tiles, hk), dim3(kTileThreads * KP), smem, stream, q,
                           k_pages, v_pages, k_scales, v_scales, o, page_indices, row_begin, row_len, tile_start, tile_rows, hq, hk, ps, sl);
        return launch_status();
    };
    auto grouped = [&](auto format) {
        if constexpr (QT == 1) {
            const long long blocks = static_cast<long long>(num_tiles) * hk;
            if (blocks <= 512) return run(format, std::integral_constant<int, 2>{});
        }
        return run(format, std::integral_constant<int, 1>{});
    };
    if (kv_format == PIE_HIP_KV_BF16) return grouped(std::integral_constant<int, kKvBf16>{});
    if (kv_format == PIE_HIP_KV_INT8_PER_TOKEN_HEAD) return grouped(std::integral_constant<int, kKvInt8>{});
    if (kv_format == PIE_HIP_KV_FP8_E5M2) return grouped(std::integral_constant<int, kKvBf8>{});
    return grouped(std::integral_constant<int, kKvFp8>{});
}

}  // namespace
}  // namespace pie_hip

extern "C" int pie_hip_attn_prefill_tile_rows(int num_q_heads, int num_kv_heads) {
    if (num_q_heads <= 0 || num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0) return 0;
    const int gqa = num_q_heads / num_kv_heads;
    if (gqa != 1 && gqa != 2 && gqa != 4 && gqa != 8) return 0;
    return pie_hip::kBlockRows / gqa;
}

extern "C" int pie_hip_attn_prefill_tiles_kvq(int kv_format, const uint16_t* q, const void* k_pages,
                                              const void* v_pages, const float* k_scales,
                                              const float* v_scales, uint16_t* o,
                                              const uint32_t* kv_page_indices,
                                              const uint32_t* row_page_begin, const int32_t* row_kv_len,
                                              const int32_t* tile_row_start, const int32_t* tile_num_rows,
                                              int num_tiles, int rows_per_tile, int num_q_heads,
                                              int num_kv_heads, int head_dim, int page_size,
                                              float sm_scale, void* stream) {
    using namespace pie_hip;
    if (!q || !k_pages || !v_pages || !o || !kv_page_indices || !row_page_begin || !row_kv_len ||
        !tile_row_start || !tile_num_rows || num_tiles <= 0 || page_size <= 0)
        return PIE_HIP_ERR_INVALID;
    {
        const bool scaled = kv_format == PIE_HIP_KV_INT8_PER_TOKEN_HEAD || kv_format == PIE_HIP_KV_FP8_PER_TOKEN_HEAD;
        if (kv_format != PIE_HIP_KV_BF16 && kv_format != PIE_HIP_KV_FP8_E4M3 && kv_format != PIE_HIP_KV_FP8_E5M2 && !scaled)
            return PIE_HIP_ERR_UNSUPPORTED;
        if (scaled != (k_scales != nullptr) || scaled != (v_scales != nullptr)) return PIE_HIP_ERR_INVALID;
    }
    const int cap = pie_hip_attn_prefill_tile_rows(num_q_heads, num_kv_heads);
    if (cap == 0 || page_size % 16 != 0 || num_tiles > 0x7FFFFFFF / 2 || num_kv_heads > 65535)
        return PIE_HIP_ERR_UNSUPPORTED;
    if (rows_per_tile != cap && rows_per_tile * 2 != cap) return PIE_HIP_ERR_UNSUPPORTED;
    const bool big = rows_per_tile == cap;
    const float scale = sm_scale > 0.f ? sm_scale : 1.0f / sqrtf(static_cast<float>(head_dim));
    const int gqa = num_q_heads / num_kv_heads;
    hipStream_t st = static_cast<hipStream_t>(stream);
#define PIE_TILE_CASE(DD, GG)                                                                       \
    if (head_dim == DD && gqa == GG)                                                                \
        return big ? launch_tiles<DD, GG, 2>(kv_format, q, k_pages, v_pages, k_scales, v_scales, o, \
                                             kv_page_indices, row_page_begin, row_kv_len,           \
                                             tile_row_start, tile_num_rows, num_tiles, num_q_heads, \
                                             num_kv_heads, page_size, scale, st)                    \
                   : launch_tiles<DD, GG, 1>(kv_format, q, k_pages, v_pages, k_scales, v_scales, o, \
                                             kv_page_indices, row_page_begin, row_kv_len,           \
                                             tile_row_start, tile_num_rows, num_tiles, num_q_heads, \
                                             num_kv_heads, page_size, scale, st);
    PIE_TILE_CASE(128, 1)
    PIE_TILE_CASE(128, 2)
    PIE_TILE_CASE(128, 4)
    PIE_TILE_CASE(128, 8)
    PIE_TILE_CASE(64, 1)
    PIE_TILE_CASE(64, 2)
    PIE_TILE_CASE(64, 4)
    PIE_TILE_CASE(64, 8)
#undef PIE_TILE_CASE
    return PIE_HIP_ERR_UNSUPPORTED;
}

extern "C" int pie_hip_attn_prefill_tiles(const uint16_t* q, const uint16_t* k_pages,
                                          const uint16_t* v_pages, uint16_t* o,
                                          const uint32_t* kv_page_indices,
                                          const uint32_t* row_page_begin, const int32_t* row_kv_len,
                                          const int32_t* tile_row_start, const int32_t* tile_num_rows,
                                          int num_tiles, int rows_per_tile, int num_q_heads,
                                          int num_kv_heads, int head_dim, int page_size,
                                          float sm_scale, void* stream) {
    return pie_hip_attn_prefill_tiles_kvq(PIE_HIP_KV_BF16, q, k_pages, v_pages, nullptr, nullptr, o,
                                          kv_page_indices, row_page_begin, row_kv_len, tile_row_start,
                                          tile_num_rows, num_tiles, rows_per_tile, num_q_heads,
                                          num_kv_heads, head_dim, page_size, sm_scale, stream);
}
