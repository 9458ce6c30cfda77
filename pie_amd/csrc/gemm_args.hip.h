// What the tiled GEMMs of large batches share: their arguments, and the launch of the wide form.
#pragma once

#include <type_traits>

#include "common.hip.h"

namespace pie_hip {

struct GemmArgs {
    const uint16_t* act;
    const unsigned char* w;
    const unsigned char* scale;
    uint16_t* y;
    int M, N, K, g_shift, beta, swiglu, scale_is_bf16;
    int pointwise;        // PIE_HIP_EPI_RELU2 and above: applied to the sum (0: nothing)
    PieHipGlu glu = kPlainGlu;   // swiglu
    float* partial;   // split-K: fp32 [gridDim.z][M][N] partial sums (row scale applied), else null
    // grouped: rows offsets[p] .. offsets[p + 1] of y belong to problem p (of `problems`), whose weights (scales)
    // start w_stride (scale_stride) bytes after the one before; act_rows: the activation row of each (null: the same row)
    const int32_t* offsets;
    const int32_t* act_rows;
    size_t w_stride, scale_stride;
    int problems, tiled;
    int aligned;   // wide form: y starts at a multiple of 8 bytes
    int lines;     // whole tile pairs, y on 16 bytes: see store_pair
};

#define PIE_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))
// s_waitcnt lgkmcnt(0) alone and vmcnt(n) alone, n < 64 (gfx9 encoding).  The no-op keeps the compiler's own wait for a
// value loaded before from being merged into this one: merged, it counts transfers into LDS as unordered and waits for all.
#define PIE_WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(0xC07F)
#define PIE_WAIT_VM(n)                              \
    do {                                            \
        __builtin_amdgcn_sched_barrier(0);          \
        __builtin_amdgcn_s_waitcnt(0x0F70 | ((n) & 15) | (((n) >> 4) << 14)); \
        asm volatile("s_nop 0");                    \
        __builtin_amdgcn_sched_barrier(0);          \
    } while (0)

#define PIE_FENCE() __builtin_amdgcn_sched_barrier(0)
#define PIE_MEET()                         \
    do {                                   \
        PIE_FENCE();                       \
        asm volatile("" ::: "memory");     \
        __builtin_amdgcn_s_barrier();      \
        asm volatile("" ::: "memory");     \
        PIE_FENCE();                       \
    } while (0)

__device__ __forceinline__ void to_lds(const unsigned char* from, u32x4_t* to) {
    __builtin_amdgcn_global_load_lds(from, PIE_LDS_PTR(to), 16, 0, 0);
}

// What a launch's rows become, so that a block asks once and not every store: gated pairs by the plain rule, by another, values as they are, onto a
// residual; Any asks for itself (the pointwise functions).  With the questions in every unrolled store a block of 256 x 256 had 23000 instructions in 1900 basic
// blocks, most of them run once and fetched for it.  256
// such blocks with K of 1024, before / here: fp8 as they are 51.3 / 46.3 us, gated 50.8 / 48.3, int4 51.1 / 47.7 and 51.0 / 47.9; bf16, 128 columns, 25.7 / 24.1 and 25.2 / 24.4.
// (Gated stores are bound by their instructions: 133 per four values before, 117 - 143 here.)
enum class Out { Gated, GatedRule, Plain, Residual, Any };
template <class Fn>
__device__ __forceinline__ void by_output(const GemmArgs& a, Fn&& store) {
    if (a.swiglu) {
        if (!a.glu.bias && a.glu.limit == __builtin_inff() && a.glu.alpha == 1.f && a.glu.shift == 0.f) store(std::integral_constant<Out, Out::Gated>{});
        else store(std::integral_constant<Out, Out::GatedRule>{});
    } else if (a.pointwise) {
        store(std::integral_constant<Out, Out::Any>{});
    } else if (a.beta) {
        store(std::integral_constant<Out, Out::Residual>{});
    } else {
        store(std::integral_constant<Out, Out::Plain>{});
    }
}
template <Out O>
__device__ __forceinline__ bool is_gated(const GemmArgs& a) { return O == Out::Any ? a.swiglu != 0 : O == Out::Gated || O == Out::GatedRule; }
template <Out O>
__device__ __forceinline__ bool is_residual(const GemmArgs& a) { return O == Out::Any ? a.beta != 0 : O == Out::Residual; }
// (the plain rule's limit is opaque: knowing it, the compiler folds the clamp of u into one that makes a NaN plus infinity, not minus)
template <Out O>
__device__ __forceinline__ PieHipGlu rule_of(const GemmArgs& a) {
    if constexpr (O != Out::Gated) return a.glu;
    float limit = a.glu.limit;
    asm volatile("" : "+s"(limit));
    return PieHipGlu{nullptr, limit, 1.f, 0.f};
}

// The epilogue of row m, columns n .. n + 3 (those below N; n is a multiple of 4): SwiGLU over (gate, up) pairs rounded to
// bf16 first, or a pointwise function and the residual.
template <Out O = Out::Any>
__device__ __forceinline__ void wide_store(const GemmArgs& a, int m, int n, float* v) {
    const int N = a.N, nout = is_gated<O>(a) ? N / 2 : N;
    const bool whole = N % 4 == 0 && a.aligned;   // one 8- (SwiGLU: 4-) byte store
    if (is_gated<O>(a)) {
        const PieHipGlu rule = rule_of<O>(a);
        uint16_t o[2];
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            float g = v[2 * r], u = v[2 * r + 1];
            if (rule.bias) {
                g += rule.bias[min(n + 2 * r, N - 1)];
                u += rule.bias[min(n + 2 * r + 1, N - 1)];
            }
            g = round_bf16(g);
            u = round_bf16(u);
            o[r] = f32_to_bf16_bits(glu_value(g, u, rule));
        }
        uint16_t* p = a.y + static_cast<size_t>(m) * nout + n / 2;
        if (whole) {
            *reinterpret_cast<uint32_t*>(p) = o[0] | static_cast<uint32_t>(o[1]) << 16;
        } else {
            p[0] = o[0];
            if (n + 2 < N) p[1] = o[1];
        }
        return;
    }
    uint16_t* p = a.y + static_cast<size_t>(m) * nout + n;
    if constexpr (O == Out::Any) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = epilogue_pointwise<true>(v[r], a.pointwise);
    }
    if (whole) {
        if (is_residual<O>(a)) {
            const u32x2_t old = *reinterpret_cast<const u32x2_t*>(p);
            v[0] += bf16_lo(old.x);
            v[1] += bf16_hi(old.x);
            v[2] += bf16_lo(old.y);
            v[3] += bf16_hi(old.y);
        }
        *reinterpret_cast<u32x2_t*>(p) = u32x2_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
        for (int r = 0; r < 4 && n + r < N; ++r) {
            if (is_residual<O>(a)) v[r] += bf16_bits_to_f32(p[r]);
            p[r] = f32_to_bf16_bits(v[r]);
        }
    }
}

inline int stores_lines(const uint16_t* y, int N) { return N % 32 == 0 && reinterpret_cast<uintptr_t>(y) % 16 == 0; }
// Where store_pair's row m goes, q the lane's sixteenth of the wave; sixteen rows on it is `row_step` values further.
template <Out O>
__device__ __forceinline__ uint16_t* pair_place(const GemmArgs& a, int m, int n, int q, int& row_step) {
    const int nout = is_gated<O>(a) ? a.N / 2 : a.N, at = q & 1 ? n + 12 : n;
    row_step = 16 * nout;
    return a.y + static_cast<size_t>(m) * nout + (is_gated<O>(a) ? at / 2 : at);
}
// wide_store for columns n .. n + 3 and n + 16 .. n + 19, n = 32 k + 4 q (a.lines): neighbouring sixteenths swap half of their values, the even ones end with
// eight columns of the first tile and the odd ones of the second, so that a store is 16 bytes and a row's four lanes fill 64 (SwiGLU: 8 and 32).
// `to` is pair_place's for the same O, row, n and sixteenth, and all four lanes of a row call it.
template <Out O = Out::Any>
__device__ __forceinline__ void store_pair(const GemmArgs& a, uint16_t* to, int n, float* v0, float* v1) {
    if (is_gated<O>(a)) {
        const PieHipGlu rule = rule_of<O>(a);
        uint32_t o[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float* v = i ? v1 : v0;
            float w[2];
#pragma unroll
            for (int r = 0; r < 2; ++r) {
                float g = v[2 * r], u = v[2 * r + 1];
                if (rule.bias) {
                    g += rule.bias[n + 16 * i + 2 * r];
                    u += rule.bias[n + 16 * i + 2 * r + 1];
                }
                g = round_bf16(g);
                u = round_bf16(u);
                w[r] = glu_value(g, u, rule);
            }
            o[i] = pack_bf16x2(w[0], w[1]);
        }
        const auto s = __builtin_amdgcn_permlane16_swap(o[0], o[1], false, false);
        *reinterpret_cast<u32x2_t*>(to) = u32x2_t{s[0], s[1]};
        return;
    }
    u32x4_t* p = reinterpret_cast<u32x4_t*>(to);
    if constexpr (O == Out::Any) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            v0[r] = epilogue_pointwise<true>(v0[r], a.pointwise);
            v1[r] = epilogue_pointwise<true>(v1[r], a.pointwise);
        }
    }
    if (is_residual<O>(a)) {
        const u32x4_t old = *p;
        const auto x = __builtin_amdgcn_permlane16_swap(old[0], old[2], false, false), y = __builtin_amdgcn_permlane16_swap(old[1], old[3], false, false);
        v0[0] += bf16_lo(x[0]);
        v0[1] += bf16_hi(x[0]);
        v0[2] += bf16_lo(y[0]);
        v0[3] += bf16_hi(y[0]);
        v1[0] += bf16_lo(x[1]);
        v1[1] += bf16_hi(x[1]);
        v1[2] += bf16_lo(y[1]);
        v1[3] += bf16_hi(y[1]);
    }
    const auto x = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v0[0], v0[1]), pack_bf16x2(v1[0], v1[1]), false, false);
    const auto y = __builtin_amdgcn_permlane16_swap(pack_bf16x2(v0[2], v0[3]), pack_bf16x2(v1[2], v1[3]), false, false);
    *p = u32x4_t{x[0], y[0], x[1], y[1]};
}

// q|k|v rows: adjacent columns of q and k heads are rotated, q goes to y [rows, hq * d], k and v to slot slots[row] of the pools
struct Rotation {
    const float* table = nullptr;   // [rows, d]: cos (d / 2), then sin (d / 2); null: plain outputs
    const int64_t* slots = nullptr; // negative: the row writes no K/V
    uint16_t *k_pages = nullptr, *v_pages = nullptr;
    int hq = 0, hk = 0, d = 0, half_out = 0;   // half_out: pair (2i, 2i + 1) goes to places (i, i + d / 2)
};

// Row m, columns n .. n + 3: the projection's bf16 values, then the rotation of qkv_rope_kvwrite_kernel, same operations and rounding.
__device__ __forceinline__ void store_rotated(const GemmArgs& a, const Rotation& r, int m, int n, const float* v) {
    const int shift = __builtin_ctz(static_cast<unsigned>(r.d)), head = n >> shift, dd = n & (r.d - 1);
    float b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = bf16_bits_to_f32(f32_to_bf16_bits(v[i]));
    const int64_t slot = r.slots[m];
    if (head >= r.hq + r.hk) {
        if (slot >= 0)
            *reinterpret_cast<u32x2_t*>(r.v_pages + (static_cast<size_t>(slot) * r.hk + (head - r.hq - r.hk)) * r.d + dd) =
                u32x2_t{pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3])};
        return;
    }
    if (head >= r.hq && slot < 0) return;
    const float* tab = r.table + static_cast<size_t>(m) * r.d + (dd >> 1);
    uint16_t* dst = head < r.hq ? a.y + (static_cast<size_t>(m) * r.hq + head) * r.d
                                : r.k_pages + (static_cast<size_t>(slot) * r.hk + (head - r.hq)) * r.d;
    uint32_t o[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float c = tab[i], s = tab[(r.d >> 1) + i], x = b[2 * i], y = b[2 * i + 1];
        o[i] = pack_bf16x2(x * c - y * s, y * c + x * s);
    }
    if (r.half_out) {
        *reinterpret_cast<uint32_t*>(dst + (dd >> 1)) = __builtin_amdgcn_perm(o[1], o[0], 0x05040100u);
        *reinterpret_cast<uint32_t*>(dst + (dd >> 1) + (r.d >> 1)) = __builtin_amdgcn_perm(o[1], o[0], 0x07060302u);
    } else {
        *reinterpret_cast<u32x2_t*>(dst + dd) = u32x2_t{o[0], o[1]};
    }
}
__device__ __forceinline__ void store4(const GemmArgs& a, const Rotation& r, int m, int n, float* v) {
    if (r.table) store_rotated(a, r, m, n, v);
    else wide_store(a, m, n, v);
}

// places of a row's sixteen 16-byte granules: granule c at c ^ key(row).  The lanes an LDS read serves together (0 - 3 and
// 12 - 15 of one granule's rows, 4 - 11 of the next but three) find sixteen different places.
__device__ __forceinline__ int key_of(int row) { return (row & 15) < 4 ? row & 15 : (row & 15) < 12 ? (row & 15) + 4 : (row & 15) - 8; }

// The problem and the rows [m0, m1) of block row `t` when problems are cut into blocks of `rows` rows one after
// another; false behind the last.  Every lane of the wave calls it and gets the same answer.
__device__ __forceinline__ bool grouped_place(const int32_t* __restrict__ offsets, int problems, int rows, int t, int lane,
                                              int& p, int& m0, int& m1) {
    constexpr int kAhead = 2;   // (chunks of 64 problems fetched together: their latency is most of this)
    int before = 0;
    for (int base = 0; base < problems; base += kAhead * kWave) {
        int lo[kAhead], hi[kAhead];
#pragma unroll
        for (int c = 0; c < kAhead; ++c) {
            const int e = base + c * kWave + lane;
            lo[c] = e < problems ? offsets[e] : 0;
            hi[c] = e < problems ? offsets[e + 1] : 0;
        }
#pragma unroll
        for (int c = 0; c < kAhead; ++c) {
            const int n = (hi[c] - lo[c] + rows - 1) / rows;
            int sum = n;
#pragma unroll
            for (int d = 1; d < kWave; d <<= 1) {
                const int o = __shfl_up(sum, d);
                if (lane >= d) sum += o;
            }
            const unsigned long long past = __ballot(before + sum > t);
            if (past) {
                const int at = __ffsll(past) - 1;
                p = __builtin_amdgcn_readfirstlane(base + c * kWave + at);
                m0 = __builtin_amdgcn_readfirstlane(__shfl(lo[c], at) + (t - before - __shfl(sum - n, at)) * rows);
                m1 = __builtin_amdgcn_readfirstlane(__shfl(hi[c], at));
                return true;
            }
            before += __shfl(sum, kWave - 1);
        }
    }
    return false;
}

// The wide form: blocks of 256 rows by 256 or 128 columns, over row-major bf16 or tile-major quantised weights (`scale`
// tile-major for int4); a workspace lets few blocks over a long K run in shares.  What it and the tiles of
// gemm_mfma.hip take, in microseconds (1e30: it does not take the shape).
int launch_gemm_wide(int format, const GemmArgs& a, int group_size, void* ws, size_t ws_bytes, hipStream_t stream);
// Experts' rows gathered by route, over tile-major fp8 or int8 weights (block_rows: 32, 64, 96, 128; 0: by the routes an expert has).
int launch_gemm_experts(int format, const GemmArgs& a, int routes, int block_rows, hipStream_t stream);
double gemm_wide_us(int format, int M, int N, int K, int group_size, size_t ws_bytes);
// Int4 weights with fp32 group scales, tile-major, of at least 128 values a group, in blocks of up to 64 rows; a workspace lets few blocks over a long K run
// in shares.
int launch_gemm_groups(const GemmArgs& a, int group_size, void* ws, size_t ws_bytes, hipStream_t stream);
double gemm_groups_us(int M, int N, int K, int group_size, size_t ws_bytes);
// The shares' fp32 sums in a.partial [shares, M, N], added in order, and the epilogue (N % 4 == 0, 16-byte boundaries).
int launch_shares_reduce(const GemmArgs& a, const Rotation& rot, int shares, hipStream_t stream);
double gemm_tiles_us(int format, int M, int N, int K);

}  // namespace pie_hip
