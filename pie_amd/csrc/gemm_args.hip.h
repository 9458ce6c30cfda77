// What the tiled GEMMs of large batches share: their arguments, and the launch of the wide form.
#pragma once

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
};

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
// Experts' rows gathered by route, over tile-major fp8 or int8 weights.
int launch_gemm_experts(int format, const GemmArgs& a, int routes, hipStream_t stream);
double gemm_wide_us(int format, int M, int N, int K, int group_size, size_t ws_bytes);
double gemm_tiles_us(int format, int M, int N, int K);

}  // namespace pie_hip
