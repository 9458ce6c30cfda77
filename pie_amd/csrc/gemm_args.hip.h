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

// The wide form: blocks of 256 rows by 256 or 128 columns, over row-major bf16 or tile-major quantised weights (`scale`
// tile-major for int4); a workspace lets few blocks over a long K run in shares.  What it and the tiles of
// gemm_mfma.hip take, in microseconds (1e30: it does not take the shape).
int launch_gemm_wide(int format, const GemmArgs& a, int group_size, void* ws, size_t ws_bytes, hipStream_t stream);
double gemm_wide_us(int format, int M, int N, int K, int group_size, size_t ws_bytes);
double gemm_tiles_us(int format, int M, int N, int K);

}  // namespace pie_hip
