#include "executor.hpp"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <stdexcept>
#include <string>

#include "pie_hip_kernels.h"

namespace pie_hip_driver {

#define PIE_HIP_CHECK(expr)                                                              \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess)                                                            \
            throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)

#define PIE_KERNEL(expr)                                                                     \
    do {                                                                                     \
        const int st_ = (expr);                                                              \
        if (st_ != PIE_HIP_OK)                                                               \
            throw std::runtime_error(std::string(#expr) + " failed with status " +          \
                                     std::to_string(st_));                                   \
    } while (0)

namespace {

using clk = std::chrono::steady_clock;
uint32_t us_since(clk::time_point t0) {
    return static_cast<uint32_t>(
        std::chrono::duration_cast<std::chrono::microseconds>(clk::now() - t0).count());
}

template <typename T>
T* dmalloc(size_t elems) {
    void* p = nullptr;
    PIE_HIP_CHECK(hipMalloc(&p, std::max<size_t>(elems, 1) * sizeof(T)));
    return static_cast<T*>(p);
}

size_t align_up(size_t v, size_t a) { return (v + a - 1) / a * a; }

int fmt_code(Quant q) {
    switch (q) {
        case Quant::Int4b8: return PIE_HIP_FMT_INT4B8;
        case Quant::Int8: return PIE_HIP_FMT_INT8;
        case Quant::Fp8: return PIE_HIP_FMT_FP8;
        default: return PIE_HIP_FMT_BF16;
    }
}

// Measured cost models (MI355X, microseconds, int4 8B-class shapes at 16-128 rows).  Skinny GEMM:
// ~5 us + the weights at ~2.8 TB/s for the first 16-row pass, each further (side-by-side) pass
// adding 85 % of that stream; from the tile-major copy (wave-private form) ~3.8 TB/s and 52 % per
// further pass, the pass count rounded up to a power of two.  Tiled GEMM (eight-wave blocks): K in
// 64-wide steps of ~0.60 us with 64-row block tiles (M <= 64), ~0.68 us with 128-row tiles, while
// the tiles fit the machine (512 resident blocks).  Split-K tiled GEMM: the steps of one share
// (+3 of prologue) at 1.06 / 1.36 us with two blocks per CU, per round of 512 blocks, plus ~15 us
// for the second kernel and the partials.
// More than 128 rows: the tiled GEMM's two forms say themselves what they take (pie_hip_gemm_mfma_us); over 40 shapes of 160 -
// 4096 rows in three formats a choice by these estimates loses 0.5 % against the fastest of the three each time.
enum class GemmPath { Skinny, Tiled, TiledSplitK, Wide };
bool tile_major(const Linear& w) { return w.data_tiled && (w.kind != Quant::Int4b8 || w.scale_tiled); }
struct Skinny {
    int p2, wpasses;        // passes of the wave-private form, and as the power of two they cost
    double wave_form, us;
};
Skinny skinny_cost(const Linear& w, int M) {
    const int passes = (M + 15) / 16;
    // the wave-private form runs its passes side by side: cost steps at powers of two; above 32
    // rows a pass covers 32 rows and costs 1.38 of a 16-row one
    const int wpasses = M > 32 ? (M + 31) / 32 : passes;
    int p2 = 1;
    while (p2 < wpasses) p2 <<= 1;
    // (past eight passes the machine is full: the cost grows in proportion)
    const double data = static_cast<double>(w.data_bytes());
    const double wave_form = (M > 32 ? 1.38 : 1.0) * (p2 <= 8 ? 1.0 + 0.52 * (p2 - 1) : (1.0 + 0.52 * 7) * wpasses / 8.0);
    return {p2, wpasses, wave_form, w.data_tiled ? 5.0 + data / 3.8e6 * wave_form : 5.0 + data / 2.8e6 * (1.0 + 0.85 * (passes - 1))};
}
// Microseconds of int4 weights in blocks of up to 64 rows, which scale a group's sum in fp32 as the skinny GEMM does (1e30: not
// taken).  Where the skinny GEMM is chosen and these are estimated faster, they run in its place: 320 rows of 4096 x 14336 50 us
// against 68, of 4096 x 4096 21 against 28; 2 / 16 / 32 / 96 of 28672 x 4096 14.5 / 13.8 / 17.4 / 34.5 against 18.4 / 19.8 / 21.9 / 47.4; 321 of q|k|v with the
// rotation, 6144 x 4096, 33 against 73.
double groups_cost(const Linear& w, int M, size_t ws_bytes) {
    return M >= 2 && w.kind == Quant::Int4b8 && tile_major(w) ? pie_hip_gemm_groups_us(M, w.N, w.K, w.group, ws_bytes) : 1e30;
}
// The skinny GEMM of tile-major weights as the other forms are compared with it: up to 128 rows fitted to 50 matrices (one-byte weights, and int4 to 320 rows: 15) of 1024 - 28672 x 1024 - 14336 with
// weights out of HBM, 5 - 11 % rms; bf16 over 17 matrices to 320 rows, with a copy or row-major, 8 - 13 %, past 128 rows 13 - 22.  (The estimate above prices all matrices by their bytes alone: it is 40 % above what few rows of large ones take, and
// blocks chosen by it ran 1.2 to 1.5 times as long as the passes: 2 rows of 8192 x 8192 int4 12.0 us against 9.9, 8 of 8192 x 1024 5.7 against 4.5.)
double passes_cost(const Linear& w, int M) {
    struct Fit {
        int rows;
        double fixed, rate, per_n, per_k;
    };
    constexpr Fit kFits[5][10] = {{{4, 3.21, 6.95e6, 0.061e-3, 0.288e-3},  {16, 3.65, 6.49e6, 0.056e-3, 0.390e-3}, {32, 4.22, 4.20e6, 0.089e-3, 0.337e-3},
                                  {64, 4.53, 3.47e6, 0.195e-3, 0.633e-3}, {96, 4.65, 1.93e6, 0.350e-3, 0.524e-3}, {128, 4.83, 1.72e6, 0.331e-3, 0.555e-3},
                                   {160, 3.00, 1.17e6, 0.730e-3, 0.975e-3}, {192, 3.47, 1.05e6, 0.786e-3, 0.968e-3},
                                   {256, 3.47, 1.01e6, 1.001e-3, 1.087e-3}, {320, 3.85, 0.57e6, 1.097e-3, 1.135e-3}},
                                 /* int8 */ {{8, 3.64, 5.22e6, 0.051e-3, 0.153e-3}, {16, 3.72, 5.74e6, 0.096e-3, 0.443e-3}, {32, 4.11, 4.64e6, 0.140e-3, 0.340e-3},
                                             {64, 3.87, 4.94e6, 0.447e-3, 0.727e-3}, {96, 4.22, 2.32e6, 0.471e-3, 0.563e-3}, {128, 4.31, 2.38e6, 0.582e-3, 0.686e-3}},
                                 /* fp8 */ {{8, 3.26, 5.38e6, 0.050e-3, 0.160e-3}, {16, 3.40, 5.52e6, 0.068e-3, 0.399e-3}, {32, 3.67, 4.62e6, 0.111e-3, 0.314e-3},
                                            {64, 3.26, 4.78e6, 0.357e-3, 0.683e-3}, {96, 3.57, 2.36e6, 0.359e-3, 0.529e-3}, {128, 3.42, 2.47e6, 0.497e-3, 0.712e-3}},
                                 /* bf16 */ {{8, 3.43, 5.89e6, 0.000e-3, 0.025e-3}, {16, 3.81, 5.77e6, 0.000e-3, 0.179e-3}, {32, 3.99, 4.65e6, 0.000e-3, 0.000e-3},
                                             {64, 4.21, 4.45e6, 0.116e-3, 0.246e-3}, {96, 4.38, 2.62e6, 0.014e-3, 0.117e-3}, {128, 4.70, 2.47e6, 0.082e-3, 0.074e-3},
                                             {192, 4.39, 1.53e6, 0.076e-3, 0.000e-3}, {320, 5.01, 1.21e6, 0.283e-3, 0.000e-3}},
                                 /* row-major */ {{8, 4.80, 6.01e6, 0.191e-3, 0.474e-3}, {16, 5.16, 6.06e6, 0.208e-3, 0.693e-3}, {32, 6.06, 2.93e6, 0.000e-3, 0.160e-3},
                                                  {64, 6.35, 1.97e6, 0.024e-3, 0.449e-3}, {96, 8.00, 1.43e6, 0.000e-3, 0.726e-3}, {128, 8.00, 1.04e6, 0.000e-3, 0.102e-3},
                                                  {192, 8.00, 0.77e6, 0.191e-3, 0.859e-3}, {320, 6.28, 0.46e6, 0.123e-3, 0.209e-3}}};
    // (parts of a step of K are refused, and the GEMV runs, four rows at a time: 12 / 16 int4 rows of 1536 x 8960 in blocks whose waves take the steps in turn 8.6 / 8.8 us)
    if (w.K % (w.kind == Quant::Int4b8 ? 512 : w.kind == Quant::Bf16 ? 128 : 256) != 0)
        return ((M + 3) / 4) * (3.4 + 2.5 * static_cast<double>(w.data_bytes()) / 5.5e6);
    if (w.kind == Quant::Bf16 || tile_major(w))
        for (const Fit& f : kFits[w.kind == Quant::Int4b8 ? 0 : w.kind == Quant::Int8 ? 1 : w.kind == Quant::Fp8 ? 2 : tile_major(w) ? 3 : 4])
            if (M <= f.rows)   // (a list's unused places have no rows)
                return f.fixed + static_cast<double>(w.data_bytes()) / f.rate + w.N * f.per_n + w.K * f.per_k;
    return skinny_cost(w, M).us;
}
// (up to 32 rows both are short, and ties stay where they are)
bool in_groups(const Linear& w, int M, size_t ws_bytes) {
    const double us = groups_cost(w, M, ws_bytes);
    if (us > 1e29) return false;
    if (M <= 128 && w.groups[M] >= 0) return w.groups[M] == 1;   // (measured at start-up)
    return (M <= 32 ? 1.05 : 1.0) * us < passes_cost(w, M);
}
// Microseconds of weights in blocks whose waves take the steps of K in turn (1e30: not taken); they run in the skinny GEMM's place where they
// are estimated faster than its passes and than blocks that scale groups.  Over 5 - 480 rows of 42 matrices, weights out of HBM, what is chosen takes 0.84 of what would be without
// them for int8, 0.90 for fp8, 0.94 for int4, 0.85 for bf16 and 0.74 for row-major bf16, and 0.8 - 2.6 % more than the fastest of all.
double waves_cost(const Linear& w, int M, size_t ws_bytes) {
    return M >= 5 && (w.kind == Quant::Bf16 || tile_major(w)) ? pie_hip_gemm_waves_us(fmt_code(w.kind), tile_major(w) ? 1 : 0, M, w.N, w.K, w.group, ws_bytes, 0) : 1e30;
}
double skinny_or_groups(const Linear& w, int M, size_t ws_bytes) { return in_groups(w, M, ws_bytes) ? groups_cost(w, M, ws_bytes) : passes_cost(w, M); }
// They have to be faster by more than what the estimates are off by where that was found to go against them (in graphs, 4001 points of 42 matrices; "before": what runs without this
// kernel).  Of quantised rows up to 24 both are short (20 int4 / 17 fp8 rows of 2048 x 8192 7.9 / 8.6 us before, 8.9 / 9.8 here); int4 blocks of a short K are
// estimated up to a fifth low (128 / 80 rows of 6144 x 2048 10.0 / 8.1 before, 11.9 / 9.1 here); row-major bf16 past 320 rows is compared with the passes'
// bytes alone (480 rows of 128 x 2048 7.1 before, 8.0 here).  With these and those of pick_gemm 20 points are more than 3 % slower than before, the worst by 10 % (48 bf16 rows
// of 28672 x 1024), where 110 were, the worst by 28 %; the mean gain is what it was, 6 - 26 % by format.
double waves_margin(const Linear& w, int M, size_t ws_bytes) {
    if (w.kind == Quant::Bf16) return !tile_major(w) && M > 320 ? 1.25 : 1.0;
    if (in_groups(w, M, ws_bytes)) return w.K <= 2048 ? 1.2 : 1.0;
    return M <= 24 ? 1.12 : 1.0;
}
bool in_waves(const Linear& w, int M, size_t ws_bytes) {
    const double us = waves_cost(w, M, ws_bytes);
    return us < 1e29 && waves_margin(w, M, ws_bytes) * us < skinny_or_groups(w, M, ws_bytes);
}
// Microseconds of one-byte weights in blocks of 32 to 128 rows (1e30: not taken); they take the place of the blocks of 256 rows
// where they are estimated faster.
// (from 65 rows on: of 28672 x 4096 96 int8 rows take 42 us so and 54 in blocks of 64 columns, 128 44 and 62; below 129 the estimate is 6 % low)
double rows_cost(const Linear& w, int M, size_t ws_bytes) {
    return M > 64 && tile_major(w) ? (M > 128 ? 1.0 : 1.06) * pie_hip_gemm_rows_us(fmt_code(w.kind), M, w.N, w.K, ws_bytes) : 1e30;
}
bool in_rows(const Linear& w, int M, size_t ws_bytes) {
    const double rows = rows_cost(w, M, ws_bytes);
    return rows < 1e29 && rows < pie_hip_gemm_mfma_us(fmt_code(w.kind), M, w.N, w.K, w.group, 1, ws_bytes);
}
// Microseconds of a projection whose sums do not wait for the norm.
double apart_cost(const Linear& w, int M, size_t ws_bytes) {
    const int fmt = fmt_code(w.kind);
    double us = in_waves(w, M, ws_bytes) ? waves_cost(w, M, ws_bytes) : skinny_or_groups(w, M, ws_bytes);
    if (w.kind != Quant::Int4b8) us = std::min({us, rows_cost(w, M, ws_bytes), static_cast<double>(pie_hip_gemm_mfma_us(fmt, M, w.N, w.K, w.group, 1, ws_bytes))});
    else if (M > 128) us = std::min({us, static_cast<double>(pie_hip_gemm_mfma_us(fmt, M, w.N, w.K, w.group, 0, ws_bytes)),
                                     static_cast<double>(pie_hip_gemm_mfma_us(fmt, M, w.N, w.K, w.group, 1, ws_bytes))});
    return us;
}
// Whether a projection back into the residual leaves its sums in shares of K, which the next norm's kernel adds up
// (pie_hip_shares_rmsnorm), for 5 rows and more: int4 4096 x 14336 and the norm of 16 / 40 / 64 / 96 rows 18.3 / 23.3 / 25.4 / 30.5 us in two launches
// without shares, 13.4 / 17.5 / 19.9 / 24.2 with them; 4096 x 4096 9.8 / 12.9 / 13.0 / 15.0 and 9.1 / 11.2 / 11.7 / 14.4.  (1e30: not taken, by the products' kernels or the norm's)
double groups_shares_cost(const Linear& w, int M, size_t ws_bytes) {
    return w.kind == Quant::Int4b8 ? pie_hip_gemm_groups_shares_us(M, w.N, w.K, w.group, ws_bytes) : 1e30;
}
double waves_shares_cost(const Linear& w, int M, size_t ws_bytes) { return pie_hip_gemm_waves_us(fmt_code(w.kind), 1, M, w.N, w.K, w.group, ws_bytes, 1); }
double shares_cost(const Linear& w, int M, size_t ws_bytes) {
    if (M < 5 || !tile_major(w) || w.N % 8 != 0 || w.N > 16384) return 1e30;
    return std::min(groups_shares_cost(w, M, ws_bytes), waves_shares_cost(w, M, ws_bytes));
}
bool in_shares(const Linear& w, int M, size_t ws_bytes) {
    const double us = shares_cost(w, M, ws_bytes);
    if (us > 1e29) return false;
    if (M <= 128 && w.shares[M] >= 0) return w.shares[M] == 1;   // (measured at start-up)
    // (a product apart reads and writes the residual too: with 0.4 us for that the choice is 0.2 - 1.4 % over the fastest of all on average over 2144 products and norms, without 0.8 - 1.5;
    // 64 int4 rows of 4096 x 4096 11.3 us in shares, 12.0 apart)
    return us - 0.4 < apart_cost(w, M, ws_bytes);
}
bool close(double a, double b) { return std::max(a, b) < 1.2 * std::min(a, b); }
// Whether a start times the skinny GEMM's passes against the blocks that scale groups: estimates less than a fifth apart, and neither gives way to blocks
// whose waves take the steps in turn, which both settings would then run.
bool measures_groups(const Linear& w, int M, size_t ws_bytes) {
    const double groups = groups_cost(w, M, ws_bytes), passes = passes_cost(w, M);
    return groups < 1e29 && close(groups, passes) && waves_cost(w, M, ws_bytes) >= std::max(groups, passes);
}
// Likewise shares that meet in the norm's kernel against a product and the norm, where blocks that scale groups make the shares.  Blocks whose waves take the steps in
// turn are chosen by estimate alone: over 160 such pairs of seven drivers that loses 0.7 % on average to the faster of a pair's smallest times (at most 14 %), about the tenth
// that a measurement needs to overrule an estimate, and of 177 pairs with shares 0.6 % (20 %).  Timed, they differed from start to start, and with them the
// kernels' rounding: 40 of the 528 measured row counts in eight starts of each driver, 12 so, seven of which run the same kernel either way (19 before there were such blocks).
bool measures_shares(const Linear& w, int M, size_t ws_bytes, bool routed_as_estimated) {
    const double us = groups_shares_cost(w, M, ws_bytes);
    return shares_cost(w, M, ws_bytes) < 1e29 && us < 1e29 && us <= waves_shares_cost(w, M, ws_bytes) && !in_waves(w, M, ws_bytes) &&
           (!routed_as_estimated || close(us, apart_cost(w, M, ws_bytes)));
}
// The tiled GEMM, up to 128 rows (bf16 weights at most as fast as they stream: 24 - 77 rows of 28672 x 4096 53 - 56 us, of 32000 x 4096 58 - 70).
double tiled_cost(const Linear& w, int M) {
    const double us = 2.0 + w.K / 64 * (M <= 64 ? 0.60 : 0.68) * std::max(1.0, (w.N + 127) / 128 / 512.0);
    return w.kind == Quant::Bf16 ? std::max(us, 2.6 + static_cast<double>(w.data_bytes()) / 4.6e6) : us;
}
GemmPath pick_gemm(const Linear& w, int M, size_t ws_bytes) {
    if (w.K % 64 != 0 || M < 17) return GemmPath::Skinny;
    const auto [p2, wpasses, wave_form, passes] = skinny_cost(w, M);
    const bool one_byte = w.kind == Quant::Int8 || w.kind == Quant::Fp8;
    const double waves = in_waves(w, M, ws_bytes) ? waves_cost(w, M, ws_bytes) : 1e30;   // (in the skinny GEMM's place)
    // (against the blocks of the larger batches: 112 int8 rows of 16384 x 2048 20.1 us in those, 21.9 here)
    const double skinny = std::min(w.kind != Quant::Int4b8 ? passes_cost(w, M) : passes, (one_byte ? 1.06 : 1.0) * waves);
    const double data = static_cast<double>(w.data_bytes()), groups = groups_cost(w, M, ws_bytes);
    const int steps = w.K / 64;
    if (M > 128) {
        // Int4 weights: the skinny GEMM multiplies the codes and scales a group's sum in fp32, the blocks round every code times
        // its scale to bf16 first, which takes a product's error from 0.0017 of its norm to 0.0022 (K of 4096, groups of 128).
        // So int4 weights leave fp32 scales only where the skinny GEMM is estimated slower than 128-row tiles, at 512 of them to a
        // round: 28672 x 4096 at once, 6144 x 4096 from 481 rows on, 4096 x 4096 from 705, 4096 x 14336 from 769.  (At 381 rows of
        // these skinny / wide blocks take 169 / 120, 45 / 42, 28 / 31 and 73 / 68 us.)
        const double high = static_cast<double>((w.N + 127) / 128) * ((M + 127) / 128);
        if (w.kind == Quant::Int4b8 && skinny <= 2.0 + steps * 0.68 * std::max(1.0, high / 512.0)) return GemmPath::Skinny;
        // (prompts' passes cost in powers of two up to 32, 17 - 31 passes a fifth worse than 32, and are bound by the products and
        // the decoding, not by the weights' width)
        const double bytes = w.kind == Quant::Bf16 ? data : (w.kind == Quant::Int8 ? 0.63 : w.kind == Quant::Fp8 ? 0.57 : 0.5) * w.N * static_cast<double>(w.K);
        const double prompt_form = p2 <= 8 ? wave_form : 1.38 * (1.0 + 0.52 * 7) * 0.9 * (p2 <= 32 ? p2 : wpasses) / 8.0 * (p2 == 32 && wpasses < 32 ? 1.2 : 1.0);
        const double rows_us = w.data_tiled ? (M > 256 ? 7.0 : 5.0) + bytes / 3.8e6 * prompt_form : w.kind != Quant::Int4b8 ? passes_cost(w, M) : passes;
        const int fmt = fmt_code(w.kind);
        const double tiles = pie_hip_gemm_mfma_us(fmt, M, w.N, w.K, w.group, 0, ws_bytes);
        const double rows = rows_cost(w, M, ws_bytes), wide = tile_major(w) ? static_cast<double>(pie_hip_gemm_mfma_us(fmt, M, w.N, w.K, w.group, 1, ws_bytes)) : tiles;
        const double blocks = std::min(rows, wide);
        // (bf16 rows are estimated a fifth low where their blocks come in two rounds, and the tiled GEMM a tenth high: 136 of 16384 x 2048 24.8 us in tiles, 31.1 here; more
        // so of a short K: 352 of 4096 x 512 11.2 and 12.2; not of a long one: 288 of 2048 x 8192 29.7 and 26.0, estimated 29.6; one-byte rows of a short K likewise: 192 of
        // 8192 x 512 8.0 in blocks of rows, 9.8 here)
        const double margin = w.kind == Quant::Bf16 ? (w.K <= 768 ? 1.3 : w.K < 8192 ? 1.12 : 1.0) : one_byte && w.K <= 1024 ? 1.2 : 1.0;
        if (margin * waves < std::min({rows, wide, tiles})) return GemmPath::Skinny;
        // (on narrow outputs blocks of few rows and the passes are close, and the passes' estimate is the one that is too high: 160 rows of 3072 x 4096 and
        // 320 of 2048 x 2048 fp8 13.9 and 13.7 us in passes, 17.0 and 14.7 in blocks)
        if (rows_us < std::min(1.12 * rows, wide) || groups < std::min({skinny, blocks, tiles})) return GemmPath::Skinny;
        return blocks < tiles ? GemmPath::Wide : GemmPath::Tiled;
    }
    const double tiles = static_cast<double>((w.N + 127) / 128), tiled = tiled_cost(w, M);
    double split = 1e30;
    const size_t need = pie_hip_gemm_mfma_workspace_bytes(M, w.N, w.K);
    if (need && need <= ws_bytes) {
        const int shares = static_cast<int>(need / (static_cast<size_t>(M) * w.N * sizeof(float)));
        const int per = (steps + shares - 1) / shares;
        split = 15.0 + (per + 3) * (M <= 64 ? 1.06 : 1.36) * std::ceil(tiles * shares / 512.0);
        if (w.kind == Quant::Bf16) split = std::max(split, 8.0 + data / 4.6e6);   // (24 / 64 rows of 32000 x 4096 62 - 66 / 73)
    }
    if (w.kind == Quant::Int4b8) {   // (blocks with fp32 group scales run in the skinny GEMM's place; up to 48 rows of wide outputs that is the wide GEMM's own form)
        if (std::min(waves, groups) < std::min(split, tiled))
            return M <= 48 && w.N >= 16384 && waves > 1e29 && in_groups(w, M, ws_bytes) ? GemmPath::Wide : GemmPath::Skinny;
    } else if (tile_major(w) && std::min(rows_cost(w, M, ws_bytes), static_cast<double>(pie_hip_gemm_mfma_us(fmt_code(w.kind), M, w.N, w.K, w.group, 1, ws_bytes))) <
                                    std::min({skinny, split, tiled})) {
        return GemmPath::Wide;
    }
    if (split < skinny && split < tiled) return GemmPath::TiledSplitK;
    return tiled < skinny ? GemmPath::Tiled : GemmPath::Skinny;
}

// The fitted cost model's kernel for M rows of `w`: 0 GEMV, 1 skinny GEMM, 2 tiled GEMM, 3 tiled GEMM
// in K shares, 4 tiled GEMM over the tile-major copy.  Two to four rows: the GEMV pays its dot products once per row, the skinny GEMM over
// the tile-major copy does not but needs the norm as its own launch (~4.8 us).  Costs fitted to
// the 8B shapes decide (decode steps of 2 / 3 / 4 rows over 512-token contexts: 1.91 / 2.46 /
// 2.79 ms with the GEMV everywhere, 2.01 / 2.08 / 2.14 ms with the skinny GEMM everywhere);
// without a tile-major copy the GEMV keeps all four.
int model_route(const Linear& w, int M, bool has_norm, size_t ws_bytes) {
    if (M <= 4) {
        if (M < 2 || !w.data_tiled) return 0;
        const double bytes = static_cast<double>(w.data_bytes());
        const double t_gemv = 3.4 + bytes / 5.5e6 * (M == 2 ? 1.35 : 1.0 + 0.5 * (M - 1));   // (a second row costs the GEMV less than the third and fourth)
        const double t_skinny = std::min(4.4 + bytes / 4.2e6, in_groups(w, M, ws_bytes) ? groups_cost(w, M, ws_bytes) : 1e30) + (has_norm ? 4.8 : 0.0);
        if (t_gemv <= t_skinny) return 0;
    }
    const GemmPath p = pick_gemm(w, M, ws_bytes);
    return p == GemmPath::Skinny ? 1 : p == GemmPath::Tiled ? 2 : p == GemmPath::TiledSplitK ? 3 : 4;
}

// (PIE_GEMV_MAX_ROWS = n: rows up to n take the GEMV, more the skinny GEMM, whatever the costs say)
int forced_gemv_rows() {
    static const int forced_rows = [] { const char* e = getenv("PIE_GEMV_MAX_ROWS"); return e ? atoi(e) : -1; }();
    return forced_rows;
}

// Whether linear_fused sends M rows of this linear to the GEMV (its first choice, before any
// refusal by the kernel).
bool routes_to_gemv(const Linear& w, int M, bool has_norm, size_t ws_bytes) {
    const int tuned = M <= 128 ? w.tuned[M] : -1;
    if (tuned >= 0) return tuned == 0 && M <= 4;
    if (forced_gemv_rows() >= 0) return M <= std::min(forced_gemv_rows(), 4);
    return model_route(w, M, has_norm, ws_bytes) == 0;
}

// y = epilogue(rmsnorm?(act) · W^T) by the weight's storage format — the dispatcher role of
// gemm_act_x_w (driver/cuda/src/ops/gemm.cpp:1414-1583).  Up to four rows: the weight-streaming
// GEMV with the norm riding in its activation staging and SwiGLU in its epilogue.  More rows
// (norm as its own kernel into `norm_tmp`): the matrix-core skinny GEMM, which streams the
// weights once per 16 rows, or the tiled matrix-core GEMM where its cost model wins; shapes those do
// not take fall back to the GEMV path.
// `force`: -1 = pick (the start-up measurement when there is one, else the cost model); 0..4 = that
// kernel whatever the costs (the tuner's own launches).  Returns false when a forced kernel does
// not take the shape.
}  // namespace

bool linear_fused(const Linear& w, const uint16_t* act, const uint16_t* norm_w, float eps,
                  uint16_t* y, int M, int beta, int swiglu, uint16_t* norm_tmp, void* gemm_ws,
                  size_t gemm_ws_bytes, hipStream_t s, int force, const PieHipGlu* glu) {
    const int fmt = fmt_code(w.kind);
    const int sbf = w.scale_bf16 ? 1 : 0;
    const int forced_rows = forced_gemv_rows();
    int tuned = force >= 0 ? force : (M <= 128 ? w.tuned[M] : -1);
    bool gemv;
    if (tuned >= 0) {
        gemv = tuned == 0 && M <= 4;
    } else if (forced_rows >= 0) {
        gemv = M <= std::min(forced_rows, 4);
    } else {
        tuned = model_route(w, M, norm_w != nullptr, gemm_ws_bytes);
        gemv = tuned == 0;
    }
    if (gemv) {
        const int st = pie_hip_linear_fused_glu(fmt, act, norm_w, eps, w.data, w.scale, sbf, w.group, y, M, w.N, w.K,
                                                beta, swiglu, glu, s);
        if (st == PIE_HIP_OK) return true;
        if (st != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(st);
        if (force >= 0) return false;
        // (a row too long for the GEMV's staged activations: the matrix-core kernels take any K)
    }
    {
        const uint16_t* a = act;
        if (norm_w) {
            PIE_KERNEL(pie_hip_rmsnorm(act, norm_w, norm_tmp, M, w.K, eps, s));
            a = norm_tmp;
        }
        const GemmPath path = tuned == 1   ? GemmPath::Skinny
                              : tuned == 2 ? GemmPath::Tiled
                              : tuned == 3 ? GemmPath::TiledSplitK
                              : tuned == 4 ? GemmPath::Wide
                                           : pick_gemm(w, M, gemm_ws_bytes);   // (forced row limit, GEMV refusal)
        if (path == GemmPath::Skinny && in_waves(w, M, gemm_ws_bytes)) {
            const int sv = w.data_tiled ? pie_hip_gemm_waves_tiled(fmt, a, w.data_tiled, w.scale_tiled ? w.scale_tiled : w.scale, sbf, w.group, y, M, w.N, w.K, beta,
                                                                   swiglu, glu, gemm_ws, gemm_ws_bytes, s)
                                        : pie_hip_gemm_waves_bf16(a, w.data, y, M, w.N, w.K, beta, swiglu, glu, gemm_ws, gemm_ws_bytes, s);
            if (sv == PIE_HIP_OK) return true;
            if (sv != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(sv);
        }
        if (path == GemmPath::Skinny && in_groups(w, M, gemm_ws_bytes)) {
            const int sg = pie_hip_gemm_groups_tiled(a, w.data_tiled, w.scale_tiled, w.group, y, M, w.N, w.K, beta, swiglu, glu,
                                                     gemm_ws, gemm_ws_bytes, s);
            if (sg == PIE_HIP_OK) return true;
            if (sg != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(sg);
        }
        if (path == GemmPath::Wide && in_rows(w, M, gemm_ws_bytes)) {
            const int sr = pie_hip_gemm_rows_tiled(fmt, a, w.data_tiled, w.scale, sbf, y, M, w.N, w.K, beta, swiglu, glu, gemm_ws, gemm_ws_bytes, s);
            if (sr == PIE_HIP_OK) return true;
            if (sr != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(sr);
        }
        if (path == GemmPath::Wide) {
            const int sw = pie_hip_gemm_mfma_tiled(fmt, a, w.data_tiled, w.scale_tiled ? w.scale_tiled : w.scale, sbf, w.group, y, M,
                                                   w.N, w.K, beta, swiglu, glu, gemm_ws, gemm_ws_bytes, s);
            if (sw == PIE_HIP_OK) return true;
            if (sw != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(sw);
            if (force >= 0) return false;
        }
        if (path != GemmPath::Skinny) {
            // the tiled GEMM (weights dequantised to bf16 while staged), in K shares for a
            // decode batch whose output has few tiles
            const bool split = path == GemmPath::TiledSplitK || M > 128;
            const int sg = pie_hip_gemm_mfma_glu(fmt, a, w.data, w.scale, sbf, w.group, y, M, w.N, w.K, beta, swiglu, glu,
                                                 split ? gemm_ws : nullptr, split ? gemm_ws_bytes : 0, s);
            if (sg == PIE_HIP_OK) return true;
            if (sg != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(sg);
            if (force >= 0) return false;
        }
        const int st = pie_hip_gemm_skinny_glu(fmt, a, w.data_tiled ? w.data_tiled : w.data,
                                               w.data_tiled && w.scale_tiled ? w.scale_tiled : w.scale, sbf, w.group, y, M,
                                               w.N, w.K, beta, swiglu, w.data_tiled ? 1 : 0, glu, s);
        if (st == PIE_HIP_OK) return true;
        if (st != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(st);
        if (force >= 0) return false;
        PIE_KERNEL(pie_hip_linear_fused_glu(fmt, a, nullptr, eps, w.data, w.scale, sbf, w.group, y, M,
                                            w.N, w.K, beta, swiglu, glu, s));
    }
    return true;
}

// Staged inputs are packed back to back in an order that makes every offset a function of
// (rows, sampled rows) only — the page list goes last — so one contiguous host-to-device copy
// feeds a forward and a captured graph's pointers stay valid for its (rows, sampled rows) key.
Executor::Inputs Executor::input_layout(int N, int S) const {
    Inputs in{};
    size_t off = 0;
    in.off_tokens = off;       off = align_up(off + static_cast<size_t>(N) * 4, 256);
    in.off_positions = off;    off = align_up(off + static_cast<size_t>(N) * 4, 256);
    in.off_slots = off;        off = align_up(off + static_cast<size_t>(N) * 8, 256);
    in.off_row_begin = off;    off = align_up(off + static_cast<size_t>(N) * 4, 256);
    in.off_row_len = off;      off = align_up(off + static_cast<size_t>(N) * 4, 256);
    in.off_sample_rows = off;  off = align_up(off + static_cast<size_t>(S) * 4, 256);
    const size_t per_row = model_.cfg().is_stack() ? 4 : 0;
    in.off_row_req = off;      off = align_up(off + N * per_row, 256);
    in.off_pair = off;         off = align_up(off + N * per_row, 256);
    in.off_qo = off;           off = align_up(off + (N + 1) * per_row, 256);
    in.off_rs_slot = off;      off = align_up(off + N * per_row, 256);
    in.off_rs_fresh = off;     off = align_up(off + N * per_row, 256);
    in.off_pages = off;
    in.total = off;
    return in;
}

Executor::Executor(const DriverConfig& cfg, Model& model) : cfg_(cfg), model_(model) {
    PIE_HIP_CHECK(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking));
    page_size_ = cfg.batching.kv_page_size;
    total_pages_ = cfg.batching.total_pages;
    max_tokens_ = cfg.batching.max_forward_tokens;
    max_page_refs_ = 4 * total_pages_ + max_tokens_;
    kv_format_ = kv_format_code(cfg.batching.kv_cache_dtype);
    dt_ = model.cfg().f32() ? PIE_HIP_DT_F32 : PIE_HIP_DT_BF16;
    alloc_kv();
    cpu_pages_ = std::max(0, cfg.batching.cpu_pages);
    if (cpu_pages_ > 0 && swap_page_bytes_ > 0) {
        const size_t bytes = swap_page_bytes_ * static_cast<size_t>(cpu_pages_);
        PIE_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&swap_pool_), bytes, hipHostMallocDefault));
        std::memset(swap_pool_, 0, bytes);
    }

    if (model.cfg().is_stack()) alloc_stack();
    else alloc_uniform();

    in_ = input_layout(max_tokens_, max_tokens_);
    in_.total = align_up(in_.off_pages + static_cast<size_t>(max_page_refs_) * 4, 256);
    PIE_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&in_host_), in_.total, hipHostMallocDefault));
    PIE_HIP_CHECK(hipMalloc(reinterpret_cast<void**>(&in_dev_), in_.total));
    out_cap_ = static_cast<size_t>(max_tokens_);
    out_tokens_ = dmalloc<uint32_t>(out_cap_);
    PIE_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&out_host_), out_cap_ * 4, hipHostMallocDefault));
    tune_linears();
}

// Activation workspaces of the uniform architectures.
void Executor::alloc_uniform() {
    const ModelConfig& m = model_.cfg();
    const size_t T = static_cast<size_t>(max_tokens_);
    const int H = m.hidden, d = m.head_dim, hq = m.q_heads, hk = m.kv_heads;
    const int I = model_.is_moe() ? m.expert_intermediate : m.intermediate;
    x_ = dmalloc<uint16_t>(T * H);
    xn_ = dmalloc<uint16_t>(T * H);
    qkv_ = dmalloc<uint16_t>(T * (hq + 2 * hk) * d);
    q_ = dmalloc<uint16_t>(T * hq * d);
    attn_ = dmalloc<uint16_t>(T * hq * d);
    gu_ = dmalloc<uint16_t>(T * 2 * I);
    if (model_.is_moe()) {
        // one row per route (token, k): expert activations and per-route outputs, the router
        // logits, and the grouped layout the routing kernel builds
        const size_t R = T * m.top_k;
        act_ = dmalloc<uint16_t>(R * I);
        moe_y_ = dmalloc<uint16_t>(R * H);
        moe_logits_ = dmalloc<uint16_t>(T * m.num_experts);
        moe_idx_ = dmalloc<int32_t>(R);
        moe_w_ = dmalloc<float>(R);
        moe_offsets_ = dmalloc<int32_t>(m.num_experts + 1);
        moe_route_token_ = dmalloc<int32_t>(R);
        moe_route_pos_ = dmalloc<int32_t>(R);
    } else {
        act_ = dmalloc<uint16_t>(T * I);
    }
    rope_tab_ = dmalloc<float>(T * d);
    const size_t srows = std::min<size_t>(T, 2 * static_cast<size_t>(cfg_.batching.max_forward_requests));
    xs_ = dmalloc<uint16_t>(srows * H);
    logits_ = dmalloc<uint16_t>(srows * m.vocab);
    amax_ws_bytes_ = pie_hip_lm_head_argmax_workspace_bytes(4, m.vocab);
    if (amax_ws_bytes_) PIE_HIP_CHECK(hipMalloc(&amax_ws_, amax_ws_bytes_));
    // Bound of the split-K partial buffers over every (rows, context) the planner can pick:
    // rows * splits <= 3072/hk + rows.
    attn_ws_bytes_ = (3072 / static_cast<size_t>(hk) + 1 + T) * hq * (d + 2) * sizeof(float);
    PIE_HIP_CHECK(hipMalloc(&attn_ws_, attn_ws_bytes_));
    if (kv_format_ != PIE_HIP_KV_BF16) {
        k_rows_ = dmalloc<uint16_t>(T * hk * d);
        v_rows_ = dmalloc<uint16_t>(T * hk * d);
        iota_slots_ = dmalloc<int64_t>(T);
        std::vector<int64_t> iota(T);
        for (size_t i = 0; i < T; ++i) iota[i] = static_cast<int64_t>(i);
        PIE_HIP_CHECK(hipMemcpy(iota_slots_, iota.data(), T * sizeof(int64_t), hipMemcpyHostToDevice));
    }
    // fp32 partials of the split-K GEMM for decode batches of up to 128 rows (dense layers) and of prompts' K shares
    if (!model_.layers.empty()) {
        const LayerWeights& l0 = model_.layers[0];
        for (const Linear* w : {&l0.wqkv, &l0.wo, &l0.wgu, &l0.wdown})
            for (int rows : {64, 128})
                if (w->data && w->K % 64 == 0)
                    gemm_ws_bytes_ = std::max(gemm_ws_bytes_, pie_hip_gemm_mfma_workspace_bytes(rows, w->N, w->K));
        gemm_ws_bytes_ = std::min<size_t>(gemm_ws_bytes_, size_t(64) << 20);
        for (const Linear* w : {&l0.wqkv, &l0.wo, &l0.router, m.num_experts ? &l0.wo : &l0.wgu, m.num_experts ? &l0.wo : &l0.wdown})
            if (w->data)
                gemm_ws_bytes_ = std::max(gemm_ws_bytes_, pie_hip_gemm_mfma_tiled_workspace_bytes(static_cast<int>(T), w->N, w->K));
        if (gemm_ws_bytes_) PIE_HIP_CHECK(hipMalloc(&gemm_ws_, gemm_ws_bytes_));
    }
}

Executor::~Executor() {
    if (stream_) (void)hipStreamSynchronize(stream_);
    for (auto& kv : graphs_) (void)hipGraphExecDestroy(kv.second);
    for (const PagePool& p : page_pools_) (void)hipFree(p.base);
    for (void* p : stack_.allocs) (void)hipFree(p);
    if (rs_base_) (void)hipFree(rs_base_);
    if (rs_host_) (void)hipHostFree(rs_host_);
    for (void* p : {static_cast<void*>(x_), static_cast<void*>(xn_), static_cast<void*>(qkv_),
                    static_cast<void*>(q_), static_cast<void*>(attn_), static_cast<void*>(gu_),
                    static_cast<void*>(act_), static_cast<void*>(xs_), static_cast<void*>(logits_),
                    static_cast<void*>(rope_tab_), static_cast<void*>(out_tokens_), attn_ws_, gemm_ws_, amax_ws_,
                    static_cast<void*>(in_dev_), static_cast<void*>(copy_ids_),
                    static_cast<void*>(moe_y_), static_cast<void*>(moe_logits_),
                    static_cast<void*>(moe_idx_), static_cast<void*>(moe_w_),
                    static_cast<void*>(moe_offsets_), static_cast<void*>(moe_route_token_),
                    static_cast<void*>(moe_route_pos_), static_cast<void*>(k_rows_),
                    static_cast<void*>(v_rows_), static_cast<void*>(iota_slots_)})
        if (p) (void)hipFree(p);
    if (kv_shadow_k_) (void)hipFree(kv_shadow_k_);
    if (kv_shadow_v_) (void)hipFree(kv_shadow_v_);
    for (Growable* g : {&mask_in_host_, &mask_in_dev_, &mask_bitmap_, &tile_in_host_, &tile_in_dev_, &expand_lat_, &expand_rot_,
                        &expand_kv_, &list_host_, &list_dev_, &record_ws_}) g->release();
    for (Growable* g : {&samp_f32_, &samp_ws_, &samp_in_dev_, &samp_in_host_, &samp_out_dev_, &samp_out_host_})
        g->release();
    if (swap_pool_) (void)hipHostFree(swap_pool_);
    if (in_host_) (void)hipHostFree(in_host_);
    if (out_host_) (void)hipHostFree(out_host_);
    if (stream_) (void)hipStreamDestroy(stream_);
}

// Page sizes of the storage formats: kv_bytes_per_page / scale_bytes_per_page,
// driver/cuda/src/kv_cache_format.cpp:27-49.
size_t Executor::page_bytes() const {
    const ModelConfig& m = model_.cfg();
    const size_t elems = static_cast<size_t>(page_size_) * m.kv_heads * m.head_dim;
    if (kv_format_ == PIE_HIP_KV_FP4_BLOCK) return elems / 2;   // two codes per byte
    return elems * (kv_format_ == PIE_HIP_KV_BF16 ? 2 : 1);
}
size_t Executor::scale_page_bytes() const {
    const ModelConfig& m = model_.cfg();
    if (kv_format_ == PIE_HIP_KV_FP4_BLOCK)   // one scale per block of 16 elements
        return static_cast<size_t>(page_size_) * m.kv_heads * ((m.head_dim + 15) / 16) * sizeof(float);
    const bool scaled = kv_format_ == PIE_HIP_KV_INT8_PER_TOKEN_HEAD || kv_format_ == PIE_HIP_KV_FP8_PER_TOKEN_HEAD;
    return scaled ? static_cast<size_t>(page_size_) * m.kv_heads * sizeof(float) : 0;
}

// Start-up measurement of the decoder linears' candidate kernels.  For every role (q|k|v, wo,
// gate|up, down) and a ladder of row counts the GEMV (2-4 rows), the skinny GEMM and the tiled GEMM
// (17-128 rows; in K shares where the workspace allows; over the tile-major copy where the model expects that) run over the weights of successive layers
// (so that they come from HBM, as in a forward pass) on zeroed activations; the fastest goes into
// every layer's table for the row counts up to the next rung.
void Executor::tune_linears() {
    const ModelConfig& m = model_.cfg();
    if (model_.layers.empty() || !cfg_.runtime.tune_linears || getenv("PIE_NO_TUNE")) return;
    hipStream_t s = stream_;
    const size_t T = static_cast<size_t>(max_tokens_);
    const int H = m.hidden, d = m.head_dim, hq = m.q_heads, hk = m.kv_heads;
    const int I = model_.is_moe() ? m.expert_intermediate : m.intermediate;
    PIE_HIP_CHECK(hipMemsetAsync(x_, 0, T * H * 2, s));
    PIE_HIP_CHECK(hipMemsetAsync(attn_, 0, T * hq * d * 2, s));
    if (!model_.is_moe()) PIE_HIP_CHECK(hipMemsetAsync(act_, 0, T * I * 2, s));
    struct Role {
        Linear LayerWeights::*lin;
        uint16_t* LayerWeights::*norm;
        const uint16_t* act;
        uint16_t* y;
        int beta, swiglu;
        double tiled_handicap_us;   // what the tiled route costs beyond the GEMM (a separate RoPE launch)
    };
    std::vector<Role> roles = {
        {&LayerWeights::wqkv, &LayerWeights::attn_norm, x_, qkv_, 0, 0, 4.0},
        {&LayerWeights::wo, nullptr, attn_, x_, 1, 0, 0.0},
    };
    if (!model_.is_moe()) {
        roles.push_back({&LayerWeights::wgu, &LayerWeights::ffn_norm, x_, act_, 0, 1, 0.0});
        roles.push_back({&LayerWeights::wdown, nullptr, act_, x_, 1, 0, 0.0});
    }
    hipEvent_t e0 = nullptr, e1 = nullptr;
    PIE_HIP_CHECK(hipEventCreate(&e0));
    PIE_HIP_CHECK(hipEventCreate(&e1));
    const int L = static_cast<int>(model_.layers.size());
    int rot = 0;
    // (the smaller of two timed rounds: a round disturbed by something else on the machine would
    // otherwise decide the dispatch for the life of the process)
    auto time_us = [&](auto&& launch) -> double {   // launch(layer): false where it does not take the shape
        constexpr int kWarm = 1, kReps = 4, kRounds = 2;
        double best = 1e30;
        for (int round = 0; round < kRounds; ++round) {
            for (int i = 0; i < kWarm + kReps; ++i) {
                if (i == kWarm) PIE_HIP_CHECK(hipEventRecord(e0, s));
                if (!launch(model_.layers[static_cast<size_t>(rot++ % L)])) return 1e30;
            }
            PIE_HIP_CHECK(hipEventRecord(e1, s));
            PIE_HIP_CHECK(hipEventSynchronize(e1));
            float ms = 0.f;
            PIE_HIP_CHECK(hipEventElapsedTime(&ms, e0, e1));
            best = std::min(best, static_cast<double>(ms) * 1e3 / kReps);
        }
        return best;
    };
    auto time_route = [&](const Role& r, int M, int force) {
        return time_us([&](LayerWeights& lw) {
            const uint16_t* nw = r.norm ? lw.*(r.norm) : nullptr;
            return linear_fused(lw.*(r.lin), r.act, nw, m.rms_eps, r.y, M, r.beta, r.swiglu, xn_, gemm_ws_, gemm_ws_bytes_, s, force);
        });
    };
    // A measurement overrides the cost model only where it is clearly faster (a tenth and
    // half a microsecond): candidates that tie keep the model's kernel, so that timing noise
    // does not change which kernel — and with it which rounding — a restart gets.
    auto clearly = [](double us, double than) { return us < 0.9 * than && us + 0.5 < than; };
    const int ladder[] = {2, 3, 4, 17, 24, 32, 33, 40, 48, 56, 64, 65, 72, 80, 88, 96, 97, 104, 112, 120, 128};
    for (const Role& r : roles) {
        const Linear& l0 = model_.layers[0].*(r.lin);
        if (!l0.data || !l0.data_tiled) continue;   // (without the tile-major copy the cost model's defaults stand)
        int prev = 1;
        // llama-type layers send two to four decode rows of q|k|v to the GEMV with the RoPE
        // epilogue whatever a measurement says (Executor::body): those rungs would decide nothing
        const bool qkv_fused_rows = r.lin == &LayerWeights::wqkv && !model_.layers[0].q_norm &&
                                    (m.rope_interleaved || model_.qk_rows_paired()) && (d & (d - 1)) == 0 &&
                                    kv_format_ == PIE_HIP_KV_BF16;
        for (int M : ladder) {
            if (M > max_tokens_) break;
            if (M <= 4 && qkv_fused_rows) {
                prev = M;
                continue;
            }
            // rows 5..16 stay with the skinny GEMM; a rung decides for the row counts above the
            // previous rung up to itself
            const int lo = M <= 4 ? M : std::max(prev + 1, 17);
            auto set = [&](std::array<int8_t, 129> Linear::*table, int value, int from) {
                for (auto& lw : model_.layers)
                    for (int mm = from; mm <= M; ++mm) (lw.*(r.lin).*table)[static_cast<size_t>(mm)] = static_cast<int8_t>(value);
            };
            // int4 weights where the skinny GEMM is chosen: its passes, or the blocks that scale groups in fp32
            double skinny_t = 1e30;
            if (groups_cost(l0, M, gemm_ws_bytes_) < 1e29) {
                int form = in_groups(l0, M, gemm_ws_bytes_) ? 1 : 0;
                if (measures_groups(l0, M, gemm_ws_bytes_)) {
                    double us[2];
                    for (int f = 0; f < 2; ++f) {
                        set(&Linear::groups, f, M);
                        us[f] = time_route(r, M, 1);
                    }
                    if (clearly(us[1 - form], us[form])) form = 1 - form;
                    skinny_t = us[form];
                }
                set(&Linear::groups, form, lo);
            }
            int best = -1;
            double best_t = 1e30, model_t = 1e30;
            const int by_model = model_route(l0, M, r.norm != nullptr, gemm_ws_bytes_);
            for (int cand = M <= 4 ? 0 : 1; cand <= (M <= 4 ? 1 : 4); ++cand) {
                if (cand == 4 && by_model != 4) continue;   // (far slower where the model does not expect it)
                if (cand == 2 && by_model != 2 && l0.kind == Quant::Int4b8 && l0.data_tiled && tiled_cost(l0, M) > 2.0 * passes_cost(l0, M)) continue;   // (likewise)
                if (cand == 3 && (M > 128 || pie_hip_gemm_mfma_workspace_bytes(M, l0.N, l0.K) == 0 ||
                                  pie_hip_gemm_mfma_workspace_bytes(M, l0.N, l0.K) > gemm_ws_bytes_))
                    continue;
                if (cand >= 2 && l0.K % 64 != 0) continue;
                double t = cand == 1 && skinny_t < 1e29 ? skinny_t : time_route(r, M, cand);
                // (up to 48 rows of int4 weights the wide GEMM's form has the rotation in its epilogue too)
                if (cand >= 2 && !(cand == 4 && l0.kind == Quant::Int4b8 && M <= 48)) t += r.tiled_handicap_us;
                if (cand == by_model) model_t = t;
                if (t < best_t) {
                    best_t = t;
                    best = cand;
                }
            }
            if (model_t < 1e29 && !clearly(best_t, model_t)) best = by_model;
            if (best >= 0) set(&Linear::tuned, best, lo);
            // the projections into the residual: this route and the norm behind it, or shares of K that meet in the norm
            const bool residual = r.beta && !model_.is_moe();
            const double shares = residual ? shares_cost(l0, M, gemm_ws_bytes_) : 1e30;
            if (best >= 0 && shares < 1e29) {
                int form = in_shares(l0, M, gemm_ws_bytes_) ? 1 : 0;
                if (measures_shares(l0, M, gemm_ws_bytes_, best == by_model)) {
                    double us[2];
                    us[0] = (best == by_model ? model_t : best_t) + time_us([&](LayerWeights& lw) { return pie_hip_rmsnorm(x_, lw.ffn_norm, xn_, M, H, m.rms_eps, s) == PIE_HIP_OK; });
                    us[1] = time_us([&](LayerWeights& lw) { return project_in_shares(lw.*(r.lin), r.act, lw.ffn_norm, M); });
                    if (clearly(us[1 - form], us[form])) form = 1 - form;
                }
                set(&Linear::shares, form, lo);
            }
            prev = M;
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    PIE_HIP_CHECK(hipStreamSynchronize(s));
}

// Allocate the pools; on out-of-memory halve the page count down to 64 pages
// (driver/portable/src/entry.cpp:327-348).
void Executor::alloc_kv() {
    while (!alloc_pools()) {
        (void)hipGetLastError();
        if (total_pages_ <= 64) throw std::runtime_error("executor: cannot allocate the KV pool");
        total_pages_ = std::max(64, total_pages_ / 2);
    }
    size_t off = 0;
    for (PagePool& p : page_pools_) {
        p.host_off = off;
        off += p.page_bytes;
        // Pages start zeroed so slots no request has written hold finite values.
        PIE_HIP_CHECK(hipMemsetAsync(p.base, 0, p.page_bytes * static_cast<size_t>(total_pages_), stream_));
    }
    swap_page_bytes_ = off;
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
}

bool Executor::alloc_pools() {
    const ModelConfig& m = model_.cfg();
    auto pool = [&](size_t bytes_per_page) -> unsigned char* {
        void* p = nullptr;
        if (hipMalloc(&p, bytes_per_page * static_cast<size_t>(total_pages_)) != hipSuccess) return nullptr;
        page_pools_.push_back({static_cast<unsigned char*>(p), bytes_per_page, 0});
        return static_cast<unsigned char*>(p);
    };
    auto give_up = [&] {
        for (const PagePool& p : page_pools_) (void)hipFree(p.base);
        page_pools_.clear();
        k_pool_.clear();
        v_pool_.clear();
        k_scale_pool_.clear();
        v_scale_pool_.clear();
        run_pool_.clear();
        return false;
    };
    if (m.is_stack()) {
        for (const LayerRun& run : m.layer_runs()) {   // every pass of a looped layer has its own
            const LayerSpec& l = m.stack[static_cast<size_t>(run.layer)];
            if (l.mixer == MixerKind::LatentAttention && l.latent.kv_from >= 0) {   // (without loops layers are runs)
                run_pool_.push_back(run_pool_[static_cast<size_t>(l.latent.kv_from)]);
                continue;
            }
            run_pool_.push_back(nullptr);
            const int row = l.mixer == MixerKind::LatentAttention ? LatentShape(l.latent).ld_row
                            : l.has_attn()                        ? l.attn.kv_heads * 2 * pad_head(l.attn.widest())
                                                                  : 0;
            if (row == 0) continue;
            const size_t esize = m.f32() ? 4 : 2;
            run_pool_.back() = pool(static_cast<size_t>(page_size_) * row * esize);
            if (!run_pool_.back()) return give_up();
        }
        return true;
    }
    for (int l = 0; l < m.layers; ++l) {
        unsigned char* k = pool(page_bytes());
        unsigned char* v = k ? pool(page_bytes()) : nullptr;
        if (!v) return give_up();
        k_pool_.push_back(reinterpret_cast<uint16_t*>(k));
        v_pool_.push_back(reinterpret_cast<uint16_t*>(v));
        if (scale_page_bytes()) {
            k = pool(scale_page_bytes());
            v = k ? pool(scale_page_bytes()) : nullptr;
            if (!v) return give_up();
            k_scale_pool_.push_back(reinterpret_cast<float*>(k));
            v_scale_pool_.push_back(reinterpret_cast<float*>(v));
        }
    }
    if (kv_format_ == PIE_HIP_KV_FP4_BLOCK) {
        // the bf16 pages the attention kernels read (k_bf16_pages / v_bf16_pages of the
        // reference's layer view, driver/cuda/src/kernels/kv_paged.cu:698-770)
        const size_t shadow = static_cast<size_t>(total_pages_) * page_size_ * m.kv_heads * m.head_dim * 2;
        void *k = nullptr, *v = nullptr;
        if (hipMalloc(&k, shadow) != hipSuccess || hipMalloc(&v, shadow) != hipSuccess) {
            if (k) (void)hipFree(k);
            return give_up();
        }
        kv_shadow_k_ = static_cast<uint16_t*>(k);
        kv_shadow_v_ = static_cast<uint16_t*>(v);
        PIE_HIP_CHECK(hipMemsetAsync(kv_shadow_k_, 0, shadow, stream_));
        PIE_HIP_CHECK(hipMemsetAsync(kv_shadow_v_, 0, shadow, stream_));
    }
    return true;
}

bool Executor::few_in_blocks(Quant kind, long long routes, int experts, int hidden, int inner) {
    if ((kind != Quant::Int8 && kind != Quant::Fp8) || grouped_in_blocks(kind, routes, experts)) return false;
    auto both = [&](int blocks) {
        return pie_hip_moe_few_routes_us(fmt_code(kind), static_cast<int>(routes), experts, 2 * inner, hidden, 1, blocks) +
               pie_hip_moe_few_routes_us(fmt_code(kind), static_cast<int>(routes), experts, hidden, inner, 0, blocks);
    };
    return 1.03f * both(1) < both(0);
}

// Up to 256 tokens may take one launch, whose blocks, one per token, each read all of the router through their CU's L2 port; blocks of shares of K read
// it once for 32 tokens, in a launch more for the norm and one for the choice.  So one launch is better for few experts or few values, and longer the
// more tokens there are.  us in one launch / in shares: 8 experts of 2048 9.5 / 11.3; 48 of 2048, 8 and 64 tokens 11.4 / 11.2, 11.7 / 13.3; 64 of 4096, 8 and 128 15.1 / 13.3, 15.8 / 16.4; 96 of
// 2048, 8 and 128 14.2 / 12.4, 15.1 / 15.3; 128 of 1024, 8 and 64 14.2 / 12.5, 14.0 / 14.7; 96 of 4096, 128 18.9 / 17.7; 128 of 2048, 1, 64 and 256 15.8 / 11.7, 16.5 / 15.1, 18.9 / 17.0; 256 of 2048, 64 26.4 / 17.4.
// The more tiles of 32 tokens and 128 experts a prompt has, the fewer shares each gets (512 blocks in all), and the longer a block waits for its steps one
// by one; a product, which keeps its loads in flight, is then better, sooner with a long K and with tiles of few experts.  us in shares / as a product and the choice:
// 128 of 2048, 1237 tokens and 8192 25.9 / 36.3, 121.5 / 123.8; 256 of 2048, 4096 and 6000 76.6 / 79.9, 110.3 / 104.6; 384 of 2048, 2048 and 4096 42.1 / 45.7, 87.1 / 82.7; 32 of 4096, 8192 112.2 / 116.3;
// 128 of 4096, 4096 and 6000 76.0 / 79.6, 109.8 / 106.2; 256 of 7168, 2048 and 6000 52.2 / 54.4, 178.2 / 144.9; 8 of 4096, 2048 and 6000 24.4 / 26.2, 45.2 / 42.3.
Executor::RouteForm Executor::route_form(Quant router, int tokens, int hidden, int experts, size_t workspace_bytes) {
    if (router != Quant::Bf16) return RouteForm::Product;
    const size_t share = pie_hip_moe_router_workspace_bytes(tokens, hidden, experts);
    const bool shares = share > 0 && share <= workspace_bytes;
    const long long values = static_cast<long long>(experts) * hidden;
    if (tokens <= 256) {
        int most = 12;   // tokens of a batch that is better in shares
        if (experts < 48 || values < 48 * 2048) most = 0;
        else if (experts < 64) most = 8;
        else if (values > 128 * 1024 && (experts >= 112 || (experts >= 80 && hidden >= 4096))) most = 256;
        return shares && tokens <= most ? RouteForm::Shares : RouteForm::InOne;
    }
    const long long tiles = (tokens + 31ll) / 32 * ((experts + 127) / 128);
    const int most = hidden <= 2048 ? 256 : experts <= 8 ? 64 : experts <= 64 ? 256 : 128;
    return shares && tiles <= most ? RouteForm::Shares : RouteForm::Product;
}

// x += sum_k w_k * down_e(swiglu(gate_up_e(norm(x)))) over each token's top-k experts
// (driver/portable/src/graph_common.cpp:237-345; kernel-by-kernel form
// driver/cuda/src/model/kimi_forward.cpp:662-714): norm, router GEMM, one routing kernel, two
// grouped expert GEMMs that read every touched expert once, one combine onto the residual.
void Executor::moe_block(const LayerWeights& w, int N, const uint16_t* next_norm, hipStream_t s) {
    const ModelConfig& m = model_.cfg();
    const int H = m.hidden, E = m.num_experts, K = m.top_k, Ie = m.expert_intermediate;
    const int fmt = fmt_code(w.wgu.kind);
    const int sbf = w.wgu.scale_bf16 ? 1 : 0;
    // (PIE_MOE_FUSED=0: the separate launches, for measurement)
    static const bool fused_on = [] { const char* e = getenv("PIE_MOE_FUSED"); return !e || atoi(e) != 0; }();
    if (!fused_on) next_norm = nullptr;
    const RouteForm form = fused_on ? route_form(w.router.kind, N, H, E, gemm_ws_bytes_) : RouteForm::Product;
    int routed = PIE_HIP_ERR_UNSUPPORTED;
    if (form == RouteForm::InOne)
        routed = pie_hip_moe_norm_route(x_, w.ffn_norm, m.rms_eps, static_cast<const uint16_t*>(w.router.data), xn_, moe_logits_, moe_idx_, moe_w_,
                                        moe_offsets_, moe_route_token_, moe_route_pos_, N, H, E, K, m.norm_topk ? 1 : 0, s);
    if (routed == PIE_HIP_ERR_UNSUPPORTED) {
        PIE_KERNEL(pie_hip_rmsnorm(x_, w.ffn_norm, xn_, N, H, m.rms_eps, s));
        if (form == RouteForm::Shares)   // (their sums in the products' workspace)
            routed = pie_hip_moe_router_route(xn_, static_cast<const uint16_t*>(w.router.data), moe_logits_, moe_idx_, moe_w_, moe_offsets_,
                                              moe_route_token_, moe_route_pos_, N, H, E, K, m.norm_topk ? 1 : 0, gemm_ws_, gemm_ws_bytes_, s);
        if (routed == PIE_HIP_ERR_UNSUPPORTED) {
            linear_fused(w.router, xn_, nullptr, m.rms_eps, moe_logits_, N, 0, 0, nullptr, gemm_ws_, gemm_ws_bytes_, s);
            routed = pie_hip_moe_route_opt(moe_logits_, moe_idx_, moe_w_, moe_offsets_, moe_route_token_, moe_route_pos_, N, E, K, m.norm_topk ? 1 : 0, s);
        }
    }
    PIE_KERNEL(routed);
    const int hint = std::max(1, std::min(N, 2 * ((N * K + E - 1) / E)));
    // experts stacked along the rows: the tile-major copy of the stack keeps expert e at the same
    // byte stride (every expert has a multiple of 16 rows)
    const bool tiled = w.wgu.data_tiled && w.wdown.data_tiled && (2 * Ie) % 16 == 0 && H % 16 == 0;
    auto grouped = tiled ? pie_hip_moe_grouped_gemm_tiled : pie_hip_moe_grouped_gemm;
    auto wptr = [&](const Linear& l) { return tiled ? l.data_tiled : l.data; };
    auto sptr = [&](const Linear& l) { return tiled && l.scale_tiled ? l.scale_tiled : l.scale; };
    // many routes per expert (a prompt's tokens): blocks of an expert's routes on the tiled GEMM (widths that the passes
    // refuse stay refused); one-byte tile-major weights take smaller blocks for few routes too, by an estimate
    const int unit = w.wgu.kind == Quant::Bf16 ? 64 : 256;
    const bool fits = H % unit == 0 && Ie % unit == 0;
    bool done = false;
    if (grouped_in_blocks(w.wgu.kind, N * K, E) || (tiled && few_in_blocks(w.wgu.kind, N * K, E, H, Ie))) {
        auto blocks = [&](const Linear& l, const uint16_t* act, const int32_t* rows, uint16_t* y, int rows_out, int cols, int epilogue) {
            return pie_hip_moe_grouped_gemm_mfma_fmt(fmt, act, rows, moe_offsets_, E, N * K, wptr(l), l.data_bytes() / E, l.scale,
                                                     l.scale_bytes() / E, sbf, l.group, y, rows_out, cols, epilogue, tiled ? 1 : 0,
                                                     nullptr, 0, s);
        };
        const int st = fits ? blocks(w.wgu, xn_, moe_route_token_, act_, 2 * Ie, H, PIE_HIP_EPI_SWIGLU) : PIE_HIP_ERR_UNSUPPORTED;
        if (st == PIE_HIP_OK) {
            PIE_KERNEL(blocks(w.wdown, act_, nullptr, moe_y_, H, Ie, PIE_HIP_EPI_NONE));
            done = true;
        } else if (st != PIE_HIP_ERR_UNSUPPORTED) {
            PIE_KERNEL(st);
        }
    }
    if (!done) {
        PIE_KERNEL(grouped(fmt, xn_, moe_route_token_, moe_offsets_, E, hint, wptr(w.wgu),
                           w.wgu.data_bytes() / E, sptr(w.wgu), w.wgu.scale_bytes() / E, sbf, w.wgu.group,
                           act_, 2 * Ie, H, 1, s));
        PIE_KERNEL(grouped(fmt, act_, nullptr, moe_offsets_, E, hint, wptr(w.wdown), w.wdown.data_bytes() / E,
                           sptr(w.wdown), w.wdown.scale_bytes() / E, sbf, w.wdown.group, moe_y_, H, Ie, 0, s));
    }
    // with the next layer's attention norm riding along when that layer takes its rows normalised
    int combined = PIE_HIP_ERR_UNSUPPORTED;
    if (next_norm)
        combined = pie_hip_moe_combine_norm(moe_y_, moe_route_pos_, moe_w_, x_, next_norm, m.rms_eps, xn_, N, K, H, s);
    if (combined == PIE_HIP_ERR_UNSUPPORTED) {
        PIE_KERNEL(pie_hip_moe_combine(moe_y_, moe_route_pos_, moe_w_, x_, N, K, H, 1, s));
        xn_holds_next_norm_ = false;
    } else {
        PIE_KERNEL(combined);
        xn_holds_next_norm_ = true;
    }
}

// x_ += act · W^T in shares of K that meet in the kernel of the norm, whose rows go to xn_; false where the shape is not taken.
bool Executor::project_in_shares(const Linear& w, const uint16_t* act, const uint16_t* norm, int N) {
    const ModelConfig& m = model_.cfg();
    int shares = 0;
    const bool waves = waves_shares_cost(w, N, gemm_ws_bytes_) < groups_shares_cost(w, N, gemm_ws_bytes_);
    const int st = waves ? pie_hip_gemm_waves_shares(fmt_code(w.kind), act, w.data_tiled, w.scale_tiled ? w.scale_tiled : w.scale, w.scale_bf16 ? 1 : 0, w.group, N,
                                                     w.N, w.K, gemm_ws_, gemm_ws_bytes_, &shares, stream_)
                         : pie_hip_gemm_groups_shares(act, w.data_tiled, w.scale_tiled, w.group, N, w.N, w.K, gemm_ws_, gemm_ws_bytes_, &shares, stream_);
    if (st == PIE_HIP_ERR_UNSUPPORTED) return false;
    PIE_KERNEL(st);
    PIE_KERNEL(pie_hip_shares_rmsnorm(static_cast<const float*>(gemm_ws_), shares, x_, norm, xn_, N, m.hidden, m.rms_eps, stream_));
    return true;
}

void Executor::body(int N, int S, int max_kv_len) {
    if (model_.cfg().is_stack()) return stack_body(N, S, max_kv_len);
    xn_holds_next_norm_ = false;
    const Inputs in_ = input_layout(N, S);
    const ModelConfig& m = model_.cfg();
    const int H = m.hidden, d = m.head_dim, hq = m.q_heads, hk = m.kv_heads;
    hipStream_t s = stream_;
    const auto* tokens = reinterpret_cast<const uint32_t*>(in_dev_ + in_.off_tokens);
    const auto* positions = reinterpret_cast<const int32_t*>(in_dev_ + in_.off_positions);
    const auto* slots = reinterpret_cast<const int64_t*>(in_dev_ + in_.off_slots);
    const auto* row_begin = reinterpret_cast<const uint32_t*>(in_dev_ + in_.off_row_begin);
    const auto* row_len = reinterpret_cast<const int32_t*>(in_dev_ + in_.off_row_len);
    const auto* sample_rows = reinterpret_cast<const uint32_t*>(in_dev_ + in_.off_sample_rows);
    const auto* pages = reinterpret_cast<const uint32_t*>(in_dev_ + in_.off_pages);

    PIE_KERNEL(pie_hip_embed(tokens, model_.embed, x_, N, H, m.vocab, s));
    PIE_KERNEL(pie_hip_rope_table_scaled(positions, model_.inv_freq, rope_tab_, N, d, rope_mscale(m), s));
    // RoPE pairing as the rotation kernels take it: adjacent pairs, half-split pairs, or
    // half-split pairs over projection rows re-ordered at load (then the fused epilogues apply)
    const int pairing = m.rope_interleaved ? PIE_HIP_ROPE_ADJACENT
                        : model_.qk_rows_paired() ? PIE_HIP_ROPE_HALF_PAIRED_ROWS : PIE_HIP_ROPE_HALF;
    const bool fused_rope = pairing != PIE_HIP_ROPE_HALF && (d & (d - 1)) == 0;
    for (int l = 0; l < m.layers; ++l) {
        const LayerWeights& w = model_.layers[l];
        const bool kvq = kv_format_ != PIE_HIP_KV_BF16;
        float* ksc = kvq && !k_scale_pool_.empty() ? k_scale_pool_[l] : nullptr;
        float* vsc = kvq && !v_scale_pool_.empty() ? v_scale_pool_[l] : nullptr;
        // (the previous layer's MoE combine or down projection may have left this layer's normalised rows in xn_)
        const bool prenormed = xn_holds_next_norm_;
        xn_holds_next_norm_ = false;
        if (kvq) {
            // one-byte pools: the rotated K / V rows of this step are staged as bf16 rows (row t
            // in "slot" t) and quantised into the tokens' real slots
            linear_fused(w.wqkv, prenormed ? xn_ : x_, prenormed ? nullptr : w.attn_norm, m.rms_eps, qkv_, N, 0, 0, xn_,
                         gemm_ws_, gemm_ws_bytes_, s);
            // rotation and quantising write in one launch; head dims past 256 take the two kernels
            const int st = pie_hip_qkv_rope_kvwrite_quant(kv_format_, qkv_, q_, k_pool_[l], v_pool_[l], ksc, vsc,
                                                          w.q_norm, w.k_norm, rope_tab_, slots, N, hq, hk, d,
                                                          page_size_, pairing, m.rms_eps, s);
            if (st == PIE_HIP_ERR_UNSUPPORTED) {
                PIE_KERNEL(pie_hip_qkv_rope_kvwrite(qkv_, q_, k_rows_, v_rows_, w.q_norm, w.k_norm, rope_tab_,
                                                    iota_slots_, N, hq, hk, d, pairing, m.rms_eps, s));
                PIE_KERNEL(pie_hip_kv_write_quant(kv_format_, k_rows_, v_rows_, slots, k_pool_[l], v_pool_[l],
                                                  ksc, vsc, N, hk, d, page_size_, s));
            } else {
                PIE_KERNEL(st);
            }
        } else {
            // decode rows of llama-type layers: rotation and KV write ride in the projection
            // (a hidden size past the GEMV's staged-activation limit takes the general route)
            int fused_st = PIE_HIP_ERR_UNSUPPORTED;
            if (N <= 4 && fused_rope && !w.q_norm) {
                fused_st = pie_hip_qkv_rope_fused(fmt_code(w.wqkv.kind), x_, w.attn_norm, m.rms_eps, w.wqkv.data,
                                                  w.wqkv.scale, w.wqkv.scale_bf16 ? 1 : 0, w.wqkv.group, N, H,
                                                  rope_tab_, slots, q_, k_pool_[l], v_pool_[l], hq, hk, d,
                                                  pairing, s);
                if (fused_st != PIE_HIP_OK && fused_st != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(fused_st);
            }
            if (fused_st != PIE_HIP_OK) {
            // a decode batch of llama-type layers on the skinny GEMM: rotation and KV write ride
            // in its epilogue too (one launch less per layer)
            bool done = false;
            const int tuned_qkv = N <= 128 ? w.wqkv.tuned[N] : -1;
            const GemmPath path = tuned_qkv < 0 ? pick_gemm(w.wqkv, N, gemm_ws_bytes_) : tuned_qkv <= 1 ? GemmPath::Skinny : tuned_qkv == 4 ? GemmPath::Wide : GemmPath::Tiled;
            const bool waves = path == GemmPath::Skinny && in_waves(w.wqkv, N, gemm_ws_bytes_), groups = !waves && in_groups(w.wqkv, N, gemm_ws_bytes_);
            if (fused_rope && !w.q_norm && w.wqkv.data_tiled && (path == GemmPath::Skinny || (path == GemmPath::Wide && groups && N <= 48))) {
                if (!prenormed) PIE_KERNEL(pie_hip_rmsnorm(x_, w.attn_norm, xn_, N, H, m.rms_eps, s));
                const int st =
                    waves ? pie_hip_qkv_rope_waves_tiled(fmt_code(w.wqkv.kind), xn_, w.wqkv.data_tiled, w.wqkv.scale_tiled ? w.wqkv.scale_tiled : w.wqkv.scale,
                                                         w.wqkv.scale_bf16 ? 1 : 0, w.wqkv.group, N, H, rope_tab_, slots, q_, k_pool_[l], v_pool_[l], hq, hk, d,
                                                         pairing, gemm_ws_, gemm_ws_bytes_, s)
                    : groups
                        ? pie_hip_qkv_rope_groups_tiled(xn_, w.wqkv.data_tiled, w.wqkv.scale_tiled, w.wqkv.group, N, H, rope_tab_, slots, q_,
                                                        k_pool_[l], v_pool_[l], hq, hk, d, pairing, gemm_ws_, gemm_ws_bytes_, s)
                        : pie_hip_qkv_rope_skinny_tiled(fmt_code(w.wqkv.kind), xn_, w.wqkv.data_tiled,
                                                        w.wqkv.scale_tiled ? w.wqkv.scale_tiled : w.wqkv.scale, w.wqkv.scale_bf16 ? 1 : 0,
                                                        w.wqkv.group, N, H, rope_tab_, slots, q_, k_pool_[l], v_pool_[l], hq, hk, d,
                                                        pairing, s);
                if (st == PIE_HIP_OK) done = true;
                else if (st != PIE_HIP_ERR_UNSUPPORTED) PIE_KERNEL(st);
            }
            if (!done) {
                linear_fused(w.wqkv, prenormed ? xn_ : x_, prenormed ? nullptr : w.attn_norm, m.rms_eps, qkv_, N, 0, 0,
                             xn_, gemm_ws_, gemm_ws_bytes_, s);
                PIE_KERNEL(pie_hip_qkv_rope_kvwrite(qkv_, q_, k_pool_[l], v_pool_[l], w.q_norm, w.k_norm,
                                                    rope_tab_, slots, N, hq, hk, d, pairing, m.rms_eps, s));
            }
            }
        }
        // 4-bit blocks: the pages this batch reads become bf16 in the shared pool pair, which the
        // bf16 attention kernels then read under the same page ids
        const bool fp4 = kv_format_ == PIE_HIP_KV_FP4_BLOCK;
        if (fp4)
            PIE_KERNEL(pie_hip_kv_dequant_pages(kv_format_, k_pool_[l], v_pool_[l], ksc, vsc, kv_shadow_k_,
                                                kv_shadow_v_, pages, n_page_refs_, hk, d, page_size_, s));
        const uint16_t* kat = fp4 ? kv_shadow_k_ : k_pool_[l];
        const uint16_t* vat = fp4 ? kv_shadow_v_ : v_pool_[l];
        const bool kvq_attn = kvq && !fp4;
        // One or two decode rows whose output projection runs the GEMV: the attention stops at its
        // splits' partial results and the projection merges them while its first weights travel —
        // one launch less per layer, but EVERY block of the projection reads all the partial results,
        // so only where those are few: measured on the 1B shape (32 heads of 64, four splits, 32 KB)
        // 0.578 -> 0.560 ms per step and on the 8B shape with four splits (64 KB, contexts below 512)
        // 1.589 -> 1.553; with eight splits (128 KB) the projection grows from 4.7 to 8.8 us, more than
        // the merge launch it saves (1.580 -> 1.601).  ([runtime] attn_merge_proj = false
        // or PIE_ATTN_MERGE_PROJ=0 keeps the separate merge.)
        bool merged_into_wo = false;
        if (N <= 2 && n_tiles_ == 0 && !masked_ && cfg_.runtime.attn_merge_proj) {
            static const bool merge_on = [] { const char* e = getenv("PIE_ATTN_MERGE_PROJ"); return !e || atoi(e) != 0; }();
            int ups = 0, ns = 1;
            if (merge_on && routes_to_gemv(w.wo, N, false, gemm_ws_bytes_) &&
                pie_hip_attn_decode_plan(N, hk, max_kv_len, &ups, &ns) == PIE_HIP_OK && ns >= 2 &&
                static_cast<size_t>(N) * hq * ns * d * sizeof(float) <= kMergeProjMaxBytes &&
                pie_hip_linear_attn_merge_supported(fmt_code(w.wo.kind), N, ns, hq, d, w.wo.group)) {
                PIE_KERNEL(pie_hip_attn_rows_paged_partials(kvq_attn ? kv_format_ : PIE_HIP_KV_BF16, q_,
                                                            kvq_attn ? static_cast<const void*>(k_pool_[l]) : kat,
                                                            kvq_attn ? static_cast<const void*>(v_pool_[l]) : vat,
                                                            kvq_attn ? ksc : nullptr, kvq_attn ? vsc : nullptr, pages,
                                                            row_begin, row_len, N, hq, hk, d, page_size_, -1.f,
                                                            max_kv_len, attn_ws_, attn_ws_bytes_, s));
                PIE_KERNEL(pie_hip_linear_attn_merge(fmt_code(w.wo.kind), attn_ws_, ns, ups, row_len, hq, d, w.wo.data,
                                                     w.wo.scale, w.wo.scale_bf16 ? 1 : 0, w.wo.group, x_, N, w.wo.N, 1,
                                                     s));
                merged_into_wo = true;
            }
        }
        // rows [r.row, r.row + r.rows) one by one
        auto attend_rows = [&](const RowRun& r) {
            const size_t at = static_cast<size_t>(r.row) * hq * d;
            if (masked_) {   // (the whole batch)
                const auto* bitmap = static_cast<const uint16_t*>(mask_bitmap_.ptr);
                if (kvq_attn)
                    PIE_KERNEL(pie_hip_attn_rows_paged_kvq_masked(kv_format_, q_, k_pool_[l], v_pool_[l], ksc, vsc, attn_, nullptr,
                                                                  pages, row_begin, row_len, bitmap, mask_stride_, N, hq, hk, d,
                                                                  page_size_, -1.f, max_kv_len, attn_ws_, attn_ws_bytes_, s));
                else
                    PIE_KERNEL(pie_hip_attn_rows_paged_masked(q_, kat, vat, attn_, nullptr, pages, row_begin, row_len, bitmap,
                                                              mask_stride_, N, hq, hk, d, page_size_, -1.f, max_kv_len, attn_ws_,
                                                              attn_ws_bytes_, s));
                return;
            }
            const uint32_t* begin = row_begin + r.row;
            const int32_t* len = row_len + r.row;
            if (kvq_attn || r.uniform)
                PIE_KERNEL((r.uniform ? pie_hip_attn_rows_paged_kvq_uniform : pie_hip_attn_rows_paged_kvq)(
                    kvq_attn ? kv_format_ : PIE_HIP_KV_BF16, q_ + at, kvq_attn ? k_pool_[l] : kat, kvq_attn ? v_pool_[l] : vat,
                    kvq_attn ? ksc : nullptr, kvq_attn ? vsc : nullptr, attn_ + at, nullptr, pages, begin, len, r.rows, hq, hk, d,
                    page_size_, -1.f, r.max_len, attn_ws_, attn_ws_bytes_, s));
            else
                PIE_KERNEL(pie_hip_attn_rows_paged(q_ + at, kat, vat, attn_ + at, nullptr, pages, begin, len, r.rows, hq, hk, d,
                                                   page_size_, -1.f, r.max_len, attn_ws_, attn_ws_bytes_, s));
        };
        if (!merged_into_wo && n_tiles_ > 0) {
            const auto* td = static_cast<const int32_t*>(tile_in_dev_.ptr);
            if (kvq_attn)
                PIE_KERNEL(pie_hip_attn_prefill_tiles_kvq(kv_format_, q_, k_pool_[l], v_pool_[l], ksc, vsc, attn_,
                                                          pages, row_begin, row_len, td, td + n_tiles_, n_tiles_,
                                                          tile_rows_, hq, hk, d, page_size_, -1.f, s));
            else
                PIE_KERNEL(pie_hip_attn_prefill_tiles(q_, kat, vat, attn_, pages, row_begin, row_len, td, td + n_tiles_, n_tiles_,
                                                      tile_rows_, hq, hk, d, page_size_, -1.f, s));
        }
        if (merged_into_wo) {
        } else if (pure_decode_) {   // (max_kv_len: the bucket a graph is captured for)
            attend_rows({0, N, max_kv_len, uniform_rows_});
        } else {
            for (const RowRun& r : runs_) attend_rows(r);
        }
        // x_ += act · W^T; true if xn_ then holds the rows under `norm`
        auto project = [&](const Linear& lin, const uint16_t* act, const uint16_t* norm) {
            if (norm && in_shares(lin, N, gemm_ws_bytes_) && project_in_shares(lin, act, norm, N)) return true;
            linear_fused(lin, act, nullptr, m.rms_eps, x_, N, 1, 0, xn_, gemm_ws_, gemm_ws_bytes_, s);
            return false;
        };
        const bool ffn_normed = !merged_into_wo && project(w.wo, attn_, model_.is_moe() ? nullptr : w.ffn_norm);
        if (model_.is_moe()) {
            // the next layer's rows come normalised when that layer runs the plain projection
            // (q/k norm: no fused RoPE epilogue) on more than the GEMV's four rows
            const bool next_plain = l + 1 < m.layers && N > 4 && model_.layers[l + 1].q_norm != nullptr;
            moe_block(w, N, next_plain ? model_.layers[l + 1].attn_norm : nullptr, s);
            continue;
        }
        linear_fused(w.wgu, ffn_normed ? xn_ : x_, ffn_normed ? nullptr : w.ffn_norm, m.rms_eps, act_, N, 0, 1, xn_, gemm_ws_, gemm_ws_bytes_, s);
        xn_holds_next_norm_ = project(w.wdown, act_, l + 1 < m.layers ? model_.layers[l + 1].attn_norm : nullptr);
    }
    // lm_head only on the sampled rows (driver/portable/src/graph_qwen3.cpp:867-896)
    const int cap = static_cast<int>(std::min<size_t>(max_tokens_, 2 * static_cast<size_t>(cfg_.batching.max_forward_requests)));
    for (int s0 = 0; s0 < S; s0 += cap) {
        const int n = std::min(cap, S - s0);
        PIE_KERNEL(pie_hip_embed(sample_rows + s0, x_, xs_, n, H, N, s));  // row gather
        Linear head;
        head.kind = Quant::Bf16;
        head.data = model_.lm_head;
        head.N = m.vocab;
        head.K = H;
        // up to four rows: the GEMV keeps (largest value, row) pairs while it stores the logits
        const int fused = n <= 4 ? pie_hip_lm_head_argmax(xs_, model_.final_norm, m.rms_eps, model_.lm_head, logits_,
                                                          out_tokens_ + s0, n, m.vocab, H, amax_ws_, amax_ws_bytes_, s)
                                 : PIE_HIP_ERR_UNSUPPORTED;
        if (fused == PIE_HIP_ERR_UNSUPPORTED) {
            linear_fused(head, xs_, model_.final_norm, m.rms_eps, logits_, n, 0, 0, xn_, gemm_ws_, gemm_ws_bytes_, s);
            PIE_KERNEL(pie_hip_argmax(logits_, out_tokens_ + s0, n, m.vocab, s));
        } else {
            PIE_KERNEL(fused);
        }
        if (samp_gather_in_body_) {   // more sampled rows than one chunk: keep each chunk's f32 rows
            const auto* in = static_cast<const unsigned char*>(samp_in_dev_.ptr);
            PIE_KERNEL(pie_hip_sample_gather_logits(
                logits_, nullptr, static_cast<float*>(samp_f32_.ptr) + static_cast<size_t>(s0) * m.vocab,
                samp_.n_bounds ? reinterpret_cast<const uint32_t*>(in + samp_.bounds) : nullptr,
                samp_.n_bounds ? reinterpret_cast<const int32_t*>(in + samp_.bounds_indptr) + s0 : nullptr,
                n, m.vocab, s));
        }
    }
}

void Executor::Growable::ensure(size_t bytes) {
    if (bytes <= cap) return;
    release();
    const size_t want = std::max<size_t>(bytes, 256);
    if (pinned) PIE_HIP_CHECK(hipHostMalloc(&ptr, want, hipHostMallocDefault));
    else PIE_HIP_CHECK(hipMalloc(&ptr, want));
    cap = want;
}

void Executor::Growable::release() {
    if (ptr) (void)(pinned ? hipHostFree(ptr) : hipFree(ptr));
    ptr = nullptr;
    cap = 0;
}

namespace {

// The reference's per-slot generator (Pcg32, driver/portable/src/sampler.cpp:31-57): PCG-XSH-RR
// 64/32, seeded in the canonical two steps on the default stream; a slot draws one uniform,
// the top 24 bits of the first output.
float pcg32_first_uniform(uint64_t seed) {
    const uint64_t inc = (0xda3e39cb94b95bdbULL << 1u) | 1u;
    uint64_t state = 0;
    state = state * 6364136223846793005ULL + inc;
    state += seed;
    state = state * 6364136223846793005ULL + inc;
    const uint64_t old = state;
    const uint32_t xorshifted = static_cast<uint32_t>(((old >> 18u) ^ old) >> 27u);
    const uint32_t rot = static_cast<uint32_t>(old >> 59u);
    const uint32_t r = (xorshifted >> rot) | (xorshifted << ((32u - rot) & 31u));
    return static_cast<float>(r >> 8) * (1.0f / 16777216.0f);
}

}  // namespace

// Cuts the batch (attention_cut.hpp) and uploads its tiles.
void Executor::prepare_tiles(const BatchPlan& plan) {
    const ModelConfig& m = model_.cfg();
    const bool fits = !masked_ && !plan.pure_decode && page_size_ % 16 == 0 && (m.head_dim == 64 || m.head_dim == 128);
    const bool one_byte = kv_format_ != PIE_HIP_KV_BF16 && kv_format_ != PIE_HIP_KV_FP4_BLOCK;   // (4-bit pools are read as bf16)
    const AttentionCut cut = cut_attention(plan, m.kv_heads, m.head_dim, one_byte, fits ? pie_hip_attn_prefill_tile_rows(m.q_heads, m.kv_heads) : 0);
    runs_ = cut.runs;
    tile_rows_ = cut.tile_rows;
    n_tiles_ = static_cast<int>(cut.tiles.size());
    if (n_tiles_ == 0) return;
    const size_t n = cut.tiles.size(), bytes = 8 * n;
    tile_in_host_.pinned = true;
    tile_in_host_.ensure(bytes);
    tile_in_dev_.ensure(bytes);
    auto* h = static_cast<int32_t*>(tile_in_host_.ptr);
    for (size_t i = 0; i < n; ++i) {
        h[i] = cut.tiles[i].first;
        h[n + i] = cut.tiles[i].second;
    }
    PIE_HIP_CHECK(hipMemcpyAsync(tile_in_dev_.ptr, h, bytes, hipMemcpyHostToDevice, stream_));
}

// Custom attention masks: each row's BRLE runs become cumulative bounds, the device expands
// them into one visibility word per 16-token unit, and the layers' attention reads that.
void Executor::prepare_masks(const BatchPlan& plan) {
    const int N = plan.N;
    std::vector<int32_t> indptr(static_cast<size_t>(N) + 1, 0);
    std::vector<uint32_t> bounds;
    const bool user = static_cast<int>(plan.row_mask_runs.size()) == N;   // (absent: window only)
    for (int i = 0; i < N && user; ++i) {
        uint64_t acc = 0;
        for (uint32_t len : plan.row_mask_runs[i]) {
            acc = std::min<uint64_t>(acc + len, 0xFFFFFFFFull);
            bounds.push_back(static_cast<uint32_t>(acc));
        }
        indptr[i + 1] = static_cast<int32_t>(bounds.size());
    }
    if (!user) std::fill(indptr.begin(), indptr.end(), 0);
    const size_t off_bounds = align_up(4ull * (N + 1), 16);
    const size_t total = off_bounds + 4ull * std::max<size_t>(bounds.size(), 1);
    mask_in_host_.pinned = true;
    mask_in_host_.ensure(total);
    mask_in_dev_.ensure(total);
    mask_stride_ = std::max(1, (plan.max_kv_len + 15) / 16);
    mask_bitmap_.ensure(static_cast<size_t>(N) * mask_stride_ * sizeof(uint16_t));
    auto* h = static_cast<unsigned char*>(mask_in_host_.ptr);
    std::memcpy(h, indptr.data(), 4ull * (N + 1));
    if (!bounds.empty()) std::memcpy(h + off_bounds, bounds.data(), 4ull * bounds.size());
    PIE_HIP_CHECK(hipMemcpyAsync(mask_in_dev_.ptr, h, total, hipMemcpyHostToDevice, stream_));
    const auto* dv = static_cast<const unsigned char*>(mask_in_dev_.ptr);
    const Inputs lay = input_layout(N, static_cast<int>(plan.sample_rows.size()));   // this forward's staging layout
    const auto* row_len = reinterpret_cast<const int32_t*>(in_dev_ + lay.off_row_len);
    PIE_KERNEL(pie_hip_attn_mask_bitmap(reinterpret_cast<const uint32_t*>(dv + off_bounds),
                                        reinterpret_cast<const int32_t*>(dv), row_len,
                                        std::max(0, model_.cfg().sliding_window),
                                        static_cast<uint16_t*>(mask_bitmap_.ptr), N, mask_stride_, stream_));
}

// Host half of the sampler stage: per-slot parameter arrays, uniforms, payload ranges, BRLE
// bounds — staged in pinned memory and sent to the device ahead of the forward body.
void Executor::prepare_samplers(const BatchPlan& plan) {
    const int S = static_cast<int>(plan.sample_rows.size());
    const int V = cfg_.model.vocab;
    if (static_cast<int>(plan.slot_samplers.size()) != S)
        throw std::runtime_error("executor: one sampler per sampling slot expected");
    std::vector<int32_t> out_indptr(static_cast<size_t>(S) + 1, 0), bounds_indptr(static_cast<size_t>(S) + 1, 0);
    std::vector<uint32_t> bounds;
    for (int r = 0, s = 0; r < plan.R; ++r) {
        const auto& runs = plan.logit_mask_runs[r];
        for (; s < plan.sample_indptr[r + 1]; ++s) {
            uint64_t acc = 0;
            for (uint32_t len : runs) {
                acc = std::min<uint64_t>(acc + len, 0xFFFFFFFFull);
                bounds.push_back(static_cast<uint32_t>(acc));
            }
            bounds_indptr[s + 1] = static_cast<int32_t>(bounds.size());
        }
    }
    for (int s = 0; s < S; ++s) {
        const SlotSampler& sp = plan.slot_samplers[s];
        int n = 0;
        switch (sp.kind) {
            case PIE_SAMPLER_KIND_MULTINOMIAL: case PIE_SAMPLER_KIND_TOP_K: case PIE_SAMPLER_KIND_TOP_P:
            case PIE_SAMPLER_KIND_MIN_P: case PIE_SAMPLER_KIND_TOP_K_TOP_P: case PIE_SAMPLER_KIND_RAW_LOGITS:
                break;
            case PIE_SAMPLER_KIND_DIST:
                n = sp.top_k > 0 ? static_cast<int>(std::min<uint32_t>(sp.top_k, static_cast<uint32_t>(V))) : V;
                break;
            case PIE_SAMPLER_KIND_LOGPROB: case PIE_SAMPLER_KIND_LOGPROBS:
                n = static_cast<int>(sp.labels_end - sp.labels_begin);
                if (n == 0) throw std::runtime_error("sampler: Logprob slot has no labels");
                for (uint32_t i = sp.labels_begin; i < sp.labels_end; ++i)
                    if (plan.label_ids[i] >= static_cast<uint32_t>(V))
                        throw std::runtime_error("sampler: Logprob label id out of vocab");
                break;
            case PIE_SAMPLER_KIND_ENTROPY: n = 1; break;
            // the response has no field for it: the slot is accepted and yields nothing, as the
            // portable executor's per-slot switch leaves it (executor.cpp:1367-1392, default arm)
            case PIE_SAMPLER_KIND_EMBEDDING: break;
            default:
                throw std::runtime_error("sampler: unknown type " + std::to_string(static_cast<int>(sp.kind)));
        }
        out_indptr[s + 1] = out_indptr[s] + n;
    }
    const int payload = out_indptr[S];
    SampLayout L{};
    L.slots = S;
    L.payload = payload;
    L.n_bounds = static_cast<int>(bounds.size());
    size_t o = 0;
    auto take = [&](size_t bytes) { const size_t at = o; o = align_up(o + bytes, 16); return at; };
    L.kind = take(4ull * S);
    L.temperature = take(4ull * S);
    L.top_k = take(4ull * S);
    L.top_p = take(4ull * S);
    L.min_p = take(4ull * S);
    L.uniform = take(4ull * S);
    L.out_indptr = take(4ull * (S + 1));
    L.labels = take(4ull * std::max(payload, 1));
    L.bounds_indptr = take(4ull * (S + 1));
    L.bounds = take(4ull * std::max<size_t>(bounds.size(), 1));
    L.total = o;
    o = 0;
    L.o_tokens = take(4ull * S);
    L.o_values = take(4ull * std::max(payload, 1));
    L.o_ids = take(4ull * std::max(payload, 1));
    L.o_total = o;
    samp_ = L;

    samp_in_host_.pinned = true;
    samp_out_host_.pinned = true;
    samp_in_host_.ensure(L.total);
    samp_in_dev_.ensure(L.total);
    samp_out_dev_.ensure(L.o_total);
    samp_out_host_.ensure(L.o_total);
    samp_f32_.ensure(static_cast<size_t>(S) * V * sizeof(float));
    samp_ws_.ensure(pie_hip_sample_workspace_bytes(S, V));

    auto* h = static_cast<unsigned char*>(samp_in_host_.ptr);
    std::memset(h, 0, L.total);
    auto* kind = reinterpret_cast<int32_t*>(h + L.kind);
    auto* temp = reinterpret_cast<float*>(h + L.temperature);
    auto* top_k = reinterpret_cast<uint32_t*>(h + L.top_k);
    auto* top_p = reinterpret_cast<float*>(h + L.top_p);
    auto* min_p = reinterpret_cast<float*>(h + L.min_p);
    auto* uni = reinterpret_cast<float*>(h + L.uniform);
    auto* labels = reinterpret_cast<uint32_t*>(h + L.labels);
    for (int s = 0; s < S; ++s) {
        const SlotSampler& sp = plan.slot_samplers[s];
        kind[s] = sp.kind;
        temp[s] = sp.temperature;
        top_k[s] = sp.top_k;
        top_p[s] = sp.top_p;
        min_p[s] = sp.min_p;
        // no caller seed: a process-wide counter, as the reference's default_rng_seed (:62-65)
        const uint64_t seed = sp.seed != 0 ? sp.seed : (0x9E3779B97F4A7C15ULL ^ unseeded_draws_++);
        uni[s] = pcg32_first_uniform(seed);
        for (uint32_t i = sp.labels_begin; i < sp.labels_end; ++i)
            labels[out_indptr[s] + (i - sp.labels_begin)] = plan.label_ids[i];
    }
    std::memcpy(h + L.out_indptr, out_indptr.data(), 4ull * (S + 1));
    std::memcpy(h + L.bounds_indptr, bounds_indptr.data(), 4ull * (S + 1));
    if (!bounds.empty()) std::memcpy(h + L.bounds, bounds.data(), 4ull * bounds.size());
    PIE_HIP_CHECK(hipMemcpyAsync(samp_in_dev_.ptr, h, L.total, hipMemcpyHostToDevice, stream_));
}

// Device half, queued behind the forward body: f32 rows (+ masks) unless the body gathered them
// chunk by chunk, one sampler block per slot, results into pinned memory.
void Executor::enqueue_samplers() {
    const int S = samp_.slots, V = cfg_.model.vocab;
    const auto* in = static_cast<const unsigned char*>(samp_in_dev_.ptr);
    auto* od = static_cast<unsigned char*>(samp_out_dev_.ptr);
    float* f32 = static_cast<float*>(samp_f32_.ptr);
    if (!samp_gather_in_body_) {
        const auto* bounds = samp_.n_bounds ? reinterpret_cast<const uint32_t*>(in + samp_.bounds) : nullptr;
        const auto* indptr = samp_.n_bounds ? reinterpret_cast<const int32_t*>(in + samp_.bounds_indptr) : nullptr;
        if (stack_.logits)
            PIE_KERNEL(pie_hip_sample_gather_logits_f32(stack_.logits, nullptr, f32, bounds, indptr, S, V, stream_));
        else
            PIE_KERNEL(pie_hip_sample_gather_logits(logits_, nullptr, f32, bounds, indptr, S, V, stream_));
    }
    PIE_HIP_CHECK(hipMemsetAsync(od, 0, samp_.o_total, stream_));   // eager stage, never captured
    PIE_KERNEL(pie_hip_sample(
        f32, reinterpret_cast<const int32_t*>(in + samp_.kind), reinterpret_cast<const float*>(in + samp_.temperature),
        reinterpret_cast<const uint32_t*>(in + samp_.top_k), reinterpret_cast<const float*>(in + samp_.top_p),
        reinterpret_cast<const float*>(in + samp_.min_p), reinterpret_cast<const float*>(in + samp_.uniform),
        reinterpret_cast<const int32_t*>(in + samp_.out_indptr), reinterpret_cast<const uint32_t*>(in + samp_.labels),
        reinterpret_cast<uint32_t*>(od + samp_.o_tokens), reinterpret_cast<float*>(od + samp_.o_values),
        reinterpret_cast<uint32_t*>(od + samp_.o_ids), samp_ws_.ptr, samp_ws_.cap, S, V, stream_));
    PIE_HIP_CHECK(hipMemcpyAsync(samp_out_host_.ptr, od, samp_.o_total, hipMemcpyDeviceToHost, stream_));
}

// After the stream has drained: results out of pinned memory, RawLogits rows copied back.
void Executor::collect_samplers(const BatchPlan& plan, SampleOutputs& out) {
    const int S = samp_.slots, V = cfg_.model.vocab;
    const float* f32 = static_cast<const float*>(samp_f32_.ptr);
    const auto* oh = static_cast<const unsigned char*>(samp_out_host_.ptr);
    out.raw_logits.clear();
    size_t n_raw = 0;
    for (const SlotSampler& sp : plan.slot_samplers) n_raw += sp.kind == PIE_SAMPLER_KIND_RAW_LOGITS;
    out.raw_logits.resize(n_raw * static_cast<size_t>(V));
    size_t at = 0;
    for (int s = 0; s < S; ++s)
        if (plan.slot_samplers[s].kind == PIE_SAMPLER_KIND_RAW_LOGITS) {
            PIE_HIP_CHECK(hipMemcpy(out.raw_logits.data() + at, f32 + static_cast<size_t>(s) * V,
                                    static_cast<size_t>(V) * sizeof(float), hipMemcpyDeviceToHost));
            at += V;
        }
    const auto* tok = reinterpret_cast<const uint32_t*>(oh + samp_.o_tokens);
    out.tokens.assign(tok, tok + S);
    const auto* val = reinterpret_cast<const float*>(oh + samp_.o_values);
    out.values.assign(val, val + samp_.payload);
    const auto* ids = reinterpret_cast<const uint32_t*>(oh + samp_.o_ids);
    out.ids.assign(ids, ids + samp_.payload);
    const auto* ip = reinterpret_cast<const int32_t*>(static_cast<const unsigned char*>(samp_in_host_.ptr) + samp_.out_indptr);
    out.out_indptr.assign(ip, ip + S + 1);
}

// Captured graphs hold the old buffer's address: they are dropped with it.
void Executor::grow_outputs(size_t slots) {
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
    for (auto& kv : graphs_) (void)hipGraphExecDestroy(kv.second);
    graphs_.clear();
    const size_t cap = std::max(slots, 2 * out_cap_);
    (void)hipFree(out_tokens_);
    out_tokens_ = nullptr;
    (void)hipHostFree(out_host_);
    out_host_ = nullptr;
    out_cap_ = 0;
    out_tokens_ = dmalloc<uint32_t>(cap);
    PIE_HIP_CHECK(hipHostMalloc(reinterpret_cast<void**>(&out_host_), cap * 4, hipHostMallocDefault));
    out_cap_ = cap;
}

void Executor::forward(const BatchPlan& plan, std::vector<uint32_t>& tokens_out,
                       ForwardTimings* t, SampleOutputs* samples) {
    const int N = plan.N, S = static_cast<int>(plan.sample_rows.size());
    if (N <= 0) throw std::runtime_error("executor: empty plan");
    if (N > max_tokens_) throw std::runtime_error("executor: batch exceeds max_forward_tokens");
    if (static_cast<int>(plan.page_indices.size()) > max_page_refs_)
        throw std::runtime_error("executor: batch exceeds the page reference capacity");
    // A request may put several samplers on one row, so the sampling slots can outnumber the
    // rows: the token buffers follow the slot count.
    if (static_cast<size_t>(S) > out_cap_) grow_outputs(static_cast<size_t>(S));

    auto t0 = clk::now();
    const Inputs in = input_layout(N, S);
    const size_t used = in.off_pages + plan.page_indices.size() * 4;
    if (used > in_.total) throw std::runtime_error("executor: staged inputs exceed their buffer");
    std::memcpy(in_host_ + in.off_tokens, plan.tokens.data(), static_cast<size_t>(N) * 4);
    std::memcpy(in_host_ + in.off_positions, plan.positions.data(), static_cast<size_t>(N) * 4);
    std::memcpy(in_host_ + in.off_slots, plan.kv_slots.data(), static_cast<size_t>(N) * 8);
    std::memcpy(in_host_ + in.off_row_begin, plan.row_page_begin.data(), static_cast<size_t>(N) * 4);
    std::memcpy(in_host_ + in.off_row_len, plan.row_kv_len.data(), static_cast<size_t>(N) * 4);
    if (S) std::memcpy(in_host_ + in.off_sample_rows, plan.sample_rows.data(), static_cast<size_t>(S) * 4);
    std::memcpy(in_host_ + in.off_pages, plan.page_indices.data(), plan.page_indices.size() * 4);
    if (model_.cfg().is_stack()) prepare_stack(plan, in);
    PIE_HIP_CHECK(hipMemcpyAsync(in_dev_, in_host_, used, hipMemcpyHostToDevice, stream_));
    // a sliding window (driver/portable/src/plan.cpp:60-70: keys below p - W + 1 are hidden)
    // matters once some context is longer than the window; such batches take the masked kernels
    const int window = model_.cfg().sliding_window;
    masked_ = plan.has_user_masks || (window > 0 && plan.max_kv_len > window);
    if (masked_) prepare_masks(plan);
    prepare_tiles(plan);
    const bool sampling = !plan.all_greedy && S > 0;
    const int chunk = static_cast<int>(std::min<size_t>(max_tokens_, 2 * static_cast<size_t>(cfg_.batching.max_forward_requests)));
    samp_gather_in_body_ = false;
    if (sampling) {
        if (!samples) throw std::runtime_error("executor: a sampling plan needs a SampleOutputs");
        prepare_samplers(plan);
        samp_gather_in_body_ = S > chunk;   // logits_ keeps one chunk of rows only
    }
    if (t) t->h2d_us = us_since(t0);

    t0 = clk::now();
    n_page_refs_ = static_cast<int>(plan.page_indices.size());
    // (a graph is captured per answer)
    pure_decode_ = plan.pure_decode;
    uniform_rows_ = plan.pure_decode && !masked_ && evenly_long(plan, 0, N);
    // (4-bit blocks: the page expansion's extent changes from step to step, so no graph)
    const bool use_graph = cfg_.runtime.use_graphs && plan.pure_decode && !samp_gather_in_body_ && !masked_ &&
                           kv_format_ != PIE_HIP_KV_FP4_BLOCK;
    if (use_graph) {
        // The split grid depends on the context bound only through 512-token buckets.
        const int bucket = (plan.max_kv_len + 511) / 512 * 512;
        const auto key = std::make_tuple(N, S, bucket, uniform_rows_ ? 1 : 0);
        auto it = graphs_.find(key);
        if (it == graphs_.end()) {
            hipGraph_t graph = nullptr;
            PIE_HIP_CHECK(hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal));
            try {
                body(N, S, bucket);
            } catch (...) {
                (void)hipStreamEndCapture(stream_, &graph);
                if (graph) (void)hipGraphDestroy(graph);
                throw;
            }
            PIE_HIP_CHECK(hipStreamEndCapture(stream_, &graph));
            hipGraphExec_t exec = nullptr;
            PIE_HIP_CHECK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
            PIE_HIP_CHECK(hipGraphDestroy(graph));
            it = graphs_.emplace(key, exec).first;
        }
        PIE_HIP_CHECK(hipGraphLaunch(it->second, stream_));
    } else {
        body(N, S, plan.max_kv_len);
    }
    if (S) PIE_HIP_CHECK(hipMemcpyAsync(out_host_, out_tokens_, static_cast<size_t>(S) * 4,
                                        hipMemcpyDeviceToHost, stream_));
    if (sampling) enqueue_samplers();
    if (t) t->launch_us = us_since(t0);

    t0 = clk::now();
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
    if (t) t->sync_us = us_since(t0);
    tokens_out.assign(out_host_, out_host_ + S);
    if (sampling) {
        collect_samplers(plan, *samples);
        tokens_out = samples->tokens;
    }
    const int cap = static_cast<int>(std::min<size_t>(max_tokens_, 2 * static_cast<size_t>(cfg_.batching.max_forward_requests)));
    if (model_.cfg().is_stack()) commit_stack(plan);
    last_logit_rows_ = S == 0 ? 0 : ((S - 1) % cap) + 1;
}

void Executor::copy_pages_d2h(const uint32_t* dev_srcs, const uint32_t* host_dsts, size_t n) {
    for (size_t i = 0; i < n; ++i)
        for (const PagePool& p : page_pools_)
            PIE_HIP_CHECK(hipMemcpyAsync(swap_slot(p, host_dsts[i]), p.base + dev_srcs[i] * p.page_bytes, p.page_bytes,
                                         hipMemcpyDeviceToHost, stream_));
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
}

void Executor::copy_pages_h2d(const uint32_t* host_srcs, const uint32_t* dev_dsts, size_t n) {
    for (size_t i = 0; i < n; ++i)
        for (const PagePool& p : page_pools_)
            PIE_HIP_CHECK(hipMemcpyAsync(p.base + dev_dsts[i] * p.page_bytes, swap_slot(p, host_srcs[i]), p.page_bytes,
                                         hipMemcpyHostToDevice, stream_));
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
}

void Executor::copy_pages_h2h(const uint32_t* srcs, const uint32_t* dsts, size_t n) {
    for (size_t i = 0; i < n; ++i)
        for (const PagePool& p : page_pools_) std::memmove(swap_slot(p, dsts[i]), swap_slot(p, srcs[i]), p.page_bytes);
}

void Executor::copy_pages_d2d(const uint32_t* srcs, const uint32_t* dsts, size_t n) {
    if (n == 0) return;
    if (n > copy_ids_cap_) {
        if (copy_ids_) (void)hipFree(copy_ids_);
        copy_ids_ = dmalloc<uint32_t>(2 * n);
        copy_ids_cap_ = n;
    }
    PIE_HIP_CHECK(hipMemcpyAsync(copy_ids_, srcs, n * 4, hipMemcpyHostToDevice, stream_));
    PIE_HIP_CHECK(hipMemcpyAsync(copy_ids_ + copy_ids_cap_, dsts, n * 4, hipMemcpyHostToDevice, stream_));
    for (size_t i = 0; i < n; i += 65535) {
        const int cnt = static_cast<int>(std::min<size_t>(65535, n - i));
        for (const PagePool& p : page_pools_)
            PIE_KERNEL(pie_hip_copy_kv_pages(p.base, copy_ids_ + i, copy_ids_ + copy_ids_cap_ + i, cnt, p.page_bytes,
                                             stream_));
    }
    PIE_HIP_CHECK(hipStreamSynchronize(stream_));
}

}  // namespace pie_hip_driver

// Host-only hook on the rules that choose a linear's kernel, as pie_hip_driver_plan is on the planner: what a matrix [N, K] of
// a storage format takes at M rows before any start-up measurement (0 GEMV, 1 skinny GEMM, 2 tiled GEMM, 3 tiled GEMM in
// K shares, 4 tiled GEMM over the tile-major copy).
extern "C" int pie_hip_driver_linear_route(int format, int group, int M, int N, int K, int tile_major, size_t workspace_bytes) {
    using namespace pie_hip_driver;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || M <= 0 || N <= 0 || K <= 0) return -1;
    constexpr Quant kinds[] = {Quant::Int4b8, Quant::Int8, Quant::Fp8, Quant::Bf16};
    static_assert(PIE_HIP_FMT_INT4B8 == 0 && PIE_HIP_FMT_INT8 == 1 && PIE_HIP_FMT_FP8 == 2 && PIE_HIP_FMT_BF16 == 3, "");
    Linear w;
    w.kind = kinds[format];
    w.N = N;
    w.K = K;
    w.group = group;
    int there = 0;   // (only whether a copy is there counts)
    if (tile_major) w.data_tiled = w.scale_tiled = &there;
    return model_route(w, M, false, workspace_bytes);
}

// And in which form that kernel runs, by what a measurement said (0 or 1; -1: by estimate): bit 0 int4 rows in blocks that scale groups in fp32 (in the skinny GEMM's place), bit 1 a
// projection into the residual in shares of K that meet in the norm's kernel, bit 2 one-byte rows in blocks of 32 to 128 (in the wide GEMM's place), bit 3 rows in
// blocks whose waves take the steps of K in turn (in the skinny GEMM's place).
extern "C" int pie_hip_driver_linear_forms(int format, int group, int M, int N, int K, int measured_groups, int measured_shares,
                                           int tile_major, size_t workspace_bytes) {
    using namespace pie_hip_driver;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || M <= 0 || N <= 0 || K <= 0) return -1;
    constexpr Quant kinds[] = {Quant::Int4b8, Quant::Int8, Quant::Fp8, Quant::Bf16};
    Linear w;
    w.kind = kinds[format];
    w.N = N;
    w.K = K;
    w.group = group;
    int there = 0;
    if (tile_major) w.data_tiled = w.scale_tiled = &there;
    w.groups.fill(static_cast<int8_t>(measured_groups));
    w.shares.fill(static_cast<int8_t>(measured_shares));
    return (in_groups(w, M, workspace_bytes) ? 1 : 0) | (in_shares(w, M, workspace_bytes) ? 2 : 0) | (in_rows(w, M, workspace_bytes) ? 4 : 0) |
           (in_waves(w, M, workspace_bytes) ? 8 : 0);
}

// And which pairs of forms the start-up measurement times at a row count of its ladder: bit 0 passes and blocks that scale groups, bit 1 a product with the
// norm behind it and shares of K that meet in the norm's kernel.
extern "C" int pie_hip_driver_measured_forms(int format, int group, int M, int N, int K, size_t workspace_bytes) {
    using namespace pie_hip_driver;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || M <= 0 || N <= 0 || K <= 0) return -1;
    constexpr Quant kinds[] = {Quant::Int4b8, Quant::Int8, Quant::Fp8, Quant::Bf16};
    Linear w;
    w.kind = kinds[format];
    w.N = N;
    w.K = K;
    w.group = group;
    int there = 0;
    w.data_tiled = w.scale_tiled = &there;
    return (measures_groups(w, M, workspace_bytes) ? 1 : 0) | (measures_shares(w, M, workspace_bytes, true) ? 2 : 0);
}

// The same for a mixture's experts: whether `routes` over `experts` of a storage format run in blocks of an expert's routes (1)
// or in passes of 16 (0); with sizes (`hidden` > 0) those of tile-major experts.
extern "C" int pie_hip_driver_experts_in_blocks(int format, long long routes, int experts, int hidden, int inner) {
    using namespace pie_hip_driver;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || routes <= 0 || experts <= 0) return -1;
    constexpr Quant kinds[] = {Quant::Int4b8, Quant::Int8, Quant::Fp8, Quant::Bf16};
    return Executor::grouped_in_blocks(kinds[format], routes, experts) ||
                   (hidden > 0 && inner > 0 && Executor::few_in_blocks(kinds[format], routes, experts, hidden, inner))
               ? 1
               : 0;
}

// And for the choice of a batch's experts: 0 one launch, 1 the logits in shares of K, 2 a product.
extern "C" int pie_hip_driver_route_form(int format, int tokens, int hidden, int experts, size_t workspace_bytes) {
    using namespace pie_hip_driver;
    if (format < PIE_HIP_FMT_INT4B8 || format > PIE_HIP_FMT_BF16 || tokens <= 0 || hidden <= 0 || experts <= 0) return -1;
    constexpr Quant kinds[] = {Quant::Int4b8, Quant::Int8, Quant::Fp8, Quant::Bf16};
    return static_cast<int>(Executor::route_form(kinds[format], tokens, hidden, experts, workspace_bytes));
}

// And for a batch's attention: the rows of request r are qo_indptr[r] .. qo_indptr[r + 1] (of R requests), row i sees
// row_kv_len[i] keys.  out receives {tile height, tiles, runs}, (first row, rows) of each tile and (first row, rows, equally long) of each
// run.  Returns the number of values, or -1 where they do not fit `cap` or the lists make no batch.
extern "C" long long pie_hip_driver_attention_cut(const int* qo_indptr, int R, const int* row_kv_len, int q_heads, int kv_heads,
                                                  int head_dim, int one_byte, int* out, size_t cap) {
    using namespace pie_hip_driver;
    if (!qo_indptr || !row_kv_len || !out || R <= 0 || q_heads <= 0 || kv_heads <= 0 || qo_indptr[0] != 0) return -1;
    for (int r = 0; r < R; ++r)
        if (qo_indptr[r + 1] < qo_indptr[r]) return -1;
    try {
        BatchPlan plan;
        plan.R = R;
        plan.N = qo_indptr[R];
        plan.qo_indptr.assign(qo_indptr, qo_indptr + R + 1);
        plan.row_kv_len.assign(row_kv_len, row_kv_len + plan.N);
        plan.max_kv_len = plan.N ? *std::max_element(plan.row_kv_len.begin(), plan.row_kv_len.end()) : 0;
        const AttentionCut cut = cut_attention(plan, kv_heads, head_dim, one_byte != 0, pie_hip_attn_prefill_tile_rows(q_heads, kv_heads));
        std::vector<int> v = {cut.tile_rows, static_cast<int>(cut.tiles.size()), static_cast<int>(cut.runs.size())};
        for (const auto& t : cut.tiles) v.insert(v.end(), {t.first, t.second});
        for (const RowRun& r : cut.runs) v.insert(v.end(), {r.row, r.rows, r.uniform ? 1 : 0});
        if (v.size() > cap) return -1;
        std::copy(v.begin(), v.end(), out);
        return static_cast<long long>(v.size());
    } catch (const std::exception&) {
        return -1;
    }
}
