// Which rows of a batch run their attention as tiles of consecutive rows of one request (on the matrix cores, a block
// per tile and kv head that walks the keys once for all its rows) and which row by row (split keys, every row reading
// its own).  Host arithmetic only.
#pragma once

#include <algorithm>
#include <cstdint>
#include <utility>
#include <vector>

#include "planner.hpp"

namespace pie_hip_driver {

struct RowRun {
    int row, rows, max_len;
    bool uniform;   // about equally long
};

struct AttentionCut {
    int tile_rows = 0;                                // the kernel's tile height
    std::vector<std::pair<int32_t, int32_t>> tiles;   // (first row, rows), in the order they start
    std::vector<RowRun> runs;                         // the other rows, in runs of neighbours
};

// Rows of which the longest context is within an eighth of the mean: their attention launch may plan one round of
// equally long blocks.
inline bool evenly_long(const BatchPlan& plan, int row, int rows) {
    if (rows < 2) return false;
    long long total = 0;
    int longest = 0;
    for (int i = row; i < row + rows; ++i) {
        total += plan.row_kv_len[i];
        longest = std::max(longest, plan.row_kv_len[i]);
    }
    return 8LL * longest * rows <= 9 * total;
}

// Decoded tokens run row by row; a portion of a prompt (8 rows or more) takes tiles where they cost less.  `full_tile`: the
// rows of the kernel's larger tile, 0 where tiles cannot serve (masks, page and head sizes, decode batches); `one_byte`: the cache's
// values.
//
// The costs, in microseconds, are fits to both kernels over portions of 8 - 512 rows behind 0 - 8000 keys, alone and beside 1 - 48
// decoded tokens, and over several portions (32, 16 and 8 query heads over 8, 4 and 2 kv heads of 128 and 64, bf16 and one-byte
// pools, whose decoding costs what their smaller size saves; 2178 points):
//   row by row: 4.5, and per 512 blocks (row, kv head) of one round 0.0185 a key (from the caches; a decoded token's own keys come
//     from memory, 2.6 as much); what goes beyond the first round costs 4 per 512 blocks more, and half a round's time once;
//     a round over 3500 bf16 keys and more reads past the caches, 1.3 as much (64 rows over 8 kv heads behind 4000 keys 104, as tiles
//     86; over a one-byte cache 88 and 91);
//     every run of rows after the first costs 6 more (a launch of few blocks, behind the one before: a token over 500 - 900 keys 8 - 10);
//   tiles: 4.2 + 0.67 per 32 keys of the longest, or 1.85 of that per step and slot once 512 blocks are more than one round.
// (Heads of 64: 0.55 of the first, 0.57 per 32 keys.)  So a portion takes tiles about from where its rows fill a round, 512 blocks,
// whatever is cached: 64 / 80 rows over 8 kv heads of 128 take, row by row and as tiles, 5.1 and 6.1 / 8.2 and 7.0 us without a context, 11.1
// and 11.8 / 16.4 and 12.4 behind 256 keys, 40.5 and 46.7 / 70.1 and 46.1 behind 2000; over 4 kv heads 128 / 144 rows behind 2000 41.7 and 47.4 /
// 74.9 and 47.3.  20 decoded tokens over 800 keys, 500 rows, a token, 400 rows and a token take 105 row by row and 58 cut into three
// runs beside tiles (over 4 kv heads 65 and 55); four times a token over 500 keys and 130 rows, and a token, 42 and 56.
// Over the 1500 points of single portions the rule is 1.1 % from the faster form on average, over the others 5.3 %.
inline AttentionCut cut_attention(const BatchPlan& plan, int kv_heads, int head_dim, bool one_byte, int full_tile) {
    AttentionCut cut;
    const double size = head_dim == 64 ? 0.55 : 1.0;
    const double step_us = head_dim == 64 ? 0.57 : 0.67;
    const double block_key_us = 0.0185 * size / 512.0;
    constexpr int kMinRows = 8;
    auto rows_of = [&](int r) { return plan.qo_indptr[r + 1] - plan.qo_indptr[r]; };
    auto last_of = [&](int r) { return plan.row_kv_len[plan.qo_indptr[r + 1] - 1]; };
    // the tiled requests of a choice: portions over at most `most` keys
    auto tiled = [&](int r, int most) { return rows_of(r) >= kMinRows && last_of(r) <= most; };
    auto runs_of = [&](int most) {
        std::vector<RowRun> runs;
        for (int r = 0; r < plan.R; ++r) {
            const int q0 = plan.qo_indptr[r], q1 = plan.qo_indptr[r + 1];
            if (q0 == q1 || tiled(r, most)) continue;
            if (runs.empty() || runs.back().row + runs.back().rows != q0) runs.push_back({q0, 0, 0, false});
            runs.back().rows += q1 - q0;
            for (int i = q0; i < q1; ++i) runs.back().max_len = std::max(runs.back().max_len, plan.row_kv_len[i]);
        }
        return runs;
    };
    auto by_rows_us = [&](int rows, double keys, int longest) {   // one run
        const double rounds = rows * static_cast<double>(kv_heads) / 512.0;
        const double far = !one_byte && rounds <= 1.0 && size * rounds * longest >= 3500.0 ? 1.3 : 1.0;
        return 4.5 + far * block_key_us * kv_heads * keys + (rounds > 1.0 ? 4.0 * size * (rounds - 1.0) + 0.5 * 512.0 * block_key_us * longest : 0.0);
    };
    auto keys_of = [&](int r) {
        const int n = rows_of(r);
        return (n < kMinRows ? 2.6 : 1.0) * n * (last_of(r) - 0.5 * (n - 1));
    };
    auto tiles_us = [&](double steps, double block_steps) { return 4.2 + step_us * std::max(steps, 1.85 * block_steps / 512.0); };
    auto steps_of = [](double keys) { return keys / 32.0 + 0.5; };
    auto cost = [&](int most) {
        double us = 0.0, keys = 0.0, block_steps = 0.0, steps = 0.0;
        int rows = 0, longest = 0, runs = 0;
        auto end_run = [&] {
            if (rows) us += by_rows_us(rows, keys, longest) + (runs++ ? 6.0 : 0.0);
            rows = longest = 0;
            keys = 0.0;
        };
        for (int r = 0; r < plan.R; ++r) {
            const int n = rows_of(r);
            if (n == 0) continue;
            if (tiled(r, most)) {
                const int tiles = (2 * n + full_tile - 1) / full_tile;
                steps = std::max(steps, steps_of(last_of(r)));
                block_steps += tiles * kv_heads * steps_of(last_of(r) - 0.5 * n);
                end_run();
            } else {
                rows += n;
                keys += keys_of(r);
                longest = std::max(longest, last_of(r));
            }
        }
        end_run();
        return us + (block_steps > 0.0 ? tiles_us(steps, block_steps) : 0.0);
    };
    constexpr int kNone = -1, kAll = 0x7FFFFFFF;
    int most = kNone;
    if (full_tile > 0) {
        // every portion; those that alone would gain, and shorter ones, which ride along; none
        int gain = kNone;
        for (int r = 0; r < plan.R; ++r)
            if (rows_of(r) >= kMinRows && by_rows_us(rows_of(r), keys_of(r), last_of(r)) > tiles_us(steps_of(last_of(r)), 0.0))
                gain = std::max(gain, last_of(r));
        double best = cost(kNone);
        for (int cand : {gain, kAll}) {
            const double c = cost(cand);
            if (c < best) {
                best = c;
                most = cand;
            }
        }
    }
    if (most != kNone) cut.runs = runs_of(most);
    else cut.runs.push_back({0, plan.N, plan.max_kv_len, false});
    for (RowRun& run : cut.runs) run.uniform = !plan.pure_decode && evenly_long(plan, run.row, run.rows);
    if (most == kNone) return cut;
    long long blocks = 0;
    for (int r = 0; r < plan.R; ++r)
        if (tiled(r, most)) blocks += static_cast<long long>((rows_of(r) + full_tile - 1) / full_tile) * kv_heads;
    // fewer than three full-size blocks per CU: halve the tiles (measured on a causal prompt of
    // 2048 tokens, 512 full-size blocks: 110 -> 100 us; of 3072 tokens, 768 blocks: 169 -> 179)
    cut.tile_rows = blocks < 768 ? full_tile / 2 : full_tile;
    // Longest first: the kernel starts its blocks in tile order, and a long causal tile started
    // last would run on alone.
    for (int r = 0; r < plan.R; ++r)
        for (int t0 = plan.qo_indptr[r]; tiled(r, most) && t0 < plan.qo_indptr[r + 1]; t0 += cut.tile_rows)
            cut.tiles.emplace_back(t0, std::min(cut.tile_rows, plan.qo_indptr[r + 1] - t0));
    std::stable_sort(cut.tiles.begin(), cut.tiles.end(), [&](const auto& a, const auto& b) {
        return plan.row_kv_len[a.first + a.second - 1] > plan.row_kv_len[b.first + b.second - 1];
    });
    // More blocks than run in two groups, one to a CU: every second round of 256 the other way round, so that the blocks that
    // share a CU have about as many steps together as any others (a causal prompt of 2048 tokens, 32 heads over 8: 92 -> 83 us;
    // 3000: 167 -> 156; 4096: 273 -> 256; of 1024, 512 blocks: 34 -> 40).
    const size_t round = static_cast<size_t>(std::max(1, 256 / kv_heads));
    for (size_t at = round; cut.tiles.size() * kv_heads > 512 && at < cut.tiles.size(); at += 2 * round)
        std::reverse(cut.tiles.begin() + at, cut.tiles.begin() + std::min(at + round, cut.tiles.size()));
    return cut;
}

}  // namespace pie_hip_driver
