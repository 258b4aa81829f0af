// fixed_plan.h -- tiles and K splits of the one-group GEMMs (dense layers, LM
// head; grouped_gemm_fixed_kernel).  Plain C++ so a host build can check the
// plans (tests/fixed_plan).
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>

namespace hf {

constexpr int kGemmTileRows = 128;  // M rows per grouped-GEMM tile (kPrefillTileRows at prefill sizes)

// One-group tiles of launch_fixed_gemm: eight wavefronts of 16 cb weight rows
// each over up to fixed_tile_rows(cb) rows of A (160 and 4 column blocks, or
// 128 and 5: what a wavefront's accumulators have registers for), and their
// output columns (pair: as many columns of each of gate and up).
constexpr int fixed_tile_rows(int cb) { return cb == 5 ? 128 : 160; }
constexpr int fixed_tile_cols(int cb, bool pair) { return pair ? 64 * cb : 128 * cb; }

// How launch_fixed_gemm covers T rows x N columns: M tiles of tile_rows rows,
// N tiles, K splits (1 unless splits are worth their partials' traffic).
struct FixedPlan {
    int m_tiles = 0, tile_rows = 0, n_tiles = 0, ksplit = 1;
    double us = 0;  // estimate
};
// Tiles and K splits by an estimate of the launch's time, in us: rounds of
// items x (K stages + 3 to fill and drain) x the time of a stage, plus the
// pass that sums the splits.  A stage of 4 column blocks takes a workgroup
// 0.5 + 0.3 us per 16-row block to multiply (A as two halves: T = 777, five
// tiles of 160 rows, 99 stages in 348 us; T = 400, five of 80, 206 us), and
// its 64 KB of weights arrive at 36 GB/s on one CU and 7.2 TB/s on all (the M
// tiles of a weight tile share them): T = 16, 24576 rows x 6144 in 2 / 3 / 4 /
// 5 / 10 splits 79 / 67 / 53 / 52 / 58 us.  Neither hides the other wholly
// (third powers: T = 128 in 5 splits 78 against 79 us measured).  Tiles lower
// than need be are tried too: T = 2048 takes 16 of 128 rows in 3 whole rounds
// rather than 13 of 160 in 2.4 (864 us against 1011).
// stages: K / 64; max_splits: what the caller's partials hold (at least 1);
// blocks: CUs.
inline FixedPlan plan_fixed_gemm(int T, int N, bool pair, int cb, int stages, int max_splits, int blocks) {
    FixedPlan best;
    const int most = fixed_tile_rows(cb);
    const int n_tiles = (N + fixed_tile_cols(cb, pair) - 1) / fixed_tile_cols(cb, pair);
    const int m_min = (T + most - 1) / most;
    const double kb = 16.0 * cb;  // KB of weights per stage
    const double out_mb = (double)T * N * (pair ? 2 : 1) * 4e-6;
    for (int m = m_min; m <= 2 * m_min; ++m) {
        const int rows = ((T + m - 1) / m + 15) / 16 * 16;
        const int m_tiles = (T + rows - 1) / rows;
        const double mul = (0.5 + 0.3 * (rows / 16)) * cb / 4;
        for (int ks = 1; ks <= max_splits; ++ks) {
            const int items = m_tiles * n_tiles * ks;
            if (ks > 1 && (items > 4 * blocks || ks * 4 > stages)) break;
            const int rounds = (items + blocks - 1) / blocks;
            const double mem = std::max(kb / 36.0, kb * std::min(items, blocks) / m_tiles / 7200.0);
            const double stage = std::cbrt(mem * mem * mem + mul * mul * mul);
            const double us =
                4.0 + rounds * ((stages + ks - 1) / ks + 3) * stage + (ks > 1 ? 3.0 + 0.3 * ks * out_mb : 0.0);
            if (best.n_tiles == 0 || us < best.us) best = FixedPlan{m_tiles, rows, n_tiles, ks, us};
        }
    }
    return best;
}

constexpr int kFixedMaxSplits = 32;
// Whether a GEMM of T rows against `weights` BF16 values takes these tiles at
// all.  Below 16 MB of weights and one 128-row tile it is a few microseconds
// of latency, and the 128-row kernel's smaller workgroups start sooner
// (512 x 1536 dense layer, T = 30: 24 against 27 us; T = 300: 68 against 46
// us the other way).  From 4 GiB on its 32-bit byte offsets do not reach.
inline bool fixed_worth(int T, size_t weights) {
    return weights < ((size_t)1 << 31) && (T > kGemmTileRows || weights >= ((size_t)8 << 20));
}

}  // namespace hf
