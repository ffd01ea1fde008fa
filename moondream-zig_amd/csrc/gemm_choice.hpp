// Which tiles the f16 products with more than one form take, from their shapes alone: kept free of device code so that a host program can ask
// for the choice (tests/cxx/gemm_choice_check.cpp).
#pragma once

#include <algorithm>
#include <cstddef>

namespace {

constexpr int CHOICE_K_TILE = 64, CHOICE_COLUMNS = 128;                // of the narrow kernels
constexpr int CHOICE_THIN_ROWS = 128, CHOICE_THIN_COLUMNS = 64;        // gemm_thin.hpp
constexpr int CHOICE_WIDE_COLUMNS = 256;                               // gemm_block.hpp, by 64 mi rows

// What products take, us, launch included, with weights from HBM, kt k-tiles: fitted to 54 products of 200 to 1920 rows by 3072 to 14336 columns by 1024 or 2048.
// Over 42 weights (3072 to 24576 columns by 512 to 4096) at 8 to 1920 rows the wide and thin tiles' say 0.8 to 1.5 times what was measured (1.0 to 1.3 at the median of each K), the narrow kernels' 0.6 to 2.2 (0.9 to
// 1.2), so a choice errs towards launches apart.  432 prompts of 12 models (width 512 to 2560, 2 to 1900 rows) against those launches: 1.27 times as fast in the mean, none slower but width 2560 at 100 to 160 rows, 2.5 %
// (its rows lie 5,120 bytes apart, and a thin k-tile of 100 of them takes 1.3 times as long as of 37).
// seg_schedule.hpp prices the same loops for bf16 products, without a launch and beside other narrow kernels: each set of constants was fitted to its own measurements.
// Tiles of 64 mi x 256 in rounds over the units; f: part of the units that a round keeps busy.
inline double block_us(int cus, int mi, size_t M, size_t columns, size_t kt) {
    const size_t tiles = (M + 64 * mi - 1) / (64 * mi) * columns;
    double us = mi == 3 ? 10.5 : 11;
    for (size_t left = tiles; left > 0; left -= std::min(left, (size_t)cus)) {
        const double f = (double)std::min(left, (size_t)cus) / cus;
        us += (left < tiles ? 6 : 0) + kt * (mi == 3 ? 0.78 + 0.42 * f : 1.03 + 0.5 * f);
    }
    return us;
}
inline int block_height(int cus, size_t M, size_t columns, size_t kt, double *us) {
    const double three = block_us(cus, 3, M, columns, kt), four = block_us(cus, 4, M, columns, kt);
    *us = std::min(three, four);
    return three <= four ? 3 : 4;
}
// Tiles of 128 x 64 (gemm_thin.hpp); later rounds find their first k-tiles on their way.
inline double thin_us(int cus, size_t M, size_t N, size_t kt) {
    const size_t rows = (M + CHOICE_THIN_ROWS - 1) / CHOICE_THIN_ROWS, tiles = rows * ((N + CHOICE_THIN_COLUMNS - 1) / CHOICE_THIN_COLUMNS);
    double us = 5.5;
    for (size_t left = tiles; left > 0; left -= std::min(left, (size_t)cus))
        us += (left < tiles ? 0.85 : 1.0) * kt * (0.24 + 0.1 * std::min(left, (size_t)cus) / cus + 0.0008 * M / rows);
    return us;
}
// The narrow kernels as run_gemm takes them: 128 x 128 tiles, split in k where they are few (the reduction 6 us), otherwise a workgroup per tile of 192 or 256 rows.
inline double narrow_us(int cus, size_t M, size_t N, size_t kt) {
    const size_t columns = (N + CHOICE_COLUMNS - 1) / CHOICE_COLUMNS, t128 = (M + 127) / 128 * columns, t192 = (M + 191) / 192 * columns, t256 = (M + 255) / 256 * columns;
    if (t128 * 2 <= (size_t)cus) return 10 + 0.47 * kt / std::max<size_t>(1, std::min({(size_t)cus / t128, kt / 8, (size_t)8}));
    if (t128 <= (size_t)cus) return 4 + 0.47 * kt;
    if (t192 <= (size_t)cus && t192 > t256) return 7 + kt * (0.45 + 0.28 * t192 / cus);
    double us = 7.5;
    for (size_t left = t256; left > 0; left -= std::min(left, (size_t)cus)) us += (left < t256 ? 6 : 0) + kt * std::max(0.6, 0.28 + 0.62 * std::min(left, (size_t)cus) / cus);
    return us;
}

// A decoder's qkv projection (N columns) beside its fc1 (N1): one launch of thin tiles, of wide ones of 64 mi rows, or neither: launches apart.
struct FrontForm {
    bool thin = false;
    int mi = 0;
};
inline FrontForm front_form(int cus, size_t M, size_t N, size_t N1, size_t kt, bool fused) {
    double wide;
    const int mi = block_height(cus, M, (N + CHOICE_WIDE_COLUMNS - 1) / CHOICE_WIDE_COLUMNS + (N1 + CHOICE_WIDE_COLUMNS - 1) / CHOICE_WIDE_COLUMNS, kt, &wide);
    const double thin = thin_us(cus, M, N + N1, kt);
    // Apart: two products, the GELU of one (2.5 us) and, where the launch would do it, the rotation (4.5).
    if (std::min(wide, thin) >= narrow_us(cus, M, N, kt) + narrow_us(cus, M, N1, kt) + (fused ? 7.0 : 2.5)) return {};
    return thin < wide ? FrontForm{true, 0} : FrontForm{false, mi};
}

// out_proj beside fc2, kt_add and kt k-tiles: the tiles, how many, and the ranges of k of each (a, s; a = 0: launches apart).
enum PairTile { PAIR_THIN, PAIR_NARROW, PAIR_WIDE };
struct PairForm {
    PairTile tile = PAIR_NARROW;
    int tiles_m = 0, tiles_n = 0, a = 0, s = 0;
    double us = 1e30;
};
// Splits (a, s): all workgroups in one round, the longest run of k-tiles as short as it gets, us at `fixed` for a launch and `one` + `all` * busy units for a k-tile,
// and for every range its sums, written and read (8 TB/s: they stay in the memory-side cache).
inline PairForm pair_plan(int cus, size_t M, size_t N, int kt_add, int kt, PairTile tile, int tile_m, int tile_n, double fixed, double one, double all) {
    PairForm p;
    p.tile = tile;
    p.tiles_m = (int)((M + tile_m - 1) / tile_m);
    p.tiles_n = (int)((N + tile_n - 1) / tile_n);
    const int tiles = p.tiles_m * p.tiles_n;
    int best_len = 1 << 30;
    for (int a = 1; a <= 8 && a <= kt_add; a++)
        for (int s = 1; s <= 8 && s <= kt; s++) {
            if (tiles * (a + s) > cus) continue;
            const int len = std::max((kt_add + a - 1) / a, (kt + s - 1) / s);
            if (len < best_len || (len == best_len && a + s < p.a + p.s)) {
                best_len = len;
                p.a = a;
                p.s = s;
            }
        }
    if (p.a) p.us = fixed + best_len * (one + all * tiles * (p.a + p.s) / cus) + (p.a + p.s) * (double)M * N * 8 / 8e6;
    return p;
}
// Below 192 rows tiles of 128 x 64 (gemm_thin.hpp): 37 rows of width 2048, apart 8.3 and 15.9 us.  From there on 192 x 128, or 192 x 256 (gemm_block.hpp) where those leave few ranges of
// k: a layer of width 2048 at 850 rows 139 -> 128 us, 1025 192 -> 161, 1536 230 -> 198; at 768 rows 192 x 128 is 2 % faster, at width 1024 up to 9.
// The line at 192 rows: a layer of width 1024 and 2048 takes 32.6 and 62.4 us at 170 rows, 36.0 and 64.1 in 192 x 128.  Thin tiles go on to win up to 256 rows (230: 33.3 and 68.0, 192 x 128 36.8 and 72.8) and
// lose behind them at width 2048 (260: 91.6 and 79.9; at width 1024 40.3 and 43.1), which this line does not use.
inline PairForm pair_form(int cus, size_t M, size_t N, int kt_add, int kt) {
    if (M < 192) return pair_plan(cus, M, N, kt_add, kt, PAIR_THIN, CHOICE_THIN_ROWS, CHOICE_THIN_COLUMNS, 0, 1, 0);
    const PairForm narrow = pair_plan(cus, M, N, kt_add, kt, PAIR_NARROW, 192, CHOICE_COLUMNS, 7, 0.45, 0.28), wide = pair_plan(cus, M, N, kt_add, kt, PAIR_WIDE, 192, CHOICE_WIDE_COLUMNS, 10, 0.78, 0.42);
    return wide.us < narrow.us ? wide : narrow;
}

} // namespace
