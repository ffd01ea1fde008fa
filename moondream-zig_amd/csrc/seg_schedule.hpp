// Which tiles of a segmented product (seg_gemm.hip) a workgroup takes, and how long that takes: kept free of device-only calls so that
// a host program can walk the same schedule (tests/cxx/seg_schedule_check.cpp).
//
// Neighbouring workgroups land on different dies, so each die gets a contiguous run of the product's tiles, numbered as its slots, and
// its workgroups take the slots in rounds.  Where ranges of k differ in length the longest comes first and every other round goes
// backwards: whoever took the first, longest tile of a round takes the last of the next, and two rounds end as early as if the first
// free workgroup took the next slot (second product of a joined layer, 768 rows x 2048 x (2048 + 2048 + 3712): 54.5 us in rounds that
// all go the same way, 42 so).  Tiles of one length are better taken the same way every round (1920 rows x 16192 x 2048 and 64 experts'
// tiles: 1 and 3 % of a prompt).
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define SEG_FN __host__ __device__ __forceinline__
#else
#define SEG_FN inline
#endif

namespace {

constexpr int SEG_DIES = 8;

// n / d by a multiplication, for all 32-bit n (Granlund and Montgomery, "Division by invariant integers using multiplication", 1994,
// figure 4.1).  The scalar unit has no division: the half dozen that find a tile held up every workgroup's first copy and last
// store (products of 2 rows and width 1024, one tile per workgroup: 12.1 and 8.0 us with them, 11.2 and 7.4 without).
struct FastDiv {
    uint32_t mul;
    int first, second; // shifts
};
inline FastDiv fast_div(uint32_t d) {
    int l = 0;
    while (l < 32 && (uint64_t(1) << l) < d) l++;
    return {(uint32_t)((((uint64_t(1) << l) - d) << 32) / d + 1), l < 1 ? l : 1, l < 1 ? 0 : l - 1};
}
SEG_FN uint32_t seg_div(uint32_t n, const FastDiv &f) {
    const uint32_t t = (uint32_t)((uint64_t(n) * f.mul) >> 32);
    return (t + ((n - t) >> f.first)) >> f.second;
}

// A die's run is walked in blocks of 2 x SEG_BAND tiles: the 32 tiles that a die works on at once then share 512 to 1,024 rows of either
// operand, where whole columns of tiles (m first) read all of A again for every few columns: 117 against 123 us at 1920 x 16192 x
// 2048 in 256-row tiles, 130 against 152 in 128-row tiles, weights from HBM.  A column of up to three tiles is a block by itself
// (blocks would leave a single row of tiles behind: 1 to 2 % of a prompt of 300 rows).  Plain f32 products are walked m first: multiply-adds
// bound them and their workgroups are all in flight at once (width 512, two layers of 1301 rows: 1.35 ms in blocks, 1.32 m first).
// A list of row tiles (grouped rows, each with weights of its own) is walked n first in both types, see seg_find_listed.
constexpr int SEG_BAND = 8, SEG_COLUMN = 3;

struct SegWalk {
    int tiles_m, tiles_n, columns; // columns: m first
    int tiles, all;    // of one range of k, of all of them
    int slots;         // of a die, at most
    int per_die;       // longest_first: tiles of one range, otherwise of all of them
    int longest_first; // 1: every die takes its tiles of the longest range, then of the next, ..
    FastDiv by_run;    // longest_first: per_die, otherwise tiles
    FastDiv by_block;  // columns: tiles_m, otherwise the tiles of a band; listed row tiles: tiles_n
    FastDiv by_last;   // two rows of tiles of the last band
    int order[8];      // the ranges, longest first
};
inline void seg_order(const int *kb, int splits, int (&order)[8]) { // (of ranges of one length the last first)
    for (int s = 0; s < splits; s++) {
        int at = s;
        for (; at > 0 && kb[order[at - 1] + 1] - kb[order[at - 1]] <= kb[s + 1] - kb[s]; at--) order[at] = order[at - 1];
        order[at] = s;
    }
}
inline SegWalk seg_walk(int tiles_m, int tiles_n, bool m_first, const int *kb, int splits, int longest_first) {
    SegWalk w{};
    w.tiles_m = tiles_m;
    w.tiles_n = tiles_n;
    w.columns = m_first || tiles_m <= SEG_COLUMN;
    w.tiles = tiles_m * tiles_n;
    w.all = w.tiles * splits;
    w.longest_first = longest_first;
    w.per_die = ((longest_first ? w.tiles : w.all) + SEG_DIES - 1) / SEG_DIES;
    w.slots = longest_first ? w.per_die * splits : w.per_die;
    w.by_run = fast_div((uint32_t)(longest_first ? w.per_die : w.tiles));
    w.by_block = fast_div((uint32_t)tiles_m * (w.columns ? 1 : SEG_BAND));
    w.by_last = fast_div(2u * (uint32_t)(tiles_n - (tiles_n - 1) / SEG_BAND * SEG_BAND));
    seg_order(kb, splits, w.order);
    return w;
}
// row tiles from a list, up to tiles_m of them: how many there are is known on the device only
inline SegWalk seg_walk_listed(int tiles_m, int tiles_n) {
    const int kb[2] = {0, 1};
    SegWalk w = seg_walk(tiles_m, tiles_n, true, kb, 1, 0);
    w.by_block = fast_div((uint32_t)tiles_n);
    return w;
}
// workgroups that have something to do, when there are `most` (a multiple of SEG_DIES)
inline int seg_workgroups(const SegWalk &w, int most) { return SEG_DIES * w.slots < most ? SEG_DIES * w.slots : most; }
// the slot that workgroup i of a die's n takes in round r
SEG_FN int seg_slot(int longest_first, int i, int n, int r) { return r * n + (longest_first & r & 1 ? n - 1 - i : i); }

// A die's slot -> its tile's row and column of tiles and its range.  1: a tile, 0: nothing to do, -1: no slot from here on has one on
// this die.
SEG_FN int seg_find(const SegWalk &w, int die, int slot, int &tm, int &tn, int &range) {
    if (slot >= w.slots) return -1;
    int tile;
    if (w.longest_first) {
        const int before = (int)seg_div((uint32_t)slot, w.by_run);
        tile = die * w.per_die + slot - before * w.per_die;
        if (tile >= w.tiles) return 0;
        range = w.order[before];
    } else {
        const int at = die * w.per_die + slot;
        if (at >= w.all) return -1;
        range = (int)seg_div((uint32_t)at, w.by_run);
        tile = at - range * w.tiles;
    }
    const int block = (int)seg_div((uint32_t)tile, w.by_block);
    if (w.columns) {
        tn = block;
        tm = tile - block * w.tiles_m;
        return 1;
    }
    const int in = tile - block * w.tiles_m * SEG_BAND, wide = w.tiles_n - block * SEG_BAND < SEG_BAND ? w.tiles_n - block * SEG_BAND : SEG_BAND;
    const int pair = wide == SEG_BAND ? in / (2 * SEG_BAND) : (int)seg_div((uint32_t)in, w.by_last), rest = in - pair * 2 * wide;
    const int two = w.tiles_m - 2 * pair >= 2; // rows of tiles in this pair, less one
    tm = 2 * pair + (rest & two);
    tn = block * SEG_BAND + (rest >> two);
    return 1;
}

// The same for a list of which `there` row tiles exist.  The dies share the tiles that exist, and a row tile's columns follow each other: its
// rows stay in the die's L2 while the weights, read once, pass by.  Dealt as if the list were full, m first, a die's run held 16 % more
// tiles than the average, and every column of tiles read all rows again: 64 experts of 704, 768 rows of width 2048 with 8 choices, first
// product 101 -> 86 us, second 51 -> 45 (weights 369 and 184 MB, 72 and 36 us at a copy's rate); in f32 1010 -> 922 and 447 -> 447, at width 1024 508 -> 465 and
// 268 -> 259, of 300 rows 250 -> 253 and 122 -> 124.
SEG_FN int seg_find_listed(const SegWalk &w, int there, int die, int slot, int &tm, int &tn) {
    const int all = there * w.tiles_n, per_die = (all + SEG_DIES - 1) / SEG_DIES, at = die * per_die + slot;
    if (slot >= per_die || at >= all) return -1;
    tm = (int)seg_div((uint32_t)at, w.by_block);
    tn = at - tm * w.tiles_n;
    return 1;
}

// What a k-tile (64) and the rest of a tile take with every compute unit busy and weights from HBM, us, by tile height in 64 rows.  The
// higher tiles move fewer bytes per product, and a product's tiles seldom fill the last round, so the height is chosen by the
// rounds: 1920 rows x 16192 x 2048 take 126 us in 256-row tiles (4 rounds), 132 in 192, 140 in 128 (a workgroup per 128-row tile:
// 171); 1920 x 2048 x 7552 takes 77 us in 128-row tiles, 57 in 256-row tiles of two k ranges, whose second slab costs 3 us in row_finish.
constexpr int SEG_K_TILE = 64, SEG_TILE_COLUMNS = 128;
struct SegTime {
    double k_tile, rest;
};
inline SegTime seg_time(int mi) {
    constexpr SegTime by_height[3] = {{0.58, 1.5}, {0.78, 2.0}, {0.95, 2.5}};
    return by_height[mi - 2];
}
// us until the last workgroup is done with tiles of that height, range s being [kb[s], kb[s + 1])
inline double seg_estimate(int cus, int mi, int M, int N, const int *kb, int splits, bool longest_first) {
    const int tiles = (M + 64 * mi - 1) / (64 * mi) * ((N + SEG_TILE_COLUMNS - 1) / SEG_TILE_COLUMNS);
    const int per_die = ((longest_first ? tiles : tiles * splits) + SEG_DIES - 1) / SEG_DIES, slots = longest_first ? per_die * splits : per_die;
    const int n = cus / SEG_DIES < 1 ? 1 : cus / SEG_DIES;
    auto cost = [&](int s) { return (kb[s + 1] - kb[s]) / SEG_K_TILE * seg_time(mi).k_tile + seg_time(mi).rest; };
    // the first die has the longest walk; of even ranges (at most eight) it takes tiles of the first alone, the longest
    if (!longest_first) return (slots + n - 1) / n * cost(0);
    double longest = 0;
    int order[8];
    seg_order(kb, splits, order);
    for (int i = 0; i < n && i < slots; i++) {
        double t = 0;
        for (int r = 0, slot; (slot = seg_slot(1, i, n, r)) < slots; r++) t += cost(order[slot / per_die]);
        if (t > longest) longest = t;
    }
    return longest;
}

// The same for tiles of 64 mi x 256 (gemm_block.hpp).  A round's k-tiles take the longer the more units are busy (clock and L2): fitted to 70 products, 200 to
// 2048 rows by 5000 to 16832 columns by 1024 or 2048, of which these choose the faster kernel for 69 (the other one 1 % off); 15 to 20 % faster than narrow tiles alone where they
// choose wide ones.
struct SegBlockTime {
    double k_tile, busy, rest; // us: k-tile of a lone unit, what is added with all busy, a tile's rest
};
inline SegBlockTime seg_block_time(int mi) { return mi == 3 ? SegBlockTime{0.55, 0.75, 4.0} : SegBlockTime{1.08, 0.42, 4.5}; }
inline double seg_block_estimate(int cus, int mi, int M, int N, int K) {
    const SegBlockTime t = seg_block_time(mi);
    const int tiles = (M + 64 * mi - 1) / (64 * mi) * ((N + 255) / 256), n = cus / SEG_DIES < 1 ? 1 : cus / SEG_DIES;
    double us = 0;
    for (int left = (tiles + SEG_DIES - 1) / SEG_DIES; left > 0; left -= n) us += t.rest + K / SEG_K_TILE * (t.k_tile + t.busy * (left < n ? left : n) / n);
    return us;
}

// The same for tiles of 128 x 64 (gemm_thin.hpp) and ranges of k, at most a tile per unit, up to three rows of them: 8 to 128 rows x 16128 x 2048 narrow 20.6 to 25.6, thin 17.7 to 20.1 us;
// 61 x 2048 x 7552 in eight ranges 12.6 and 10.0, 61 x 4992 x 1024 10.1 and 7.7.  In more rounds they lose: 61 x 16832 x 2048, 263 thin tiles, 23.0 and 27.7.
constexpr int SEG_THIN_ROWS = 128;
inline double seg_thin_estimate(int cus, int M, int N, const int *kb, int splits, bool longest_first) {
    const int rows = (M + SEG_THIN_ROWS - 1) / SEG_THIN_ROWS, range = rows * ((N + 63) / 64), tiles = range * splits;
    const int slots = longest_first ? (range + SEG_DIES - 1) / SEG_DIES * splits : (tiles + SEG_DIES - 1) / SEG_DIES, n = cus / SEG_DIES < 1 ? 1 : cus / SEG_DIES;
    if (rows > 3 || slots > n) return 1e30; // (a die's slots: with ranges dealt longest first it has the same share of each, rounded up)
    int longest = 0;
    for (int s = 0; s < splits; s++) longest = kb[s + 1] - kb[s] > longest ? kb[s + 1] - kb[s] : longest;
    return 1.0 + longest / SEG_K_TILE * (0.24 + 0.1 * tiles / cus + 0.0008 * M / rows);
}

} // namespace
