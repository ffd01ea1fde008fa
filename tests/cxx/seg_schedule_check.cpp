// Host check of the schedule of the segmented products (moondream-zig_amd/csrc/seg_schedule.hpp): division by multiplication against
// the division, every tile of every range taken exactly once whatever the shape and the number of workgroups, the estimate against the
// sums along every workgroup's walk (thin tiles: none has two), and the walk against a first-free-takes-the-next one where the ranges of k differ in length.
#include "seg_schedule.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <queue>
#include <random>
#include <vector>

static int failures = 0;
static long checked = 0;
static void expect(bool ok, const char *what, int a, int b, int c, int d) {
    checked++;
    if (!ok && failures++ < 20) printf("FAILED %s: %d %d %d %d\n", what, a, b, c, d);
}

// us of every workgroup's walk; counts each (tile, range) if seen is given
static std::vector<double> walk(const SegWalk &w, int most, int mi, const int *kb, std::vector<int> *seen) {
    const int grid = seg_workgroups(w, most);
    std::vector<double> us(grid, 0.0);
    for (int b = 0; b < grid; b++)
        for (int round = 0;; round++) { // (as the kernel: until a slot says that none follows)
            int tm, tn, range;
            const int r = seg_find(w, b % SEG_DIES, seg_slot(w.longest_first, b / SEG_DIES, grid / SEG_DIES, round), tm, tn, range);
            if (r < 0) break;
            if (r == 0) continue;
            us[b] += (kb[range + 1] - kb[range]) / SEG_K_TILE * seg_time(mi).k_tile + seg_time(mi).rest;
            if (tm < 0 || tm >= w.tiles_m || tn < 0 || tn >= w.tiles_n || range < 0 || range * w.tiles >= w.all) failures++;
            else if (seen) (*seen)[range * w.tiles + tn * w.tiles_m + tm]++;
        }
    return us;
}

static double first_free(int workgroups, int tiles, int mi, const int *kb, int splits) { // the longest range first
    int order[8];
    seg_order(kb, splits, order);
    std::priority_queue<double, std::vector<double>, std::greater<double>> free(std::greater<double>(), std::vector<double>(workgroups, 0.0));
    double last = 0;
    for (int o = 0; o < splits; o++)
        for (int i = 0; i < tiles; i++) {
            const int s = order[o];
            const double t = free.top() + (kb[s + 1] - kb[s]) / SEG_K_TILE * seg_time(mi).k_tile + seg_time(mi).rest;
            free.pop();
            free.push(t);
            last = std::max(last, t);
        }
    return last;
}

int main() {
    std::mt19937_64 rng(1);
    auto in = [&](uint64_t lo, uint64_t hi) { return lo + rng() % (hi - lo + 1); };

    for (int i = 0; i < 2000000; i++) {
        const uint32_t d = (uint32_t)(i < 1000 ? i + 1 : i % 3 ? in(1, uint64_t(1) << in(1, 31)) : 0xffffffffu - in(0, 1000)); // (the compiler's own '/' is the truth)
        const uint32_t n = i % 5 == 0 ? 0xffffffffu - (uint32_t)in(0, 3) : i % 5 == 1 ? (uint32_t)(d * in(0, 0xffffffffu / d)) : (uint32_t)(rng() >> in(32, 62));
        const FastDiv f = fast_div(d);
        expect(seg_div(n, f) == n / d, "division", (int)n, (int)d, 0, 0);
        if (n) expect(seg_div(n - 1, f) == (n - 1) / d, "division", (int)(n - 1), (int)d, 0, 0);
    }

    for (int i = 0; i < 4000; i++) {
        const int mi = (int)in(2, 4), M = (int)in(1, i % 2 ? 300 : 2100), N = 64 * (int)in(1, i % 3 ? 40 : 300), splits = (int)in(1, 8), longest_first = (int)in(0, 1);
        const int cus = (int)(i % 4 ? 256 : in(8, 320)), most = cus / SEG_DIES * SEG_DIES;
        const int tiles_m = (M + 64 * mi - 1) / (64 * mi), tiles_n = (N + SEG_TILE_COLUMNS - 1) / SEG_TILE_COLUMNS;
        int kb[9] = {0};
        if (longest_first)
            for (int s = 0; s < splits; s++) kb[s + 1] = kb[s] + 64 * (int)in(1, 40);
        else { // even ones, the last shorter
            const int per = 64 * (int)in(1, 40);
            for (int s = 0; s < splits; s++) kb[s + 1] = kb[s] + per;
            kb[splits] -= 64 * (int)in(0, per / 64 - 1);
        }
        const SegWalk w = seg_walk(tiles_m, tiles_n, i % 5 == 0, kb, splits, longest_first);
        std::vector<int> seen((size_t)w.tiles * splits, 0);
        const std::vector<double> us = walk(w, most, mi, kb, &seen);
        expect(std::all_of(seen.begin(), seen.end(), [](int n) { return n == 1; }), "every tile once", M, N, splits, cus);
        const double longest = *std::max_element(us.begin(), us.end()), said = seg_estimate(cus, mi, M, N, kb, splits, longest_first);
        expect(std::fabs(said - longest) <= 1e-9 * longest, "estimate of the walk", M, N, splits, cus);
    }

    // few rows in tiles of 128 x 64: where they are priced, no workgroup has to take two
    for (int i = 0; i < 4000; i++) {
        const int M = (int)in(1, 400), N = 64 * (int)in(1, 260), splits = (int)in(1, 8), longest_first = (int)in(0, 1), cus = (int)(i % 4 ? 256 : in(8, 320));
        int kb[9] = {0};
        for (int s = 0; s < splits; s++) kb[s + 1] = kb[s] + 64 * (int)(longest_first ? in(1, 40) : 8);
        if (seg_thin_estimate(cus, M, N, kb, splits, longest_first) >= 1e30) continue;
        const SegWalk w = seg_walk((M + SEG_THIN_ROWS - 1) / SEG_THIN_ROWS, (N + 63) / 64, false, kb, splits, longest_first);
        const int grid = seg_workgroups(w, cus / SEG_DIES * SEG_DIES);
        int most = 0;
        for (int b = 0; b < grid; b++) {
            int taken = 0;
            for (int round = 0, r, tm, tn, range; (r = seg_find(w, b % SEG_DIES, seg_slot(longest_first, b / SEG_DIES, grid / SEG_DIES, round), tm, tn, range)) >= 0; round++) taken += r;
            most = std::max(most, taken);
        }
        expect(most <= 1, "a thin tile per workgroup", M, N, splits, cus);
    }

    // listed row tiles: those that exist once each, and no die with more than an eighth of them, rounded up
    for (int i = 0; i < 2000; i++) {
        const int most_tiles = (int)in(1, 640), there = (int)in(0, most_tiles), tiles_n = (int)in(1, 90), most = (int)(i % 4 ? 256 : in(8, 320) / SEG_DIES * SEG_DIES);
        const SegWalk w = seg_walk_listed(most_tiles, tiles_n);
        const int grid = seg_workgroups(w, most);
        std::vector<int> seen((size_t)most_tiles * tiles_n, 0), by_die(SEG_DIES, 0);
        for (int b = 0; b < grid; b++)
            for (int round = 0, tm, tn; seg_find_listed(w, there, b % SEG_DIES, seg_slot(0, b / SEG_DIES, grid / SEG_DIES, round), tm, tn) >= 0; round++) {
                if (tm < 0 || tm >= there || tn < 0 || tn >= tiles_n) failures++;
                else seen[(size_t)tm * tiles_n + tn]++;
                by_die[b % SEG_DIES]++;
            }
        bool once = true;
        for (size_t t = 0; t < seen.size(); t++) once = once && seen[t] == (t < (size_t)there * tiles_n);
        expect(once, "every listed tile once", most_tiles, there, tiles_n, most);
        expect(*std::max_element(by_die.begin(), by_die.end()) <= (there * tiles_n + SEG_DIES - 1) / SEG_DIES, "dies share the list", most_tiles, there, tiles_n, most);
    }

    // A joined layer's second product: three ranges, the last one of another length.  The height with the smallest estimate does as well
    // as the best height would if the first free workgroup took the next tile, as long as a workgroup has two tiles.
    for (int width : {1024, 2048})
        for (int ff : {1024, 1728, 2048, 2752, 3712, 4480})
            for (int rows = width == 1024 ? 1100 : 700; rows <= 2048; rows += 4) {
                const int kb[4] = {0, width, 2 * width, 2 * width + ff};
                double best = 1e30, best_free = 1e30;
                for (int mi = 2; mi <= 4; mi++) {
                    best = std::min(best, seg_estimate(256, mi, rows, width, kb, 3, true));
                    best_free = std::min(best_free, first_free(256, (rows + 64 * mi - 1) / (64 * mi) * (width / SEG_TILE_COLUMNS), mi, kb, 3));
                }
                expect(best <= 1.02 * best_free, "as short as first-free", width, ff, rows, (int)(100 * best / best_free));
            }
    printf("%ld checks, %d failures\n", checked, failures);
    return failures != 0;
}
