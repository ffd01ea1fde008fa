// Host check of the choice of tiles for the f16 products (moondream-zig_amd/csrc/gemm_choice.hpp): the prompts of the GPU tests take the forms that
// those tests are about, and a joint launch of out_proj and fc2 fits the units with no empty range of k, whatever the shape.
#include "gemm_choice.hpp"

#include <cstdio>
#include <random>

static int failures = 0;
static long checked = 0;
static void expect(bool ok, const char *what, int a, int b, int c, int d) {
    checked++;
    if (!ok && failures++ < 20) printf("FAILED %s: %d %d %d %d\n", what, a, b, c, d);
}

int main() {
    // width, feed-forward, rows; form of the front (0: thin tiles, 3, 4: wide ones of 192 and 256 rows, -1: launches apart), with the rotation in it and without; form of the pair (-1: not asked)
    const struct {
        int width, ffn, rows, front, unturned, pair;
    } prompts[] = {
        {192, 776, 37, 0, 0, -1},      {192, 776, 130, 0, 0, -1},     {192, 776, 385, 0, 0, -1},     {192, 832, 64, 0, 0, PAIR_THIN}, {192, 832, 129, 0, 0, PAIR_THIN},
        {192, 832, 513, 0, 0, PAIR_NARROW}, {512, 2048, 2, 0, 0, PAIR_THIN}, {512, 2048, 37, 0, 0, PAIR_THIN}, {512, 2048, 129, 0, 0, PAIR_THIN}, {512, 2048, 191, 0, 0, PAIR_THIN},
        {512, 2048, 192, 0, 0, PAIR_NARROW}, {512, 2048, 385, 0, 0, PAIR_NARROW}, {512, 2048, 700, 0, 0, PAIR_NARROW},
        {960, 3840, 129, 0, 0, PAIR_THIN}, {960, 3840, 130, 0, 0, PAIR_THIN}, {960, 3840, 897, 3, -1, PAIR_NARROW}, {960, 3840, 1729, 4, 4, PAIR_NARROW},
        {2048, 8192, 37, 0, 0, PAIR_THIN}, {2048, 8192, 700, 3, 3, PAIR_NARROW}, {2048, 8192, 769, 4, 4, PAIR_WIDE}, {2048, 8192, 1000, 4, 4, PAIR_WIDE}, {2048, 8192, 1025, 3, 3, PAIR_WIDE},
    };
    for (const auto &p : prompts) {
        for (int turned = 0; turned < 2; turned++) {
            const FrontForm f = front_form(256, p.rows, 3 * p.width, p.ffn, p.width / CHOICE_K_TILE, turned);
            expect((f.thin ? 0 : f.mi ? f.mi : -1) == (turned ? p.front : p.unturned), "form of the front", p.width, p.ffn, p.rows, turned);
        }
        if (p.pair < 0) continue;
        const PairForm f = pair_form(256, p.rows, p.width, p.width / CHOICE_K_TILE, p.ffn / CHOICE_K_TILE);
        expect(f.a && f.tile == p.pair, "form of the pair", p.width, p.ffn, p.rows, f.tile);
    }

    std::mt19937_64 rng(1);
    auto in = [&](int lo, int hi) { return lo + (int)(rng() % (hi - lo + 1)); };
    for (int i = 0; i < 200000; i++) {
        const int cus = i % 4 ? 256 : in(8, 320), M = in(2, i % 2 ? 400 : 4000), N = 8 * in(1, 256), kt[2] = {in(1, 40), in(1, 160)};
        const PairForm f = pair_form(cus, M, N, kt[0], kt[1]);
        if (!f.a) continue;
        const int rows = f.tile == PAIR_THIN ? CHOICE_THIN_ROWS : 192, columns = f.tile == PAIR_THIN ? CHOICE_THIN_COLUMNS : f.tile == PAIR_WIDE ? CHOICE_WIDE_COLUMNS : CHOICE_COLUMNS;
        expect(f.tiles_m * rows >= M && (f.tiles_m - 1) * rows < M && f.tiles_n * columns >= N && (f.tiles_n - 1) * columns < N, "tiles cover the result", M, N, f.tiles_m, f.tiles_n);
        expect(f.tiles_m * f.tiles_n * (f.a + f.s) <= cus && f.a <= kt[0] && f.s <= kt[1], "one round of ranges that are not empty", M, N, f.a, f.s);
    }
    printf("%ld checks, %d failures\n", checked, failures);
    return failures != 0;
}
