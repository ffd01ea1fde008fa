// Host check of moondream-zig_amd/csrc/whole_share.hpp: the producers of a layer's launch over the sizes, keys and units it is asked for.
#include "whole_share.hpp"

#include <cstdio>
#include <random>

static int failures = 0;
static void expect(bool ok, const char *what) {
    if (!ok && failures++ < 20) printf("FAILED %s\n", what);
}
static double pairs(const WholeWork &w, int n) { return (w.front + w.ff) / (4.0 * n); }

int main() {
    // width 1024, 16 key heads, 16 delta heads, feed-forward 1728: behind 45 keys 160 workgroups wait, behind 600 416
    const int front = (3 * 1024 + 3 * 1024 + 128) / 2 + 8;
    WholeWork joined{front, 1728, true, 32 + 16 + 128, 4, 256, 32};
    expect(whole_producers(joined) == 320, "two a unit where a wavefront has few pairs");
    joined.waiting = 256 + 16 + 128;
    expect(whole_producers(joined) == 608, "all places where two a unit leave 96 producers");
    // width 1024, feed-forward 9856: a wavefront of two a unit has nine pairs
    expect(whole_producers({2048, 9856, true, 176, 5, 256, 32}) == 1088, "all places for a large feed-forward");
    expect(whole_producers({2048, 9856, true, 176, 2, 256, 32}) == 0, "three launches where a unit holds no more than two");
    // width 2048, 32 key heads without a window: 256 + 32 a thousand keys wait
    for (int thousands = 8; thousands < 24; thousands++) {
        const WholeWork w{4096, 5504, false, 256 + 32 * thousands, 4, 256, 1000};
        const int n = whole_producers(w);
        expect(n == (thousands < 23 ? 1024 - w.waiting : 0), "what long contexts leave, until it is too little");
    }
    std::mt19937 rng(1);
    int one = 0, three = 0, all = 0;
    for (int i = 0; i < 200000; i++) {
        WholeWork w{int(rng() % 7000) + 1, rng() % 4 ? int(rng() % 10241) : 0, rng() % 2 == 0, int(rng() % 1400) + 1, int(rng() % 5) + 1, rng() % 4 ? 256 : int(rng() % 300) + 8, int(rng() % 1025)};
        const int n = whole_producers(w), places = w.per_cu * w.cus;
        if (!n) {
            three++;
            continue;
        }
        one++;
        expect(n % WHOLE_LEAVES == 0 && n >= WHOLE_LEAVES, "whole leaves");
        expect(n == WHOLE_LEAVES || n + w.waiting <= places, "producers have places of their own");
        expect(pairs(w, n) <= (w.split_keys > 512 ? 40 : 9), "few pairs a wavefront");
        if (w.narrow && n + w.waiting > 2 * w.cus && n > WHOLE_LEAVES) {
            all++;
            WholeWork two = w;
            two.per_cu = std::min(w.per_cu, 2);
            const int m = std::max((2 * w.cus - w.waiting) / WHOLE_LEAVES, 1) * WHOLE_LEAVES;
            expect(pairs(w, m) > 5 && n >= m, "more than two a unit only where those leave many pairs");
        }
    }
    expect(one && three && all, "every answer came up");
    printf("%d in one launch, %d of them with all places, %d in three, %d failures\n", one, all, three, failures);
    return failures != 0;
}
