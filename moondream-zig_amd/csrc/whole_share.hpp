// How many producers a layer's launch is given (layer_whole.hip); kept free of device-only calls so that a host program can check it
// (tests/cxx/whole_share_check.cpp).
#pragma once

#include <algorithm>

constexpr int WHOLE_LEAVES = 32; // the producers' counts come together on so many lines: their number is a multiple

struct WholeWork {
    int front, ff;           // pairs of weight rows that come first or with the gate, and of gate/up rows
    bool narrow;             // width up to 1024
    int waiting;             // workgroups that wait
    int per_cu, cus;         // workgroups of the launch that a unit holds, units
    int split_keys;          // keys of a split
};

// 0: the layer takes three launches.
// Wide layers take all the places there are.  Narrow ones take two a unit, where a wavefront has few pairs, and all otherwise (us a token of 12 layers of width 1024, 16 key
// heads, two against all: 4.2 pairs 211 / 210, 6.3 222 / 219, joined 266 / 253; 9.5 263 / 236, joined 12.7 328 / 277; 6 of feed-forward 9856 9.3 177 / 149; joined ones of 4 key
// heads 3.2 234 / 235, 3.6 259 / 261).
// A wavefront asks for a pair when the one before is summed, so its time is its pairs', and with too many of them three launches, whose workgroups all produce, are faster: one
// against three with producers taken away, behind 100 to 500 keys, 8.0 to 8.7 pairs 0.99 to 1.15 times as fast, 10 to 10.9 0.95 to 1.10, 12.4 to 13 0.89 to 1.03.  Behind long contexts the
// attention is most of the time and the three launches' is the slower one: splits of 700 to 1,000 keys, 9.4 to 16 pairs 1.08 to 1.52, 37.5 to 40 1.18 to 1.35, 75 to 78 0.95 to 0.99.
constexpr int WHOLE_FEW_PAIRS = 5, WHOLE_MOST_PAIRS = 9, WHOLE_MOST_PAIRS_LONG = 40, WHOLE_LONG_SPLIT = 512;
inline int whole_producers(const WholeWork &w) {
    const int most = (std::max(w.front, w.ff) + 3) / 4; // (a pair of rows per wavefront at least)
    auto of = [&](int places) { return std::max(std::min(places - w.waiting, most) / WHOLE_LEAVES, 1) * WHOLE_LEAVES; };
    auto over = [&](int n, int pairs) { return w.front + w.ff > 4 * n * pairs; };
    int n = of((w.narrow ? std::min(w.per_cu, 2) : w.per_cu) * w.cus);
    if (w.narrow && over(n, WHOLE_FEW_PAIRS)) n = of(w.per_cu * w.cus);
    return over(n, w.split_keys > WHOLE_LONG_SPLIT ? WHOLE_MOST_PAIRS_LONG : WHOLE_MOST_PAIRS) ? 0 : n;
}
