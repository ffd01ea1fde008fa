// How a token's keys are split over workgroups (layer_decode.hip, layer_whole.hip); kept free of device-only calls so that a host program
// can check it (tests/cxx/key_splits_check.cpp).
#pragma once

#include <algorithm>

constexpr int MIX_KEYS = 1024;     // keys of one split at most
constexpr int MIX_TARGET = 32;     // keys of one split at least
constexpr int MIX_SPLITS = 16;     // splits at most, unless MIX_KEYS asks for more: what the merge requests at once

// wgs: workgroups that a split takes
inline int mix_splits(int n_keys, int wgs, int cus) {
    const int S = std::min(std::min((n_keys + MIX_TARGET - 1) / MIX_TARGET, MIX_SPLITS), std::max(1, cus / wgs));
    return std::max(S, (n_keys + MIX_KEYS - 1) / MIX_KEYS);
}
inline int mix_split_keys(int n_keys, int splits) { return (n_keys + splits - 1) / splits; }
// Of any split behind up to n_keys keys.  Not always those of the last position: where MIX_KEYS asks for one split more, each gets fewer (16,384 keys are 16 times
// 1,024, 16,385 17 times 964).
inline int mix_most_split_keys(int n_keys, int wgs, int cus) {
    const int S = mix_splits(n_keys, wgs, cus);
    return S > 1 && S > mix_splits((S - 1) * MIX_KEYS, wgs, cus) ? std::max(MIX_KEYS, mix_split_keys(n_keys, S)) : mix_split_keys(n_keys, S);
}
