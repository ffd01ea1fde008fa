// Host check of moondream-zig_amd/csrc/key_splits.hpp: what sizes a launch for all positions of a session holds at every one of them.
#include "key_splits.hpp"

#include <cstdio>

static int failures = 0;
static void expect(bool ok, const char *what, int n, int wgs) {
    if (!ok && failures++ < 20) printf("FAILED %s: %d keys, %d workgroups a split\n", what, n, wgs);
}

int main() {
    int fewer = 0;
    for (const int cus : {256, 64, 8})
        for (const int wgs : {1, 2, 3, 4, 5, 8, 11, 16, 20, 32, 33, 64, 128, 200, 256, 300}) {
            int most = 0, splits = 0;
            for (int n = 1; n <= 40000; n++) {
                const int S = mix_splits(n, wgs, cus), keys = mix_split_keys(n, S);
                expect(S >= splits, "splits never get fewer with more keys", n, wgs);
                expect(keys <= MIX_KEYS && S * keys >= n, "the splits hold all keys", n, wgs);
                fewer += keys < most;
                splits = S;
                most = std::max(most, keys);
                const int said = std::max(MIX_TARGET, mix_most_split_keys(n, wgs, cus));
                expect(said >= most, "no split has more keys at an earlier position", n, wgs);
                expect(said == std::max(MIX_TARGET, most), "and some split has as many", n, wgs);
            }
        }
    printf("%d positions with fewer keys a split than an earlier one, %d failures\n", fewer, failures);
    return failures != 0 || !fewer;
}
