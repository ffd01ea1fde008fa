// Host check of moondream-zig_amd/csrc/launch_counts.hpp: whatever becomes of a launch, the counters on the device are what the next launch's targets start from,
// or the error word says that they are not.
#include "launch_counts.hpp"

#include <cstdio>
#include <cstring>
#include <random>

static int failures = 0;
static void expect(bool ok, const char *what) {
    if (!ok && failures++ < 20) printf("FAILED %s\n", what);
}

int main() {
    std::mt19937 rng(1);
    int ran = 0, lost = 0, stray = 0, broken = 0;
    LaunchTargets at, device;
    volatile uint32_t error = 0;
    for (int i = 0; i < 20000; i++) {
        LaunchTargets add;
        for (uint32_t &v : add.leaf) v = rng() % 3 * 7;
        for (uint32_t &v : add.reached) v = rng() % 3 ? 0x10000000u + rng() % 64 : 0; // (counts wrap)
        LaunchTargets next = at;
        for (int k = 0; k < 2; k++) next.leaf[k] += add.leaf[k];
        for (int k = 0; k < 3; k++) next.reached[k] += add.reached[k];
        const int kind = rng() % 8; // 0: never ran; 1: ran, with an earlier call's error; 2: never ran, and the clear fails; others run
        const int rc = launch_counted(
            &at, next, &error,
            [&] {
                if (kind == 0 || kind == 2) return 5;
                for (int k = 0; k < 2; k++) device.leaf[k] += add.leaf[k];
                for (int k = 0; k < 3; k++) device.reached[k] += add.reached[k];
                return kind == 1 ? 5 : 0;
            },
            [&] {
                if (kind == 2) return 7;
                device = LaunchTargets{};
                return 0;
            });
        (kind == 0 ? lost : kind == 1 ? stray : kind == 2 ? broken : ran)++;
        expect(rc == (kind < 3 ? 5 : 0), "the launch's own result comes back");
        if (kind == 2) {
            expect(error == 1, "a clear that failed is remembered");
            device = at = LaunchTargets{}; // (what the session's reset does)
            error = 0;
        }
        expect(error == 0 && !memcmp(&at, &device, sizeof at), "targets and counters agree");
    }
    expect(ran && lost && stray && broken, "every case came up");
    printf("%d ran, %d never, %d with a stray error, %d not cleared, %d failures\n", ran, lost, stray, broken, failures);
    return failures != 0;
}
