// Host check of moondream-zig_amd/csrc/wait_places.hpp with the decode kernels' own numbers on a device of 8 dies with 32 units each: four
// workgroups per unit, 768 of the 2,048-wide layer's wait, 384 of the 1,024-wide one's, 256 of the two-launch front kernel's.
#include "wait_places.hpp"

#include <atomic>
#include <cstdio>
#include <random>
#include <thread>

static std::atomic<int> failures{0};
static void expect(bool ok, const char *what) {
    if (!ok && failures++ < 20) printf("FAILED %s\n", what);
}

int main() {
    const WaitNeed wide{96, 128}, narrow{48, 128}, front{32, 128}, half{20, 64};
    {
        WaitPlaces p;
        expect(p.take(narrow) && p.take(narrow), "two narrow sessions decode in whole-layer launches");
        expect(!p.take(narrow) && !p.take(wide), "a third does not, nor a wide one");
        p.give(narrow);
        expect(!p.take(wide) && p.take(narrow), "a narrow one again when one of them is done");
        p.give(narrow);
        p.give(narrow);
        expect(p.take(wide) && !p.take(wide) && !p.take(front) && !p.take(narrow), "a wide one beside nothing else");
        p.give(wide);
        expect(p.take(front) && p.take(front) && p.take(front) && !p.take(front), "three front kernels: 96 of 128 wait");
    }
    {
        WaitPlaces p; // a kernel of which a die holds fewer sets the limit for all
        expect(p.take(half) && p.take(half) && p.take(half) && !p.take(half), "60 of 64");
        expect(!p.take(narrow), "48 more would fill units that hold two of the larger");
        p.give(half);
        p.give(half);
        p.give(half);
        expect(p.take(narrow) && !p.take(half), "20 beside 48: over 64");
    }
    { // calls with a crowd count those that run without places too
        const WaitNeed wide_list{48, 128, 1}, narrow_list{48, 128, 2};
        for (const WaitNeed &n : {wide_list, narrow_list}) {
            WaitPlaces p;
            expect(p.enter(n) && p.enter(n), "two fit");
            expect(!p.enter(n), "a third does not");
            p.leave(n, true); // one of the first two is over and begins anew beside one with places and one without
            const bool again = p.enter(n);
            expect(again == (n.crowd > 1), "144 of 128 run");
            p.leave(n, true);
            expect(p.enter(n) == (n.crowd > 1), "the other one likewise");
            for (int i = 0; i < 2; i++) p.leave(n, n.crowd > 1);
            p.leave(n, false);
            expect(p.enter(n), "none is left behind");
        }
        WaitPlaces p;
        for (int i = 0; i < 5; i++) expect(p.enter(narrow_list) == (i < 2), "five, 240 of 256");
        p.leave(narrow_list, true);
        expect(p.enter(narrow_list), "no crowd yet");
        expect(!p.enter(narrow_list), "a sixth");
        p.leave(narrow_list, true);
        expect(!p.enter(narrow_list), "288 of 256 run");
        expect(p.enter(front) && !p.enter(wide), "without a crowd the places alone count: 32 beside 48, but not 96");
        p.leave(narrow_list, true);
        p.leave(front, true);
        expect(p.enter(wide), "96 where nobody holds any");
    }
    // threads that come and go: whatever is held at once leaves a place
    WaitPlaces p;
    std::atomic<int> waiting{0}, taken{0}, refused{0};
    std::vector<std::thread> threads;
    for (int t = 0; t < 8; t++)
        threads.emplace_back([&, t] {
            std::mt19937 rng(t);
            for (int i = 0; i < 20000; i++) {
                const WaitNeed &n = rng() % 4 ? narrow : rng() % 2 ? front : wide;
                if (!p.take(n)) {
                    refused++;
                    std::this_thread::yield();
                    continue;
                }
                taken++;
                expect((waiting += n.waiting) < 128, "all that wait at once");
                if (rng() % 2) std::this_thread::yield();
                waiting -= n.waiting;
                p.give(n);
            }
        });
    for (std::thread &t : threads) t.join();
    expect(taken > 0 && refused > 0, "both answers came up");
    expect(p.take(wide), "everything was given back");
    printf("%d taken, %d refused, %d failures\n", taken.load(), refused.load(), failures.load());
    return failures != 0;
}
