// How workgroups of one launch wait for each other: counters that only rise, polled by one thread, every wait bounded.
#pragma once
#include "epilogue.hpp"

namespace {

constexpr int LAYER_LINE = 32;                       // uint32 per 128-byte line
// The two counters that all the output workgroups wait for ("fc1 leaves complete", "heads merged") exist in LAYER_COPIES copies
// each: whoever completes a leaf or merges a head adds to every copy (one atomic instruction, a lane per copy), and an output
// workgroup polls the copy of its index.  512 workgroups polling one line keep the memory channel that holds it busy (a poll
// is a read at the memory side), and everything else that lives in that channel, a 128th of the weight stream included,
// waits behind them: with the polls of these two counters replaced by fixed delays (timing only) the launch was 4.7 %
// shorter.  The copies are LAYER_COPY_STRIDE words apart (4 KiB + 256 B), which lands them in different channels whether the
// channels interleave by 256 bytes or by pages.
constexpr int LAYER_COPIES = 64;
constexpr int LAYER_COPY_STRIDE = 1088;
constexpr long long FRONT_TIMEOUT_TICKS = 100000000LL; // 1 s of the 100 MHz wall clock

// thread 0 of the workgroup polls *word until it reaches target; the clock and the error word are looked at once in
// 64 polls.  Returns (to every thread) whether the wait succeeded.  report: for the host, written only where a wait fails.
// error lies in the device's memory: with hundreds of workgroups that looked at a page-locked word, any wait of more than 64 polls (about 20 us) became some 10 us longer
// (list decoders' layers in one launch: 12 without a feed-forward, width 1024 299 us a token in place of 189, 4 behind 5,000 keys 146 in place of 106).
__device__ __forceinline__ bool wait_reached(uint32_t *word, uint32_t target, uint32_t *error, int *s_flag, uint32_t *report = nullptr) {
    lds_barrier();
    if (threadIdx.x == 0) {
        const long long t0 = wall_clock64();
        int ok = 1;
        for (unsigned polls = 1;; polls++) {
            if ((int)(__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) >= 0) break; // (a count may wrap)
            if ((polls & 63u) == 0) {
                if (__hip_atomic_load(error, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) {
                    ok = 0;
                    break;
                }
                if (wall_clock64() - t0 > FRONT_TIMEOUT_TICKS) {
                    __hip_atomic_store(error, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    ok = 0;
                    break;
                }
            }
        }
        if (!ok && report) __hip_atomic_store(report, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        *s_flag = ok;
    }
    lds_barrier();
    return *s_flag != 0;
}

} // namespace
