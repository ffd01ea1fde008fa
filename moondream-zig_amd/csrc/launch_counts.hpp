// What the counters of launches whose workgroups wait for each other count to; kept free of device-only calls so that a host program can
// check it (tests/cxx/launch_counts_check.cpp).
#pragma once

#include <cstdint>

struct LaunchTargets { // so far: the counters only rise, and every launch waits for targets of its own
    uint32_t leaf[2] = {}, reached[3] = {};
};

// launch(): queues the launch that counts to `next`; clear(): sets the counters to zero behind all that is queued, and has them so when it returns; both return 0 if
// they have.  A launch that reports an error may not run, or may run all the same (the runtime reports earlier calls' errors, too), so counters and targets start over
// together.  Where even that fails, *error is raised as by a wait that has run out: whoever waits gives up, and the session is refused until a clear succeeds.
template <class Launch, class Clear> int launch_counted(LaunchTargets *at, const LaunchTargets &next, volatile uint32_t *error, Launch launch, Clear clear) {
    const int rc = launch();
    if (rc == 0) *at = next;
    else if (clear() == 0) *at = LaunchTargets{};
    else *error = 1;
    return rc;
}
