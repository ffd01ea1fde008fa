// Workgroups that wait for others of their launch, counted over all launches that a device runs at once; kept free of device-only calls
// so that a host program can check it (tests/cxx/wait_places_check.cpp).
//
// A waiting workgroup holds its place on a compute unit until workgroups that never wait have done their part, and those need a place too.
// One launch leaves them some (its launcher has checked that); launches of several contexts together might not, and would then stand
// still until their waits time out.  So a call that is about to queue such launches takes their places here for as long as it runs, and
// where they are not to be had it takes kernels that do not wait.  A context has one stream, so each call in flight has one such launch
// running at most.  Workgroups are dealt to the dies in turn: the count is per die.
#pragma once

#include <algorithm>
#include <mutex>
#include <vector>

struct WaitNeed {
    int waiting = 0; // workgroups of one launch that may wait on a die at once
    int places = 0;  // workgroups of that kernel that a die holds
};

class WaitPlaces {
  public:
    // If all those that may wait are fewer than the places that the largest of these kernels has, some compute unit holds fewer of them than
    // it has places for the largest, so a workgroup of any of these kernels still fits there.
    bool take(const WaitNeed &n) {
        std::lock_guard<std::mutex> lock(mu);
        int waiting = n.waiting, places = n.places;
        for (const WaitNeed &h : held) {
            waiting += h.waiting;
            places = std::min(places, h.places);
        }
        if (waiting >= places) return false;
        held.push_back(n);
        return true;
    }
    void give(const WaitNeed &n) {
        std::lock_guard<std::mutex> lock(mu);
        for (size_t i = 0; i < held.size(); i++)
            if (held[i].waiting == n.waiting && held[i].places == n.places) {
                held.erase(held.begin() + i);
                return;
            }
    }

  private:
    std::mutex mu;
    std::vector<WaitNeed> held;
};
