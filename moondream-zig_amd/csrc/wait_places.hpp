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
    int crowd = 0;   // not 0: waiting workgroups of all calls that run, in multiples of the places, from which on the call takes kernels that do not wait (enter)
};

class WaitPlaces {
  public:
    // A call begins: true if it has its places until leave().  Calls that found none run beside those that did, and where many do, launches whose workgroups wait are slower for
    // all of them than kernels that do not: those hold units that the others' weights could stream through.  So a call with a crowd counts everybody that runs, with
    // places or without.  Tokens/s of several contexts' list decoders together, as many as fit in one launch a layer and the others in three, against all in three: width 2048, 8 key
    // heads, 48 of 128 places each, two contexts (both fit) 1.13, three 0.93, eight 0.97; with 32 delta heads (52 each) 1.07, 0.88, 0.94; 32 key heads (64 each) two 0.97, three 0.95.  Width 1024, 16 key
    // heads (48 each), three 1.11, five 1.03, six 1.00, eight 0.95; four key heads (24 of 160) eight 1.10, with delta heads (26 of 128) 1.07.
    // With a crowd of 1 at width 2048 and of 2 below, those that were slower are at 0.99 to 1.00 (three joined ones 0.96: each one's first call of six still began beside fewer).
    bool enter(const WaitNeed &n) {
        int waiting = n.waiting, places = n.places;
        {
            std::lock_guard<std::mutex> lock(mu);
            for (const WaitNeed &r : running) {
                waiting += r.waiting;
                places = std::min(places, r.places);
            }
            running.push_back(n);
        }
        return !(n.crowd && waiting >= n.crowd * places) && take(n);
    }
    void leave(const WaitNeed &n, bool took) {
        if (took) give(n);
        std::lock_guard<std::mutex> lock(mu);
        remove(running, n);
    }
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
        remove(held, n);
    }

  private:
    std::mutex mu;
    std::vector<WaitNeed> held, running;
    static void remove(std::vector<WaitNeed> &from, const WaitNeed &n) {
        for (size_t i = 0; i < from.size(); i++)
            if (from[i].waiting == n.waiting && from[i].places == n.places) {
                from.erase(from.begin() + i);
                return;
            }
    }
};
