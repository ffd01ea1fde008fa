// Choice of experts for one token by one wavefront, in f32: scores sigmoid(z), the `top` largest of score + correction (the
// lower index wins a tie), weights score / (sum of the chosen scores + EXPERT_WEIGHT_EPS).
#pragma once
#include "epilogue.hpp"
#include "layer_list.hpp"
#include "lm_types.hpp"

constexpr int ROUTER_MAX_EXPERTS = 512; // LDS of the kernels that route: 2 floats per expert and wavefront

// scores: 2 * E floats of LDS owned by this wavefront; ids / weight may be global memory or LDS
// A chain of `top` dependent choices ahead of the chosen experts' weights: the largest by cross-lane moves, its lane by a mask.  As a tree of
// shuffles, each a trip through LDS, eight choices of 64 took 4 us: one token's decode_mix (46 MB) 18.0 -> 13.6 us, a prompt's route_kernel
// (768 rows) 8.5 -> 4.8.
__device__ __forceinline__ void route_wave(const float *logits, const float *correction, int E, int top, float *scores, int lane, int *ids,
                                           float *weight) {
    float sum = 0.0f;
    if (E <= 64) { // an expert per lane, in registers; the k-th choice ends up in lane k
        const float s = lane < E ? lm_sigmoid(logits[lane]) : 0.0f, c = lane < E ? s + correction[lane] : -INFINITY;
        float left = c > -INFINITY ? c : -INFINITY, chosen = 0.0f; // (what is not a number is never the largest)
        int id = 0;
        for (int k = 0; k < top; k++) {
            const unsigned long long best = __ballot(left == wave_max(left) && left > -INFINITY);
            const int idx = best ? __ffsll(best) - 1 : k;
            const float v = read_lane(s, idx);
            if (lane == idx) left = -INFINITY;
            if (lane == k) {
                id = idx;
                chosen = v;
            }
            sum += v;
        }
        if (lane < top) {
            ids[lane] = id;
            weight[lane] = chosen * (1.0f / (sum + EXPERT_WEIGHT_EPS));
        }
        return;
    }
    float *choice = scores + E;
    for (int e = lane; e < E; e += 64) {
        const float s = lm_sigmoid(logits[e]);
        scores[e] = s;
        choice[e] = s + correction[e];
    }
    for (int k = 0; k < top; k++) { // (a lane only ever looks for the largest among the entries it wrote itself)
        float best = -INFINITY;
        int mine = 0x7fffffff, idx;
        for (int e = lane; e < E; e += 64)
            if (choice[e] > best) {
                best = choice[e];
                mine = e;
            }
        // the lowest index of the lanes with the largest choice
        const float most = wave_max(best);
        unsigned long long tied = __ballot(best == most);
        idx = 0x7fffffff;
        for (; tied; tied &= tied - 1) idx = min(idx, __builtin_amdgcn_readlane(mine, __ffsll(tied) - 1));
        if (idx >= E) idx = k; // (scores that are not numbers: stay within the experts)
        const float s = scores[idx]; // (another lane's: LDS serves a wavefront in order)
        if (lane == (idx & 63)) choice[idx] = -INFINITY;
        if (lane == 0) {
            ids[k] = idx;
            weight[k] = s;
        }
        sum += s;
    }
    const float inv = 1.0f / (sum + EXPERT_WEIGHT_EPS);
    if (lane == 0)
        for (int k = 0; k < top; k++) weight[k] *= inv;
}
