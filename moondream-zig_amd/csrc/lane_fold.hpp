// Sums of several values at once over the lanes of a wavefront.
#pragma once
#include "epilogue.hpp"

constexpr int DPP_ROW_ROR8 = 0x128; // the lane 8 away within a row of 16

// Maximum of a lane's value and the one 32 lanes away (no trip through LDS)
__device__ __forceinline__ float half_max(float v) {
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    const unsigned r0 = r[0], r1 = r[1];
    return fmaxf(__builtin_bit_cast(float, r0), __builtin_bit_cast(float, r1));
}

// A lane's value plus that of the lane 8, 16 or 32 away: the additions of v + __shfl_xor(v, n) without its trip through LDS
__device__ __forceinline__ float add_8_away(float v) { return v + dpp_move<DPP_ROW_ROR8>(v); }
__device__ __forceinline__ float add_16_away(float v) {
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const unsigned r0 = r[0], r1 = r[1];
    return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float add_32_away(float v) {
    const unsigned b = __builtin_bit_cast(unsigned, v);
    const auto r = __builtin_amdgcn_permlane32_swap(b, b, false, false);
    const unsigned r0 = r[0], r1 = r[1];
    return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}

// Of four wavefronts' values, value l of the one 2 h + w in element 2 (l / 32) + h of lane 32 w + l % 32: (wave_sum(0) + wave_sum(1)) + (wave_sum(2) + wave_sum(3)), the
// same additions.  From the second step on lane 4 i + k has element k's sums.
__device__ __forceinline__ float quarters_sum(const float (&v)[4], int lane) {
    constexpr int QUAD_REVERSED = 0x1B; // and mirrored within 8: the lane 4 away
    const bool odd = lane & 1, upper = lane & 2;
    const float a = (odd ? v[1] : v[0]) + dpp_move<DPP_QUAD_XOR1>(odd ? v[0] : v[1]), b = (odd ? v[3] : v[2]) + dpp_move<DPP_QUAD_XOR1>(odd ? v[2] : v[3]);
    float s = (upper ? b : a) + dpp_move<DPP_QUAD_XOR2>(upper ? a : b);
    s += dpp_move<DPP_ROW_HALF_MIRROR>(dpp_move<QUAD_REVERSED>(s));
    s = add_16_away(add_8_away(s));
    s += dpp_move<DPP_QUAD_XOR2>(s);
    s = add_32_away(s);
    return s + dpp_move<DPP_QUAD_XOR1>(s);
}

// Sum over this lane and those below it (no trip through LDS): within rows of 16, then the last lanes of the rows before.
__device__ __forceinline__ int lane_prefix_sum(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false); // from 1, 2, 4 and 8 lanes below within the row, zero where there is none
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false); // lane 15 of a row to the second and fourth row
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false); // lane 31 to the upper half
    return v;
}

// Sum over aligned groups of n lanes (a power of two, the same in every lane); every lane of a group returns it.
__device__ __forceinline__ float group_sum(float v, int n) {
    if (n >= 2) v += dpp_move<DPP_QUAD_XOR1>(v);
    if (n >= 4) v += dpp_move<DPP_QUAD_XOR2>(v);
    if (n >= 8) v += dpp_move<DPP_ROW_HALF_MIRROR>(v);
    if (n >= 16) v += dpp_move<DPP_ROW_MIRROR>(v);
    if (n >= 32) v = add_16_away(v);
    if (n >= 64) v = add_32_away(v);
    return v;
}

// Sums of N values over the lanes that differ in the bits of OFF and below down to `stop` (a power of two, the same in every lane).
// At every step a lane hands one half of its values to its partner and keeps the other, so N / 2 + N / 4 + .. exchanges do; done(i, sum)
// is called for the values that end up in this lane (by several lanes where there are fewer values than lanes).
template <int N, int OFF, class Done>
__device__ __forceinline__ void fold_lanes(float (&v)[N], int lane, int stop, int base, Done done) {
    if (OFF < stop) {
#pragma unroll
        for (int i = 0; i < N; i++) done(base + i, v[i]);
        return;
    }
    const bool upper = lane & OFF;
    if constexpr (N > 1) {
        float half[N / 2];
        if constexpr (OFF == 32 || OFF == 16) {
            // one instruction swaps the upper rows of one value with the lower rows of the other (no trip through LDS)
#pragma unroll
            for (int i = 0; i < N / 2; i++) {
                const unsigned a = __builtin_bit_cast(unsigned, v[i]), b = __builtin_bit_cast(unsigned, v[i + N / 2]);
                const auto r = OFF == 32 ? __builtin_amdgcn_permlane32_swap(a, b, false, false) : __builtin_amdgcn_permlane16_swap(a, b, false, false);
                const unsigned r0 = r[0], r1 = r[1];
                half[i] = __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
            }
        } else if constexpr (OFF == 8) {
#pragma unroll
            for (int i = 0; i < N / 2; i++) half[i] = (upper ? v[i + N / 2] : v[i]) + dpp_move<DPP_ROW_ROR8>(upper ? v[i] : v[i + N / 2]);
        } else
#pragma unroll
        for (int i = 0; i < N / 2; i++) half[i] = (upper ? v[i + N / 2] : v[i]) + __shfl_xor(upper ? v[i] : v[i + N / 2], OFF);
        if constexpr (OFF > 1) fold_lanes<N / 2, OFF / 2>(half, lane, stop, base + (upper ? N / 2 : 0), done);
        else
#pragma unroll
            for (int i = 0; i < N / 2; i++) done(base + (upper ? N / 2 : 0) + i, half[i]);
    } else {
        v[0] += __shfl_xor(v[0], OFF);
        if constexpr (OFF > 1) fold_lanes<1, OFF / 2>(v, lane, stop, base, done);
        else done(base, v[0]);
    }
}
