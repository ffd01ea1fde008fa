// What the workgroups of the decode launches do (layer_decode.hip, layer_whole.hip): shares of rows, dots of weight rows with a vector,
// a row's norm, one token's attention and one token of the gated delta rule.
#pragma once
#include "delta_math.hpp"
#include "key_splits.hpp"
#include "lane_fold.hpp"
#include "layer_list.hpp"
#include "lm_types.hpp"
#include "norm.hpp"

#include <algorithm>

namespace {

__device__ __forceinline__ void share(int n, int parts, int i, int &begin, int &end) {
    const int q = n / parts, r = n % parts;
    begin = i * q + min(i, r);
    end = begin + q + (i < r ? 1 : 0);
}

// dots of RG weight rows with a vector in LDS (T, pieces * 16 bytes); every lane returns all of them.  rows[j] null: skipped.
template <class T, int RG, int U>
struct RowDots {
    lm_u32x4 w[RG][U];
    __device__ __forceinline__ void request(const T *const (&rows)[RG], int p0, int pieces, int lane) {
#pragma unroll
        for (int j = 0; j < RG; j++)
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int g = p0 + u * 64 + lane;
                w[j][u] = lm_u32x4{0, 0, 0, 0};
                if (g < pieces && rows[j]) w[j][u] = __builtin_nontemporal_load(reinterpret_cast<const lm_u32x4 *>(rows[j]) + g);
            }
    }
    __device__ __forceinline__ void add(const T *vec, int p0, int pieces, int lane, float (&acc)[RG]) const {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int g = p0 + u * 64 + lane;
            lm_u32x4 x = {0, 0, 0, 0};
            if (g < pieces) x = *reinterpret_cast<const lm_u32x4 *>(vec + size_t(g) * Piece<T>::N);
#pragma unroll
            for (int j = 0; j < RG; j++) acc[j] = dot_piece<T>(w[j][u], x, acc[j]);
        }
    }
};

// Row of gate/up column pair i (half 0: gate, 1: up) in the interleaved weights
__device__ __forceinline__ int pair_row(int i, int half) { return (i >> 5) * 64 + half * 32 + (i & 31); }

// The norm of a token's row x (or of its embedding row) by a workgroup that holds NV times four elements a thread: widths of up to 1024 NV, a
// multiple of 4.  JOIN: where p.y is set, x is completed with a joined layer's results first.  request() asks for everything, finish() leaves
// h in LDS; `write`: the workgroup that also writes x and h to memory.
template <class T, int NV, bool JOIN, bool COH> struct NormRow {
    float4_t xv[NV], gv[NV], bv[NV], jl[JOIN ? NV : 1], jr[JOIN ? NV : 1], wl[JOIN ? NV : 1], wr[JOIN ? NV : 1];
    __device__ __forceinline__ void request(const DecodeProj &p, const T *er, int tid) {
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int i = (k * 256 + tid) * 4, j = i < p.width ? i : 0;
            if (er) {
#pragma unroll
                for (int e = 0; e < 4; e++) xv[k][e] = (float)er[j + e];
            } else xv[k] = *reinterpret_cast<const float4_t *>(p.x + j);
            if (JOIN && (!COH || p.y)) {
                jl[k] = *reinterpret_cast<const float4_t *>(p.y + j);
                jr[k] = *reinterpret_cast<const float4_t *>(p.y + p.dp + j);
                xv[k] += *reinterpret_cast<const float4_t *>(p.y + 2 * p.dp + j);
                wl[k] = *reinterpret_cast<const float4_t *>(p.out_l + j);
                wr[k] = *reinterpret_cast<const float4_t *>(p.out_r + j);
            }
            gv[k] = *reinterpret_cast<const float4_t *>(p.gamma + j);
            bv[k] = p.beta ? *reinterpret_cast<const float4_t *>(p.beta + j) : float4_t{0, 0, 0, 0};
        }
    }
    static __device__ __forceinline__ void store(float *at, const float4_t &v) {
        if (!COH) *reinterpret_cast<float4_t *>(at) = v;
        else
#pragma unroll
            for (int e = 0; e < 4; e++) st_f<true>(at + e, v[e]);
    }
    __device__ __forceinline__ void finish(const DecodeProj &p, bool embedded, bool write, T *s_h, float *s_red, int tid) {
        const int lane = tid & 63, wave = tid >> 6;
        float s = 0.0f, m2 = 0.0f;
        if (JOIN && (!COH || p.y)) {
            float ss[2] = {0.0f, 0.0f}; // of the two results
#pragma unroll
            for (int k = 0; k < NV; k++)
                if ((k * 256 + tid) * 4 < p.width)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        ss[0] = fmaf(jl[k][e], jl[k][e], ss[0]);
                        ss[1] = fmaf(jr[k][e], jr[k][e], ss[1]);
                    }
            join_factors(p, ss, s_red, lane, wave);
#pragma unroll
            for (int k = 0; k < NV; k++) {
                const int i = (k * 256 + tid) * 4;
#pragma unroll
                for (int e = 0; e < 4; e++) xv[k][e] += jl[k][e] * ss[0] * wl[k][e] + jr[k][e] * ss[1] * wr[k][e];
                if (i < p.width && write) store(p.x_new + i, xv[k]);
            }
        }
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int i = (k * 256 + tid) * 4;
            if (embedded) xv[k] *= p.embed_scale;
            if (i >= p.width) xv[k] = float4_t{0, 0, 0, 0};
            else if (embedded && write) store(p.x + i, xv[k]);
            s += (xv[k][0] + xv[k][1]) + (xv[k][2] + xv[k][3]);
        }
        const float mean = p.beta ? block_sum(s, s_red) / (float)p.width : 0.0f; // (an RMS norm takes no mean off)
#pragma unroll
        for (int k = 0; k < NV; k++)
            if ((k * 256 + tid) * 4 < p.width) {
                xv[k] -= mean;
#pragma unroll
                for (int e = 0; e < 4; e++) m2 = fmaf(xv[k][e], xv[k][e], m2);
            }
        const float rstd = 1.0f / sqrtf(block_sum(m2, s_red) / (float)p.width + p.eps);
#pragma unroll
        for (int k = 0; k < NV; k++) {
            const int i = (k * 256 + tid) * 4;
            if (i >= p.dp) continue;
            typedef T vec4 __attribute__((ext_vector_type(4)));
            vec4 v;
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] = i < p.width ? (T)(xv[k][e] * rstd * gv[k][e] + bv[k][e]) : (T)0.0f;
            *reinterpret_cast<vec4 *>(s_h + i) = v;
            if (p.h && write) *reinterpret_cast<vec4 *>(reinterpret_cast<T *>(p.h) + i) = v;
        }
    }
    // squares of the two results, a thread's share -> the factors of both
    static __device__ __forceinline__ void join_factors(const DecodeProj &p, float (&ss)[2], float *s_red, int lane, int wave) {
        ss[0] = wave_sum(ss[0]);
        ss[1] = wave_sum(ss[1]);
        if (lane == 0) {
            s_red[8 + wave] = ss[0];
            s_red[12 + wave] = ss[1];
        }
        lds_barrier();
        ss[0] = 0.5f / sqrtf(((s_red[8] + s_red[9]) + (s_red[10] + s_red[11])) / (float)p.width + p.eps);
        ss[1] = 0.5f / sqrtf(((s_red[12] + s_red[13]) + (s_red[14] + s_red[15])) / (float)p.width + p.eps);
    }
};

constexpr int MIX_HEADS = 8;       // query heads one workgroup serves
__host__ __device__ __forceinline__ int mix_head_blocks(int per_group) { return (per_group + MIX_HEADS - 1) / MIX_HEADS; }

__device__ __forceinline__ int next_pow2(int v) { return v <= 1 ? 1 : 1 << (32 - __builtin_clz(v - 1)); }

// LDS of an attention workgroup, in floats: q [NH][dimp], new k [dimp], new v [vdimp], scores [NH][keys], reduction [4][NH][vdimp], misc
__host__ __device__ __forceinline__ size_t mix_lds_floats(int nh, int dimp, int vdimp, int keys) {
    return size_t(nh) * dimp + dimp + vdimp + size_t(nh) * keys + size_t(4) * nh * vdimp + 4 * nh + 8; // (launch_decode_mix: at least nh * S before the misc)
}

// How a role meets the others.  In a launch of its own it starts with everything it reads in memory and leaves its results to the next one.
struct Apart {
    static constexpr bool SHARED = false;
    __device__ __forceinline__ bool wait() const { return true; }
    __device__ __forceinline__ bool wait_gate() const { return true; }
    __device__ __forceinline__ void done() const {}
};
template <bool COH> __device__ __forceinline__ float4_t ld_f4(const float *p) {
    if (!COH) return *reinterpret_cast<const float4_t *>(p);
    union {
        unsigned long long u[2];
        float4_t f;
    } v;
    const unsigned long long *q = reinterpret_cast<const unsigned long long *>(p);
    v.u[0] = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    v.u[1] = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return v.f;
}
template <bool COH, class T> __device__ __forceinline__ void st_t(T *p, T v) {
    if (!COH) *p = v;
    else if constexpr (sizeof(T) == 2) __hip_atomic_store(reinterpret_cast<unsigned short *>(p), __builtin_bit_cast(unsigned short, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    else __hip_atomic_store(reinterpret_cast<unsigned *>(p), __builtin_bit_cast(unsigned, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Attention of one token: kv head g, query heads h0 .. h0 + nh - 1, split `split` of S.  Keys are numbered: the blocks that lie before
// the window, then the window's tokens.  WHOLE: the mechanisms of the last part of DecodeMix.  LONG: head sizes of more than 64 pieces.
// Every phase runs once or twice per launch, so what bounds it is latency, instruction fetches among it: nothing here is unrolled that
// need not be, and cache rows are found without divisions.
// D: the padded head sizes, where the launch is for these only (0: any).  Meet: Apart, or how the workgroup waits for the token's projections and
// reports a merged head; the projections and the heads then pass by the dies' caches.
template <class T, int NH, bool WHOLE, bool LONG, int D, class Meet>
__device__ __forceinline__ void mix_attention(const DecodeMix &p, int g, int hb, int split, int S, int keys_max, float *lds, const Meet &meet) {
    constexpr bool COH = Meet::SHARED;
    const int dimp = D ? D : p.dimp, vdimp = D ? D : p.vdimp;
    const int per = p.H / p.G, n_hb = mix_head_blocks(per), h0 = g * per + hb * MIX_HEADS, nh = min(MIX_HEADS, per - hb * MIX_HEADS);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pos = p.pos_dev ? (int)p.pos_dev[0] : (int)p.pos;
    const int lo = p.window ? max(0, pos - p.window + 1) : 0, blocks = WHOLE && p.pool ? lo / p.pool : 0, n_keys = blocks + pos - lo + 1;
    const int chunk = (n_keys + S - 1) / S, j0 = split * chunk, j1 = min(j0 + chunk, n_keys), cnt = max(0, j1 - j0);
    const bool own = !(WHOLE && p.borrowed);    // the token's key and value are not in the cache yet
    const int newest = own ? n_keys - 1 : -1;   // their number
    float *s_q = lds, *s_k = s_q + NH * dimp, *s_v = s_k + dimp, *s_s = s_v + vdimp, *s_r = s_s + NH * keys_max, *s_ml = s_r + 4 * NH * vdimp;
    T *t_k = reinterpret_cast<T *>(s_k), *t_v = reinterpret_cast<T *>(s_v); // the token's key and value as the cache holds them
    T *ck = reinterpret_cast<T *>(p.ck) + size_t(g) * p.cap * dimp, *cv = reinterpret_cast<T *>(p.cv) + size_t(g) * p.cap * vdimp;
    const T *pk_rows = reinterpret_cast<const T *>(p.pk) + size_t(g) * p.blocks * dimp, *pv_rows = reinterpret_cast<const T *>(p.pv) + size_t(g) * p.blocks * vdimp;
    const bool has_new = own && cnt > 0 && j1 == n_keys;
    // K: lpk lanes per key, V: lpv lanes per key (powers of two); a step is the keys the four wavefronts take at once.  The first
    // PF steps' rows are requested before anything else: they do not depend on the new token.
    constexpr int PE = Piece<T>::N, PF = 4;
    const int kp = dimp / PE, lpk = min(64, next_pow2(kp)), kpw = 64 / lpk, sub = lane / lpk, c0 = lane % lpk;
    const int vp = vdimp / PE, lpv = min(64, next_pow2(vp)), vpw = 64 / lpv, vsub = lane / lpv, vc0 = lane % lpv;
    const int base_row = lo % p.cap; // (a window's tokens are at most cap)
    auto token_row = [&](int j) { return base_row + j >= p.cap ? base_row + j - p.cap : base_row + j; };
    const int new_row = token_row(pos - lo);
    auto k_piece = [&](int key, int c) {
        const T *row = WHOLE && key < blocks ? pk_rows + size_t(key) * dimp : ck + size_t(token_row(key - blocks)) * dimp;
        return *reinterpret_cast<const lm_u32x4 *>(row + c * PE);
    };
    auto v_piece = [&](int key, int c) {
        const T *row = WHOLE && key < blocks ? pv_rows + size_t(key) * vdimp : cv + size_t(token_row(key - blocks)) * vdimp;
        return *reinterpret_cast<const lm_u32x4 *>(row + c * PE);
    };
    // The token's own projections first: a wavefront's loads return in order, and the cache rows come from further away.  This lane's
    // first element of the wavefront's tasks (query heads, the new key, the new value).
    constexpr int TASKS = (NH + 2 + 3) / 4;
    const int n_tasks = nh + (has_new ? 2 : 0);
    auto task_src = [&](int task) { return p.proj + (task == nh + 1 ? p.ov + g * vdimp : task < nh ? (h0 + task) * dimp : p.ok + g * dimp); };
    float first[TASKS];
    auto request_first = [&]() {
#pragma unroll
        for (int i = 0; i < TASKS; i++) {
            const int task = wave + 4 * i;
            first[i] = task < n_tasks && lane < (task == nh + 1 ? vdimp : dimp) ? ld_f<COH>(task_src(task) + lane) : 0.0f;
        }
    };
    // (the first mixing layer's value of this position: an earlier launch's)
    T first_v1 = (T)0.0f;
    const T *v1 = !WHOLE && p.mixes && has_new ? reinterpret_cast<const T *>(p.v_first) + (size_t(g) * p.cap_first + pos % p.cap_first) * vdimp : nullptr;
    if (COH && v1 && lane < vdimp) first_v1 = v1[lane];
    if (!COH) request_first();
    auto task_half = [&](int task) { return WHOLE ? task == nh + 1 ? (p.rotv ? p.vdim / 2 : 0) : p.rot ? p.rot_dims / 2 : 0 : 0; }; // pairs that turn
    float first_w[WHOLE ? TASKS : 1];
    float2 first_cs[WHOLE ? TASKS : 1];
    if (WHOLE) {
#pragma unroll
        for (int i = 0; i < TASKS; i++) {
            const int task = wave + 4 * i, half = task_half(task);
            first_w[i] = 1.0f;
            first_cs[i] = float2{1.0f, 0.0f};
            if (task >= n_tasks) continue;
            if (p.whole && task <= nh && lane < dimp) first_w[i] = task < nh ? p.qn[(h0 + task) * dimp + lane] : p.kn[g * dimp + lane];
            if (lane < 2 * half) first_cs[i] = (task == nh + 1 ? p.rotv : p.rot)[size_t(pos) * half + lane % half];
        }
    }
    // (all of q and k are normed together: every workgroup adds their squares up)
    constexpr int SQ = 2; // 4,096 bytes of q at a time
    const int nq = WHOLE && p.whole ? p.H * dimp : 0, nk = WHOLE && p.whole && has_new ? p.G * dimp : 0;
    float4_t sq_q[WHOLE ? SQ : 1], sq_k = {0, 0, 0, 0};
    auto request_squares = [&]() {
        if (!WHOLE) return;
#pragma unroll
        for (int i = 0; i < SQ; i++) sq_q[i] = tid * 4 + 1024 * i < nq ? ld_f4<COH>(p.proj + tid * 4 + 1024 * i) : float4_t{0, 0, 0, 0};
        if (tid * 4 < nk) sq_k = ld_f4<COH>(p.proj + p.ok + tid * 4);
    };
    if (!COH) request_squares();
    lm_u32x4 pk[PF], pv[PF];
    auto request_rows = [&]() {
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int key = j0 + (i * 4 + wave) * kpw + sub;
            pk[i] = lm_u32x4{0, 0, 0, 0};
            if (key < j1 && key != newest && c0 < kp) pk[i] = k_piece(key, c0);
        }
#pragma unroll
        for (int i = 0; i < PF; i++) {
            const int key = j0 + (i * 4 + wave) * vpw + vsub;
            pv[i] = lm_u32x4{0, 0, 0, 0};
            if (key < j1 && key != newest && vc0 < vp) pv[i] = v_piece(key, vc0);
        }
    };
    if (COH) { // the cache's rows wait for nothing, but a poll returns behind what its wavefront has asked for before
        if (wave != 0) request_rows();
        if (!meet.wait()) return;
        request_first();
        request_squares();
        if (wave == 0) request_rows();
    } else request_rows();
    // element d of a head x, times its weight w, turned by its pair's angle
    auto turned = [&](const float *x, const float *w, int d, const float2 *table, int half) {
        float y = w ? x[d] * w[d] : x[d];
        if (!table || d >= 2 * half) return y;
        const int m = d < half ? d : d - half, other = d < half ? d + half : m;
        const float2 cs = table[size_t(pos) * half + m];
        const float z = w ? x[other] * w[other] : x[other];
        return d < half ? y * cs.x - z * cs.y : y * cs.x + z * cs.y;
    };
    // where the outputs turn back: the angle of this thread's first element, requested early
    const int back = WHOLE && p.rotv ? p.vdim / 2 : 0;
    float2 back_cs = {1.0f, 0.0f};
    if (WHOLE && back && tid % vdimp < 2 * back) back_cs = p.rotv[size_t(pos) * back + tid % vdimp % back];
    if constexpr (WHOLE) {
        // q and k are normed as a whole: the heads go to LDS turned and weighted, the norms' factors come last
        float ss[2] = {0.0f, 0.0f};
        auto squares = [](const float4_t &v) { return (v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]); };
#pragma unroll
        for (int i = 0; i < SQ; i++) ss[0] += squares(sq_q[i]);
        ss[1] = squares(sq_k);
        for (int i = tid * 4 + 1024 * SQ; i < nq; i += 1024) ss[0] += squares(ld_f4<COH>(p.proj + i));
        for (int i = tid * 4 + 1024; i < nk; i += 1024) ss[1] += squares(ld_f4<COH>(p.proj + p.ok + i));
#pragma unroll
        for (int i = 0; i < TASKS; i++) {
            const int task = wave + 4 * i, half = task_half(task);
            if (task >= n_tasks) continue;
            const bool is_v = task == nh + 1, is_q = task < nh;
            const int size = is_v ? vdimp : dimp;
            float *dst = is_v ? s_v : is_q ? s_q + task * dimp : s_k;
            if (size <= 64) { // the other element of a pair is another lane's
                const float y = first[i] * first_w[i], z = __shfl(y, lane < half ? lane + half : lane - half);
                if (lane < size) dst[lane] = lane >= 2 * half ? y : lane < half ? y * first_cs[i].x - z * first_cs[i].y : y * first_cs[i].x + z * first_cs[i].y;
                continue;
            }
            const float *src = task_src(task), *w = is_v || !p.whole ? nullptr : is_q ? p.qn + (h0 + task) * dimp : p.kn + g * dimp;
            for (int d = lane; d < size; d += 64) dst[d] = turned(src, w, d, is_v ? p.rotv : p.rot, half);
        }
        ss[0] = wave_sum(ss[0]);
        ss[1] = wave_sum(ss[1]);
        if (lane == 0) {
            s_r[2 * wave] = ss[0];
            s_r[2 * wave + 1] = ss[1];
        }
        lds_barrier();
        const float f_q = p.whole ? 1.0f / sqrtf(((s_r[0] + s_r[2]) + (s_r[4] + s_r[6])) / (float)(p.H * p.dim) + p.eps) : 1.0f;
        const float f_k = p.whole ? 1.0f / sqrtf(((s_r[1] + s_r[3]) + (s_r[5] + s_r[7])) / (float)(p.G * p.dim) + p.eps) : 1.0f;
        for (int i = tid; i < nh * dimp; i += 256) s_q[i] = (float)(T)(s_q[i] * f_q);
        if (has_new)
            for (int i0 = 0; i0 < dimp + vdimp; i0 += 256) { // (in rounds: the rounded values lie over the others)
                const int i = i0 + tid;
                const bool is_v = i >= dimp, live = i < dimp + vdimp;
                const int d = is_v ? i - dimp : i;
                const T c = (T)(live ? is_v ? s_v[d] : s_k[d] * f_k : 0.0f);
                lds_barrier();
                if (!live) continue;
                (is_v ? t_v : t_k)[d] = c;
                if (hb == 0) (is_v ? cv + size_t(new_row) * vdimp : ck + size_t(new_row) * dimp)[d] = c;
            }
    } else
#pragma unroll
    for (int i = 0; i < TASKS; i++) {
        const int task = wave + 4 * i;
        if (task >= n_tasks) continue;
        const float *src = task_src(task);
        if (task == nh + 1) { // the new value
            for (int d = lane; d < vdimp; d += 64) {
                float v = (float)(T)(d == lane ? first[i] : ld_f<COH>(src + d));
                if (v1) v = (1.0f - p.lambda) * v + p.lambda * (float)(COH && d == lane ? first_v1 : v1[d]);
                const T c = (T)v;
                t_v[d] = c;
                if (hb == 0) cv[size_t(new_row) * vdimp + d] = c;
            }
        } else { // a query head or the new key
            const bool is_q = task < nh;
            float ss = first[i] * first[i];
            for (int d = lane + 64; d < dimp; d += 64) {
                const float y = ld_f<COH>(src + d);
                ss = fmaf(y, y, ss);
            }
            const float f = p.qk_rms ? 1.0f / sqrtf(wave_sum(ss) / (float)p.dim + p.eps) : 1.0f;
            for (int d = lane; d < dimp; d += 64) {
                const T c = (T)((d == lane ? first[i] : ld_f<COH>(src + d)) * f);
                if (is_q) s_q[task * dimp + d] = (float)c;
                else {
                    t_k[d] = c;
                    if (hb == 0) ck[size_t(new_row) * dimp + d] = c;
                }
            }
        }
    }
    lds_barrier();
    if (WHOLE && p.pool && has_new && hb == 0 && (pos + 1) % p.pool == 0) { // the token completes a block (no window reaches past it yet)
        const int b = pos / p.pool;
        for (int i = tid; i < dimp + vdimp; i += 256) {
            const bool is_v = i >= dimp;
            const int d = is_v ? i - dimp : i, size = is_v ? vdimp : dimp;
            const T *rows = is_v ? cv : ck;
            float sum = 0.0f;
#pragma unroll 4
            for (int j = b * p.pool; j < pos; j++) sum += (float)rows[size_t(j % p.cap) * size + d];
            sum += (float)(is_v ? t_v : t_k)[d];
            reinterpret_cast<T *>(is_v ? p.pv : p.pk)[(size_t(g) * p.blocks + b) * size + d] = (T)(sum / (float)p.pool);
        }
    }
    float scale[NH];
#pragma unroll
    for (int h = 0; h < NH; h++) scale[h] = WHOLE && p.temp && h < nh ? p.scale * p.temp[h0 + h] : p.scale;
    auto score_step = [&](int key, const lm_u32x4 &first) {
        float acc[NH];
#pragma unroll
        for (int h = 0; h < NH; h++) acc[h] = 0.0f;
        for (int c = c0; c < kp; c += LONG ? lpk : kp) {
            float kf[PE];
            lm_u32x4 piece = first;
            if (LONG && c != c0 && key < j1 && key != newest) piece = k_piece(key, c);
            if (key == newest) piece = *reinterpret_cast<const lm_u32x4 *>(t_k + c * PE);
            Piece<T>::unpack(piece, kf);
#pragma unroll
            for (int h = 0; h < NH; h++) // (heads past nh: whatever LDS holds, never stored)
#pragma unroll
                for (int e = 0; e < PE; e++) acc[h] = fmaf(kf[e], s_q[h * dimp + c * PE + e], acc[h]);
        }
#pragma unroll
        for (int h = 0; h < NH; h++) {
            acc[h] = group_sum(acc[h], lpk);
            if (key < j1 && c0 == 0 && h < nh) s_s[h * keys_max + key - j0] = acc[h] * scale[h];
        }
    };
#pragma unroll
    for (int i = 0; i < PF; i++)
        if (j0 + (i * 4 + wave) * kpw < j1) score_step(j0 + (i * 4 + wave) * kpw + sub, pk[i]);
#pragma unroll 1
    for (int j = j0 + (PF * 4 + wave) * kpw; j < j1; j += 4 * kpw) {
        const int key = j + sub;
        lm_u32x4 first = {0, 0, 0, 0};
        if (key < j1 && key != newest && c0 < kp) first = k_piece(key, c0);
        score_step(key, first);
    }
    lds_barrier();
    for (int h = wave; h < nh; h += 4) {
        float m = -INFINITY;
        for (int i = lane; i < cnt; i += 64) m = fmaxf(m, s_s[h * keys_max + i]);
        m = wave_max(m);
        float l = 0.0f;
        for (int i = lane; i < cnt; i += 64) {
            const float e = expf(s_s[h * keys_max + i] - m);
            s_s[h * keys_max + i] = e;
            l += e;
        }
        l = wave_sum(l);
        if (lane == 0) {
            s_ml[2 * h] = m;
            s_ml[2 * h + 1] = l;
        }
    }
    lds_barrier();
    for (int c = vc0; c < (LONG ? (vp + lpv - 1) / lpv * lpv : lpv); c += lpv) {
        float acc[NH][PE];
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int e = 0; e < PE; e++) acc[h][e] = 0.0f;
        auto value_step = [&](int key, lm_u32x4 piece) {
            float vf[PE];
            if (key == newest) piece = *reinterpret_cast<const lm_u32x4 *>(t_v + c * PE);
            Piece<T>::unpack(piece, vf);
#pragma unroll
            for (int h = 0; h < NH; h++) { // (heads past nh as above)
                const float w = s_s[h * keys_max + key - j0];
#pragma unroll
                for (int e = 0; e < PE; e++) acc[h][e] = fmaf(w, vf[e], acc[h][e]);
            }
        };
        if (c < vp) {
#pragma unroll
            for (int i = 0; i < PF; i++) {
                const int key = j0 + (i * 4 + wave) * vpw + vsub;
                if (key < j1) value_step(key, LONG && c != vc0 && key != newest ? v_piece(key, c) : pv[i]);
            }
#pragma unroll 1
            for (int key = j0 + (PF * 4 + wave) * vpw + vsub; key < j1; key += 4 * vpw) value_step(key, key == newest ? pv[0] : v_piece(key, c));
        }
        float flat[NH * PE];
#pragma unroll
        for (int h = 0; h < NH; h++)
#pragma unroll
            for (int e = 0; e < PE; e++) flat[h * PE + e] = acc[h][e];
        fold_lanes<NH * PE, 32>(flat, lane, lpv, 0, [&](int i, float v) {
            if (c < vp && i / PE < nh) s_r[(wave * NH + i / PE) * vdimp + c * PE + i % PE] = v;
        });
    }
    lds_barrier();
    // This split's sums and (m, l) per head to memory; the workgroup that counts in last adds the splits up.
    const int stride = vdimp + 2;
    float *part = p.partial + size_t(g * n_hb + hb) * S * MIX_HEADS * stride;
    for (int i = tid; i < nh * vdimp; i += 256) {
        const int h = i / vdimp, d = i % vdimp;
        const float v = (s_r[(0 * NH + h) * vdimp + d] + s_r[(1 * NH + h) * vdimp + d]) + (s_r[(2 * NH + h) * vdimp + d] + s_r[(3 * NH + h) * vdimp + d]);
        st_f<true>(part + (size_t(split) * MIX_HEADS + h) * stride + d, v);
    }
    if (tid < 2 * nh) st_f<true>(part + (size_t(split) * MIX_HEADS + (tid >> 1)) * stride + vdimp + (tid & 1), s_ml[tid]);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // stored before the workgroup counts in
    int *s_last = reinterpret_cast<int *>(s_ml + 2 * NH);
    __syncthreads();
    if (tid == 0) {
        uint32_t *counter = p.counter + g * n_hb + hb;
        const uint32_t old = __hip_atomic_fetch_add(counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *s_last = old + 1 == (uint32_t)S;
        if (*s_last) __hip_atomic_store(counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); // ready for the next launch
    }
    __syncthreads();
    if (!*s_last) return;
    // Every head's splits: this thread's elements of the first splits, all (m, l) and the gate are requested together; the weight of each
    // split (a lane per split) goes through LDS.
    constexpr int AT_ONCE = MIX_SPLITS, HW = (NH + 3) / 4;
    const size_t pitch = size_t(MIX_HEADS) * stride; // floats between splits
    float *s_w = lds; // [nh][S], over what the phases before have used
    float v[AT_ONCE], m0[HW], l0[HW], sink[HW], gate0 = 0.0f;
    const int i_first = min(tid, nh * vdimp - 1);
    {
        const float *ph = part + size_t(i_first / vdimp) * stride + i_first % vdimp;
#pragma unroll
        for (int u = 0; u < AT_ONCE; u++) v[u] = ld_f<true>(ph + min(u, S - 1) * pitch);
    }
#pragma unroll
    for (int i = 0; i < HW; i++) {
        const int h = wave + 4 * i;
        const float *ph = part + size_t(h) * stride + vdimp;
        sink[i] = m0[i] = -INFINITY;
        l0[i] = 0.0f;
        if (h < nh && p.sink) sink[i] = p.sink[h0 + h];
        if (h < nh && lane < S) {
            m0[i] = ld_f<true>(ph + lane * pitch);
            l0[i] = ld_f<true>(ph + lane * pitch + 1);
        }
    }
    if (p.gate) {
        if (!meet.wait_gate()) return;
        gate0 = ld_f<COH>(p.proj + p.og + h0 * vdimp + i_first);
    }
#pragma unroll
    for (int i = 0; i < HW; i++) {
        const int h = wave + 4 * i;
        if (h >= nh) continue;
        const float *ph = part + size_t(h) * stride + vdimp;
        float m = fmaxf(sink[i], m0[i]), l = 0.0f;
        for (int s = lane + 64; s < S; s += 64) m = fmaxf(m, ld_f<true>(ph + s * pitch));
        m = wave_max(m);
        for (int s = lane; s < S; s += 64) { // (an empty split: m = -inf, weight 0)
            const float w = expf((s == lane ? m0[i] : ld_f<true>(ph + s * pitch)) - m);
            l = fmaf(s == lane ? l0[i] : ld_f<true>(ph + s * pitch + 1), w, l);
            s_w[h * S + s] = w;
        }
        l = wave_sum(l) + (p.sink ? expf(sink[i] - m) : 0.0f);
        if (lane == 0) s_ml[h] = 1.0f / l;
    }
    lds_barrier();
    float *s_o = s_r; // (free again)
    for (int i = tid; i < nh * vdimp; i += 256) {
        const int h = i / vdimp, d = i % vdimp;
        const float *ph = part + size_t(h) * stride + d;
        float o = 0.0f;
        for (int s0 = 0; s0 < S; s0 += AT_ONCE) {
            if (s0 || i != tid)
#pragma unroll
                for (int u = 0; u < AT_ONCE; u++) v[u] = ld_f<true>(ph + min(s0 + u, S - 1) * pitch);
#pragma unroll
            for (int u = 0; u < AT_ONCE; u++)
                if (s0 + u < S) o = fmaf(v[u], s_w[h * S + s0 + u], o);
        }
        o *= s_ml[h];
        if (WHOLE && p.rotv) {
            s_o[i] = o;
            continue;
        }
        if (p.gate) o *= lm_sigmoid(i == tid ? gate0 : ld_f<COH>(p.proj + p.og + (h0 + h) * vdimp + d));
        st_t<COH>(reinterpret_cast<T *>(p.out) + (h0 + h) * vdimp + d, (T)o);
    }
    if (!(WHOLE && p.rotv)) return meet.done();
    lds_barrier();
    for (int i = tid; i < nh * vdimp; i += 256) { // the outputs turn back
        const int h = i / vdimp, d = i % vdimp;
        float o = s_o[i];
        if (d < 2 * back) {
            const float2 cs = i == tid ? back_cs : p.rotv[size_t(pos) * back + d % back];
            o = d < back ? o * cs.x + s_o[i + back] * cs.y : o * cs.x - s_o[i - back] * cs.y;
        }
        if (p.gate) o *= lm_sigmoid(i == tid ? gate0 : ld_f<COH>(p.proj + p.og + (h0 + h) * vdimp + d));
        st_t<COH>(reinterpret_cast<T *>(p.out) + (h0 + h) * vdimp + d, (T)o);
    }
    meet.done();
}

// One token of the gated delta rule (delta_rows.hip has the equations): head h, whole.  A thread holds four columns of every rp-th row of
// the state, up to DELTA_ROWS of them in registers (REG); larger states are read again for the update.
constexpr int DELTA_ROWS = 16;
// LDS in floats: q, k, decay [ddimp], v, gate, u [dvdimp], sums [1024], 8 more, then the two-step projections' inner vectors
__host__ __device__ __forceinline__ size_t delta_lds_floats(int dimp, int vdimp, int kd) { return size_t(3) * dimp + 3 * vdimp + 1024 + 8 + kd; }
template <class T, bool REG, class Meet>
__device__ __forceinline__ void mix_delta(const DecodeMix &p, int h, float *lds, const Meet &meet) {
    constexpr bool COH = Meet::SHARED;
    constexpr int PE = Piece<T>::N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, dimp = p.ddimp, vdimp = p.dvdimp;
    const int pos = p.pos_dev ? (int)p.pos_dev[0] : (int)p.pos, per = p.dH / p.dG, c = h / per;
    // Behind the end of a generation (the loop's state says so) launches may still come: they must leave the recurrence as it is.
    const bool keep = !(p.pos_dev && p.pos_dev[3]);
    const int vq = vdimp / 4, rp = 256 / vq, col = tid % vq, r0 = tid / vq;
    const bool on = tid < rp * vq;
    float *s_q = lds, *s_k = s_q + dimp, *s_g = s_k + dimp, *s_v = s_g + dimp, *s_gate = s_v + vdimp, *s_u = s_gate + vdimp, *s_sum = s_u + vdimp, *s_misc = s_sum + 1024;
    T *s_in = reinterpret_cast<T *>(s_misc + 8);
    float4_t *state = reinterpret_cast<float4_t *>(p.state + size_t(h) * dimp * vdimp) + col;
    float4_t S[REG ? DELTA_ROWS : 1];
    auto load = [&](int row) { return pos && on && row < dimp ? state[size_t(row) * vq] : float4_t{0, 0, 0, 0}; };
    if (REG)
#pragma unroll
        for (int i = 0; i < DELTA_ROWS; i++) S[i] = load(r0 + i * rp);
    if (!meet.wait()) return;
    // convolutions
    const T *ring = reinterpret_cast<const T *>(p.ring);
    for (int i = tid; i < 2 * dimp + vdimp; i += 256) {
        const int ch = i < dimp ? c * dimp + i : i < 2 * dimp ? (p.dG + c) * dimp + i - dimp : 2 * p.dG * dimp + h * vdimp + i - 2 * dimp;
        const T now = (T)ld_f<COH>(p.proj + p.oc + ch);
        float acc = 0.0f;
        for (int tap = 0; tap + 1 < p.taps; tap++) {
            const int at = pos - (p.taps - 1) + tap;
            if (at >= 0) acc = fmaf(p.conv[size_t(tap) * p.channels + ch], (float)ring[size_t(at % p.taps) * p.channels + ch], acc);
        }
        acc = delta_silu(fmaf(p.conv[size_t(p.taps - 1) * p.channels + ch], (float)now, acc));
        (i < dimp ? s_q + i : i < 2 * dimp ? s_k + i - dimp : s_v + i - 2 * dimp)[0] = acc;
        if (keep && (i >= 2 * dimp || h % per == 0)) reinterpret_cast<T *>(p.ring)[size_t(pos % p.taps) * p.channels + ch] = now; // (no tap reads this row)
    }
    for (int i = tid; i < p.kd; i += 256) s_in[i] = i < p.rank_a + p.rank_g ? (T)ld_f<COH>(p.proj + p.od + i) : (T)0.0f;
    const float beta = lm_sigmoid(ld_f<COH>(p.beta + h)), rate = expf(p.a_log[h]);
    lds_barrier();
    if (wave < 2) { // unit vectors
        float *x = wave ? s_k : s_q, ss = 0.0f;
        for (int d = lane; d < dimp; d += 64) ss = fmaf(x[d], x[d], ss);
        float f = 1.0f / sqrtf(wave_sum(ss) + DELTA_UNIT_EPS);
        if (!wave) f *= 1.0f / sqrtf((float)p.ddim);
        for (int d = lane; d < dimp; d += 64) x[d] *= f;
    }
    { // second steps of the decay's and the gate's projections, 8 lanes a row
        const int a_end = (p.rank_a + PE - 1) / PE, g_begin = p.rank_a / PE, g_end = (p.rank_a + p.rank_g + PE - 1) / PE, rows = dimp + vdimp;
        constexpr int RU = 4; // rows a lane works on at a time
        for (int base = tid >> 3; base < (rows + 31) / 32 * 32; base += 32 * RU) {
            float acc[RU];
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int i = base + 32 * u;
                const bool is_a = i < dimp;
                acc[u] = 0.0f;
                if (i >= rows) continue;
                const T *w = reinterpret_cast<const T *>(p.wlr) + size_t(is_a ? p.lr16 + h * dimp + i : h * vdimp + i - dimp) * p.kd;
                const int end = is_a ? a_end : g_end, first = (is_a ? 0 : g_begin) + (tid & 7); // (the other step's columns are zero)
                for (int q = first; q < end; q += 8)
                    acc[u] = dot_piece<T>(reinterpret_cast<const lm_u32x4 *>(w)[q], *reinterpret_cast<const lm_u32x4 *>(s_in + q * PE), acc[u]);
            }
#pragma unroll
            for (int off = 4; off >= 1; off >>= 1)
#pragma unroll
                for (int u = 0; u < RU; u++) acc[u] += __shfl_xor(acc[u], off);
#pragma unroll
            for (int u = 0; u < RU; u++) {
                const int i = base + 32 * u;
                if ((tid & 7) || i >= rows) continue;
                if (i < dimp) s_g[i] = delta_decay(rate, acc[u] + p.dt_bias[h * dimp + i]);
                else s_gate[i - dimp] = lm_sigmoid(acc[u]);
            }
        }
    }
    lds_barrier();
    auto sum_rows = [&](const float4_t &mine, auto done) { // four columns per thread, summed over the row groups
        if (on) *reinterpret_cast<float4_t *>(s_sum + r0 * vdimp + col * 4) = mine;
        lds_barrier();
        for (int d = tid; d < vdimp; d += 256) {
            float t = 0.0f;
            for (int r = 0; r < rp; r++) t += s_sum[r * vdimp + d];
            done(d, t);
        }
        lds_barrier();
    };
    float4_t w = {0, 0, 0, 0}, o = {0, 0, 0, 0};
    if (REG) {
#pragma unroll
        for (int i = 0; i < DELTA_ROWS; i++) {
            const int row = r0 + i * rp;
            if (row >= dimp) continue;
            S[i] *= s_g[row];
            w += S[i] * s_k[row];
        }
    } else
        for (int row = r0; row < dimp; row += rp) w += load(row) * (s_g[row] * s_k[row]);
    sum_rows(w, [&](int d, float t) { s_u[d] = beta * (s_v[d] - t); });
    if (on) {
        const float4_t u = *reinterpret_cast<const float4_t *>(s_u + col * 4);
        auto update = [&](int row, float4_t s) {
            s += u * s_k[row];
            o += s * s_q[row];
            if (keep) state[size_t(row) * vq] = s;
        };
        if (REG) {
#pragma unroll
            for (int i = 0; i < DELTA_ROWS; i++)
                if (r0 + i * rp < dimp) update(r0 + i * rp, S[i]);
        } else
            for (int row = r0; row < dimp; row += rp) update(row, load(row) * s_g[row]);
    }
    sum_rows(o, [&](int d, float t) { s_u[d] = t; });
    float ss = 0.0f;
    for (int d = lane; d < vdimp; d += 64) ss = fmaf(s_u[d], s_u[d], ss); // (every wavefront by itself)
    const float f = 1.0f / sqrtf(wave_sum(ss) / (float)p.dvdim + p.eps);
    for (int d = tid; d < vdimp; d += 256) st_t<COH>(reinterpret_cast<T *>(p.dout) + h * vdimp + d, (T)(s_u[d] * f * p.dnorm[d] * s_gate[d]));
    meet.done();
}


// ---- host: what the launches of one token's attention have in common
inline bool mix_whole(const DecodeMix &p) { return p.whole || p.rot || p.rotv || p.pool || p.temp || p.borrowed || p.dH; }
inline int mix_keys(const DecodeMix &p, size_t pos) {
    const int n_win = (int)(p.window ? std::min(pos + 1, (size_t)p.window) : pos + 1);
    return n_win + (p.pool ? (int)(pos + 1 - n_win) / p.pool : 0);
}
inline int check_decode_mix(moon_ctx *ctx, const DecodeMix &p) {
    if (p.pool && ((p.pos + 1) / p.pool > (size_t)p.blocks || (p.pos + 1 >= (size_t)p.pool && p.pool > p.cap))) return moon_fail(ctx, MOON_EINVAL_DIM, "decode attention: %d pooled blocks kept", p.blocks);
    if (mix_whole(p) && (p.qk_rms || p.mixes)) return moon_fail(ctx, MOON_EINVAL, "decode attention: norms per head or mixed values beside rotation, blocks or a norm of all of q");
    if (p.dH && (p.dH % p.dG || p.ddimp % 16 || p.dvdimp % 16 || p.ddimp > (int)DELTA_MAX_DIM || p.dvdimp > (int)DELTA_MAX_DIM || p.oc % 8 || p.kd % 64))
        return moon_fail(ctx, MOON_EINVAL_DIM, "decode: delta rule with head sizes %d and %d", p.ddimp, p.dvdimp);
    return MOON_OK;
}

} // namespace
