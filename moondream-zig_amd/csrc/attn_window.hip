// Causal attention of several query rows over a KV cache, with a sliding window, pooled blocks before it, grouped key/value heads, a
// sink in the softmax denominator, a factor per head on the scale, outputs that turn back by their position's angles (where the values
// were turned by theirs) and an output gate; each of them is an argument.  The cache of a layer is [G][cap][head size]; the keys of
// position p lie in row p % cap, so a windowed layer needs no more rows than its window and one call's rows together.
//
// bf16 runs on the matrix cores, arranged like the kernel of attn_prefill.hip: a 256-thread workgroup owns 32 query rows of one
// head, its four wavefronts take every fourth tile of 64 keys of the range the rows can see, each with an online softmax of its
// own over private LDS staging, and the four results are merged at the end.  Per tile, with v_mfma_f32_32x32x16_bf16 and f32
// accumulation,
//     S^T[key][q] = K . Q^T     (a lane holds 32 scores of ONE query)
//     O^T[d][q]  += V^T . P^T   (V row-major in LDS, transposed by the LDS load)
// Scores and weights are f32.  A weight enters the second product as two bf16 terms, its rounding and the remainder, so the
// product sees 16 bits of it.  Heads of 64 in calls with enough rows share their tiles between four wavefronts instead
// (window_attn_shared_kernel).
// f32, and head sizes above 256, take one wavefront per (row, head) with plain multiply-adds.
#include "lane_fold.hpp"
#include "layer_list.hpp"
#include "lm_types.hpp"
#include "tile_copy.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace {

// Blocks that lie wholly before the window of position pos: block b ends at b pool + pool - 1 <= pos - window
__device__ __forceinline__ int blocks_seen(int pos, int window, int pool) { return max(0, pos - window + 1) / pool; }

constexpr int WA_KT = 64, WA_Q = 32, WA_WAVES = 4; // keys per tile, query rows and wavefronts per workgroup
typedef short wa_short4_t __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

template <int P> struct WaCfg { // P: head sizes up to P (a multiple of 32), rows zero padded to it
    static constexpr int KSTEPS = P / 16, DT = P / 32, G = P / 8;
    static constexpr int KS = P + 8; // K row stride: 128-bit reads of consecutive rows are conflict free
    // V rows are unpadded.  The transposing reads take 16 dwords of each of 4 consecutive rows: rows of 16 or 48 dwords lie apart
    // mod 64 by themselves, in the others granule c of row r sits at c ^ SWZ * (r % 4).
    static constexpr int VS = P, SWZ = P == 64 ? 2 : P >= 128 ? 4 : 0;
    static constexpr int WAVE_ELEMS = WA_KT * KS; // K is only read before the scores, V only after: they share the area
    static constexpr int LOADS = G;  // 16-byte pieces per lane and operand tile
    static constexpr bool AHEAD = P <= 128; // the next tile's pieces wait in registers (above, there are too many)
    static constexpr int SD = P + 4; // merge: O as [wave][q][SD] floats, (m, l) [wave][q] behind them
    static constexpr size_t TILE_BYTES = size_t(WA_WAVES) * WAVE_ELEMS * 2, MERGE_BYTES = size_t(WA_WAVES) * WA_Q * SD * 4;
    static constexpr size_t ML_OFFSET = TILE_BYTES > MERGE_BYTES ? TILE_BYTES : MERGE_BYTES;
    static constexpr size_t LDS_BYTES = ML_OFFSET + 2 * WA_WAVES * WA_Q * 4;
};

__device__ __forceinline__ wa_short4_t wa_read_tr(const bf16_t *p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) wa_short4_t *)(p));
}

// Two weights as two bf16 terms each: a packed conversion, its two halves back as f32, the remainders
__device__ __forceinline__ uint2 split_pair(float w0, float w1) {
    const unsigned hi = __builtin_bit_cast(unsigned, __builtin_convertvector(float2_t{w0, w1}, bf16x2_t));
    const float2_t rest = {w0 - __builtin_bit_cast(float, hi << 16), w1 - __builtin_bit_cast(float, hi & 0xffff0000u)};
    return uint2{hi, __builtin_bit_cast(unsigned, __builtin_convertvector(rest, bf16x2_t))};
}

// POOL: the tiles of the blocks' keys come first, in the same softmax
template <int P, bool POOL>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(P <= 64 ? 2 : 1))) void window_attn_kernel(WindowAttn p) {
    using C = WaCfg<P>;
    extern __shared__ __attribute__((aligned(16))) bf16_t wa_lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), col = lane & 31, hf = lane >> 5;
    const int n_qb = (p.n + WA_Q - 1) / WA_Q;
    // Workgroups are dealt to the eight dies round robin: where the count divides, a die takes whole stretches of the (head, block)
    // list, so heads that share keys and values meet in one L2.  Late blocks see the most keys: they start first.
    int item = blockIdx.x;
    const int n_items = n_qb * p.H;
    if (n_items % 8 == 0) item = (item % 8) * (n_items / 8) + item / 8;
    int h = item / n_qb, qb = item % n_qb;
    if (n_items % 8 == 0 && (n_items / 8) % n_qb == 0) { // whole heads per die: their blocks walk together
        const int per_die = n_items / 8, heads = per_die / n_qb, j = item % per_die;
        h = item / per_die * heads + j % heads;
        qb = j / heads;
    }
    qb = n_qb - 1 - qb;
    const int g = h / (p.H / p.G), row0 = qb * WA_Q;
    const int first_pos = p.pos0 + row0, last_pos = p.pos0 + min(row0 + WA_Q, p.n) - 1, pos = first_pos + col; // pos: this lane's query
    const int lo_key = p.window ? max(0, first_pos - p.window + 1) : 0;
    // tiles start at multiples of 64 positions; POOL: tile numbers below t_window stand for blocks (of the first one, from 0 on)
    const int seen = POOL ? blocks_seen(last_pos, p.window, p.pool) : 0, t_blocks = (seen + WA_KT - 1) / WA_KT;
    const int t_begin = POOL ? lo_key / WA_KT - t_blocks : lo_key / WA_KT, t_end = last_pos / WA_KT + 1;
    const int t_window = POOL ? lo_key / WA_KT : 0;
    // the head's cache rows as buffers: a 32-bit offset per piece, and what must not be read is an offset past the end (zeros)
    const int k_bytes = p.cap * p.dimp * 2, v_bytes = p.cap * p.vdimp * 2;
    const __amdgpu_buffer_rsrc_t kr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(reinterpret_cast<const bf16_t *>(p.ck) + size_t(g) * p.cap * p.dimp), 0, k_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(reinterpret_cast<const bf16_t *>(p.cv) + size_t(g) * p.cap * p.vdimp), 0, v_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t pkr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(reinterpret_cast<const bf16_t *>(p.pk) + size_t(g) * p.blocks * p.dimp), 0, POOL ? p.blocks * p.dimp * 2 : 0, 0x00020000);
    const __amdgpu_buffer_rsrc_t pvr = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(reinterpret_cast<const bf16_t *>(p.pv) + size_t(g) * p.blocks * p.vdimp), 0, POOL ? p.blocks * p.vdimp * 2 : 0, 0x00020000);
    bf16_t *Ks = wa_lds + wave * C::WAVE_ELEMS, *Vs = Ks;

    constexpr int NOWHERE = 0x7fffffff; // past the end of either buffer
    lm_u32x4 rk[C::LOADS], rv[C::LOADS];
    int k_off[C::LOADS], v_off[C::LOADS]; // this lane's pieces of a tile whose first row is row 0
#pragma unroll
    for (int i = 0; i < C::LOADS; i++) {
        const int x = i * 64 + lane, row = x / C::G, c = x % C::G;
        k_off[i] = c * 8 < p.dimp ? (row * p.dimp + c * 8) * 2 : NOWHERE;
        v_off[i] = c * 8 < p.vdimp ? (row * p.vdimp + c * 8) * 2 : NOWHERE;
    }
    auto load = [&](lm_u32x4 (&r)[C::LOADS], const __amdgpu_buffer_rsrc_t rs, const __amdgpu_buffer_rsrc_t blocks, const int (&offs)[C::LOADS], int d, int t) {
        if (POOL && t < t_window) {
            const int b0 = __builtin_amdgcn_readfirstlane((t - t_begin) * WA_KT);
#pragma unroll
            for (int i = 0; i < C::LOADS; i++) {
                const int off = offs[i] == NOWHERE || b0 + (i * 64 + lane) / C::G >= seen ? NOWHERE : offs[i] + b0 * d * 2;
                r[i] = __builtin_bit_cast(lm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(blocks, off, 0, 0));
            }
            return;
        }
        const int key0 = __builtin_amdgcn_readfirstlane(t * WA_KT), slot0 = key0 < p.cap ? key0 : key0 % p.cap, row_bytes = d * 2;
        if (key0 >= lo_key && key0 + WA_KT - 1 <= last_pos && slot0 + WA_KT <= p.cap) { // the whole tile, in one piece
#pragma unroll
            for (int i = 0; i < C::LOADS; i++) r[i] = __builtin_bit_cast(lm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, offs[i], slot0 * row_bytes, 0));
        } else {
#pragma unroll
            for (int i = 0; i < C::LOADS; i++) {
                const int row = (i * 64 + lane) / C::G, key = key0 + row;
                int off = (offs[i] == NOWHERE ? 0 : offs[i]) + slot0 * row_bytes;
                if (slot0 + row >= p.cap) off -= p.cap * row_bytes; // (a cache that wraps has more rows than a tile)
                if (offs[i] == NOWHERE || key < lo_key || key > last_pos) off = NOWHERE;
                r[i] = __builtin_bit_cast(lm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
            }
        }
    };
    auto store = [&](const lm_u32x4 (&r)[C::LOADS], bf16_t *dst, int stride, int swz) {
#pragma unroll
        for (int i = 0; i < C::LOADS; i++) {
            const int x = i * 64 + lane, row = x / C::G;
            *reinterpret_cast<lm_u32x4 *>(dst + row * stride + (x % C::G ^ swz * (row & 3)) * 8) = r[i];
        }
    };
    int t = t_begin + wave;
    if (C::AHEAD && t < t_end) load(rk, kr, pkr, k_off, p.dimp, t);
    const float scale = p.temp ? p.scale * p.temp[h] : p.scale;
    bf16x8_t qf[C::KSTEPS]; // the MFMA "B" operand: Q[row0 + col][16 s + 8 hf .. + 7]
    {
        const bf16_t *q = reinterpret_cast<const bf16_t *>(p.q) + size_t(min(row0 + col, p.n - 1)) * p.ldq + h * p.dimp;
#pragma unroll
        for (int s = 0; s < C::KSTEPS; s++) {
            lm_u32x4 v = {0, 0, 0, 0};
            if (16 * s + 8 * hf < p.dimp) v = *reinterpret_cast<const lm_u32x4 *>(q + 16 * s + 8 * hf);
            if (scale < 0.0f) v ^= 0x80008000u; // scores are kept unscaled and the scale enters as its magnitude: the sign goes here
            qf[s] = __builtin_bit_cast(bf16x8_t, v);
        }
    }
    if (C::AHEAD && t < t_end) load(rv, vr, pvr, v_off, p.vdimp, t);
    int voff[C::DT]; // where this lane points the transposing loads: key 4 hf + (lane % 16) / 4, columns 32 dt + 16 ((lane / 16) % 2) + 4 (lane % 4)
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++) {
        const int rq = (lane & 15) >> 2, d = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        voff[dt] = (4 * hf + rq) * C::VS + ((d >> 3 ^ C::SWZ * rq) << 3 | (d & 7));
    }

    float16_t o[C::DT];
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[dt][v] = 0.0f;
    constexpr float LOG2E = 1.4426950408889634f;
    const float c2 = fmaxf(fabsf(scale) * LOG2E, 1e-37f); // > 0: the maximum of the scaled scores is the scaled maximum, -inf stays -inf
    const float sink = p.sink ? p.sink[h] * LOG2E : -INFINITY;
    float m_run = -INFINITY, l_run = 0.0f; // m_run: scaled, in base-2 units; l_run: this lane's half of the row's sum

    for (; t < t_end; t += WA_WAVES) {
        const int key0 = t * WA_KT;
        if (!C::AHEAD) load(rk, kr, pkr, k_off, p.dimp, t);
        asm volatile("" ::: "memory"); // the V tile of the round before has been read: the K tile takes its place
        store(rk, Ks, C::KS, 0);
        if (C::AHEAD && t + WA_WAVES < t_end) load(rk, kr, pkr, k_off, p.dimp, t + WA_WAVES);
        if (!C::AHEAD) load(rv, vr, pvr, v_off, p.vdimp, t);
        float16_t s[2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
#pragma unroll
            for (int v = 0; v < 16; v++) s[kt][v] = 0.0f;
#pragma unroll
            for (int st = 0; st < C::KSTEPS; st++)
                s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t *>(Ks + (32 * kt + col) * C::KS + 16 * st + 8 * hf), qf[st],
                                                                s[kt], 0, 0, 0);
        }
        // s[kt][v]: key key0 + 32 kt + 8 (v / 4) + 4 hf + v % 4 against this lane's query
        float mx = -INFINITY;
        if (POOL && t < t_window) {
            const int mine = blocks_seen(pos, p.window, p.pool) - (t - t_begin) * WA_KT - 4 * hf;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float x = 32 * kt + 8 * (v >> 2) + (v & 3) < mine ? s[kt][v] : -INFINITY;
                    s[kt][v] = x;
                    mx = fmaxf(mx, x);
                }
        } else if (key0 + WA_KT - 1 > first_pos || (p.window && key0 < last_pos - p.window + 1)) { // some row does not see the whole tile
            const int age0 = pos - key0 - 4 * hf; // how far back this lane's first key is
            const unsigned ages = p.window ? (unsigned)p.window : 0x7fffffffu;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) { // (a key ahead of the query wraps to a large age)
                    const float x = (unsigned)(age0 - (32 * kt + 8 * (v >> 2) + (v & 3))) < ages ? s[kt][v] : -INFINITY;
                    s[kt][v] = x;
                    mx = fmaxf(mx, x);
                }
        } else {
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[kt][v]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx * c2), m_use = m_new == -INFINITY ? 0.0f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
        const bool rescale = __any(m_new != m_run);
        m_run = m_new;
        float psum = 0.0f;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][v], c2, -m_use));
                s[kt][v] = e;
                psum += e;
            }
        l_run = l_run * alpha + psum;
        if (rescale)
#pragma unroll
            for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++) o[dt][v] *= alpha;
        asm volatile("" ::: "memory"); // the K tile has been read (LDS serves a wavefront in order): V takes its place
        store(rv, Vs, C::VS, C::SWZ);
        if (C::AHEAD && t + WA_WAVES < t_end) load(rv, vr, pvr, v_off, p.vdimp, t + WA_WAVES);
        // contraction step (kt, sp) uses the keys a lane holds in s[kt][8 sp .. 8 sp + 7]: key0 + 32 kt + 16 sp + {4 hf + 0..3, 8 + 4 hf + 0..3}
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int sp = 0; sp < 2; sp++) {
                lm_u32x4 hi_bits, lo_bits;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const uint2 pair = split_pair(s[kt][8 * sp + 2 * e], s[kt][8 * sp + 2 * e + 1]);
                    hi_bits[e] = pair.x;
                    lo_bits[e] = pair.y;
                }
                const bf16x8_t hi = __builtin_bit_cast(bf16x8_t, hi_bits), lo = __builtin_bit_cast(bf16x8_t, lo_bits);
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++) {
                    const bf16_t *vp = Vs + voff[dt] + (32 * kt + 16 * sp) * C::VS;
                    const wa_short4_t a0 = wa_read_tr(vp), a1 = wa_read_tr(vp + 8 * C::VS);
                    const bf16x8_t a = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, lo, o[dt], 0, 0, 0);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, hi, o[dt], 0, 0, 0);
                }
            }
    }

    // this thread's gate values (and angles) for the merged result, requested before the merge
    const int q = tid & 31, row = row0 + q, d0 = (tid >> 5) * 8;
    const bf16_t *gate = p.gate ? reinterpret_cast<const bf16_t *>(p.gate) + size_t(min(row, p.n - 1)) * p.ldq + h * p.vdimp : nullptr;
    bf16x8_t gz = {};
    if (gate && d0 < p.vdimp) gz = *reinterpret_cast<const bf16x8_t *>(gate + d0);
    const bool pairs = P == 64 && p.rotv && p.vdim == 64; // (eight pairs lie in two granules: 37.1 -> 33 us at 1301 rows of 32 rotated heads)
    float4_t turn[4] = {}; // and its angles: cos, sin, cos, sin
    if (P == 64 && pairs)
#pragma unroll
        for (int e = 0; e < 4; e++) turn[e] = reinterpret_cast<const float4_t *>(p.rotv + size_t(p.pos0 + min(row, p.n - 1)) * 32 + (d0 & 31))[e];
    // merge the wavefronts' results; the sink is one more term of the denominator
    const float l_wave = l_run + __shfl_xor(l_run, 32);
    float *so = reinterpret_cast<float *>(wa_lds), *sm = reinterpret_cast<float *>(reinterpret_cast<char *>(wa_lds) + C::ML_OFFSET), *sl = sm + WA_WAVES * WA_Q;
    if (hf == 0) {
        sm[wave * WA_Q + col] = m_run;
        sl[wave * WA_Q + col] = l_wave;
    }
    __syncthreads(); // every wavefront is done with its staging area
    float m_all = sink;
#pragma unroll
    for (int w = 0; w < WA_WAVES; w++) m_all = fmaxf(m_all, sm[w * WA_Q + col]);
    const float f = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_all);
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int j = 0; j < 4; j++) { // o[dt][4 j .. 4 j + 3] are elements 32 dt + 8 j + 4 hf .. + 3
            const float4 r = {o[dt][4 * j] * f, o[dt][4 * j + 1] * f, o[dt][4 * j + 2] * f, o[dt][4 * j + 3] * f};
            *reinterpret_cast<float4 *>(so + (wave * WA_Q + col) * C::SD + 32 * dt + 8 * j + 4 * hf) = r;
        }
    __syncthreads();
    if (row >= p.n) return;
    float l_all = p.sink ? __builtin_amdgcn_exp2f(sink - m_all) : 0.0f;
#pragma unroll
    for (int w = 0; w < WA_WAVES; w++) {
        const float mw = sm[w * WA_Q + q];
        if (mw != -INFINITY) l_all += __builtin_amdgcn_exp2f(mw - m_all) * sl[w * WA_Q + q];
    }
    const float inv = 1.0f / l_all;
    bf16_t *out = reinterpret_cast<bf16_t *>(p.out) + size_t(row) * p.ldo + h * p.vdimp;
    for (int d = d0; d < p.vdimp; d += 64) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < WA_WAVES; w++)
#pragma unroll
            for (int e = 0; e < 8; e++) acc[e] += so[(w * WA_Q + q) * C::SD + d + e];
#pragma unroll
        for (int e = 0; e < 8; e++) acc[e] *= inv;
        if (P == 64 && pairs) { // the other ones of eight pairs lie 32 elements away
            float other[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WA_WAVES; w++)
#pragma unroll
                for (int e = 0; e < 8; e++) other[e] += so[(w * WA_Q + q) * C::SD + (d ^ 32) + e];
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float c = turn[e / 2][2 * (e & 1)], sn = turn[e / 2][2 * (e & 1) + 1], z = other[e] * inv;
                acc[e] = d & 32 ? acc[e] * c - z * sn : acc[e] * c + z * sn;
            }
        } else if (p.rotv) { // each element with the other one of its pair
            const int half = p.vdim / 2;
#pragma unroll
            for (int e = 0; e < 8; e++)
                if (d + e < 2 * half) {
                    const bool second = d + e >= half;
                    const int m = second ? d + e - half : d + e, other = second ? m : m + half;
                    const float2 cs = p.rotv[size_t(p.pos0 + row) * half + m];
                    float z = 0.0f;
#pragma unroll
                    for (int w = 0; w < WA_WAVES; w++) z += so[(w * WA_Q + q) * C::SD + other];
                    z *= inv;
                    acc[e] = second ? acc[e] * cs.x - z * cs.y : acc[e] * cs.x + z * cs.y;
                }
        }
        bf16x8_t r;
        if (gate && d != d0) gz = *reinterpret_cast<const bf16x8_t *>(gate + d);
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = (bf16_t)(acc[e] * (gate ? lm_sigmoid((float)gz[e]) : 1.0f));
        *reinterpret_cast<bf16x8_t *>(out + d) = r;
    }
}

constexpr int WS_PAIRED = 64; // workgroups of a die that are there at once: two per unit

// Heads of 64 in calls with many rows.  A workgroup takes four units of 32 query rows, heads that read the same keys where a group has
// them, else the next rows; a unit's wavefront walks all of its keys, so the four share every tile and nothing is merged over rows.  Two
// such groups of wavefronts take every other tile, merged once at the end: with one, the wavefronts of a call that puts one workgroup on a
// unit are alone on their SIMDs and spend 1.5 us a tile, mostly waiting; with two, 1.9 us for two.  Tiles are copied straight to LDS
// (tile_copy.hpp), the next one while one is worked on, with a barrier per tile.
// A window of 1024 is 17 tiles: the kernel above gives a wavefront four of them, and its first loads, scores' masks and merge cost as much
// as the tiles.  What bounds this one is the vector unit (of about 1,370 cycles a tile and wavefront, exponentials 510, the weights' second
// term 380) and, in calls of one workgroup per unit, latency: start and end take 7 us.
// Times, above -> here: 32 heads on 8 key heads, window 1024, 1920 rows 52.2 -> 38.2 us, 1301 rows 35.2 -> 28.2, with blocks 34.9 -> 26.6, rotated 34.7 -> 26.5; with 32
// key heads 52.2 -> 39.8, 35.2 -> 29.4, 34.8 -> 29.0, 34.6 -> 27.4.
// Measured and not kept: 64 rows per wavefront in the arrangement above (43.5 us at 1920 rows; better, by 15 %, only around 768); two
// wavefronts instead of four there (46.9); remainders of the weights by two-element dot products (1 to 3 us slower); wave priorities.
struct WsCfg {
    static constexpr int D = 64, KSTEPS = D / 16, DT = D / 32, G = D / 8, STAGES = 2, GROUPS = 2;
    static constexpr int TILE = WA_KT * D, COPIES = WA_KT * G / 64 / WA_WAVES; // elements of a K or V tile, copies of each per wavefront
    static constexpr size_t TILE_BYTES = size_t(GROUPS) * STAGES * 2 * TILE * 2, LDS_BYTES = TILE_BYTES + GROUPS * WA_WAVES * sizeof(int);
};
__host__ __device__ __forceinline__ int ws_heads(int per_group) { return per_group % 4 == 0 ? 4 : per_group % 2 == 0 ? 2 : 1; } // heads per workgroup
__host__ __device__ __forceinline__ int ws_rows(int per_group) { return WA_Q * WA_WAVES / ws_heads(per_group); }                 // rows per workgroup

// The lane's number, asked for anew: a value that the compiler does not keep in a register (or in memory) across what came before
__device__ __forceinline__ int lane_again() {
    int lane;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
    return lane;
}

// APART: wavefronts of one workgroup have different rows (fewer than four heads read the same keys)
template <bool POOL, bool APART>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(4))) void window_attn_shared_kernel(WindowAttn p) {
    using C = WsCfg;
    constexpr int D = C::D, ROW = D * 2; // ROW: bytes of a cache row
    extern __shared__ __attribute__((aligned(16))) bf16_t wa_lds[];
    const int tid = threadIdx.x, kg = __builtin_amdgcn_readfirstlane(tid >> 8), wave = __builtin_amdgcn_readfirstlane(tid >> 6 & 3);
    const int per = p.H / p.G, nh = ws_heads(per), rows = ws_rows(per), n_qb = (p.n + rows - 1) / rows, n_hb = p.H / nh;
    // which heads and rows: a die takes whole stretches of the (heads, block) list, late blocks first
    int item = blockIdx.x;
    const int n_items = n_qb * n_hb;
    int hb = item / n_qb, qb = item % n_qb;
    if (n_items % 8 == 0 && (n_items / 8) % n_qb == 0) { // whole heads per die: their blocks walk together
        const int per_die = n_items / 8, heads = per_die / n_qb;
        int j = item / 8;
        if (per_die <= WS_PAIRED && j >= WS_PAIRED / 2) j = per_die - 1 - (j - WS_PAIRED / 2); // two per unit: the lightest beside the heaviest
        hb = item % 8 * heads + j % heads;
        qb = j / heads;
    }
    qb = n_qb - 1 - qb;
    const int h = hb * nh + wave % nh, g = h / per, wg_row0 = qb * rows, row0 = wg_row0 + wave / nh * WA_Q;
    const int wg_first = p.pos0 + wg_row0, last_pos = p.pos0 + min(wg_row0 + rows, p.n) - 1; // positions of the workgroup's first and last row
    const int first_pos = p.pos0 + row0;                                                      // and of the wavefront's first row
    const int lo_key = p.window ? max(0, wg_first - p.window + 1) : 0;
    const int seen = POOL ? blocks_seen(last_pos, p.window, p.pool) : 0, t_blocks = (seen + WA_KT - 1) / WA_KT;
    const int t_begin = POOL ? lo_key / WA_KT - t_blocks : lo_key / WA_KT, t_end = last_pos / WA_KT + 1;
    const int t_window = POOL ? lo_key / WA_KT : 0;
    const int lo_mine = p.window ? max(0, first_pos - p.window + 1) : 0, seen_mine = POOL ? blocks_seen(first_pos + WA_Q - 1, p.window, p.pool) : 0; // of the wavefront's 32 rows
    const size_t head_rows = size_t(g) * p.cap * ROW, head_blocks = POOL ? size_t(g) * p.blocks * ROW : 0;
    const char *ck = reinterpret_cast<const char *>(p.ck) + head_rows, *cv = reinterpret_cast<const char *>(p.cv) + head_rows;
    const char *pk = reinterpret_cast<const char *>(p.pk) + head_blocks, *pv = reinterpret_cast<const char *>(p.pv) + head_blocks;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<unsigned long>((__attribute__((address_space(3))) const bf16_t *)wa_lds));
    constexpr float LOG2E = 1.4426950408889634f;
    const float scale = p.temp ? p.scale * p.temp[h] : p.scale;
    const float c2 = fmaxf(fabsf(scale) * LOG2E, 1e-37f);
    const float sink = p.sink ? p.sink[h] * LOG2E : -INFINITY;
    float16_t o[C::DT];
    float m_run, l_run;

    // STRICT: values that none of the wavefront's 32 rows read are zero.  A tile may have some for the workgroup's other rows, whose weights here are
    // zero; zero times infinity is not.
    auto walk = [&](auto strict, int lane) {
        constexpr bool STRICT = decltype(strict)::value;
        const int col = lane & 31, hf = lane >> 5, pos = first_pos + col; // pos: this lane's query
        int off[C::COPIES]; // this lane's granules of a tile, from its first row (K and V lie alike)
#pragma unroll
        for (int i = 0; i < C::COPIES; i++) {
            const int row = (wave * C::COPIES + i) * 8 + (lane >> 3);
            off[i] = row * ROW + ((lane & 7) ^ row64_swizzle(row)) * 16;
        }
        // This wavefront's part of tile t to stage t % STAGES; rows that must not be read are offsets past the end, which bring zeros.
        constexpr int NOWHERE = 0x7fffffff;
        auto copy = [&](int t, int stage) {
            const unsigned k_lds = lds0 + (kg * C::STAGES + stage) * 2 * C::TILE * 2 + wave * C::COPIES * 1024, v_lds = k_lds + C::TILE * 2;
            const bool blocks = POOL && t < t_window;
            const int key0 = blocks ? (t - t_begin) * WA_KT : t * WA_KT, lo = blocks ? 0 : lo_key, hi = blocks ? seen - 1 : last_pos, rows = blocks ? p.blocks : p.cap;
            const int slot0 = key0 < rows ? key0 : key0 % rows;
            const bool whole = key0 >= lo && key0 + WA_KT - 1 <= hi && slot0 + WA_KT <= rows; // in one piece
            int offs[C::COPIES];
#pragma unroll
            for (int i = 0; i < C::COPIES; i++) {
                const int row = (wave * C::COPIES + i) * 8 + (lane >> 3), key = key0 + row;
                offs[i] = off[i] + slot0 * ROW;
                if (whole) continue;
                if (slot0 + row >= rows) offs[i] -= rows * ROW; // (a cache that wraps has more rows than a tile)
                if (key < lo || key > hi) offs[i] = NOWHERE;
            }
            tile_copy(blocks ? pk : ck, rows * ROW, k_lds, offs);
            tile_copy(blocks ? pv : cv, rows * ROW, v_lds, offs);
        };
        if (t_begin + kg < t_end) copy(t_begin + kg, 0);
        bf16x8_t qf[C::KSTEPS]; // the MFMA "B" operand: Q[row0 + col][16 s + 8 hf .. + 7]
        {
            const bf16_t *q = reinterpret_cast<const bf16_t *>(p.q) + size_t(min(row0 + col, p.n - 1)) * p.ldq + h * D;
#pragma unroll
            for (int s = 0; s < C::KSTEPS; s++) {
                lm_u32x4 v = *reinterpret_cast<const lm_u32x4 *>(q + 16 * s + 8 * hf);
                if (scale < 0.0f) v ^= 0x80008000u; // (as in window_attn_kernel)
                qf[s] = __builtin_bit_cast(bf16x8_t, v);
            }
        }
        int voff[2][C::DT]; // where this lane points the transposing loads: keys 4 hf + (lane % 16) / 4 (+ 8), columns 32 dt + 16 ((lane / 16) % 2) + 4 (lane % 4)
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int dt = 0; dt < C::DT; dt++) {
                const int key = 8 * j + 4 * hf + ((lane & 15) >> 2), c = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
                voff[j][dt] = key * D + ((c >> 3 ^ row64_swizzle(key)) << 3 | (c & 7));
            }
        __builtin_amdgcn_s_waitcnt(0xf70); // vmcnt(0): the query rows have arrived (else the compiler waits for them, and every copy, in each round)
        const int mine0 = POOL ? blocks_seen(pos, p.window, p.pool) - 1 - 4 * hf : 0; // the last block that this lane's row sees, from its first one
        m_run = -INFINITY;
        l_run = 0.0f;
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[dt][v] = 0.0f;
        for (int left = (t_end - t_begin + C::GROUPS - 1) / C::GROUPS, stage = 0, t = t_begin + kg; left > 0; left--, t += C::GROUPS, stage ^= 1) {
            const int key0 = t * WA_KT;
            tile_handed_over();
            if (t + C::GROUPS < t_end) copy(t + C::GROUPS, stage ^ 1);
            if (t >= t_end) continue;
            const bool blocks = POOL && t < t_window;
            if (!blocks && (key0 > first_pos + WA_Q - 1 || (p.window && key0 + WA_KT <= first_pos - p.window + 1))) continue; // no row sees any of it
            const bf16_t *Ks = wa_lds + (kg * C::STAGES + stage) * 2 * C::TILE, *Vs = Ks + C::TILE;
            float16_t s[2];
            bf16x8_t a[2][C::KSTEPS];
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int st = 0; st < C::KSTEPS; st++) a[kt][st] = *reinterpret_cast<const bf16x8_t *>(Ks + (32 * kt + col) * D + ((2 * st + hf) ^ row64_swizzle(col)) * 8);
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) s[kt][v] = 0.0f;
#pragma unroll
            for (int st = 0; st < C::KSTEPS; st++)
#pragma unroll
                for (int kt = 0; kt < 2; kt++) s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[kt][st], qf[st], s[kt], 0, 0, 0);
            // s[kt][v]: key key0 + 32 kt + 8 (v / 4) + 4 hf + v % 4 against this lane's query
            if (blocks || key0 + WA_KT - 1 > first_pos || (p.window && key0 <= first_pos + WA_Q - 1 - p.window)) { // some row does not see the whole tile
                const int age0 = blocks ? mine0 - (t - t_begin) * WA_KT : pos - key0 - 4 * hf; // how far back this lane's first key (block) is
                const unsigned ages = !blocks && p.window ? (unsigned)p.window : 0x7fffffffu;
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) // (a key ahead of the query wraps to a large age)
                        s[kt][v] = (unsigned)(age0 - (32 * kt + 8 * (v >> 2) + (v & 3))) < ages ? s[kt][v] : -INFINITY;
            }
            asm volatile("" : "+v"(s[0]), "+v"(s[1])); // (in these registers on both paths: left alone, the scores are copied on each)
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[kt][v]);
            mx = half_max(mx);
            const float m_new = fmaxf(m_run, mx * c2), m_use = m_new == -INFINITY ? 0.0f : m_new;
            float alpha = 1.0f;
            if (__any(m_new != m_run)) {
                alpha = __builtin_amdgcn_exp2f(m_run - m_use);
                m_run = m_new;
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) o[dt][v] *= alpha;
            }
            float psum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kt][v], c2, -m_use));
                    s[kt][v] = e;
                    psum += e;
                }
            l_run = l_run * alpha + psum;
            // contraction step (kt, sp) uses the keys a lane holds in s[kt][8 sp .. 8 sp + 7], as in window_attn_kernel
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int sp = 0; sp < 2; sp++) {
                    lm_u32x4 hi_bits, lo_bits;
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint2 pair = split_pair(s[kt][8 * sp + 2 * e], s[kt][8 * sp + 2 * e + 1]);
                        hi_bits[e] = pair.x;
                        lo_bits[e] = pair.y;
                    }
                    const bf16x8_t hi = __builtin_bit_cast(bf16x8_t, hi_bits), lo = __builtin_bit_cast(bf16x8_t, lo_bits);
                    bf16x8_t v[C::DT];
#pragma unroll
                    for (int dt = 0; dt < C::DT; dt++) {
                        const wa_short4_t a0 = wa_read_tr(Vs + voff[0][dt] + (32 * kt + 16 * sp) * D), a1 = wa_read_tr(Vs + voff[1][dt] + (32 * kt + 16 * sp) * D);
                        v[dt] = __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7));
                    }
                    if (STRICT) {
                        const int from = (blocks ? 0 : lo_mine - key0) - 4 * hf; // the first value that the 32 rows read, counted from this lane's first
                        const int count = blocks ? max(0, seen_mine - (t - t_begin) * WA_KT) : first_pos + WA_Q - lo_mine; // and how many there are
                        lm_u32x4 read;
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const int key = 32 * kt + 16 * sp + 8 * (e >> 1) + 2 * (e & 1) - from;
                            read[e] = ((unsigned)key < (unsigned)count ? 0xffffu : 0u) | ((unsigned)(key + 1) < (unsigned)count ? 0xffff0000u : 0u);
                        }
#pragma unroll
                        for (int dt = 0; dt < C::DT; dt++) v[dt] = __builtin_bit_cast(bf16x8_t, __builtin_bit_cast(lm_u32x4, v[dt]) & read);
                    }
#pragma unroll
                    for (int dt = 0; dt < C::DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[dt], lo, o[dt], 0, 0, 0);
#pragma unroll
                    for (int dt = 0; dt < C::DT; dt++) o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v[dt], hi, o[dt], 0, 0, 0);
                }
        }
    };
    walk(std::false_type(), tid & 63);
    const int lane = lane_again(), col = lane & 31, hf = lane >> 5;

    // o[dt][4 j + e] is element 32 dt + 8 j + 4 hf + e of this lane's row.  The second group hands its result over, [wave][register][lane].
    float *so = reinterpret_cast<float *>(wa_lds) + wave * (C::DT * 16 + 2) * 64 + lane;
    l_run += __shfl_xor(l_run, 32);
    // what the results still need, requested before the merge: this lane's gate granules 4 dt + 2 i + hf, cos and sin of two pairs each
    const int row = row0 + col, at_row = min(row, p.n - 1);
    const bf16_t *gate = p.gate ? reinterpret_cast<const bf16_t *>(p.gate) + size_t(at_row) * p.ldq + h * D : nullptr;
    bf16x8_t gz[C::DT][2];
    float4_t turn[4][2];
    auto request = [&] {
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int i = 0; i < 2; i++) gz[dt][i] = kg == 0 && gate ? *reinterpret_cast<const bf16x8_t *>(gate + (4 * dt + 2 * i + hf) * 8) : bf16x8_t{};
        if (kg == 0 && p.rotv) // (over all of the head: the other one of a pair is 32 elements away)
#pragma unroll
            for (int j = 0; j < 4; j++)
#pragma unroll
                for (int e = 0; e < 2; e++) turn[j][e] = reinterpret_cast<const float4_t *>(p.rotv + size_t(p.pos0 + at_row) * (D / 2))[4 * j + 2 * hf + e];
    };
    request();
    // Where wavefronts have different rows and a result is not finite, once more: it may be a value that only the others read.  (Zeros put in place of
    // such values in every tile that may have some, by a choice per step, took 10 to 27 % more; this check takes up to 1 us: 32 heads with keys of their own,
    // window 1024, 768 rows 19.9 -> 20.4 us, 1301 rows 28.1 -> 28.8, 1920 rows 37.8 -> 38.9.)
    int *redo = reinterpret_cast<int *>(reinterpret_cast<char *>(wa_lds) + C::TILE_BYTES);
    if (APART) {
        float zero[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) zero[v & 3] = __builtin_fmaf(o[dt][v], 0.0f, zero[v & 3]);
        const bool again = __any((zero[0] + zero[1]) + (zero[2] + zero[3]) != 0.0f);
        if (lane == 0) redo[kg * WA_WAVES + wave] = again;
    }
    __syncthreads(); // every wavefront is done with the tiles
    if (APART && __builtin_expect(__any(redo[lane % (C::GROUPS * WA_WAVES)]), 0)) { // (its code behind everything else: in between it costs 1 us of instruction fetches)
        walk(std::true_type(), lane_again()); // (nothing of the first walk is kept for this one)
        l_run += __shfl_xor(l_run, 32);
        request();
        __syncthreads();
    }
    if (kg == 1) {
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) so[(16 * dt + v) * 64] = o[dt][v];
        so[C::DT * 16 * 64] = m_run;
        so[(C::DT * 16 + 1) * 64] = l_run;
    }
    __syncthreads();
    if (kg == 1) return;
    // (the sink is one more term of the denominator)
    const float m_other = so[C::DT * 16 * 64], m_all = fmaxf(fmaxf(sink, m_run), m_other);
    const float f = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_all), f_other = m_other == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_other - m_all);
    const float inv = 1.0f / (l_run * f + so[(C::DT * 16 + 1) * 64] * f_other + (p.sink ? __builtin_amdgcn_exp2f(sink - m_all) : 0.0f));
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[dt][v] = (o[dt][v] * f + so[(16 * dt + v) * 64] * f_other) * inv;
    if (p.rotv) {
#pragma unroll
        for (int j = 0; j < 4; j++)
#pragma unroll
            for (int e = 0; e < 4; e += 2) {
                const float4_t cs = turn[j][e / 2];
#pragma unroll
                for (int k = 0; k < 2; k++) {
                    const float x = o[0][4 * j + e + k], y = o[1][4 * j + e + k];
                    o[0][4 * j + e + k] = x * cs[2 * k] + y * cs[2 * k + 1];
                    o[1][4 * j + e + k] = y * cs[2 * k] - x * cs[2 * k + 1];
                }
            }
    }
    bf16_t *out = reinterpret_cast<bf16_t *>(p.out) + size_t(at_row) * p.ldo + h * D;
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int i = 0; i < 2; i++) { // halves of two granules against whole ones: the lower lanes take granule 4 dt + 2 i, the upper the next
            bf16x8_t r;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const auto x = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, (float)o[dt][8 * i + e]), __builtin_bit_cast(unsigned, (float)o[dt][8 * i + 4 + e]), false, false);
                const unsigned x0 = x[0], x1 = x[1];
                r[e] = (bf16_t)(__builtin_bit_cast(float, x0) * (gate ? lm_sigmoid((float)gz[dt][i][e]) : 1.0f));
                r[4 + e] = (bf16_t)(__builtin_bit_cast(float, x1) * (gate ? lm_sigmoid((float)gz[dt][i][4 + e]) : 1.0f));
            }
            if (row < p.n) *reinterpret_cast<bf16x8_t *>(out + (4 * dt + 2 * i + hf) * 8) = r;
        }
}

// One wavefront per (row, head): 64 keys at a time, one per lane for the scores, one element per lane for the values.
constexpr int ROW_MAX_D = 1024; // elements of a head the values' accumulators cover
template <class T>
__global__ __launch_bounds__(256) void window_attn_rows_kernel(WindowAttn p) {
    __shared__ float s_q[4][ROW_MAX_D], s_w[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, task = blockIdx.x * 4 + wave;
    if (task >= p.n * p.H) return; // (wavefronts share nothing)
    const int row = task / p.H, h = task % p.H, g = h / (p.H / p.G), pos = p.pos0 + row, lo = p.window ? max(0, pos - p.window + 1) : 0;
    const T *q = reinterpret_cast<const T *>(p.q) + size_t(row) * p.ldq + h * p.dimp;
    const T *ck = reinterpret_cast<const T *>(p.ck) + size_t(g) * p.cap * p.dimp, *cv = reinterpret_cast<const T *>(p.cv) + size_t(g) * p.cap * p.vdimp;
    for (int d = lane; d < p.dimp; d += 64) s_q[wave][d] = (float)q[d];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const float scale = p.temp ? p.scale * p.temp[h] : p.scale;
    const int seen = p.pool ? blocks_seen(pos, p.window, p.pool) : 0; // the blocks come first, then the tokens from lo on
    const T *pk = reinterpret_cast<const T *>(p.pk) + size_t(g) * p.blocks * p.dimp, *pv = reinterpret_cast<const T *>(p.pv) + size_t(g) * p.blocks * p.vdimp;
    float m = p.sink ? p.sink[h] : -INFINITY, l = p.sink ? 1.0f : 0.0f;
    float o[ROW_MAX_D / 64];
#pragma unroll
    for (int i = 0; i < ROW_MAX_D / 64; i++) o[i] = 0.0f;
    const int total = seen + pos - lo + 1;
    for (int k0 = 0; k0 < total; k0 += 64) {
        const int key = k0 + lane, n_keys = min(64, total - k0);
        float s = -INFINITY;
        if (key < total) {
            const T *kr = key < seen ? pk + size_t(key) * p.dimp : ck + size_t((key - seen + lo) % p.cap) * p.dimp;
            s = 0.0f;
            for (int d = 0; d < p.dimp; d++) s = fmaf(s_q[wave][d], (float)kr[d], s);
            s *= scale;
        }
        const float m_new = fmaxf(m, wave_max(s)), alpha = expf(m - m_new), w = key < total ? expf(s - m_new) : 0.0f;
        l = l * alpha + wave_sum(w);
        m = m_new;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        s_w[wave][lane] = w;
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < ROW_MAX_D / 64; i++) {
            const int d = 64 * i + lane;
            if (64 * i >= p.vdimp) continue;
            float acc = o[i] * alpha;
            if (d < p.vdimp)
                for (int j = 0; j < n_keys; j++) {
                    const int at = k0 + j;
                    acc = fmaf(s_w[wave][j], (float)(at < seen ? pv + size_t(at) * p.vdimp : cv + size_t((at - seen + lo) % p.cap) * p.vdimp)[d], acc);
                }
            o[i] = acc;
        }
    }
#pragma unroll
    for (int i = 0; i < ROW_MAX_D / 64; i++)
        if (64 * i + lane < p.vdimp) s_q[wave][64 * i + lane] = o[i] / l; // (the query is not needed any more)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int half = p.rotv ? p.vdim / 2 : 0;
    for (int d = lane; d < p.vdimp; d += 64) {
        float r = s_q[wave][d];
        if (d < 2 * half) {
            const int m = d < half ? d : d - half;
            const float2 cs = p.rotv[size_t(pos) * half + m];
            r = d < half ? r * cs.x + s_q[wave][d + half] * cs.y : r * cs.x - s_q[wave][m] * cs.y;
        }
        if (p.gate) r *= lm_sigmoid((float)reinterpret_cast<const T *>(p.gate)[size_t(row) * p.ldq + h * p.vdimp + d]);
        reinterpret_cast<T *>(p.out)[size_t(row) * p.ldo + h * p.vdimp + d] = (T)r;
    }
}

// Where the shared tiles pay.  The kernel with merged wavefronts spreads any call over the device: its time goes with the tiles that all rows walk
// (x: rows times tiles, per unit) and with the rounds of 64 rows per unit.  The other's goes with the longest walk, T tiles of about 1 us, behind a start
// and an end of 6 us, 9 with a gate.  On 256 units, merged -> shared (us), r rows per unit:
//   gate, 32 heads     window 1024  600 rows (r 75, T 10, x 390) 17.9 -> 18.4, 768 (96, 12, 624) 20.6 -> 21.2, 960 (120, 15, 960) 23.8 -> 24.4, 1024 (128, 16, 1088) 24.1 -> 24.6,
//                      1100 (138, 18, 1250) 28.9 -> 26.7, 1920 52.2 -> 38.2; window 512  600 (75, 10, 387) 18.0 -> 18.6, 768 (96, 9, 576) 21.0 -> 19.2; window 256  600 (75, 6, 295) 16.5 -> 15.1
//   gate, other heads  16, window 256  900 (56, 6, 241) 13.2 -> 14.2; 16, window 512  1100 (69, 10, 475) 17.8 -> 18.5, 1300 (81, 10, 587) 20.7 -> 18.8; 16, window 1024  1400 (88, 17, 944)
//                      24.6 -> 26.0, 1700 (106, 17, 1262) 26.7 -> 26.8; 64, 256 rows (64, 4, 160) 9.3 -> 12.7, 300 (75, 5, 215) 15.1 -> 14.3
//   none, rotated      64, 256 rows (64, 4, 160) 8.6 -> 9.8; 16, window 256  900 (56, 6, 241) 12.9 -> 11.8; 32, window 1024  768 (96, 12, 624) 18.8 -> 17.5, 960 22.7 -> 21.5, 1920 51 -> 36
bool shares_tiles(moon_ctx *ctx, const WindowAttn &p) {
    if (p.dimp != WsCfg::D || p.vdimp != WsCfg::D || (p.rotv && p.vdim != WsCfg::D)) return false;
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    auto walk = [&](int first, int last) { // tiles of the block of rows that has these positions
        const int lo = p.window ? std::max(0, first - p.window + 1) : 0, seen = p.pool ? std::max(0, last - p.window + 1) / p.pool : 0;
        return last / WA_KT - lo / WA_KT + 1 + (seen + WA_KT - 1) / WA_KT;
    };
    const int end = p.pos0 + p.n, longest = walk(std::max(0, end - WA_Q), end - 1);
    if ((long long)p.n * p.H < (7 * longest + 10) * (long long)cus) return false;
    const long long rows = (long long)p.n * p.H;
    if (p.gate && (rows <= 64LL * cus || rows > 128LL * cus)) return rows > 64LL * cus;
    long long walked = 0;
    for (int first = p.pos0; first < end; first += WA_Q) walked += std::min(WA_Q, end - first) * walk(first, std::min(first + WA_Q, end) - 1);
    return walked * p.H >= (p.gate ? 93 * longest - 381 : 30 * longest + 50) * (long long)cus;
}

template <class Kernel> int launch_as(moon_ctx *ctx, const WindowAttn &p, Kernel kernel, std::atomic<bool> (&attr_set)[64], size_t lds, int workgroups, int threads) {
    const int dev = ctx->device >= 0 && ctx->device < 64 ? ctx->device : -1; // the opt-in to this much dynamic LDS is per device (and per kernel)
    if (dev < 0 || !attr_set[dev].load()) {
        MOON_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        if (dev >= 0) attr_set[dev].store(true);
    }
    hipLaunchKernelGGL(kernel, dim3((unsigned)workgroups), dim3(threads), lds, ctx->stream, p);
    MOON_HIP(ctx, hipGetLastError());
    return MOON_OK;
}
template <int P, bool POOL> int launch_mfma_as(moon_ctx *ctx, const WindowAttn &p) {
    if constexpr (P == 64)
        if (shares_tiles(ctx, p)) {
            static std::atomic<bool> attr_set[64], attr_apart[64];
            const int per = p.H / p.G, rows = ws_rows(per);
            const int workgroups = (p.n + rows - 1) / rows * (p.H / ws_heads(per));
            if (rows > WA_Q) MOON_TRY(launch_as(ctx, p, window_attn_shared_kernel<POOL, true>, attr_apart, WsCfg::LDS_BYTES, workgroups, 512));
            else MOON_TRY(launch_as(ctx, p, window_attn_shared_kernel<POOL, false>, attr_set, WsCfg::LDS_BYTES, workgroups, 512));
            MOON_NOTE_ATTENTION(ctx, "window_attn_shared_kernel %d rows of %d heads%s", rows, ws_heads(per), POOL ? ", blocks" : "");
            return MOON_OK;
        }
    static std::atomic<bool> attr_set[64];
    MOON_TRY(launch_as(ctx, p, window_attn_kernel<P, POOL>, attr_set, WaCfg<P>::LDS_BYTES, (p.n + WA_Q - 1) / WA_Q * p.H, 256));
    MOON_NOTE_ATTENTION(ctx, "window_attn_kernel<%d>", P);
    return MOON_OK;
}
// (a call before whose window no block lies yet takes the kernel without them)
template <int P> int launch_mfma(moon_ctx *ctx, const WindowAttn &p) { return p.pool && p.pos0 + p.n - p.window >= p.pool ? launch_mfma_as<P, true>(ctx, p) : launch_mfma_as<P, false>(ctx, p); }

} // namespace

int launch_window_attention(moon_ctx *ctx, int dtype, const WindowAttn &p) {
    if (p.n <= 0) return MOON_OK;
    if (p.H % p.G || p.dimp % 8 || p.vdimp % 8 || p.dimp > ROW_MAX_D || p.vdimp > ROW_MAX_D)
        return moon_fail(ctx, MOON_EINVAL_DIM, "window attention: %d heads over %d, head sizes %d and %d", p.H, p.G, p.dimp, p.vdimp);
    if ((p.window ? p.window - 1 + p.n : p.pos0 + p.n) > p.cap && p.pos0 + p.n > p.cap)
        return moon_fail(ctx, MOON_EINVAL_DIM, "window attention: %d rows behind a window of %d do not fit %d cache rows", p.n, p.window, p.cap);
    if (p.pool && (!p.window || (p.pos0 + p.n - p.window) / p.pool > p.blocks)) // (no block is seen before it is whole)
        return moon_fail(ctx, MOON_EINVAL_DIM, "window attention: blocks of %d before a window of %d, %d of them kept", p.pool, p.window, p.blocks);
    const int big = std::max(p.dimp, p.vdimp);
    if (dtype == MOON_DTYPE_BF16 && big <= 256 && size_t(std::max(p.cap, p.blocks)) * big * 2 < (size_t(1) << 30)) { // (32-bit offsets within a head's rows)
        if (big <= 32) return launch_mfma<32>(ctx, p);
        if (big <= 64) return launch_mfma<64>(ctx, p);
        if (big <= 96) return launch_mfma<96>(ctx, p);
        if (big <= 128) return launch_mfma<128>(ctx, p);
        return launch_mfma<256>(ctx, p);
    }
    const dim3 grid((unsigned)((size_t(p.n) * p.H + 3) / 4));
    if (dtype == MOON_DTYPE_BF16) hipLaunchKernelGGL(window_attn_rows_kernel<bf16_t>, grid, dim3(256), 0, ctx->stream, p);
    else hipLaunchKernelGGL(window_attn_rows_kernel<float>, grid, dim3(256), 0, ctx->stream, p);
    MOON_HIP(ctx, hipGetLastError());
    MOON_NOTE_ATTENTION(ctx, "window_attn_rows_kernel");
    return MOON_OK;
}
