// Matrix-core attention for multi-token queries: the causal prefill of the text decoder (32 heads x 64,
// attention.multiMaskedSDPA with the mask of createAttentionMask, attention.zig:256-281, 416-541) and the
// non-causal 729-token vision attention (16 heads x 72, attention.multiMasklessSDPA, attention.zig:125-234).
//
// One 256-thread workgroup owns 32 query rows of one head (64 in flash_attn64_kernel and 96 in flash_attn96_kernel, for large calls).  Its four wavefronts split the key range in tiles
// of 64 keys (wave w takes tiles w, w+4, ...), each running an online-softmax pass of its own over private LDS
// staging, so the main loop has no workgroup barrier; the four partial results (m, l, O) are merged through
// LDS at the end.  Per tile a wave computes, with v_mfma_f32_32x32x16_f16 and f32 accumulation,
//     S^T[key][q] = K . Q^T          (keys are the MFMA rows, so a lane holds 32 scores of ONE query and the
//                                      row maximum / sum are in-register reductions plus one cross-half exchange)
//     O^T[d][q]  += V^T . P^T        (P rounded to f16 for the matrix core; V is staged row-major and transposed by
//                                      the LDS load that feeds the matrix core)
// The scale 1/sqrt(D) multiplies the f32 product (attention.zig:192-194, 487-489), masked scores are -inf, the
// result is divided by the f32 row sum and rounded once to f16.
#include "epilogue.hpp"
#include "lane_fold.hpp"
#include "tile_copy.hpp"

#include <atomic>

namespace {

typedef tile_u32x4 u32x4;
typedef _Float16 half4_t __attribute__((ext_vector_type(4)));

constexpr int FA_Q = 32;     // query rows per workgroup
constexpr int FA_KT = 64;    // keys per tile
constexpr int FA_WAVES = 4;

template <int D>
struct FaCfg {
    static constexpr int DK = (D + 15) / 16 * 16; // contraction length of K.Q^T, zero padded
    static constexpr int KSTEPS = DK / 16;
    static constexpr int DT = (D + 31) / 32;      // 32-row tiles of O^T, rows >= D are zero
    static constexpr int G = D / 8;               // 16-byte granules per row
    static constexpr int KS = DK + 8;             // K tile row stride in halfs: 36 or 44 dwords, conflict-free b128 reads
    // The V tile stays row-major, [key][d], and is read with the transposing LDS load (ds_read_tr16_b64).  Per half-wavefront
    // such a load touches 4 consecutive keys x 32 consecutive d: with D = 64 the rows are unpadded (32 dwords) and the 16-byte
    // granule c of key row r sits at granule c ^ 2*(r & 3), so those 4 x 4 granules fall on distinct banks and the b128
    // stores of two consecutive rows do too; otherwise the row stride is 48 dwords (rows 0..3 start at banks 0, 48, 32, 16).
    static constexpr bool V_SWIZZLE = (D == 64);
    static constexpr int VS = V_SWIZZLE ? D : 96; // V tile row stride in halfs
    static constexpr int K_HALFS = FA_KT * KS;
    static constexpr int V_HALFS = FA_KT * VS;
    // the K tile and the V tile of a wavefront share their LDS: K is only read before the scores, V only after
    static constexpr int WAVE_HALFS = K_HALFS > V_HALFS ? K_HALFS : V_HALFS;
    static constexpr int K_LOADS = (FA_KT * G + 63) / 64;       // 16-byte loads per lane for a K tile
    static constexpr bool FA_FULL_K = (FA_KT * G) % 64 == 0;    // every lane takes part in every K load
    // merge of the four wavefronts: O as [wave][q][SD] floats over the tiles (row stride D + 4: the 16-byte accesses of 16
    // consecutive q fall on distinct banks), the maxima and sums [wave][q] behind them in an area of their own
    static constexpr int SD = D + 4;
    static constexpr size_t MERGE_BYTES = size_t(FA_WAVES) * FA_Q * SD * sizeof(float);
    static constexpr size_t TILE_BYTES = size_t(FA_WAVES) * WAVE_HALFS * sizeof(half_t);
    static constexpr size_t ML_OFFSET = TILE_BYTES > MERGE_BYTES ? TILE_BYTES : MERGE_BYTES;
    static constexpr size_t LDS_BYTES = ML_OFFSET + 2 * FA_WAVES * FA_Q * sizeof(float);
};

struct FaArgs {
    const half_t *q, *k, *v;
    half_t *out;
    int H, Lq, Lkv;
    size_t q_head_stride, q_row_stride;   // element (h, r, d) of q sits at q[h * q_head_stride + r * q_row_stride + d]
    size_t kv_head_stride, kv_row_stride; // same for k and v
    long causal_pos; // key j is visible to query row r when causal_pos < 0 or j <= causal_pos + r
    int out_merged;  // 0: out[h][r][d], 1: out[r][h][d]
    float scale;
};

template <int D>
struct FaTileRegs {
    u32x4 k[FaCfg<D>::K_LOADS];
    u32x4 v[FaCfg<D>::K_LOADS];
};

// The K / V rows of a head are addressed as a buffer: a scalar descriptor of the head's rows, one 32-bit byte offset per
// lane that does not change from tile to tile, and the tile's first row as the scalar offset (fewer address registers
// and instructions than a 64-bit pointer per load, and the loads of a wavefront whose SIMD feeds the matrix core issue
// faster in this form).  Rows past the head's last read as zero (the descriptor ends there); their scores are masked.
typedef unsigned int fa_u32x4 __attribute__((ext_vector_type(4)));
template <int D>
__device__ __forceinline__ void fa_load_k(FaTileRegs<D> &r, __amdgpu_buffer_rsrc_t rs, int row_bytes, int key0, int lane) {
    using C = FaCfg<D>;
    const int tile_off = __builtin_amdgcn_readfirstlane(key0 * row_bytes); // (the same in every lane: a scalar operand)
#pragma unroll
    for (int i = 0; i < C::K_LOADS; i++) {
        const int g = i * 64 + lane;
        if (C::FA_FULL_K || g < FA_KT * C::G) {
            const int row = g / C::G, c = g % C::G;
            r.k[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, row * row_bytes + c * 16, tile_off, 0));
        }
    }
}
template <int D>
__device__ __forceinline__ void fa_load_v(FaTileRegs<D> &r, __amdgpu_buffer_rsrc_t rs, int row_bytes, int key0, int lane) {
    using C = FaCfg<D>;
    const int tile_off = __builtin_amdgcn_readfirstlane(key0 * row_bytes);
#pragma unroll
    for (int i = 0; i < C::K_LOADS; i++) {
        const int g = i * 64 + lane;
        if (C::FA_FULL_K || g < FA_KT * C::G) {
            const int row = g / C::G, c = g % C::G;
            r.v[i] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, row * row_bytes + c * 16, tile_off, 0));
        }
    }
}

template <int D>
__device__ __forceinline__ void fa_store_k(const FaTileRegs<D> &r, half_t *Ks, int lane) {
    using C = FaCfg<D>;
#pragma unroll
    for (int i = 0; i < C::K_LOADS; i++) {
        const int g = i * 64 + lane;
        if (C::FA_FULL_K || g < FA_KT * C::G) {
            const int row = g / C::G, c = g % C::G;
            *reinterpret_cast<u32x4 *>(Ks + row * C::KS + c * 8) = r.k[i];
        }
    }
    if (C::DK > D) { // zero padding of the contraction, columns [D, DK): one row per lane (the V tile overwrote it)
        static_assert(C::DK - D == 8 || C::DK == D, "one 16-byte granule of padding");
        *reinterpret_cast<u32x4 *>(Ks + lane * C::KS + D) = u32x4{0, 0, 0, 0};
    }
}
template <int D>
__device__ __forceinline__ void fa_store_v(const FaTileRegs<D> &r, half_t *Vs, int lane) {
    using C = FaCfg<D>;
#pragma unroll
    for (int i = 0; i < C::K_LOADS; i++) {
        const int g = i * 64 + lane;
        if (C::FA_FULL_K || g < FA_KT * C::G) {
            const int row = g / C::G, c = g % C::G;
            const int cs = C::V_SWIZZLE ? (c ^ (2 * (row & 3))) : c;
            *reinterpret_cast<u32x4 *>(Vs + row * C::VS + cs * 8) = r.v[i];
        }
    }
}
// Transposing LDS load: the 16 lanes of a quarter-wavefront each name 4 consecutive halfs; lane i of the quarter receives
// element i % 4 of the halfs named by lanes i / 4, i / 4 + 4, i / 4 + 8, i / 4 + 12.  When lane n names key n / 4, d-columns
// 4 * (n % 4) .. + 3 of a 4 x 16 block of row-major V, lane i ends up with column i of keys 0..3: V^T as the matrix core reads it.
__device__ __forceinline__ half4_t fa_read_tr(const half_t *p) {
    typedef short short4_t __attribute__((ext_vector_type(4)));
    return __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) short4_t *)(p)));
}

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void flash_attn_kernel(FaArgs p) {
    using C = FaCfg<D>;
    extern __shared__ __attribute__((aligned(16))) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6); // (wave: a scalar)
    const int col = lane & 31, hf = lane >> 5;
    const bool causal = p.causal_pos >= 0;
    // Workgroups are dealt to the eight accelerator dies round robin, and each die has an L2 of its own: when the count
    // divides, die x takes the x-th eighth of the (head, query block) list, so a head's K and V are fetched into one or two
    // L2s instead of all eight.
    int item = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int n_items = (int)(gridDim.x * gridDim.y);
    if (n_items % 8 == 0) item = (item % 8) * (n_items / 8) + item / 8;
    int h = item / (int)gridDim.x, bx = item % (int)gridDim.x;
    // Late query blocks see the most keys: start them first.  Where a die's share is whole heads, its workgroups walk the
    // query blocks of all its heads together (block 23 of heads 0-3, block 22 of heads 0-3, ...): what is still to start when
    // the first workgroups leave is then the lightest blocks of every head, not all of the last head's.
    if (causal && n_items % 8 == 0 && (n_items / 8) % (int)gridDim.x == 0) {
        const int per_die = n_items / 8, heads_per_die = per_die / (int)gridDim.x, j = item % per_die;
        h = (item / per_die) * heads_per_die + j % heads_per_die;
        bx = j / heads_per_die;
    }
    const int qb = causal ? (int)gridDim.x - 1 - bx : bx;
    const int q0 = qb * FA_Q;
    half_t *Ks = smem + wave * C::WAVE_HALFS;
    half_t *Vs = Ks; // (shared with the K tile)
    // where this lane points the transposing loads of O^T row tile dt (see fa_read_tr): key 4*hf + (lane % 16) / 4 of the 8 keys
    // of a contraction half-step, d-columns 32*dt + 16*((lane / 16) % 2) + 4*(lane % 4) .. + 3.  Rows of O^T at or past D are
    // dropped, so the lanes that would name columns past the row name its last four instead.
    int voff[C::DT];
    {
        const int rq = (lane & 15) >> 2;
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++) {
            int colh = 32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
            if (C::V_SWIZZLE) colh = (((colh >> 3) ^ (2 * rq)) << 3) | (colh & 7);
            else colh = min(colh, D - 4);
            voff[dt] = (4 * hf + rq) * C::VS + colh;
        }
    }
    // this head's rows: (Lkv - 1) row strides and one row of D halfs
    const int row_bytes = (int)p.kv_row_stride * 2, head_bytes = (p.Lkv - 1) * row_bytes + D * 2;
    const __amdgpu_buffer_rsrc_t kh = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(p.k + size_t(h) * p.kv_head_stride), 0, head_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t vh = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(p.v + size_t(h) * p.kv_head_stride), 0, head_bytes, 0x00020000);

    // keys any row of this block can see
    long kv_end = p.Lkv;
    if (causal && p.causal_pos + q0 + FA_Q < kv_end) kv_end = p.causal_pos + q0 + FA_Q;
    const int n_tiles = (int)((kv_end + FA_KT - 1) / FA_KT);

    // The first K tile is requested before the query rows and the first V tile after them: the scores wait for K and Q only,
    // and the one round trip to memory that this wavefront cannot hide covers all three.
    FaTileRegs<D> regs;
    if (wave < n_tiles) fa_load_k<D>(regs, kh, row_bytes, wave * FA_KT, lane);

    // this lane's query row as the MFMA "B" operand: Q[q0 + col][16*s + 8*hf .. +7]
    half8_t qf[C::KSTEPS];
    {
        const int qrow = min(q0 + col, p.Lq - 1);
        const half_t *qp = p.q + size_t(h) * p.q_head_stride + size_t(qrow) * p.q_row_stride;
#pragma unroll
        for (int s = 0; s < C::KSTEPS; s++) {
            const int d = 16 * s + 8 * hf;
#pragma unroll
            for (int e = 0; e < 8; e++) qf[s][e] = (half_t)0.0f;
            if (d < D) qf[s] = *reinterpret_cast<const half8_t *>(qp + d);
        }
    }
    if (wave < n_tiles) fa_load_v<D>(regs, vh, row_bytes, wave * FA_KT, lane);

    float16_t o[C::DT];
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[dt][v] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f; // l_run: this lane's half of the row sum

    for (int t = wave; t < n_tiles; t += FA_WAVES) {
        asm volatile("" ::: "memory"); // the V tile of the previous iteration has been read: the K tile takes its place
        fa_store_k<D>(regs, Ks, lane);
        if (t + FA_WAVES < n_tiles) fa_load_k<D>(regs, kh, row_bytes, (t + FA_WAVES) * FA_KT, lane);
        const int key0 = t * FA_KT;

        float16_t s[2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
#pragma unroll
            for (int v = 0; v < 16; v++) s[kt][v] = 0.0f;
#pragma unroll
            for (int st = 0; st < C::KSTEPS; st++) {
                const half8_t a = *reinterpret_cast<const half8_t *>(Ks + (32 * kt + col) * C::KS + 16 * st + 8 * hf);
                s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[st], s[kt], 0, 0, 0);
            }
        }
        // s[kt][v] = score of key key0 + 32*kt + 8*(v/4) + 4*hf + v%4 against query q0 + col
        const bool edge = (key0 + FA_KT > p.Lkv) || (causal && (long)(key0 + FA_KT - 1) > p.causal_pos + q0);
        float mx = -INFINITY;
        // Scores stay unscaled in s; the scale (times log2 e) enters in the one fma that feeds exp2.  The running maximum
        // m_run is kept in those units (scaled, base 2).
        if (edge) { // (a tile that needs no masking takes the other path: no compare, no branch per score)
            const long last_visible = causal ? min((long)p.Lkv - 1, p.causal_pos + q0 + col) : (long)p.Lkv - 1;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const int key = key0 + 32 * kt + 8 * (v >> 2) + 4 * hf + (v & 3);
                    const float x = (long)key > last_visible ? -INFINITY : s[kt][v];
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
        const float c2 = p.scale * 1.4426950408889634f; // > 0: the maximum of the scaled scores is the scaled maximum
        const float m_new = fmaxf(m_run, mx * c2);
        const float m_use = (m_new == -INFINITY) ? 0.0f : m_new; // a row that has seen no key yet
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_use);
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
        // (rows of O^T at or past D are never read: in the last row tile only the registers of rows below D are rescaled;
        // the others hold whatever accumulates, each on its own)
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++)
                if (32 * dt + 8 * (v >> 2) < D) o[dt][v] *= alpha;

        asm volatile("" ::: "memory"); // the K tile has been read (LDS serves a wavefront in order): V takes its place
        fa_store_v<D>(regs, Vs, lane);
        if (t + FA_WAVES < n_tiles) fa_load_v<D>(regs, vh, row_bytes, (t + FA_WAVES) * FA_KT, lane);
        // O^T += V^T . P^T : contraction step (kt, sp) uses the keys a lane already holds in s[kt][8*sp .. 8*sp+7],
        // i.e. key0 + 32*kt + 16*sp + {4*hf + 0..3, 8 + 4*hf + 0..3}
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int sp = 0; sp < 2; sp++) {
                half8_t pb;
#pragma unroll
                for (int e = 0; e < 8; e++) pb[e] = (half_t)s[kt][8 * sp + e];
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++) {
                    const half_t *vp = Vs + voff[dt] + (32 * kt + 16 * sp) * C::VS;
                    const half4_t lo = fa_read_tr(vp);
                    const half4_t hi = fa_read_tr(vp + 8 * C::VS);
                    half8_t a;
                    a[0] = lo[0]; a[1] = lo[1]; a[2] = lo[2]; a[3] = lo[3];
                    a[4] = hi[0]; a[5] = hi[1]; a[6] = hi[2]; a[7] = hi[3];
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb, o[dt], 0, 0, 0);
                }
            }
    }

    // merge the four waves' partial results
    const float l_wave = l_run + __shfl_xor(l_run, 32);
    float *so = reinterpret_cast<float *>(smem);                                                        // [wave][q][SD]
    float *sm = reinterpret_cast<float *>(reinterpret_cast<char *>(smem) + C::ML_OFFSET);               // [wave][q]
    float *sl = sm + FA_WAVES * FA_Q;                                                                   // [wave][q]
    if (hf == 0) {
        sm[wave * FA_Q + col] = m_run;
        sl[wave * FA_Q + col] = l_wave;
    }
    __syncthreads(); // every wave is done with its staging area, which O takes over, and has published its maximum
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < FA_WAVES; w++) m_all = fmaxf(m_all, sm[w * FA_Q + col]);
    const float f = (m_run == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_all); // (maxima are in base-2 units)
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int d = 32 * dt + 8 * j + 4 * hf; // o[dt][4*j .. 4*j+3] are rows d .. d+3 of O^T
            if (32 * dt + 8 * j < D) {
                float4 r;
                r.x = o[dt][4 * j] * f;
                r.y = o[dt][4 * j + 1] * f;
                r.z = o[dt][4 * j + 2] * f;
                r.w = o[dt][4 * j + 3] * f;
                *reinterpret_cast<float4 *>(so + (wave * FA_Q + col) * C::SD + d) = r;
            }
        }
    __syncthreads();
    {
        const int q = tid & 31;
        float l_all = 0.0f;
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) {
            const float mw = sm[w * FA_Q + q];
            if (mw != -INFINITY) l_all += __builtin_amdgcn_exp2f(mw - m_all) * sl[w * FA_Q + q];
        }
        const float inv = 1.0f / l_all;
        const int row = q0 + q;
        if (row < p.Lq) {
            for (int dg = tid >> 5; dg < C::G; dg += 8) {
                float acc[8];
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] = 0.0f;
#pragma unroll
                for (int w = 0; w < FA_WAVES; w++) {
                    const float4 a = *reinterpret_cast<const float4 *>(so + (w * FA_Q + q) * C::SD + dg * 8);
                    const float4 b = *reinterpret_cast<const float4 *>(so + (w * FA_Q + q) * C::SD + dg * 8 + 4);
                    acc[0] += a.x; acc[1] += a.y; acc[2] += a.z; acc[3] += a.w;
                    acc[4] += b.x; acc[5] += b.y; acc[6] += b.z; acc[7] += b.w;
                }
                half8_t r;
#pragma unroll
                for (int e = 0; e < 8; e++) r[e] = (half_t)(acc[e] * inv);
                const size_t oi = p.out_merged ? (size_t(row) * p.H + h) * D + dg * 8 : (size_t(h) * p.Lq + row) * D + dg * 8;
                *reinterpret_cast<half8_t *>(p.out + oi) = r;
            }
        }
    }
}

// Sixty-four query rows per workgroup, for calls with enough of them.  The kernel above spends as long on bringing a tile from the L2
// into LDS and out of it as on the matrix instructions; here a fragment of K or V read from LDS serves both blocks of 32 rows,
// which halves that, and the copies go to LDS directly, whose rows need no padding (no staging registers, for which 64 rows have
// no room).  What bounds it now: the exponentials and what goes with them, whose time in the vector unit two wavefronts per SIMD
// hardly overlap with the matrix core's (32 heads x 4096 x 4096 of 72, counted: vector instructions issued in 63 % of the cycles,
// matrix core busy in 42 %, no bank conflicts; of 64: 68 and 35 %).  Calls back to back, 32 rows -> 64: 16 heads of 72, 1458 rows
// 25.6 -> 23.8 us; 32 heads of 64, 1024 causal rows 15.2 -> 13.9, 2000 rows 38.9 -> 33.8.  Tried and slower: the exponentials of one
// block between the matrix instructions of the other, in program order (5 to 8 %).  The denominator is summed in f32, as above: taken
// from the matrix core it is a sum of rounded probabilities, 5 % faster for heads of 72, and loses the faint keys of a long call.
// Each row goes through the same operations in the same order as above: the same bits (tested).
template <int D>
struct FbCfg {
    static constexpr int QS = 2;                  // blocks of 32 query rows per workgroup
    static constexpr int Q = 32 * QS;             // query rows per workgroup
    static constexpr int DK = (D + 15) / 16 * 16; // contraction length of K.Q^T, zero padded
    static constexpr int KSTEPS = DK / 16;
    static constexpr int DT = (D + 31) / 32;      // 32-row tiles of O^T, rows >= D are zero
    static constexpr int G = D / 8;               // 16-byte granules per row
    static constexpr int TILE = FA_KT * D;        // halfs of a K or V tile
    static constexpr int COPIES = FA_KT * G / 64; // copies of 64 granules that bring a tile
    static_assert((FA_KT * G) % 64 == 0 && (D == 64 || D == 72), "whole copies, and a bank layout of its own for each row length");
    // merge of the four wavefronts: O as [wave][q][SD] floats over the tiles (row stride D + 4: the 16-byte accesses of 16
    // consecutive q fall on distinct banks), the maxima and sums [wave][q] behind them in an area of their own
    static constexpr int SD = D + 4;
    static constexpr size_t MERGE_BYTES = size_t(FA_WAVES) * Q * SD * sizeof(float);
    static constexpr size_t TILE_BYTES = size_t(FA_WAVES) * 2 * TILE * sizeof(half_t);
    static constexpr size_t ML_OFFSET = TILE_BYTES > MERGE_BYTES ? TILE_BYTES : MERGE_BYTES;
    static constexpr size_t LDS_BYTES = ML_OFFSET + 2 * FA_WAVES * Q * sizeof(float);
    static_assert(2 * LDS_BYTES <= 160 * 1024, "two workgroups per compute unit");
};

// Where a tile's granules lie in LDS.  The copies fill it in order, 64 granules of 16 bytes at a time, so rows are unpadded and
// the choice is which key a slot holds (D = 72) or which granule of its row (D = 64).  A K read takes one granule of each of
// 16 consecutive keys, a transposing V read 4 granules of each of 4 consecutive keys; 16 granules are all 64 banks.
//   D = 72: slot s starts at granule 9 s.  Slots 4 apart start 4 granules apart mod 16, so keys 4 a + b of a group of 16 sit in slot
//           4 b + a (its own inverse): four consecutive keys fill the banks, and so do 16 with one granule each.
//   D = 64: slot s is key s and starts at granule 8 s.  Granule c sits at c ^ row64_swizzle(s).
template <int D> __device__ __forceinline__ int fb_slot(int key) { return D == 72 ? (key & ~15) | (key & 3) << 2 | (key >> 2 & 3) : key; }
template <int D> __device__ __forceinline__ int fb_swizzle(int key) { return D == 72 ? 0 : row64_swizzle(key); }

template <int D>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void flash_attn64_kernel(FaArgs p) {
    using C = FbCfg<D>;
    constexpr int QS = C::QS;
    extern __shared__ __attribute__((aligned(16))) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6); // (wave: a scalar)
    const int col = lane & 31, hf = lane >> 5;
    const bool causal = p.causal_pos >= 0;
    // which head and rows: as in flash_attn_kernel
    int item = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int n_items = (int)(gridDim.x * gridDim.y);
    if (n_items % 8 == 0) item = (item % 8) * (n_items / 8) + item / 8;
    int h = item / (int)gridDim.x, bx = item % (int)gridDim.x;
    if (causal && n_items % 8 == 0 && (n_items / 8) % (int)gridDim.x == 0) {
        const int per_die = n_items / 8, heads_per_die = per_die / (int)gridDim.x, j = item % per_die;
        h = (item / per_die) * heads_per_die + j % heads_per_die;
        bx = j / heads_per_die;
    }
    const int qb = causal ? (int)gridDim.x - 1 - bx : bx;
    const int q0 = qb * C::Q;
    const half_t *Ks = smem + wave * 2 * C::TILE, *Vs = Ks + C::TILE;
    const unsigned k_lds = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<unsigned long>((__attribute__((address_space(3))) const half_t *)Ks));
    const unsigned v_lds = k_lds + C::TILE * sizeof(half_t);
    // where this lane points the transposing loads of O^T row tile dt (see fa_read_tr): keys 4 hf + (lane % 16) / 4 of the 8 keys
    // of a contraction half-step (and, second, 8 keys on), d-columns 32 dt + 16 ((lane / 16) % 2) + 4 (lane % 4) .. + 3.  Rows of
    // O^T at or past D take no V, so the lanes that would name columns past the row name its last four instead.
    int voff[2][C::DT];
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++) {
            const int key = (D == 72 ? 0 : 8 * j) + 4 * hf + ((lane & 15) >> 2), c = min(32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3), D - 4);
            voff[j][dt] = fb_slot<D>(key) * D + ((c >> 3 ^ fb_swizzle<D>(key)) << 3 | (c & 7)) + (D == 72 ? j * fb_slot<D>(8) * D : 0);
        }
    // this head's rows: (Lkv - 1) row strides and one row of D halfs
    const int row_bytes = (int)p.kv_row_stride * 2, head_bytes = (p.Lkv - 1) * row_bytes + D * 2;
    const half_t *kh = p.k + size_t(h) * p.kv_head_stride, *vh = p.v + size_t(h) * p.kv_head_stride;
    int off[C::COPIES]; // this lane's granules of a tile, from its first row (K and V lie alike)
#pragma unroll
    for (int i = 0; i < C::COPIES; i++) {
        const int x = i * 64 + lane, key = fb_slot<D>(x / C::G); // (the slot of a slot's number is its key)
        off[i] = key * row_bytes + (x % C::G ^ fb_swizzle<D>(key)) * 16;
        asm volatile("" : "+v"(off[i])); // (one register each: the compiler would keep the 64-bit products)
    }

    // keys any row of this block can see
    long kv_end = p.Lkv;
    if (causal && p.causal_pos + q0 + C::Q < kv_end) kv_end = p.causal_pos + q0 + C::Q;
    const int n_tiles = (int)((kv_end + FA_KT - 1) / FA_KT);
    const size_t tile_stride = size_t(FA_KT) * p.kv_row_stride;

    if (wave < n_tiles) {
        tile_copy(kh + wave * tile_stride, head_bytes - wave * FA_KT * row_bytes, k_lds, off);
        tile_copy(vh + wave * tile_stride, head_bytes - wave * FA_KT * row_bytes, v_lds, off);
    }
    // this lane's query rows as the MFMA "B" operand: Q[q0 + 32 u + col][16*s + 8*hf .. +7]
    half8_t qf[QS][C::KSTEPS];
#pragma unroll
    for (int u = 0; u < QS; u++) {
        const int qrow = min(q0 + 32 * u + col, p.Lq - 1);
        const half_t *qp = p.q + size_t(h) * p.q_head_stride + size_t(qrow) * p.q_row_stride;
#pragma unroll
        for (int s = 0; s < C::KSTEPS; s++) {
            const int d = 16 * s + 8 * hf;
#pragma unroll
            for (int e = 0; e < 8; e++) qf[u][s][e] = (half_t)0.0f;
            if (d < D) qf[u][s] = *reinterpret_cast<const half8_t *>(qp + d);
        }
    }
    // Tell the compiler that the query rows have arrived: it would wait for them at their first use, in every round of the loop,
    // by counting to zero, and with them for the tile that is on its way.  (One round trip brings all three.)
    __builtin_amdgcn_s_waitcnt(0xf70); // vmcnt(0), the other counters at their maxima

    float16_t o[QS][C::DT];
    float m_run[QS], l_run[QS]; // l_run: this lane's half of the row sum
#pragma unroll
    for (int u = 0; u < QS; u++) {
        m_run[u] = -INFINITY;
        l_run[u] = 0.0f;
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int v = 0; v < 16; v++) o[u][dt][v] = 0.0f;
    }
    const float c2 = p.scale * 1.4426950408889634f; // > 0: the maximum of the scaled scores is the scaled maximum

    for (int t = wave; t < n_tiles; t += FA_WAVES) {
        const int key0 = t * FA_KT;
        const bool more = t + FA_WAVES < n_tiles;
        const half_t *k_next = kh + (t + FA_WAVES) * tile_stride, *v_next = vh + (t + FA_WAVES) * tile_stride;
        const int left = head_bytes - (t + FA_WAVES) * FA_KT * row_bytes;
        tile_landed<C::COPIES>(); // the K tile (the V tile's copies are newer)

        float16_t s[QS][2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
#pragma unroll
            for (int u = 0; u < QS; u++)
#pragma unroll
                for (int v = 0; v < 16; v++) s[u][kt][v] = 0.0f;
            const half_t *row = Ks + fb_slot<D>(32 * kt + col) * D;
#pragma unroll
            for (int st = 0; st < C::KSTEPS; st++) {
                const bool past = 16 * st + 8 >= D; // the second half of the wavefront has no granule here: zeros
                const int g = past ? 2 * st : (2 * st + hf) ^ fb_swizzle<D>(col);
                u32x4 a = *reinterpret_cast<const u32x4 *>(row + g * 8);
                if (past && hf) a = u32x4{0, 0, 0, 0};
#pragma unroll
                for (int u = 0; u < QS; u++) s[u][kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), qf[u][st], s[u][kt], 0, 0, 0);
            }
        }
        if (more) tile_copy(k_next, left, k_lds, off);
#pragma unroll
        for (int u = 0; u < QS; u++) {
            // s[u][kt][v] = score of key key0 + 32*kt + 8*(v/4) + 4*hf + v%4 against query q0 + 32 u + col
            const bool edge = (key0 + FA_KT > p.Lkv) || (causal && (long)(key0 + FA_KT - 1) > p.causal_pos + q0 + 32 * u);
            float mx = -INFINITY;
            // Scores stay unscaled in s; the scale (times log2 e) enters in the one fma that feeds exp2.  m_run is kept in those
            // units (scaled, base 2).
            if (edge) { // (a tile that needs no masking takes the other path: no compare, no branch per score)
                const int first = causal ? (int)min((long)p.Lkv, p.causal_pos + q0 + 32 * u) : p.Lkv; // the last key that row 32 u sees
                const int seen = min(p.Lkv - 1, first + col) - key0 - 4 * hf;                         // keys past this one of the tile are masked
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) {
                        const float x = 32 * kt + 8 * (v >> 2) + (v & 3) > seen ? -INFINITY : s[u][kt][v];
                        s[u][kt][v] = x;
                        mx = fmaxf(mx, x);
                    }
            } else {
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[u][kt][v]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            // (A reference that may lag behind the maximum, by less than f16 minds, would spare most of the rescaling, but the largest
            // probability would no longer be exactly 1: error against 64 bits 5 to 11 % larger at 729 and 1458 rows.)
            const float m_new = fmaxf(m_run[u], mx * c2);
            float alpha = 1.0f;
            if (__any(m_new != m_run[u])) {
                alpha = __builtin_amdgcn_exp2f(m_run[u] - (m_new == -INFINITY ? 0.0f : m_new));
                m_run[u] = m_new;
                // (in the last row tile only the registers of rows below D are rescaled)
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
                    for (int v = 0; v < 16; v++)
                        if (32 * dt + 8 * (v >> 2) < D) o[u][dt][v] *= alpha;
            }
            const float m_use = m_run[u] == -INFINITY ? 0.0f : m_run[u]; // a row that has seen no key yet
            // (the denominator is the sum of the probabilities before they are rounded for the matrix core)
            float psum = 0.0f;
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) {
                    const float e = __builtin_amdgcn_exp2f(__builtin_fmaf(s[u][kt][v], c2, -m_use));
                    s[u][kt][v] = e;
                    psum += e;
                }
            l_run[u] = l_run[u] * alpha + psum;
        }

        if (more) tile_landed<C::COPIES>(); // the V tile
        else tile_landed<0>();
        // O^T += V^T . P^T : contraction step (kt, sp) uses the keys a lane already holds in s[u][kt][8*sp .. 8*sp+7],
        // i.e. key0 + 32*kt + 16*sp + {4*hf + 0..3, 8 + 4*hf + 0..3}
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int sp = 0; sp < 2; sp++) {
                half8_t pb[QS];
#pragma unroll
                for (int u = 0; u < QS; u++)
#pragma unroll
                    for (int e = 0; e < 8; e++) pb[u][e] = (half_t)s[u][kt][8 * sp + e];
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++) {
                    const half4_t lo = fa_read_tr(Vs + voff[0][dt] + (32 * kt + 16 * sp) * D);
                    const half4_t hi = fa_read_tr(Vs + voff[1][dt] + (32 * kt + 16 * sp) * D);
                    const half8_t a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
                    for (int u = 0; u < QS; u++) o[u][dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[u], o[u][dt], 0, 0, 0);
                }
            }
        if (more) tile_copy(v_next, left, v_lds, off);
    }

    // merge the four waves' partial results
    float *so = reinterpret_cast<float *>(smem);                                                        // [wave][q][SD]
    float *sm = reinterpret_cast<float *>(reinterpret_cast<char *>(smem) + C::ML_OFFSET);               // [wave][q]
    float *sl = sm + FA_WAVES * C::Q;                                                                   // [wave][q]
#pragma unroll
    for (int u = 0; u < QS; u++) {
        const float l_wave = l_run[u] + __shfl_xor(l_run[u], 32);
        if (hf == 0) {
            sm[wave * C::Q + 32 * u + col] = m_run[u];
            sl[wave * C::Q + 32 * u + col] = l_wave;
        }
    }
    __syncthreads(); // every wave is done with its staging area, which O takes over, and has published its maximum
#pragma unroll
    for (int u = 0; u < QS; u++) {
        float m_all = -INFINITY;
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) m_all = fmaxf(m_all, sm[w * C::Q + 32 * u + col]);
        const float f = (m_run[u] == -INFINITY) ? 0.0f : __builtin_amdgcn_exp2f(m_run[u] - m_all); // (maxima are in base-2 units)
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int d = 32 * dt + 8 * j + 4 * hf; // o[u][dt][4*j .. 4*j+3] are rows d .. d+3 of O^T
                if (32 * dt + 8 * j < D) {
                    float4 r;
                    r.x = o[u][dt][4 * j] * f;
                    r.y = o[u][dt][4 * j + 1] * f;
                    r.z = o[u][dt][4 * j + 2] * f;
                    r.w = o[u][dt][4 * j + 3] * f;
                    *reinterpret_cast<float4 *>(so + (wave * C::Q + 32 * u + col) * C::SD + d) = r;
                }
            }
    }
    __syncthreads();
    {
        const int q = tid % C::Q;
        float m_all = -INFINITY, l_all = 0.0f;
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) m_all = fmaxf(m_all, sm[w * C::Q + q]);
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) {
            const float mw = sm[w * C::Q + q];
            if (mw != -INFINITY) l_all += __builtin_amdgcn_exp2f(mw - m_all) * sl[w * C::Q + q];
        }
        const float inv = 1.0f / l_all;
        const int row = q0 + q;
        if (row < p.Lq) {
            for (int dg = tid / C::Q; dg < C::G; dg += 256 / C::Q) {
                float acc[8];
#pragma unroll
                for (int e = 0; e < 8; e++) acc[e] = 0.0f;
#pragma unroll
                for (int w = 0; w < FA_WAVES; w++) {
                    const float4 a = *reinterpret_cast<const float4 *>(so + (w * C::Q + q) * C::SD + dg * 8);
                    const float4 b = *reinterpret_cast<const float4 *>(so + (w * C::Q + q) * C::SD + dg * 8 + 4);
                    acc[0] += a.x; acc[1] += a.y; acc[2] += a.z; acc[3] += a.w;
                    acc[4] += b.x; acc[5] += b.y; acc[6] += b.z; acc[7] += b.w;
                }
                half8_t r;
#pragma unroll
                for (int e = 0; e < 8; e++) r[e] = (half_t)(acc[e] * inv);
                const size_t oi = p.out_merged ? (size_t(row) * p.H + h) * D + dg * 8 : (size_t(h) * p.Lq + row) * D + dg * 8;
                *reinterpret_cast<half8_t *>(p.out + oi) = r;
            }
        }
    }
}

// The same for calls of which 96 rows of a head per workgroup still fit one round, one workgroup to a compute unit (heads of 72): three
// blocks of 32 rows, each walked by four wavefronts as in flash_attn_kernel, twelve in all; the three with the same tiles share them.  With 64
// rows per workgroup such a call puts two workgroups on some units and one on others (16 heads, 1458 rows: 368 on 256), and
// the units with two decide.  Here every SIMD has three wavefronts of six tiles each.  A tile of each (256 keys) takes 2.2 us, launch, first tiles and
// merge 5.7 (256 to 1,536 keys, 256 workgroups).  Inside the encoder the vector unit has 48 % of a unit's busy cycles, the matrix core 28, LDS 18;
// a wavefront waits for 48 % of its own, among others for its LDS operands, which are read one step at a time.
// Calls back to back, 64 rows -> 96: 16 heads, 1100 rows 19.8 -> 15.0 us, 1250 20.6 -> 15.8, 1458 23.0 -> 18.6 (28.7 -> 23.6
// inside the encoder); 32 heads, 600 rows 14.5 -> 11.0, 729 15.1 -> 11.8; 8 heads, 2916 rows 39.8 -> 32.0.  In two rounds it loses (16 x 2000: 31.9 against 43.3, 32 x 1000: 19.0
// against 25.8) or gains little (32 x 1250: 31.8 and 30.7), and where 32 rows per workgroup fit one round they are better (16 x 1024: 12.5 and 13.4, 32 x 512: 8.7 and 9.3).
// Tried and slower: three blocks per wavefront, the accumulators in both halves of the registers (42.5 us at 1458 rows).
// Each row goes through the same operations in the same order as above: the same bits (tested).
constexpr int FC_BLOCKS = 3, FC_THREADS = 64 * FC_BLOCKS * FA_WAVES;
template <int D>
struct FcCfg {
    static constexpr int BLOCKS = FC_BLOCKS, Q = 32 * BLOCKS, STAGES = 2;
    static constexpr int DK = (D + 15) / 16 * 16, KSTEPS = DK / 16, DT = (D + 31) / 32, G = D / 8;
    static constexpr int TILE = FA_KT * D;                  // halfs of a K or V tile
    static constexpr int COPIES = FA_KT * G / 64 / BLOCKS;  // copies of 64 granules that a wavefront makes of each
    static_assert(FA_KT * G == 64 * BLOCKS * COPIES, "whole copies");
    static constexpr int SD = D + 4;
    static constexpr size_t MERGE_BYTES = size_t(FA_WAVES) * Q * SD * sizeof(float);
    static constexpr size_t TILE_BYTES = size_t(FA_WAVES) * STAGES * 2 * TILE * sizeof(half_t);
    static constexpr size_t ML_OFFSET = TILE_BYTES > MERGE_BYTES ? TILE_BYTES : MERGE_BYTES;
    static constexpr size_t LDS_BYTES = ML_OFFSET + 2 * FA_WAVES * Q * sizeof(float);
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

template <int D>
__global__ __launch_bounds__(FC_THREADS) __attribute__((amdgpu_waves_per_eu(3))) void flash_attn96_kernel(FaArgs p) {
    using C = FcCfg<D>;
    extern __shared__ __attribute__((aligned(16))) half_t smem[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), block = wave % C::BLOCKS, group = wave / C::BLOCKS;
    const int col = lane & 31, hf = lane >> 5;
    // which head and rows: a die takes whole stretches of the (head, block) list
    int item = (int)(blockIdx.y * gridDim.x + blockIdx.x);
    const int n_items = (int)(gridDim.x * gridDim.y);
    if (n_items % 8 == 0) item = (item % 8) * (n_items / 8) + item / 8;
    const int h = item / (int)gridDim.x, q0 = item % (int)gridDim.x * C::Q;
    const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<unsigned long>((__attribute__((address_space(3))) const half_t *)smem));
    int voff[2][C::DT]; // where this lane points the transposing loads, as in flash_attn64_kernel
#pragma unroll
    for (int j = 0; j < 2; j++)
#pragma unroll
        for (int dt = 0; dt < C::DT; dt++) {
            const int key = (D == 72 ? 0 : 8 * j) + 4 * hf + ((lane & 15) >> 2), c = min(32 * dt + 16 * ((lane >> 4) & 1) + 4 * (lane & 3), D - 4);
            voff[j][dt] = fb_slot<D>(key) * D + ((c >> 3 ^ fb_swizzle<D>(key)) << 3 | (c & 7)) + (D == 72 ? j * fb_slot<D>(8) * D : 0);
        }
    const int row_bytes = (int)p.kv_row_stride * 2, head_bytes = (p.Lkv - 1) * row_bytes + D * 2;
    const half_t *kh = p.k + size_t(h) * p.kv_head_stride, *vh = p.v + size_t(h) * p.kv_head_stride;
    int off[C::COPIES]; // this lane's granules of a tile, from its first row (K and V lie alike)
#pragma unroll
    for (int i = 0; i < C::COPIES; i++) {
        const int x = (block * C::COPIES + i) * 64 + lane, key = fb_slot<D>(x / C::G);
        off[i] = key * row_bytes + (x % C::G ^ fb_swizzle<D>(key)) * 16;
    }
    const int n_tiles = (p.Lkv + FA_KT - 1) / FA_KT;
    const size_t tile_stride = size_t(FA_KT) * p.kv_row_stride;
    auto copy = [&](int t, int stage) {
        const unsigned k_lds = lds0 + (group * C::STAGES + stage) * 2 * C::TILE * 2 + block * C::COPIES * 1024;
        tile_copy(kh + t * tile_stride, head_bytes - t * FA_KT * row_bytes, k_lds, off);
        tile_copy(vh + t * tile_stride, head_bytes - t * FA_KT * row_bytes, k_lds + C::TILE * 2, off);
    };
    int t = group;
    if (t < n_tiles) copy(t, 0);
    half8_t qf[C::KSTEPS]; // this lane's query row as the MFMA "B" operand: Q[q0 + 32 block + col][16*s + 8*hf .. +7]
    {
        const half_t *qp = p.q + size_t(h) * p.q_head_stride + size_t(min(q0 + 32 * block + col, p.Lq - 1)) * p.q_row_stride;
#pragma unroll
        for (int s = 0; s < C::KSTEPS; s++) {
            const int d = 16 * s + 8 * hf;
#pragma unroll
            for (int e = 0; e < 8; e++) qf[s][e] = (half_t)0.0f;
            if (d < D) qf[s] = *reinterpret_cast<const half8_t *>(qp + d);
        }
    }
    // (as in flash_attn64_kernel; without it every round waited for the tile just asked for: back to back, with K and V in the L2, 1 % or nothing, inside
    // the encoder 1458 rows 24.5 -> 23.6 us)
    __builtin_amdgcn_s_waitcnt(0xf70);
    float16_t o[C::DT];
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int v = 0; v < 16; v++) o[dt][v] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f; // l_run: this lane's half of the row sum
    const float c2 = p.scale * 1.4426950408889634f; // > 0: the maximum of the scaled scores is the scaled maximum

    for (int left = (n_tiles + FA_WAVES - 1) / FA_WAVES, stage = 0; left > 0; left--, t += FA_WAVES, stage ^= 1) {
        tile_handed_over();
        if (t + FA_WAVES < n_tiles) copy(t + FA_WAVES, stage ^ 1);
        if (t >= n_tiles) continue;
        const half_t *Ks = smem + (group * C::STAGES + stage) * 2 * C::TILE, *Vs = Ks + C::TILE;
        const int key0 = t * FA_KT;
        float16_t s[2];
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
#pragma unroll
            for (int v = 0; v < 16; v++) s[kt][v] = 0.0f;
            const half_t *row = Ks + fb_slot<D>(32 * kt + col) * D;
#pragma unroll
            for (int st = 0; st < C::KSTEPS; st++) {
                const bool past = 16 * st + 8 >= D; // the second half of the wavefront has no granule here: zeros
                const int g = past ? 2 * st : (2 * st + hf) ^ fb_swizzle<D>(col);
                u32x4 a = *reinterpret_cast<const u32x4 *>(row + g * 8);
                if (past && hf) a = u32x4{0, 0, 0, 0};
                s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a), qf[st], s[kt], 0, 0, 0);
            }
        }
        // s[kt][v] = score of key key0 + 32*kt + 8*(v/4) + 4*hf + v%4; from here on as in flash_attn64_kernel
        if (key0 + FA_KT > p.Lkv) {
            const int seen = p.Lkv - 1 - key0 - 4 * hf; // keys past this one of the tile are masked
#pragma unroll
            for (int kt = 0; kt < 2; kt++)
#pragma unroll
                for (int v = 0; v < 16; v++) s[kt][v] = 32 * kt + 8 * (v >> 2) + (v & 3) > seen ? -INFINITY : s[kt][v];
        }
        asm volatile("" : "+v"(s[0]), "+v"(s[1])); // (in these registers on both paths: left alone, the scores are copied on each)
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int v = 0; v < 16; v++) mx = fmaxf(mx, s[kt][v]);
        mx = half_max(mx);
        const float m_new = fmaxf(m_run, mx * c2);
        float alpha = 1.0f;
        if (__any(m_new != m_run)) {
            alpha = __builtin_amdgcn_exp2f(m_run - (m_new == -INFINITY ? 0.0f : m_new));
            m_run = m_new;
#pragma unroll
            for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
                for (int v = 0; v < 16; v++)
                    if (32 * dt + 8 * (v >> 2) < D) o[dt][v] *= alpha;
        }
        const float m_use = m_run == -INFINITY ? 0.0f : m_run;
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
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
            for (int sp = 0; sp < 2; sp++) {
                half8_t pb;
#pragma unroll
                for (int e = 0; e < 8; e++) pb[e] = (half_t)s[kt][8 * sp + e];
#pragma unroll
                for (int dt = 0; dt < C::DT; dt++) {
                    const half4_t lo = fa_read_tr(Vs + voff[0][dt] + (32 * kt + 16 * sp) * D);
                    const half4_t hi = fa_read_tr(Vs + voff[1][dt] + (32 * kt + 16 * sp) * D);
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7), pb, o[dt], 0, 0, 0);
                }
            }
    }

    // merge the four groups' results, as in flash_attn64_kernel
    float *so = reinterpret_cast<float *>(smem);                                          // [group][q][SD]
    float *sm = reinterpret_cast<float *>(reinterpret_cast<char *>(smem) + C::ML_OFFSET); // [group][q]
    float *sl = sm + FA_WAVES * C::Q;                                                     // [group][q]
    const int mine = group * C::Q + 32 * block + col;
    const float l_wave = l_run + __shfl_xor(l_run, 32);
    if (hf == 0) {
        sm[mine] = m_run;
        sl[mine] = l_wave;
    }
    __syncthreads(); // every wavefront is done with the tiles, which O takes over, and has published its maximum
    float m_all = -INFINITY;
#pragma unroll
    for (int w = 0; w < FA_WAVES; w++) m_all = fmaxf(m_all, sm[w * C::Q + 32 * block + col]);
    const float f = m_run == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m_run - m_all); // (maxima are in base-2 units)
#pragma unroll
    for (int dt = 0; dt < C::DT; dt++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (32 * dt + 8 * j < D) // o[dt][4*j .. 4*j+3] are rows 32 dt + 8 j + 4 hf .. + 3 of O^T
                *reinterpret_cast<float4 *>(so + mine * C::SD + 32 * dt + 8 * j + 4 * hf) = float4{o[dt][4 * j] * f, o[dt][4 * j + 1] * f, o[dt][4 * j + 2] * f, o[dt][4 * j + 3] * f};
    __syncthreads();
    for (int i = tid; i < C::Q * C::G; i += FC_THREADS) {
        const int q = i % C::Q, dg = i / C::Q, row = q0 + q;
        if (row >= p.Lq) continue;
        float most = -INFINITY, l_all = 0.0f;
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) most = fmaxf(most, sm[w * C::Q + q]);
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++) {
            const float mw = sm[w * C::Q + q];
            if (mw != -INFINITY) l_all += __builtin_amdgcn_exp2f(mw - most) * sl[w * C::Q + q];
        }
        const float inv = 1.0f / l_all;
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < FA_WAVES; w++)
#pragma unroll
            for (int e = 0; e < 8; e++) acc[e] += so[(w * C::Q + q) * C::SD + dg * 8 + e];
        half8_t r;
#pragma unroll
        for (int e = 0; e < 8; e++) r[e] = (half_t)(acc[e] * inv);
        *reinterpret_cast<half8_t *>(p.out + (p.out_merged ? (size_t(row) * p.H + h) * D : (size_t(h) * p.Lq + row) * D) + dg * 8) = r;
    }
}

template <int D>
int launch_flash(moon_ctx *ctx, const FaArgs &p) {
    // Two workgroups fit a compute unit.  Sixty-four rows from where 32 rows would take a second round (rows of all heads > 64 per unit),
    // for heads of 64, whose tiles cost less to bring, from the third half round (96), and where a row sees only the keys before it, so
    // that the light blocks fill up the first round, from 112.  Times of a call, 32 rows -> 64, on 256 units:
    //   heads of 72           16 x 1024 (64 per unit) 14.1 -> 14.3 us, 16 x 1100 21.6 -> 20.9, 32 x 512 (64) 9.4 -> 9.7, 32 x 550 15.3 -> 14.6
    //   heads of 64           32 x 600 13.4 -> 13.9, 32 x 768 (96) 14.2 -> 14.3, 32 x 832 19.0 -> 16.1, 16 x 1664 29.8 -> 24.4
    //   heads of 64, causal   32 x 768 (96) 12.0 -> 11.5, 32 x 800 12.4 -> 12.7, 32 x 832 12.8 -> 13.0, 16 x 1600 17.4 -> 18.3, 8 x 3328 (104) 28.8 -> 29.4;
    //                         32 x 896 (112) 13.6 -> 13.4, 16 x 1792 (112) 20.0 -> 18.9, 8 x 3584 (112) 31.9 -> 31.5, 32 x 1024 15.4 -> 13.9
    // Past the line the two kernels' rounds end at different sizes, so a few sizes lose up to 2 % (32 heads of 64: 1360 causal rows 22.6 ->
    // 23.0, 1056 rows 26.5 -> 27.1); from there on up to 25 % are gained (32 x 2048: 65.7 -> 52.6; of 72: 79.6 -> 61.7).
    // Well below the line the chip is better filled with 32: 16 heads of 72, 512 rows 7.6 us against 9.5.
    const size_t rows = (size_t)p.Lq * p.H, cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const bool two = p.causal_pos >= 0 ? rows >= 112 * cus : rows > (D == 64 ? 96 : 64) * cus;
    auto go = [&](auto kernel, std::atomic<bool> (&attr_set)[64], int rows_wg, int threads, size_t lds, const char *name) -> int {
        const unsigned blocks = (unsigned)((p.Lq + rows_wg - 1) / rows_wg);
        const int dev = ctx->device >= 0 && ctx->device < 64 ? ctx->device : -1; // the opt-in to this much dynamic LDS is per device (and per kernel)
        if (dev < 0 || !attr_set[dev].load()) {
            MOON_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            if (dev >= 0) attr_set[dev].store(true);
        }
        hipLaunchKernelGGL(kernel, dim3(blocks, (unsigned)p.H), dim3(threads), lds, ctx->stream, p);
        MOON_HIP(ctx, hipGetLastError());
        MOON_NOTE_ATTENTION(ctx, "%s %d workgroups", name, (int)blocks * p.H);
        return MOON_OK;
    };
    static std::atomic<bool> set32[64], set64[64], set96[64];
    if constexpr (D == 72)
        if (two && p.causal_pos < 0 && size_t(p.Lq + 95) / 96 * p.H <= cus)
            return go(flash_attn96_kernel<D>, set96, FcCfg<D>::Q, FC_THREADS, FcCfg<D>::LDS_BYTES, "flash_attn96_kernel<72>");
    if (two) return go(flash_attn64_kernel<D>, set64, FbCfg<D>::Q, 256, FbCfg<D>::LDS_BYTES, D == 64 ? "flash_attn64_kernel<64>" : "flash_attn64_kernel<72>");
    return go(flash_attn_kernel<D>, set32, FA_Q, 256, FaCfg<D>::LDS_BYTES, D == 64 ? "flash_attn_kernel<64>" : "flash_attn_kernel<72>");
}

} // namespace

// Takes the call when the shape is one the matrix-core kernel is built for; otherwise *handled stays false and the
// caller falls back to the shape-generic kernel.
int launch_sdpa_mfma(moon_ctx *ctx, const half_t *q, const half_t *k, const half_t *v, half_t *out, size_t H, size_t Lq, size_t Lkv,
                     size_t D, size_t kv_head_stride, long causal_pos, bool out_merged, bool *handled) {
    *handled = false;
    if ((D != 64 && D != 72) || Lq < 16 || Lkv == 0 || H == 0 || H > 65535) return MOON_OK;
    if (((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)out) % 16 || (kv_head_stride * sizeof(half_t)) % 16) return MOON_OK;
    if (Lkv * D * sizeof(half_t) >= (size_t(1) << 31)) return MOON_OK; // a head's rows are addressed with 32-bit offsets
    FaArgs p{q, k, v, out, (int)H, (int)Lq, (int)Lkv, Lq * D, D, kv_head_stride, D, causal_pos, out_merged ? 1 : 0, 1.0f / sqrtf((float)D)};
    *handled = true;
    return D == 64 ? launch_flash<64>(ctx, p) : launch_flash<72>(ctx, p);
}

// Non-causal attention straight from a packed projection qkv[T][3 * H * D] (row = q | k | v, heads side by side inside each
// third: vision_model.zig:285-314 splits and transposes it into three tensors first) to the merged layout out[T][H * D]
// that the output projection reads (vision_model.zig:326-335).  *handled stays false for shapes the kernel does not cover.
int launch_sdpa_packed_qkv(moon_ctx *ctx, const half_t *qkv, half_t *out, size_t H, size_t T, size_t D, bool *handled) {
    *handled = false;
    if ((D != 64 && D != 72) || T < 16 || H == 0 || H > 65535) return MOON_OK;
    if (((uintptr_t)qkv | (uintptr_t)out) % 16) return MOON_OK;
    const size_t d = H * D;
    if (T * 3 * d * sizeof(half_t) >= (size_t(1) << 31)) return MOON_OK; // (32-bit offsets within a head's rows)
    FaArgs p{qkv, qkv + d, qkv + 2 * d, out, (int)H, (int)T, (int)T, D, 3 * d, D, 3 * d, -1, 1, 1.0f / sqrtf((float)D)};
    *handled = true;
    return D == 64 ? launch_flash<64>(ctx, p) : launch_flash<72>(ctx, p);
}
