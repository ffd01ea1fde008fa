// One token through a layer of a layer-list decoder, in three launches:
//   decode_proj   h = norm(x) (or of the embedding row; behind a layer of two joined mixers x is completed first), then the layer's
//                 first product: q, k, v, gate, router logits, or a dense feed-forward's silu(gate) * up.  With only f32 rows it is
//                 the LM head.
//   decode_mix    the token's attention over the cache (norm of q and k, rotation, value mixing, cache update, sink, output gate), keys
//                 split over workgroups, the one that finishes last merging; beside it, in workgroups of their own, the router's choice
//                 and the chosen experts' silu(gate) * up, or one token of the gated delta rule, a head per workgroup; and the dense
//                 activation's part of the second product, which needs nothing of the attention.
//   decode_out    x += W2 . (heads | dense activation) + the chosen experts' weighted down products, or the parts of W2 . (..) that
//                 the next decode_proj joins; without what decode_mix has left.
// The attention is a chain of dependent steps that keeps a few units busy for 8 to 9 us, whatever it reads, while the stream of the dense
// columns (22.5 of the second product's 30.9 MB at width 2048, feed-forward 5504) takes about as long: together 0.844 instead of
// 0.908 ms per token behind 768 cached keys, 0.802 instead of 0.847 behind 60.  In the chain itself the projections are requested ahead of the
// cache rows (loads return in order), lanes are summed with cross-lane moves instead of trips through LDS, the newest key is a piece like
// the others and rows are found without divisions: 0.771 and 0.747 ms.  One split for a short context, which would save the merge, is slower
// (0.785 against 0.747 at 60 to 90 keys): a step of 32 keys costs more than the hop.
// Every role of decode_mix has the attention's LDS and the experts' registers.  It pays all the same: with heads of 512, which leave a unit one
// workgroup, eight layers (8 heads on one key head) went from 819 to 631 us per token behind 60 keys and from 1,907 to 1,200 behind 1,900; a
// kernel without the experts' part, which lets three or four workgroups of the down product share a unit, is 1.4 to 2 % slower (heads of 64).
// All are bound by HBM: weights are read once with 128-bit non-temporal loads.  No workgroup waits for another.
#include "decode_roles.hpp"
#include "kernel_args.hpp"
#include "router.hpp"

#include <algorithm>
#include <type_traits>

namespace {

// NV: 16-byte pieces of x, gamma and beta a thread holds (rows of up to 1024 NV elements, a multiple of 4); 0: any row, from memory.
// JOIN: x is completed with a joined layer's results first.
template <class T, int U, int NV, bool JOIN>
__global__ __launch_bounds__(256) void decode_proj_kernel(DecodeProj) {
    const DecodeProj &p = fetch_arguments<DecodeProj>();
    extern __shared__ __attribute__((aligned(16))) char s_raw[]; // h: T [dp], then (NV = 0) x: float [width]
    T *s_h = reinterpret_cast<T *>(s_raw);
    float *s_x = reinterpret_cast<float *>(s_raw + size_t(p.dp) * sizeof(T));
    __shared__ float s_red[16];
    constexpr int RG = 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const T *W = reinterpret_cast<const T *>(p.w1);
    const int pieces = p.dp / Piece<T>::N;
    // The rows in groups of four: the used rows of the 16-bit and the f32 segment (each rounded up to whole groups), then two
    // gate/up pairs per group.
    const int g16 = (p.n16_used + 3) / 4, g32 = g16 + (p.n32_used + 3) / 4, groups = g32 + (p.ff + 1) / 2;
    int g_begin, g_end;
    share(groups, gridDim.x * 4, blockIdx.x * 4 + wave, g_begin, g_end);
    const T *rows[RG];
    auto locate = [&](int g) {
#pragma unroll
        for (int j = 0; j < RG; j++) {
            int row;
            if (g < g16) row = 4 * g + j;
            else if (g < g32) row = p.n16 + 4 * (g - g16) + j;
            else row = p.n32 + pair_row(2 * (g - g32) + (j >> 1), j & 1);
            rows[j] = W + size_t(row) * p.dp; // (segments are padded to whole groups)
        }
    };
    // The norm's inputs are requested first, then the first weights: loads return in order, so the weights stream in while the
    // norm is computed.
    const T *er = p.token ? reinterpret_cast<const T *>(p.embed) + size_t(p.token[0]) * p.dp : nullptr;
    NormRow<T, NV ? NV : 1, JOIN, false> norm;
    if (NV) norm.request(p, er, tid);
    RowDots<T, RG, U> dots;
    if (g_begin < g_end) {
        locate(g_begin);
        dots.request(rows, 0, pieces, lane);
    }
    if (NV) norm.finish(p, er, blockIdx.x == 0, s_h, s_red, tid);
    else {
        if (JOIN) {
            float ss[2] = {0.0f, 0.0f};
            for (int i = tid; i < p.width; i += 256) {
                ss[0] = fmaf(p.y[i], p.y[i], ss[0]);
                ss[1] = fmaf(p.y[p.dp + i], p.y[p.dp + i], ss[1]);
            }
            norm.join_factors(p, ss, s_red, lane, wave);
            for (int i = tid; i < p.width; i += 256) {
                s_x[i] = p.x[i] + p.y[2 * p.dp + i] + (p.y[i] * ss[0] * p.out_l[i] + p.y[p.dp + i] * ss[1] * p.out_r[i]);
                if (blockIdx.x == 0) p.x_new[i] = s_x[i];
            }
        }
        float s = 0.0f, m2 = 0.0f;
        for (int i = tid; i < p.width; i += 256) {
            const float v = er ? (float)er[i] * p.embed_scale : JOIN ? s_x[i] : p.x[i];
            if (er && blockIdx.x == 0) p.x[i] = v;
            s_x[i] = v;
            s += v;
        }
        const float mean = p.beta ? block_sum(s, s_red) / (float)p.width : 0.0f;
        for (int i = tid; i < p.width; i += 256) {
            const float d = s_x[i] - mean;
            m2 = fmaf(d, d, m2);
        }
        const float rstd = 1.0f / sqrtf(block_sum(m2, s_red) / (float)p.width + p.eps);
        for (int i = tid; i < p.dp; i += 256) {
            const T v = i < p.width ? (T)((s_x[i] - mean) * rstd * p.gamma[i] + (p.beta ? p.beta[i] : 0.0f)) : (T)0.0f;
            s_h[i] = v;
            if (p.h && blockIdx.x == 0) reinterpret_cast<T *>(p.h)[i] = v;
        }
    }
    lds_barrier();
    for (int g = g_begin; g < g_end; g++) {
        float acc[RG] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p0 = 0;;) {
            dots.add(s_h, p0, pieces, lane, acc);
            p0 += 64 * U;
            if (p0 >= pieces) break;
            dots.request(rows, p0, pieces, lane);
        }
        if (g + 1 < g_end) {
            locate(g + 1);
            dots.request(rows, 0, pieces, lane);
        }
#pragma unroll
        for (int j = 0; j < RG; j++) acc[j] = wave_sum(acc[j]);
        if (lane == 0) {
            if (g < g16) *reinterpret_cast<float4 *>(p.proj + 4 * g) = float4{acc[0], acc[1], acc[2], acc[3]};
            else if (g < g32) {
                float4 z = {acc[0], acc[1], acc[2], acc[3]};
                if (p.softcap > 0.0f) z = {lm_softcap(z.x, p.softcap), lm_softcap(z.y, p.softcap), lm_softcap(z.z, p.softcap), lm_softcap(z.w, p.softcap)};
                *reinterpret_cast<float4 *>(p.logits + 4 * (g - g16)) = z;
            }
            else {
                T *o = reinterpret_cast<T *>(p.glu) + 2 * (g - g32); // (the activation is padded like the weights)
                o[0] = (T)(lm_silu(acc[0]) * acc[1]);
                o[1] = (T)(lm_silu(acc[2]) * acc[3]);
            }
        }
    }
}

constexpr int MIX_DOWN_ROWS = 4;   // rows of the dense activation's product per workgroup

// The chosen experts' gate and up rows, by the launch's expert workgroups.
template <class T, int U>
__device__ __forceinline__ void mix_experts(const DecodeMix &p, int wg, int n_wgs, char *lds) {
    constexpr int RG = 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, pieces = p.dp / Piece<T>::N;
    T *s_h = reinterpret_cast<T *>(lds);
    float *s_scores = reinterpret_cast<float *>(lds + size_t(p.dp) * sizeof(T)); // [2 E]
    float *s_w = s_scores + 2 * p.E;                                              // [top]
    int *s_ids = reinterpret_cast<int *>(s_w + p.top);                            // [top]
    for (int i = tid; i < pieces; i += 256) reinterpret_cast<lm_u32x4 *>(s_h)[i] = reinterpret_cast<const lm_u32x4 *>(p.h)[i];
    if (wave == 0) route_wave(p.logits, p.correction, p.E, p.top, s_scores, lane, s_ids, s_w);
    __syncthreads();
    if (wg == 0)
        for (int k = tid; k < p.top; k += 256) {
            p.ids[k] = s_ids[k];
            p.weight[k] = s_w[k];
        }
    const int per_expert = (p.ff + 1) / 2; // groups of two pairs
    int g_begin, g_end;
    share(p.top * per_expert, n_wgs * 4, wg * 4 + wave, g_begin, g_end);
    RowDots<T, RG, U> dots;
    const T *rows[RG];
    auto locate = [&](int g) {
        const int k = g / per_expert, i = 2 * (g % per_expert);
        const T *W = reinterpret_cast<const T *>(p.wgu) + size_t(s_ids[k]) * 2 * p.ffp * p.dp;
#pragma unroll
        for (int j = 0; j < RG; j++) rows[j] = W + size_t(pair_row(i + (j >> 1), j & 1)) * p.dp;
    };
    if (g_begin < g_end) {
        locate(g_begin);
        dots.request(rows, 0, pieces, lane);
    }
    for (int g = g_begin; g < g_end; g++) {
        float acc[RG] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (int p0 = 0;;) {
            dots.add(s_h, p0, pieces, lane, acc);
            p0 += 64 * U;
            if (p0 >= pieces) break;
            dots.request(rows, p0, pieces, lane);
        }
        if (g + 1 < g_end) {
            locate(g + 1);
            dots.request(rows, 0, pieces, lane);
        }
#pragma unroll
        for (int j = 0; j < RG; j++) acc[j] = wave_sum(acc[j]);
        if (lane == 0) {
            T *o = reinterpret_cast<T *>(p.act) + size_t(g / per_expert) * p.ffp + 2 * (g % per_expert);
            o[0] = (T)(lm_silu(acc[0]) * acc[1]);
            o[1] = (T)(lm_silu(acc[2]) * acc[3]);
        }
    }
}

typedef float OutSums[4][3][4]; // [wavefront][part][row]
// Rows [row0, row0 + RW) of W2 against columns [c0, c1) of a (16-byte pieces), and of the chosen experts' down matrices against their
// activations.  A workgroup owns the rows; its four wavefronts share each row's pieces, so a lane reads its part of the vectors once
// for all rows.  PARTS = 3: the sums over three stretches of the columns are kept apart.  done(k, r, sum) is called by one thread per
// sum.
template <class T, int RW, int U, int PARTS, class Done>
__device__ __forceinline__ void out_rows(const DecodeOut &p, int row0, int c0, int c1, OutSums &s_part, Done done) {
    constexpr int PE = Piece<T>::N;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int pa = c1 - c0, pf = p.top ? p.ffp / PE : 1, total = pa + p.top * pf;
    int begin, end;
    share(total, 4, wave, begin, end);
    float acc[PARTS][RW];
#pragma unroll
    for (int k = 0; k < PARTS; k++)
#pragma unroll
        for (int r = 0; r < RW; r++) acc[k][r] = 0.0f;
    for (int base = begin; base < end; base += 64 * U) {
        lm_u32x4 w[U][RW], x[U];
        float scale[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int i = base + u * 64 + lane;
            x[u] = lm_u32x4{0, 0, 0, 0};
            scale[u] = 1.0f;
#pragma unroll
            for (int r = 0; r < RW; r++) w[u][r] = lm_u32x4{0, 0, 0, 0};
            if (i < end) {
                const T *m;
                size_t pitch;
                if (i < pa) {
                    x[u] = reinterpret_cast<const lm_u32x4 *>(p.a)[c0 + i];
                    m = reinterpret_cast<const T *>(p.w2) + size_t(row0) * p.k0 + size_t(c0 + i) * PE;
                    pitch = p.k0;
                } else {
                    const int k = (i - pa) / pf, c = (i - pa) % pf;
                    x[u] = reinterpret_cast<const lm_u32x4 *>(p.act)[size_t(k) * pf + c];
                    scale[u] = p.weight[k];
                    m = reinterpret_cast<const T *>(p.wd) + (size_t(p.ids[k]) * p.dp + row0) * p.ffp + size_t(c) * PE;
                    pitch = p.ffp;
                }
#pragma unroll
                for (int r = 0; r < RW; r++) // (rows are padded to 64)
                    w[u][r] = __builtin_nontemporal_load(reinterpret_cast<const lm_u32x4 *>(m + r * pitch));
            }
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int r = 0; r < RW; r++) {
                const float d = dot_piece<T>(w[u][r], x[u], 0.0f);
                const int i = c0 + base + u * 64 + lane;
                if (PARTS == 1) acc[0][r] = fmaf(d, scale[u], acc[0][r]);
                else
#pragma unroll
                    for (int k = 0; k < PARTS; k++) acc[k][r] += (i >= p.k1 / PE) + (i >= p.k2 / PE) == k ? d : 0.0f;
            }
    }
#pragma unroll
    for (int k = 0; k < PARTS; k++)
#pragma unroll
        for (int r = 0; r < RW; r++) {
            const float s = wave_sum(acc[k][r]);
            if (lane == 0) s_part[wave][k][r] = s;
        }
    lds_barrier();
    const int k = tid / RW, r = tid % RW;
    if (k >= PARTS || row0 + r >= p.width) return;
    done(k, row0 + r, (s_part[0][k][r] + s_part[1][k][r]) + (s_part[2][k][r] + s_part[3][k][r]));
}

// x += W2 . a, but for what decode_mix has left in p.down already.
template <class T, int RW, int U, int PARTS>
__global__ __launch_bounds__(256) void decode_out_kernel(DecodeOut p) {
    __shared__ OutSums s_part;
    const int row = blockIdx.x * RW + threadIdx.x % RW;
    float down = 0.0f;
    if (PARTS == 1 && p.down && threadIdx.x < RW && row < p.width) down = p.down[row]; // (requested before the weights)
    out_rows<T, RW, U, PARTS>(p, blockIdx.x * RW, 0, (p.down ? p.k2 : p.k0) / Piece<T>::N, s_part, [&](int k, int n, float s) {
        if (PARTS == 1) p.x[n] += s + down;
        else if (k < 2 || !p.down) p.y[k * p.dp + n] = s;
    });
}

struct MixArgs {
    DecodeMix p;
    DecodeOut o;
    int S, keys_max, n_attn, n_expert;
};
template <class T, int NH, int U, bool WHOLE, bool LONG>
__global__ __launch_bounds__(256) void decode_mix_kernel(MixArgs given) {
    // (WHOLE has so many that addresses of the compiler's own serve it better, once the lines are there: 793 against 805 us a token at width 2048)
    const MixArgs &fetched = fetch_arguments<MixArgs>(), &args = WHOLE ? given : fetched;
    if (WHOLE) __builtin_amdgcn_sched_barrier(0);
    const DecodeMix &p = args.p;
    const DecodeOut &o = args.o;
    const int S = args.S, keys_max = args.keys_max, n_attn = args.n_attn, n_expert = args.n_expert;
    extern __shared__ __attribute__((aligned(16))) char s_mix[]; // (all there is: heads may fill a compute unit's)
    // attention first: it is a chain of dependent steps, the experts' part and the dense activation's product are long streams
    const int i = blockIdx.x, n_hb = mix_head_blocks(p.H / p.G), n_delta = WHOLE ? p.dH : 0;
    if (i < n_attn) mix_attention<T, NH, WHOLE, LONG, 0>(p, i / S / n_hb, i / S % n_hb, i % S, S, keys_max, reinterpret_cast<float *>(s_mix), Apart{});
    else if (WHOLE && i < n_attn + n_delta) {
        const int h = i - n_attn;
        if (p.ddimp <= DELTA_ROWS * (256 / (p.dvdimp / 4))) mix_delta<T, true>(p, h, reinterpret_cast<float *>(s_mix), Apart{});
        else mix_delta<T, false>(p, h, reinterpret_cast<float *>(s_mix), Apart{});
    } else if (i < n_attn + n_delta + n_expert) mix_experts<T, U>(p, i - n_attn - n_delta, n_expert, s_mix);
    else
        out_rows<T, MIX_DOWN_ROWS, 4, 1>(o, (i - n_attn - n_delta - n_expert) * MIX_DOWN_ROWS, o.k2 / Piece<T>::N, o.k0 / Piece<T>::N,
                                         *reinterpret_cast<OutSums *>(s_mix),
                                         [&](int, int n, float s) { o.down[n] = s; });
}

template <class T, int NH, bool WHOLE> int mix_launch_as(moon_ctx *ctx, const DecodeMix &p, const DecodeOut &o, int S, int keys_max, int n_attn, int n_expert, size_t lds) {
    const bool longer = std::max(p.dimp, p.vdimp) > 64 * Piece<T>::N;
    auto kern = longer ? decode_mix_kernel<T, NH, 4, WHOLE, true> : p.dp / Piece<T>::N > 64 ? decode_mix_kernel<T, NH, 4, WHOLE, false> : decode_mix_kernel<T, NH, 1, WHOLE, false>;
    if (lds > 64 * 1024) MOON_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int n_down = o.down ? (o.width + MIX_DOWN_ROWS - 1) / MIX_DOWN_ROWS : 0;
    hipLaunchKernelGGL(kern, dim3(n_attn + n_expert + (WHOLE ? p.dH : 0) + n_down), dim3(256), lds, ctx->stream, MixArgs{p, o, S, keys_max, n_attn, n_expert});
    MOON_HIP(ctx, hipGetLastError());
    return MOON_OK;
}
template <class T, int NH> int mix_launch(moon_ctx *ctx, const DecodeMix &p, const DecodeOut &o, int S, int keys_max, int n_attn, int n_expert, size_t lds) {
    return mix_whole(p) ? mix_launch_as<T, NH, true>(ctx, p, o, S, keys_max, n_attn, n_expert, lds)
                        : mix_launch_as<T, NH, false>(ctx, p, o, S, keys_max, n_attn, n_expert, lds);
}

template <class T> int proj_launch(moon_ctx *ctx, const DecodeProj &p) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const int groups = (p.n16_used + 3) / 4 + (p.n32_used + 3) / 4 + (p.ff + 1) / 2;
    const dim3 grid((unsigned)std::max(1, std::min(2 * cus, (groups + 3) / 4)));
    const int ch = (p.dp / Piece<T>::N + 63) / 64, nv = p.width % 4 || p.dp > 4096 || (reinterpret_cast<uintptr_t>(p.x) & 15) ? 0 : (p.dp + 1023) / 1024;
    const size_t lds = size_t(p.dp) * sizeof(T) + (nv ? 0 : size_t(p.width) * sizeof(float));
    if (lds > 60 * 1024) return moon_fail(ctx, MOON_EINVAL_DIM, "decode: width %d too large", p.width);
    auto pick = [&](auto u) {
        constexpr int U = decltype(u)::value;
        if (p.y) return nv == 0 ? decode_proj_kernel<T, U, 0, true> : nv == 1 ? decode_proj_kernel<T, U, 1, true> : nv == 2 ? decode_proj_kernel<T, U, 2, true> : decode_proj_kernel<T, U, 4, true>;
        return nv == 0 ? decode_proj_kernel<T, U, 0, false> : nv == 1 ? decode_proj_kernel<T, U, 1, false> : nv == 2 ? decode_proj_kernel<T, U, 2, false> : decode_proj_kernel<T, U, 4, false>;
    };
    auto kern = ch == 1 ? pick(std::integral_constant<int, 1>{}) : ch == 2 ? pick(std::integral_constant<int, 2>{}) : ch == 3 ? pick(std::integral_constant<int, 3>{})
                                                                                                                          : pick(std::integral_constant<int, 4>{});
    hipLaunchKernelGGL(kern, grid, dim3(256), lds, ctx->stream, p);
    MOON_HIP(ctx, hipGetLastError());
    return MOON_OK;
}

template <class T> int out_launch(moon_ctx *ctx, const DecodeOut &p) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    auto go = [&](auto parts) {
        constexpr int N = decltype(parts)::value;
        if (p.width >= 4 * 2 * cus) hipLaunchKernelGGL((decode_out_kernel<T, 4, 4, N>), dim3((p.width + 3) / 4), dim3(256), 0, ctx->stream, p);
        else if (p.width >= 2 * 2 * cus) hipLaunchKernelGGL((decode_out_kernel<T, 2, 6, N>), dim3((p.width + 1) / 2), dim3(256), 0, ctx->stream, p);
        else hipLaunchKernelGGL((decode_out_kernel<T, 1, 8, N>), dim3(p.width), dim3(256), 0, ctx->stream, p);
    };
    if (p.down && (p.top || p.k2 % 64 || p.k2 >= p.k0)) return moon_fail(ctx, MOON_EINVAL, "decode: no dense columns behind %d of %d", p.k2, p.k0);
    if (p.y && (p.top || p.k1 % 64 || p.k2 % 64 || p.k1 > p.k2 || p.k2 > p.k0)) return moon_fail(ctx, MOON_EINVAL, "decode: columns in parts %d %d %d", p.k1, p.k2, p.k0);
    if (p.y) go(std::integral_constant<int, 3>{});
    else go(std::integral_constant<int, 1>{});
    MOON_HIP(ctx, hipGetLastError());
    return MOON_OK;
}

} // namespace

int launch_decode_proj(moon_ctx *ctx, int dtype, const DecodeProj &p) {
    return dtype == MOON_DTYPE_BF16 ? proj_launch<bf16_t>(ctx, p) : proj_launch<float>(ctx, p);
}

int launch_decode_out(moon_ctx *ctx, int dtype, const DecodeOut &p) {
    return dtype == MOON_DTYPE_BF16 ? out_launch<bf16_t>(ctx, p) : out_launch<float>(ctx, p);
}

size_t decode_mix_counters(size_t heads, size_t kv_heads) { return kv_heads * mix_head_blocks((int)(heads / kv_heads)); }
size_t decode_mix_partial_floats(moon_ctx *ctx, size_t heads, size_t kv_heads, size_t vdimp, size_t max_keys) {
    const size_t cus = ctx->cu_count > 0 ? ctx->cu_count : 256, wgs = decode_mix_counters(heads, kv_heads);
    return std::max(std::max(wgs, cus), wgs * ((max_keys + MIX_KEYS - 1) / MIX_KEYS)) * MIX_HEADS * (vdimp + 2);
}

int launch_decode_mix(moon_ctx *ctx, int dtype, const DecodeMix &p, const DecodeOut &o) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256, per = p.H / p.G, wgs = p.G * mix_head_blocks(per), n_keys = mix_keys(p, p.pos), S = mix_splits(n_keys, wgs, cus);
    MOON_TRY(check_decode_mix(ctx, p));
    if (size_t(wgs) * S * MIX_HEADS * (p.vdimp + 2) > p.partial_floats) return moon_fail(ctx, MOON_ESEQ_TOO_LONG, "decode attention: %d keys", n_keys);
    const int keys_max = mix_split_keys(n_keys, S);
    if (p.E && (p.top < 1 || p.top > p.E || p.E > ROUTER_MAX_EXPERTS)) return moon_fail(ctx, MOON_EINVAL_DIM, "router: %d of %d experts", p.top, p.E);
    const int groups = p.E ? p.top * ((p.ff + 1) / 2) : 0;
    const int n_expert = std::min((groups + 3) / 4, std::max(cus, 2 * cus - wgs * S)); // (together two workgroups per CU: more measured slower)
    const int nh = std::min(per, MIX_HEADS), NH = nh <= 1 ? 1 : nh <= 2 ? 2 : nh <= 4 ? 4 : 8;
    const size_t el = dtype == MOON_DTYPE_BF16 ? sizeof(bf16_t) : sizeof(float);
    const size_t lds = std::max(std::max(mix_lds_floats(NH, p.dimp, p.vdimp, keys_max) * sizeof(float),
                                         p.E ? size_t(p.dp) * el + (size_t(2) * p.E + 2 * p.top) * sizeof(float) : 0),
                                p.dH ? delta_lds_floats(p.ddimp, p.dvdimp, p.kd) * sizeof(float) : 0);
    static_assert(sizeof(OutSums) <= (8 + 8 + 8 + 1 + 4 * 8 + 4 + 8) * sizeof(float), "the smallest heads leave room for the down product's sums");
    if (size_t(NH) * S > mix_lds_floats(NH, p.dimp, p.vdimp, keys_max) - 4 * NH - 8) return moon_fail(ctx, MOON_ESEQ_TOO_LONG, "decode attention: %d splits", S);
    if (lds > 160 * 1024) return moon_fail(ctx, MOON_EINVAL_DIM, "decode attention: heads of %d and %d", p.dimp, p.vdimp);
    auto go = [&](auto tag) -> int {
        using T = decltype(tag);
        switch (NH) {
        case 1: return mix_launch<T, 1>(ctx, p, o, S, keys_max, wgs * S, n_expert, lds);
        case 2: return mix_launch<T, 2>(ctx, p, o, S, keys_max, wgs * S, n_expert, lds);
        case 4: return mix_launch<T, 4>(ctx, p, o, S, keys_max, wgs * S, n_expert, lds);
        default: return mix_launch<T, 8>(ctx, p, o, S, keys_max, wgs * S, n_expert, lds);
        }
    };
    return dtype == MOON_DTYPE_BF16 ? go(bf16_t{}) : go(float{});
}
