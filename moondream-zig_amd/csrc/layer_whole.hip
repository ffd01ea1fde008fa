// One token through a whole layer of a layer-list decoder in ONE launch (layer_decode.hip has the same in three).  Workgroups take roles by index:
//   producers   h = norm(x), their rows of the first product: first q, k, v (and a delta rule's columns), counted by themselves, then the gate's and the
//               feed-forward's silu(gate) * up
//   attention   a split of a key head's keys each, and the delta rule's heads: ask for cache rows and states, wait for the first count, and report every
//               merged head
//   output      rows of the second product, two per wavefront: most of them (19 of 30 KB at width 2048, feed-forward 5504) is in registers by the time that the
//               activation is there, the rest streams while the attention is still under way; the heads' part comes last
// A layer of 97 MB (width 2048, 8 key heads, feed-forward 5504) took 14.6 + 11 + 4.6 us and three launches' starts, ends and gaps; the weights of its later phases stream while
// the earlier ones run here.  A token, LM head included, three launches a layer -> one: 24 layers behind 61 keys 724 -> 628 us, 12 behind 900 401 -> 351; 32 key heads 413 -> 370, 4 key heads and feed-forward
// 2048 372 -> 313; width 1024, 24 layers 500 -> 393, rotated and joined 549 -> 444 (width 2048, 12 layers 440 -> 386).  What bounds it is the chain q, k, v -> attention -> merge -> output beside the stream: 4 TB/s.
// Measured and not kept (8 key heads 592 us without the LM head, 32 335 of 12 layers at the time): one row per output wavefront, which leaves the producers half of the places (603 and 373; with 192
// producers 4 key heads took 1,202); gate rows ahead of the attention (615; 12 layers behind 900 keys 352 against 327); a delta rule's taps, ranks and vectors asked for ahead of the wait (no difference); the first count on 8 or 16 lines that all heads' workgroups poll, a hop less, in place of 64 copies (660, 635: 130 pollers on
// a line hold up the stream); no pauses between the lots of an output row, longer ones, and no wave priority: 0 to 2 % either way; three workgroups a unit at width 1024 in place of two: 0 to 2 % slower.
// The same for routed experts (a role that waits for the router's logits, chooses and streams the gate and up rows; output workgroups that choose too and ask for the chosen down rows)
// took 33.3 to 34.3 us a layer with 8 of 64 experts of 704 where the three launches take 32.1: the choice and the two streams behind it follow each other all the same.  Front rows spread evenly over the
// producers, on one producer a unit, or output workgroups that start 1.3 to 5 us late: 0 to 3 % slower.
// Progress: producers never wait and come first in the grid, so on every die they have their places before any workgroup that waits; the
// attention's workgroups wait for producers, the output's for both, in the grid's order (a merge also waits for the gate: producers again).  Workgroups of several launches could all the same fill the dies
// with some that wait for another die's: calls take their places beforehand (wait_places.hpp) and run in three launches where there are
// none.  Launches that nobody counts together, of several processes, are not kept apart so: each may hold the place that another's producers or heads need, and their
// waits then run out.  Their sessions ask for three launches (moon_text_set_decode_mode).  Every wait is bounded.
// Exchanged vectors are written through to memory; the attention reads what it needs of the projections past the dies' caches, the output
// workgroups read the two long vectors through them (no line of either is read before its count is complete).
#include "decode_roles.hpp"
#include "kernel_args.hpp"
#include "launch_waits.hpp"
#include "whole_share.hpp"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int WHOLE_D = 64;      // padded head sizes
// Loads of a row of the dense activation's weights at most (10,240 columns: the layers of a joined list whose weights are in the feed-forward have 6,464 at
// width 2048; in three launches, as with 12 loads, half of such a list's layers were, and a token of 12 layers took 392 us in place of 355 at the time), ..
constexpr int WHOLE_GLU = 20;
constexpr int WHOLE_HELD = 12;   // .. and those of an output wavefront's first row that wait in registers
constexpr int WHOLE_ROWS = 2;    // rows of an output wavefront
constexpr int WHOLE_SLEEP = 6;   // units of 64 cycles between two lots of them
enum { WHOLE_FRONT, WHOLE_ACT, WHOLE_HEADS, WHOLE_COUNTS };
constexpr int WHOLE_COPIES_AT = 2 * WHOLE_LEAVES * LAYER_LINE; // behind the leaves of the first two

struct WholeArgs {
    DecodeProj p;
    DecodeMix m;
    DecodeOut o;
    int S, keys_max, n_prod, n_attn;
    int front16;              // rows of the 16-bit segment that the heads begin with; the gate's behind them come with the activation
    uint32_t *sync, *report;
    LaunchTargets at;         // what the leaves and the copies count to
};

__device__ __forceinline__ uint32_t *whole_copy(const WholeArgs &a, int which, int i) { return a.sync + WHOLE_COPIES_AT + (which * LAYER_COPIES + i) * LAYER_COPY_STRIDE; }

constexpr int WHOLE_ERROR_AT = WHOLE_COPIES_AT + WHOLE_COUNTS * LAYER_COPIES * LAYER_COPY_STRIDE; // in a line of its own
__device__ __forceinline__ uint32_t *whole_error(const WholeArgs &a) { return a.sync + WHOLE_ERROR_AT; }

struct Within {
    static constexpr bool SHARED = true;
    const WholeArgs &a;
    int *s_flag;
    __device__ __forceinline__ bool wait() const {
        return wait_reached(whole_copy(a, WHOLE_FRONT, blockIdx.x % LAYER_COPIES), a.at.reached[WHOLE_FRONT], whole_error(a), s_flag, a.report);
    }
    __device__ __forceinline__ bool wait_gate() const {
        return a.front16 == a.p.n16_used || wait_reached(whole_copy(a, WHOLE_ACT, blockIdx.x % LAYER_COPIES), a.at.reached[WHOLE_ACT], whole_error(a), s_flag, a.report);
    }
    __device__ __forceinline__ void done() const {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the heads are stored
        lds_barrier();
        if (threadIdx.x < LAYER_COPIES) __hip_atomic_fetch_add(whole_copy(a, WHOLE_HEADS, threadIdx.x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};

// This producer's rows of a phase are stored: counted on its leaf, and by the leaf's last one on every copy
__device__ __forceinline__ void whole_report(const WholeArgs &a, int phase) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    if (threadIdx.x >= 64) return;
    int full = 0;
    if (threadIdx.x == 0)
        full = __hip_atomic_fetch_add(a.sync + (phase * WHOLE_LEAVES + blockIdx.x % WHOLE_LEAVES) * LAYER_LINE, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1 == a.at.leaf[phase];
    if (__builtin_amdgcn_readfirstlane(full)) __hip_atomic_fetch_add(whole_copy(a, phase, threadIdx.x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int U> __device__ __forceinline__ void whole_producer(const WholeArgs &a, char *lds, float *s_red) {
    typedef bf16_t T;
    const DecodeProj &p = a.p;
    T *s_h = reinterpret_cast<T *>(lds);
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = a.n_prod * 4, gw = blockIdx.x * 4 + wave;
    const T *W = reinterpret_cast<const T *>(p.w1);
    const int pieces = p.dp / 8;
    const T *er = p.token ? reinterpret_cast<const T *>(p.embed) + size_t(p.token[0]) * p.dp : nullptr;
    NormRow<T, U / 2, true, true> norm;
    norm.request(p, er, tid);
    // pairs of rows (segments are padded).  The first phase: what the heads begin with, and the f32 rows; the second: gate rows, then a gate/up pair each,
    // its longer shares to the wavefronts that had the shorter ones
    const int g16 = (a.front16 + 1) / 2, later = (p.n16_used - a.front16 + 1) / 2;
    int g, g_end, i, i_end;
    share(g16 + (p.n32_used + 1) / 2, waves, gw, g, g_end);
    share(later + p.ff, waves, waves - 1 - gw, i, i_end);
    RowDots<T, 2, U> dots;
    const T *rows[2];
    auto request = [&](int row, int apart) {
        rows[0] = W + size_t(row) * p.dp;
        rows[1] = rows[0] + size_t(apart) * p.dp;
        dots.request(rows, 0, pieces, lane);
    };
    auto front = [&](int g) { request(g < g16 ? 2 * g : p.n16 + 2 * (g - g16), 1); };
    auto second = [&](int i) { i < later ? request(a.front16 + 2 * i, 1) : request(p.n32 + pair_row(i - later, 0), 32); };
    if (g < g_end) front(g);
    norm.finish(p, er, blockIdx.x == 0, s_h, s_red, tid);
    lds_barrier();
    lm_u32x4 x[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const int at = u * 64 + lane;
        x[u] = lm_u32x4{0, 0, 0, 0};
        if (at < pieces) x[u] = *reinterpret_cast<const lm_u32x4 *>(s_h + at * 8);
    }
    float acc[2];
    auto sums = [&]() {
        acc[0] = acc[1] = 0.0f;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int j = 0; j < 2; j++) acc[j] = dot_piece<T>(dots.w[j][u], x[u], acc[j]);
    };
    auto store = [&](float *to) {
        if (lane < 2) st_f<true>(to + lane, lane ? acc[1] : acc[0]);
    };
    for (; g < g_end; g++) {
        sums();
        if (g + 1 < g_end) front(g + 1);
        acc[0] = wave_sum(acc[0]);
        acc[1] = wave_sum(acc[1]);
        store(g < g16 ? p.proj + 2 * g : p.logits + 2 * (g - g16));
    }
    whole_report(a, WHOLE_FRONT);
    if (!(later + p.ff)) return;
    if (i < i_end) second(i);
    for (; i < i_end; i++) {
        sums();
        if (i + 1 < i_end) second(i + 1);
        acc[0] = wave_sum(acc[0]);
        acc[1] = wave_sum(acc[1]);
        if (i < later) store(p.proj + a.front16 + 2 * i);
        else if (lane == 0) st_t<true>(reinterpret_cast<T *>(p.glu) + i - later, (T)(lm_silu(acc[0]) * acc[1]));
    }
    whole_report(a, WHOLE_ACT);
}

// 16 bytes a lane of a stretch of `bytes`; zeros behind its end
enum { LOAD_DIE = 1, LOAD_STREAM = 2 }; // from the die's cache on; not to be kept
template <int HOW> __device__ __forceinline__ lm_u32x4 stretch_load(__amdgpu_buffer_rsrc_t r, int at, int base) {
    return __builtin_bit_cast(lm_u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, at, base, HOW));
}
__device__ __forceinline__ __amdgpu_buffer_rsrc_t stretch(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, bytes, 0x00020000);
}

// A row's sums are those of out_rows, addition for addition, so one launch and three give the same bits.  There four wavefronts take a quarter of a stretch's pieces
// each, lane l of one its pieces l, l + 64, ..  Here one wavefront takes all four, half a wavefront a quarter: lane 32 w + j of load c has piece 32 (c / 2) + j of quarter
// 2 (c % 2) + w, which is lane 32 (c / 2 % 2) + j there.  So a lane keeps four sums, element c % 4, and quarters_sum adds them up.
// A token takes 1 % longer than with whole KiB in any order (24 layers of width 2048, feed-forward 5504 598 us against 590, 12 of 32 key heads 335 against 333, width
// 1024 382 against 381).  Measured and not kept: loads of 64 pieces of one quarter (597, 340, 385), of 16 of each (599, 336, 400); whole KiB, their dots turned by
// ds_bpermute where a quarter ends (648, 360, 435) or through LDS (596, 338, 386).
constexpr int NOWHERE = 1 << 30; // no buffer is as long: loads zeros
struct Quarters {
    int pieces, mine, at; // of a quarter; this lane's first; its byte
    __device__ __forceinline__ Quarters(int bytes, int lane) : pieces(bytes / 64), mine(lane % 32), at((lane / 32 * (bytes / 64) + lane % 32) * 16) {}
    __device__ __forceinline__ bool any(int c) const { return c * 16 < pieces; } // (c even: loads c and c + 1)
    __device__ __forceinline__ int offset(int c) const { return c / 2 * 512 + c % 2 * 2 * pieces * 16; }
    __device__ __forceinline__ int piece(int c) const { return (at + offset(c)) / 16; }
    template <int HOW> __device__ __forceinline__ lm_u32x4 load(__amdgpu_buffer_rsrc_t r, int c) const { return stretch_load<HOW>(r, c / 2 * 32 + mine < pieces ? at : NOWHERE, offset(c)); }
};

// QW: loads of a row's part for the heads, of which the delta rule's come behind the attention's.  A wavefront owns WHOLE_ROWS rows: their parts for the
// heads and the beginning of the first one's for the dense activation (HOLD loads) are in registers by the time that the activation is there, the rest streams
// while the attention is still under way.  Where eight loads a row are for the heads, the second row's come behind the dense activation's: with both from the start, up to 24 registers lay in scratch (12
// layers of width 2048, joined and rotated in turn, 380 us a token in place of 358), or a unit held three workgroups in place of four (6 joined layers of 32 key heads behind 300 keys 261 in place of 207).
template <int QW, bool DELTA> __device__ __forceinline__ void whole_output(const WholeArgs &a, int wg, int n_wgs, char *lds, int *s_flag) {
    typedef bf16_t T;
    constexpr int R = WHOLE_ROWS, HOLD = QW > 4 ? 8 : WHOLE_HELD;
    const DecodeOut &o = a.o;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), first = wg * 4 + wave, b = blockIdx.x % LAYER_COPIES;
    const bool fresh = a.p.token || a.p.y; // a producer writes x in this launch
    const int n_h = o.k2 * 2, n_f = (o.k0 - o.k2) * 2; // bytes of a row's parts
    const Quarters h(n_h, lane), f(n_f, lane);
    auto row = [&](int r) { return first + r * n_wgs * 4; };
    // (rows behind the width are padding: there are dp, a multiple of 64)
    auto weights = [&](int r, int column, int bytes) { return stretch(reinterpret_cast<const T *>(o.w2) + size_t(row(r)) * o.k0 + column, bytes); };
    lm_u32x4 wh[R][QW], wf[HOLD];
    float old[R];
    const bool more = QW > 4 && h.pieces > 64; // than four loads (6 rotated layers of width 2048, 32 key heads, 300 keys 182 -> 176 us)
    auto heads_weights = [&](int r) {
        const auto w = weights(r, 0, n_h);
#pragma unroll
        for (int c = 0; c < QW; c++)
            if (c < 4 || more) wh[r][c] = h.load<LOAD_STREAM>(w, c);
    };
    constexpr int EARLY = QW > 4 ? 1 : R;
#pragma unroll
    for (int r = 0; r < R; r++) {
        old[r] = 0.0f;
        if (!fresh && !o.y && row(r) < o.width) old[r] = o.x[row(r)];
        if (r < EARLY) heads_weights(r);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    float dot_f[R] = {};
    if (n_f) {
        auto request = [&](__amdgpu_buffer_rsrc_t w, int base, int c) { // loads base + c .. base + c + 3
#pragma unroll
            for (int m = c; m < c + 4; m += 2)
                if (f.any(base + m)) {
                    wf[m] = f.load<LOAD_STREAM>(w, base + m);
                    wf[m + 1] = f.load<LOAD_STREAM>(w, base + m + 1);
                }
        };
        {
            const auto w = weights(0, o.k2, n_f);
#pragma unroll
            for (int c = 0; c < HOLD; c += 4) {
                request(w, 0, c);
                if (c + 4 < HOLD) {
                    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_sleep(WHOLE_SLEEP);
                }
            }
        }
        if (!wait_reached(whole_copy(a, WHOLE_ACT, b), a.at.reached[WHOLE_ACT], whole_error(a), s_flag, a.report)) return;
        const auto act = stretch(reinterpret_cast<const T *>(o.a) + o.k2, n_f);
        auto copy = [&](auto from, auto to) { // the vector as the lanes meet it, 4 KiB a step, all requested before any is waited for
            constexpr int FROM = decltype(from)::value, N = decltype(to)::value - FROM;
            lm_u32x4 v[N];
#pragma unroll
            for (int c = 0; c < N; c++) v[c] = f.load<LOAD_DIE>(act, (FROM + c) * 4 + wave);
#pragma unroll
            for (int c = 0; c < N; c++) reinterpret_cast<lm_u32x4 *>(lds)[(FROM + c) * 256 + tid] = v[c];
        };
        copy(std::integral_constant<int, 0>{}, std::integral_constant<int, WHOLE_HELD / 4>{});
        if (n_f > WHOLE_HELD * 1024) copy(std::integral_constant<int, WHOLE_HELD / 4>{}, std::integral_constant<int, WHOLE_GLU / 4>{});
        lds_barrier();
#pragma unroll
        for (int r = 0; r < R; r++) {
            const auto w = weights(r, o.k2, n_f);
            float part[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 1
            for (int base = 0; f.any(base); base += HOLD) {
#pragma unroll
                for (int c = 0; c < HOLD; c += 4)
                    if (r || base) request(w, base, c);
#pragma unroll
                for (int c = 0; c < HOLD; c += 2)
                    if (f.any(base + c))
#pragma unroll
                        for (int m = c; m < c + 2; m++) part[m % 4] += dot_piece<T>(wf[m], reinterpret_cast<const lm_u32x4 *>(lds)[(base + m) * 64 + lane], 0.0f);
            }
            dot_f[r] = quarters_sum(part, lane);
        }
    }
#pragma unroll
    for (int r = EARLY; r < R; r++) heads_weights(r);
    if (!wait_reached(whole_copy(a, WHOLE_HEADS, b), a.at.reached[WHOLE_HEADS], whole_error(a), s_flag, a.report)) return;
    const auto heads = stretch(o.a, n_h);
    lm_u32x4 xh[QW];
    if (fresh && !o.y)
#pragma unroll
        for (int r = 0; r < R; r++)
            if (row(r) < o.width) old[r] = ld_f<true>(o.x + row(r));
#pragma unroll
    for (int c = 0; c < QW; c++)
        if (c < 4 || more) xh[c] = h.load<LOAD_DIE>(heads, c);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const int n = row(r);
        float part[4] = {0.0f, 0.0f, 0.0f, 0.0f}, part_d[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < QW; c++)
            if (c < 4 || more) {
                const float d = dot_piece<T>(wh[r][c], xh[c], 0.0f);
                const bool delta = DELTA && h.piece(c) >= o.k1 / 8; // (no layer without a delta rule has columns there)
                part[c % 4] += delta ? 0.0f : d;
                if (DELTA) part_d[c % 4] += delta ? d : 0.0f;
            }
        const float dot = quarters_sum(part, lane), dot_d = DELTA ? quarters_sum(part_d, lane) : 0.0f;
        if (lane || n >= o.width) continue;
        if (o.y) {
            o.y[n] = dot;
            o.y[o.dp + n] = dot_d;
            o.y[2 * o.dp + n] = dot_f[r];
        } else o.x[n] = old[r] + (dot + dot_f[r]);
    }
}

template <int NH, int U, bool WHOLE>
__global__ __launch_bounds__(256, NH > 4 ? 3 : U > 2 || WHOLE ? 4 : 5) void decode_whole_kernel(WholeArgs) {
    const WholeArgs &a = fetch_arguments<WholeArgs>();
    extern __shared__ __attribute__((aligned(16))) char s_whole[];
    __shared__ float s_red[16];
    __shared__ int s_flag;
    const int b = blockIdx.x, n_delta = WHOLE ? a.m.dH : 0;
    if (b < a.n_prod) return whole_producer<U>(a, s_whole, s_red);
    int i = b - a.n_prod;
    if (i < a.n_attn + n_delta) {
        __builtin_amdgcn_s_setprio(3); // the chain that the launch waits for longest
        const Within meet{a, &s_flag};
        float *lds = reinterpret_cast<float *>(s_whole);
        if (i < a.n_attn) {
            const int n_hb = mix_head_blocks(a.m.H / a.m.G);
            return mix_attention<bf16_t, NH, WHOLE, false, WHOLE_D>(a.m, i / a.S / n_hb, i / a.S % n_hb, i % a.S, a.S, a.keys_max, lds, meet);
        }
        if (WHOLE) mix_delta<bf16_t, true>(a.m, i - a.n_attn, lds, meet);
        return;
    }
    whole_output<(WHOLE ? 2 * U : U), WHOLE>(a, i - a.n_attn - n_delta, gridDim.x - a.n_prod - a.n_attn - n_delta, s_whole, &s_flag);
}

typedef void (*WholeKernel)(WholeArgs);
template <int U, bool WHOLE> WholeKernel whole_kernel_of(int NH) {
    return NH == 1 ? decode_whole_kernel<1, U, WHOLE> : NH == 2 ? decode_whole_kernel<2, U, WHOLE> : NH == 4 ? decode_whole_kernel<4, U, WHOLE> : decode_whole_kernel<8, U, WHOLE>;
}

struct WholePlan {
    WholeKernel kern;
    int S, keys_max, n_prod, n_attn, merges, grid, waiting;
    size_t lds;
};
// A layer's launch with n_keys keys; false: not in one launch.  per_cu: workgroups that a compute unit holds (0: what launches with up to n_keys keys need at most).  No producers: three
// launches are faster.
bool whole_plan(moon_ctx *ctx, const DecodeProj &p, const DecodeMix &m, const DecodeOut &o, int n_keys, int per_cu, WholePlan *w) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256, U = p.dp <= 1024 ? 2 : 4;
    if (m.E || m.dimp != WHOLE_D || m.vdimp != WHOLE_D || p.width % 4 || p.dp > 2048 || (reinterpret_cast<uintptr_t>(p.x) & 15)) return false;
    if (o.k1 > 512 * U || o.k2 - o.k1 > 512 * U || o.k0 - o.k2 > 512 * WHOLE_GLU || (o.k0 > o.k2) != (p.ff > 0)) return false;
    if (m.dH && (m.ddimp > DELTA_ROWS * (256 / (m.dvdimp / 4)))) return false;
    const int per = m.H / m.G, wgs = m.G * mix_head_blocks(per), nh = std::min(per, MIX_HEADS), NH = nh <= 1 ? 1 : nh <= 2 ? 2 : nh <= 4 ? 4 : 8;
    w->S = mix_splits(n_keys, wgs, cus);
    w->keys_max = std::max(MIX_TARGET, per_cu ? mix_split_keys(n_keys, w->S) : mix_most_split_keys(n_keys, wgs, cus)); // (fewer keys: the LDS of so many all the same)
    w->lds = std::max({size_t(p.dp) * 2, mix_lds_floats(NH, WHOLE_D, WHOLE_D, w->keys_max) * sizeof(float), size_t(!p.ff ? 0 : o.k0 - o.k2 > 512 * WHOLE_HELD ? WHOLE_GLU * 1024 : WHOLE_HELD * 1024),
                       m.dH ? delta_lds_floats(m.ddimp, m.dvdimp, m.kd) * sizeof(float) : 0});
    if (w->lds > 60 * 1024 || size_t(NH) * w->S > mix_lds_floats(NH, WHOLE_D, WHOLE_D, w->keys_max) - 4 * NH - 8) return false;
    w->kern = mix_whole(m) ? (U == 2 ? whole_kernel_of<2, true>(NH) : whole_kernel_of<4, true>(NH)) : (U == 2 ? whole_kernel_of<2, false>(NH) : whole_kernel_of<4, false>(NH));
    w->n_attn = wgs * w->S;
    w->merges = wgs + m.dH;
    w->waiting = w->n_attn + m.dH + (o.width + 4 * WHOLE_ROWS - 1) / (4 * WHOLE_ROWS);
    w->n_prod = whole_producers({(p.n16_used + 1) / 2 + (p.n32_used + 1) / 2, p.ff, U == 2, w->waiting, per_cu, cus, w->keys_max});
    w->grid = w->n_prod + w->waiting;
    return size_t(w->n_attn) * MIX_HEADS * (WHOLE_D + 2) <= m.partial_floats;
}

} // namespace

size_t decode_whole_sync_words() { return WHOLE_ERROR_AT + 1; }

bool decode_whole_supported(moon_ctx *ctx, int dtype, const DecodeProj &p, const DecodeMix &m, const DecodeOut &o, size_t max_seq, int *per_cu, WaitNeed *need) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    WholePlan w;
    // (the splits never get fewer with more keys)
    if (dtype != MOON_DTYPE_BF16 || !max_seq || !whole_plan(ctx, p, m, o, mix_keys(m, max_seq - 1), 0, &w)) return false;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(per_cu, reinterpret_cast<const void *>(w.kern), 256, w.lds) != hipSuccess) return false;
    *need = {(w.waiting + 7) / 8, *per_cu * cus / 8};
    return need->waiting < need->places;
}

int launch_decode_whole(moon_ctx *ctx, const DecodeProj &p, const DecodeMix &m, const DecodeOut &o, int per_cu, WholeCounts *counts, bool *launched) {
    *launched = false;
    MOON_TRY(check_decode_mix(ctx, m));
    WholePlan w;
    if (!whole_plan(ctx, p, m, o, mix_keys(m, m.pos), per_cu, &w)) return moon_fail(ctx, MOON_EINVAL, "decode: a layer that does not run in one launch");
    if (!w.n_prod) return MOON_OK;
    const int front16 = m.gate && !m.dH ? m.og : p.n16_used; // (a delta rule's columns come behind the gate's)
    LaunchTargets next = counts->at;
    next.leaf[WHOLE_FRONT] += w.n_prod / WHOLE_LEAVES;
    next.reached[WHOLE_FRONT] += WHOLE_LEAVES;
    if (p.ff || front16 < p.n16_used) {
        next.leaf[WHOLE_ACT] += w.n_prod / WHOLE_LEAVES;
        next.reached[WHOLE_ACT] += WHOLE_LEAVES;
    }
    next.reached[WHOLE_HEADS] += w.merges;
    auto launch = [&]() -> int {
        hipLaunchKernelGGL(w.kern, dim3(w.grid), dim3(256), w.lds, ctx->stream, WholeArgs{p, m, o, w.S, w.keys_max, w.n_prod, w.n_attn, front16, counts->sync, counts->error, next});
        MOON_HIP(ctx, hipGetLastError());
        return MOON_OK;
    };
    auto clear = [&]() -> int {
        if (launch_fill_uniform_u32(ctx, counts->sync, decode_whole_sync_words(), 0, 0, 1) != MOON_OK) return MOON_EHIP;
        return hipStreamSynchronize(ctx->stream) == hipSuccess ? MOON_OK : MOON_EHIP;
    };
    MOON_TRY(launch_counted(&counts->at, next, counts->error, launch, clear));
    *launched = true;
    MOON_NOTE_KERNEL(ctx, "decode_whole_kernel %d splits of the keys", w.S);
    return MOON_OK;
}
