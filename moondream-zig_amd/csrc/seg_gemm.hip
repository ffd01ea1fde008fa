// Products of the layer-list decoders: C[M, N] = A . W^T with the columns in segments (16-bit, f32, gated pairs), rows gathered
// and grouped where a router asks for it.  bf16 runs on the matrix cores through the stream of tiles of gemm_stream.hpp; f32 is computed with f32 multiply-adds (no reduced-precision mode).
#include "gemm_block.hpp"
#include "gemm_stream.hpp"
#include "gemm_thin.hpp"
#include "layer_list.hpp"
#include "lm_types.hpp"
#include "seg_schedule.hpp"

#include <algorithm>
#include <atomic>

namespace {

static_assert(SEG_K_TILE == BK && SEG_TILE_COLUMNS == BN && SEG_MAX_SPLITS <= SEG_DIES, "what the schedule's estimate takes for granted");

struct TilePos {
    int m0, m_end, n0, group, split;
    bool lone; // of a list: the group has no other row tile
};
// A die's slot (seg_schedule.hpp) -> its tile; returns what seg_find does.
__device__ __forceinline__ int seg_tile(const SegGemm &p, const SegWalk &w, bool listed, int die, int slot, int tile_m, int tile_n, TilePos &t) {
    int tm, tn;
    if (listed) { // (scalar loads: a launch does not write its own list, and a vector load would wait for the copies in flight)
        typedef const __attribute__((address_space(4))) int *list_t;
        auto entry = [&](const int *list, int i) { return ((list_t)list)[i]; };
        if (const int r = seg_find_listed(w, entry(p.n_tiles, 0), die, slot, tm, tn); r <= 0) return r;
        t.split = 0;
        t.group = entry(p.tile_group, tm);
        t.m0 = entry(p.tile_row, tm);
        const int end = entry(p.tile_end, tm);
        t.m_end = min(t.m0 + tile_m, end);
        t.lone = end <= t.m0 + tile_m && (tm == 0 || entry(p.tile_group, tm - 1) != t.group);
    } else {
        if (const int r = seg_find(w, die, slot, tm, tn, t.split); r <= 0) return r;
        t.group = 0;
        t.m0 = tm * tile_m;
        t.m_end = min(t.m0 + tile_m, p.M);
    }
    t.n0 = tn * tile_n;
    return 1;
}

// Four consecutive columns of one row of a wavefront's 32-row blocks of accumulators: piece i (of eight) of lane l has row row(l, i) and
// columns 4 column4(l, i) .. + 3; piece i < 4 holds columns below 32, piece i + 4 those 32 behind it.
struct Pieces32 { // 32 x 32 products (gemm_stream.hpp): acc[32 columns][32 rows]
    static __device__ __forceinline__ int row(int lane, int) { return lane & 31; }
    static __device__ __forceinline__ int column4(int lane, int i) { return 2 * i + (lane >> 5); }
    template <int MI> static __device__ __forceinline__ float4_t get(const float16_t (&acc)[2][MI], int mi, int i) {
        const float16_t &a = acc[i >> 2][mi];
        const int q = i & 3;
        return float4_t{a[4 * q], a[4 * q + 1], a[4 * q + 2], a[4 * q + 3]};
    }
};
struct Pieces16 { // 16 x 16 products (gemm_block.hpp): acc[16 columns][16 rows]
    static __device__ __forceinline__ int row(int lane, int i) { return 16 * (i & 1) + (lane & 15); }
    static __device__ __forceinline__ int column4(int lane, int i) { return 4 * (i >> 1) + (lane >> 4); }
    template <int M2> static __device__ __forceinline__ float4_t get(const float4_t (&acc)[4][M2], int mi, int i) { return acc[i >> 1][2 * mi + (i & 1)]; }
};

// A multiplier wavefront's accumulators -> their segment, 32 rows at a time through its 4 KiB of LDS so that the stores are whole
// lines: rows of 128 (gated pairs: 64) bytes, the 16-byte granules XOR-swizzled by row.
typedef bf16_t bf16x4_t __attribute__((ext_vector_type(4)));
template <class P, int MI, class Acc>
__device__ __forceinline__ void seg_store(const SegGemm &p, const Acc &acc, const TilePos &t, int wm, int wn, int lane, char *scratch) {
    asm volatile("" : "+v"(lane)); // (per tile: kept over the products, a lane's addresses would not fit the registers, and scratch loads held up each tile by 1 us)
    const int n = t.n0 + wn * 64;
    if (n >= p.N) return;
    const int m_wave = t.m0 + wm * 32 * MI, row8 = lane >> 3, g8 = lane & 7;
    // the wavefront reads back what its own lanes wrote; its next writes come behind those reads, LDS serves it in order
    auto written = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); };
    auto fence = [] { asm volatile("" ::: "memory"); };
    if (n < p.n16) {
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float4_t a = P::get(acc, mi, i);
                const int r = P::row(lane, i), c = P::column4(lane, i);
                bf16x4_t o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (bf16_t)a[e];
                *reinterpret_cast<bf16x4_t *>(scratch + r * 128 + ((c >> 1) ^ (r & 7)) * 16 + (c & 1) * 8) = o;
            }
            written();
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int ml = r * 8 + row8, m = m_wave + mi * 32 + ml;
                const lm_u32x4 v = *reinterpret_cast<const lm_u32x4 *>(scratch + ml * 128 + (g8 ^ (ml & 7)) * 16);
                if (m < t.m_end) *reinterpret_cast<lm_u32x4 *>(reinterpret_cast<bf16_t *>(p.c16) + size_t(m) * p.ld16 + n + g8 * 8) = v;
            }
            fence();
        }
    } else if (n < p.n32) {
        float *dst = p.c32 + size_t(t.split) * p.M * p.ld32 + (n - p.n16) + g8 * 4;
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++) {
#pragma unroll
                for (int i = 4 * ni; i < 4 * ni + 4; i++) {
                    float4_t o = P::get(acc, mi, i);
                    const int r = P::row(lane, i), c = P::column4(lane, i) & 7;
                    if (p.softcap > 0.0f) o = float4_t{lm_softcap(o[0], p.softcap), lm_softcap(o[1], p.softcap), lm_softcap(o[2], p.softcap), lm_softcap(o[3], p.softcap)};
                    *reinterpret_cast<float4_t *>(scratch + r * 128 + (c ^ (r & 7)) * 16) = o;
                }
                written();
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int ml = r * 8 + row8, m = m_wave + mi * 32 + ml;
                    const float4_t v = *reinterpret_cast<const float4_t *>(scratch + ml * 128 + (g8 ^ (ml & 7)) * 16);
                    if (m < t.m_end) *reinterpret_cast<float4_t *>(dst + size_t(m) * p.ld32 + ni * 32) = v;
                }
                fence();
            }
    } else {
        const int row4 = lane >> 2, g4 = lane & 3;
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float4_t gate = P::get(acc, mi, i), up = P::get(acc, mi, i + 4);
                const int r = P::row(lane, i), c = P::column4(lane, i);
                bf16x4_t o;
#pragma unroll
                for (int e = 0; e < 4; e++) o[e] = (bf16_t)(lm_silu(gate[e]) * up[e]);
                *reinterpret_cast<bf16x4_t *>(scratch + r * 64 + ((c >> 1) ^ ((r >> 1) & 3)) * 16 + (c & 1) * 8) = o;
            }
            written();
#pragma unroll
            for (int r = 0; r < 2; r++) {
                const int ml = r * 16 + row4, m = m_wave + mi * 32 + ml;
                const lm_u32x4 v = *reinterpret_cast<const lm_u32x4 *>(scratch + ml * 64 + (g4 ^ ((ml >> 1) & 3)) * 16);
                if (m < t.m_end) *reinterpret_cast<lm_u32x4 *>(reinterpret_cast<bf16_t *>(p.glu) + size_t(m) * p.ldg + (n - p.n32) / 2 + g4 * 8) = v;
            }
            fence();
        }
    }
}

// LISTED: row tiles from a list.  A kernel of its own: with both ways to a tile in one, the plain products of a prompt of 768 rows lost
// 0.4 to 0.8 us each.
template <int MI, bool LISTED>
__global__ __launch_bounds__(DMA_THREADS) void seg_gemm_bf16_kernel(SegGemm p, SegWalk w) {
    extern __shared__ __attribute__((aligned(16))) half_t lds_stream[]; // (the tile product addresses LDS from 0: nothing static beside it)
    using S = Stream<MI>;
    const int lane = threadIdx.x & 63, role_wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    int round = 0;
    auto next = [&](TilePos &t) { // (both roles walk the same tiles)
        for (;;) {
            const int r = seg_tile(p, w, LISTED, blockIdx.x % SEG_DIES, seg_slot(w.longest_first, blockIdx.x / SEG_DIES, gridDim.x / SEG_DIES, round++), S::ROWS, BN, t);
            if (r != 0) return r > 0;
        }
    };
    if (threadIdx.x >= 256) {
        stream_load<MI, LISTED, TilePos>(lds_stream, role_wave, next, [&](const TilePos &t, StreamSource<MI> &s) {
            // (the launcher has checked that both operands fit a descriptor)
            const bf16_t *weights = reinterpret_cast<const bf16_t *>(p.W) + size_t(t.group) * p.w_group;
            s.a = __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p.A), 0, p.a_rows * p.lda * 2, 0x00020000);
            s.w = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t *>(weights), 0, p.N * p.K * 2, 0x00020000);
#pragma unroll
            for (int j = 0; j < 2 * MI; j++) {
                const int r = stream_row_a(MI, role_wave, j, lane), m = min(t.m0 + r, t.m_end - 1);
                s.off_a[j] = ((p.rows ? (int)p.rows[m] : m) * p.lda + swz(r, lane & 7) * 8) * 2;
            }
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int r = 32 * role_wave + 8 * j + (lane >> 3);
                s.off_w[j] = (min(t.n0 + r, p.N - 1) * p.K + swz(r, lane & 7) * 8) * 2;
            }
            s.k = p.kb[t.split] * 2;
            s.n_ktiles = (p.kb[t.split + 1] - p.kb[t.split]) / BK;
            // A group's only row tile: 64 experts of 704, 8 a row, width 2048, us a layer with all copies ordinary, all non-temporal, and by this rule: 61 rows 158, 143, 143, 768 rows 234, 248, 225,
            // 1025 rows 270, not tried, 261 with random choices; 768 rows over the experts evenly 229, 218, 218.  A second row tile finds what the first one left in the L2.
            s.once = LISTED && t.lone;
        });
        return;
    }
    const int wm = role_wave & 1, wn = role_wave >> 1;
    char *scratch = reinterpret_cast<char *>(lds_stream) + S::STAGES * S::STAGE_BYTES + role_wave * STREAM_SCRATCH_BYTES;
    stream_multiply<MfmaBf16, MI, TilePos>(wm, wn, lane, next, [&](const TilePos &t) { return (p.kb[t.split + 1] - p.kb[t.split]) / BK; },
                                           [&](const TilePos &t, const float16_t (&acc)[2][MI]) { seg_store<Pieces32, MI>(p, acc, t, wm, wn, lane, scratch); });
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t seg_rows(const void *from, int first, int n, int pitch) { // n rows (the launcher has checked that both operands fit a descriptor)
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<const char *>(from)) + size_t(first) * pitch, 0, n * pitch, 0x00020000);
}

// The same in tiles of 64 MI x 256 (gemm_block.hpp); no gathered rows and no list.
template <int MI>
__global__ __launch_bounds__(DMA_THREADS) void seg_gemm_bf16_block_kernel(SegGemm p, SegWalk w) {
    extern __shared__ __attribute__((aligned(16))) half_t lds_stream[];
    using S = Block<MI>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    auto next = [&](TilePos &t, int &round) {
        for (;;) {
            const int r = seg_tile(p, w, false, blockIdx.x % SEG_DIES, seg_slot(w.longest_first, blockIdx.x / SEG_DIES, gridDim.x / SEG_DIES, round++), S::ROWS, S::COLUMNS, t);
            if (r != 0) return r > 0;
        }
    };
    auto ktiles = [&](const TilePos &t) { return (p.kb[t.split + 1] - p.kb[t.split]) / BK; };
    auto open = [&](const TilePos &t, BlockSource &s) {
        s.a = seg_rows(p.A, t.m0, t.m_end - t.m0, p.lda * 2);
        s.w = seg_rows(p.W, t.n0, min(p.N - t.n0, S::COLUMNS), p.K * 2);
        s.k = p.kb[t.split] * 2;
        s.n_ktiles = ktiles(t);
    };
    char *scratch = reinterpret_cast<char *>(lds_stream) + 2 * S::STAGE_BYTES + wave * S::SCRATCH_BYTES;
    block_stream<BlockBf16, MI, TilePos>(lds_stream, wave, lane, p.lda * 2, p.K * 2, next, open, ktiles,
                                         [&](const TilePos &t, int wm, int wn, const float4_t (&acc)[4][2 * MI]) { seg_store<Pieces16, MI>(p, acc, t, wm, wn, lane, scratch); });
}

// The same for few rows in tiles of 128 x 64 (gemm_thin.hpp); no gathered rows and no list.
__global__ __launch_bounds__(DMA_THREADS) void seg_gemm_bf16_thin_kernel(SegGemm p, SegWalk w) {
    extern __shared__ __attribute__((aligned(16))) half_t lds_stream[];
    using S = Thin;
    const int lane = threadIdx.x & 63, role_wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3);
    int round = 0;
    auto next = [&](TilePos &t) {
        for (;;) {
            const int r = seg_tile(p, w, false, blockIdx.x % SEG_DIES, seg_slot(w.longest_first, blockIdx.x / SEG_DIES, gridDim.x / SEG_DIES, round++), S::ROWS, S::COLUMNS, t);
            if (r != 0) return r > 0;
        }
    };
    auto ktiles = [&](const TilePos &t) { return (p.kb[t.split + 1] - p.kb[t.split]) / BK; };
    if (threadIdx.x >= 256) {
        thin_load<TilePos>(lds_stream, role_wave, lane, next, [&](const TilePos &t, BlockSource &s, int &pitch_a, int &pitch_w) {
            pitch_a = p.lda * 2;
            pitch_w = p.K * 2;
            s.a = seg_rows(p.A, t.m0, t.m_end - t.m0, pitch_a);
            s.w = seg_rows(p.W, t.n0, min(p.N - t.n0, S::COLUMNS), pitch_w);
            s.k = p.kb[t.split] * 2;
            s.n_ktiles = ktiles(t);
        });
        return;
    }
    char *scratch = reinterpret_cast<char *>(lds_stream) + S::STAGES * S::STAGE_BYTES + role_wave * S::SCRATCH_BYTES;
    thin_multiply<BlockBf16, TilePos>(role_wave, lane, next, ktiles, [&](const TilePos &t, const float4_t (&acc)[4][2]) { seg_store<Pieces16, 1>(p, acc, t, role_wave, 0, lane, scratch); });
}

// f32: 64 x 64 tile, a thread owns rows ty, ty + 16, .. and columns tx, tx + 16, tx + 32, tx + 48 (so a gate column and its up
// column are in one thread).  Tile lists are 128 rows high: two passes over m.
constexpr int F32_K = 16;
__global__ __launch_bounds__(256) void seg_gemm_f32_kernel(SegGemm p, SegWalk w) {
    __shared__ float sa[F32_K][64 + 4], sw[F32_K][64 + 4];
    TilePos t;
    if (seg_tile(p, w, p.tile_group != nullptr, blockIdx.x % SEG_DIES, blockIdx.x / SEG_DIES, SEG_TILE_ROWS, 64, t) <= 0) return;
    const int k_begin = p.kb[t.split], k_end = p.kb[t.split + 1];
    const int tid = threadIdx.x, tx = tid & 15, ty = tid >> 4, lr = tid >> 2, lk = (tid & 3) * 4;
    const float *A = reinterpret_cast<const float *>(p.A), *W = reinterpret_cast<const float *>(p.W) + size_t(t.group) * p.w_group;
    for (int mb = t.m0; mb < t.m_end; mb += 64) {
        float acc[4][4] = {};
        const int m_src = min(mb + lr, t.m_end - 1);
        const float *arow = A + size_t(p.rows ? (int)p.rows[m_src] : m_src) * p.lda, *wrow = W + size_t(t.n0 + lr) * p.K;
        for (int k = k_begin; k < k_end; k += F32_K) {
            const float4 a = *reinterpret_cast<const float4 *>(arow + k + lk), b = *reinterpret_cast<const float4 *>(wrow + k + lk);
            __syncthreads();
            sa[lk][lr] = a.x; sa[lk + 1][lr] = a.y; sa[lk + 2][lr] = a.z; sa[lk + 3][lr] = a.w;
            sw[lk][lr] = b.x; sw[lk + 1][lr] = b.y; sw[lk + 2][lr] = b.z; sw[lk + 3][lr] = b.w;
            __syncthreads();
#pragma unroll
            for (int kk = 0; kk < F32_K; kk++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int j = 0; j < 4; j++) acc[i][j] = fmaf(sa[kk][ty + 16 * i], sw[kk][tx + 16 * j], acc[i][j]);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int m = mb + ty + 16 * i;
            if (m >= t.m_end) continue;
            if (t.n0 < p.n16)
                for (int j = 0; j < 4; j++) reinterpret_cast<float *>(p.c16)[size_t(m) * p.ld16 + t.n0 + tx + 16 * j] = acc[i][j];
            else if (t.n0 < p.n32)
                for (int j = 0; j < 4; j++) p.c32[(size_t(t.split) * p.M + m) * p.ld32 + t.n0 - p.n16 + tx + 16 * j] = p.softcap > 0.0f ? lm_softcap(acc[i][j], p.softcap) : acc[i][j];
            else
                for (int j = 0; j < 2; j++)
                    reinterpret_cast<float *>(p.glu)[size_t(m) * p.ldg + (t.n0 - p.n32) / 2 + tx + 16 * j] = lm_silu(acc[i][j]) * acc[i][j + 2];
        }
        __syncthreads();
    }
}

} // namespace

// The tile for a product whose ranges are set: its height in 64 rows, + SEG_BLOCK where it is 256 columns wide, + SEG_THIN where it is 64.  Plain f32 results keep the
// narrow tiles: wide ones need more ranges of k to fill the chip, and each range's sums cost a slab (1920 x 2048 x 7552: 58 us in two ranges of 256 x 128, 57 in
// three of 192 x 256, whose third slab costs 3 us in row_finish; 768 rows 31 in four ranges, 32 in eight).
static int seg_choose(moon_ctx *ctx, const SegGemm &p) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    int best = 2;
    double t = 1e30;
    for (int mi = 2; mi <= 4; mi++)
        if (const double e = seg_estimate(cus, mi, p.M, p.N, p.kb, p.splits, p.longest_first); e < t) {
            t = e;
            best = mi;
        }
    if (p.tile_group || p.rows) return best;
    if (const double e = seg_thin_estimate(cus, p.M, p.N, p.kb, p.splits, p.longest_first); e < t) {
        t = e;
        best = SEG_THIN + 2;
    }
    if (p.splits > 1 || (!p.n16 && p.n32 == p.N)) return best;
    for (int mi = 3; mi <= 4; mi++)
        if (const double e = seg_block_estimate(cus, mi, p.M, p.N, p.K); e < t) {
            t = e;
            best = SEG_BLOCK + mi;
        }
    return best;
}

static void even_ranges(int K, int splits, int *kb) {
    for (int s = 0, per = (int)pad_to((K + splits - 1) / splits, BK); s <= splits; s++) kb[s] = std::min(K, s * per);
}

// f32: its multiply-adds take ten times as long as a range's slab, and ranges even out what the units get, so as many as there is room
// for.  Two layers of a prompt, us, with the bf16 kernel's estimate -> so: width 1024, feed-forward 2752, 500 rows 928 -> 904, 640 rows
// 1238 -> 1192; 2048, 5504: 640 rows 3170 -> 3060, 1301 rows 7800 -> 7760.
int seg_gemm_splits(moon_ctx *ctx, int dtype, size_t M, size_t N, size_t K, size_t max_rows) {
    const int cus = ctx->cu_count > 0 ? ctx->cu_count : 256;
    const double slab = (double)M * N * 8 / 4.5e6; // another range's sums, written and read, us at 4.5 TB/s
    int best = 1;
    double t = 1e30;
    for (int splits = 1; splits <= SEG_MAX_SPLITS && (splits == 1 || (K / splits >= 512 && splits * M <= max_rows)); splits++) {
        int kb[SEG_MAX_SPLITS + 1];
        even_ranges((int)K, splits, kb);
        if (kb[splits - 1] >= kb[splits]) continue;
        if (dtype != MOON_DTYPE_BF16) {
            best = splits;
            continue;
        }
        for (int mi = 2; mi <= 4; mi++)
            if (const double e = seg_estimate(cus, mi, (int)M, (int)N, kb, splits, false) + (splits - 1) * slab; e < t) {
                t = e;
                best = splits;
            }
        if (const double e = seg_thin_estimate(cus, (int)M, (int)N, kb, splits, false) + (splits - 1) * slab; e < t) {
            t = e;
            best = splits;
        }
    }
    return best;
}

int launch_seg_gemm(moon_ctx *ctx, int dtype, SegGemm p) {
    if (p.M <= 0 || p.N <= 0) return MOON_OK;
    if (p.N % 64 || p.K % 64 || p.K <= 0 || p.n16 % 64 || p.n32 % 64 || p.n16 > p.n32 || p.n32 > p.N || p.lda < p.K)
        return moon_fail(ctx, MOON_EINVAL_DIM, "segmented product: sizes must be padded to 64 (N %d, K %d, segments %d %d)", p.N, p.K, p.n16, p.n32);
    if (p.splits < 1) p.splits = 1;
    if (p.splits > 1 && (p.n16 || p.n32 != p.N || p.tile_group)) return moon_fail(ctx, MOON_EINVAL, "segmented product: only a plain f32 result splits k");
    if (p.splits > 1 && (long long)p.splits * p.M > p.c32_rows) return moon_fail(ctx, MOON_EINVAL, "segmented product: %d slabs of %d rows, room for %d", p.splits, p.M, p.c32_rows);
    if (p.splits > SEG_MAX_SPLITS) return moon_fail(ctx, MOON_EINVAL, "segmented product: %d k splits", p.splits);
    if (!p.kb[p.splits]) even_ranges(p.K, p.splits, p.kb);
    for (int s = 0; s < p.splits; s++)
        if (p.kb[0] || p.kb[s] >= p.kb[s + 1] || p.kb[s + 1] % BK || p.kb[p.splits] != p.K)
            return moon_fail(ctx, MOON_EINVAL, "segmented product: %d k splits leave one empty", p.splits);
    int rows = 64, columns = 64;
    if (dtype == MOON_DTYPE_BF16) {
        const size_t lim = (size_t(1) << 31) - 4096;
        if (size_t(p.a_rows) * p.lda * 2 >= lim || size_t(p.N) * p.K * 2 >= lim)
            return moon_fail(ctx, MOON_EINVAL_DIM, "segmented product: an operand of 2 GiB or more");
        const int tile = p.tile_group ? 2 : p.tile ? p.tile : seg_choose(ctx, p), mi = tile % SEG_BLOCK;
        if (tile != SEG_THIN + 2 && (mi < (tile > SEG_BLOCK ? 3 : 2) || mi > 4 || tile > SEG_BLOCK + 4)) return moon_fail(ctx, MOON_EINVAL, "segmented product: tile form %d", tile);
        if (tile > 4 && p.rows) return moon_fail(ctx, MOON_EINVAL, "segmented product: tile form %d", tile);
        columns = tile > SEG_THIN ? Thin::COLUMNS : tile > SEG_BLOCK ? 256 : BN;
        rows = 64 * mi;
        auto go = [&](auto kern, size_t lds, std::atomic<bool> (&attr_set)[64]) -> int {
            const int dev = ctx->device >= 0 && ctx->device < 64 ? ctx->device : -1;
            if (dev < 0 || !attr_set[dev].load()) {
                MOON_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
                if (dev >= 0) attr_set[dev].store(true);
            }
            const int cus = std::max(SEG_DIES, (ctx->cu_count > 0 ? ctx->cu_count : 256) / SEG_DIES * SEG_DIES);
            const int tiles_n = (p.N + columns - 1) / columns;
            const SegWalk w = p.tile_group ? seg_walk_listed(p.max_tiles, tiles_n) : seg_walk((p.M + rows - 1) / rows, tiles_n, false, p.kb, p.splits, p.longest_first);
            hipLaunchKernelGGL(kern, dim3((unsigned)seg_workgroups(w, cus)), dim3(DMA_THREADS), lds, ctx->stream, p, w);
            return MOON_OK;
        };
        static std::atomic<bool> set_listed[64], set2[64], set3[64], set4[64], wide3[64], wide4[64], thin2[64];
        if (p.tile_group) MOON_TRY(go(seg_gemm_bf16_kernel<2, true>, Stream<2>::LDS_BYTES, set_listed));
        else if (tile == SEG_THIN + 2) MOON_TRY(go(seg_gemm_bf16_thin_kernel, Thin::LDS_BYTES, thin2));
        else if (tile == SEG_BLOCK + 4) MOON_TRY(go(seg_gemm_bf16_block_kernel<4>, Block<4>::LDS_BYTES, wide4));
        else if (tile == SEG_BLOCK + 3) MOON_TRY(go(seg_gemm_bf16_block_kernel<3>, Block<3>::LDS_BYTES, wide3));
        else if (mi == 4) MOON_TRY(go(seg_gemm_bf16_kernel<4, false>, Stream<4>::LDS_BYTES, set4));
        else if (mi == 3) MOON_TRY(go(seg_gemm_bf16_kernel<3, false>, Stream<3>::LDS_BYTES, set3));
        else MOON_TRY(go(seg_gemm_bf16_kernel<2, false>, Stream<2>::LDS_BYTES, set2));
    } else {
        const SegWalk w = p.tile_group ? seg_walk_listed(p.max_tiles, p.N / 64) : seg_walk((p.M + SEG_TILE_ROWS - 1) / SEG_TILE_ROWS, p.N / 64, true, p.kb, p.splits, p.longest_first);
        hipLaunchKernelGGL(seg_gemm_f32_kernel, dim3((unsigned)(SEG_DIES * w.slots)), dim3(256), 0, ctx->stream, p, w);
    }
    MOON_HIP(ctx, hipGetLastError());
    MOON_NOTE_KERNEL(ctx, "%s %d rows a tile, k split %d", dtype != MOON_DTYPE_BF16 ? "seg_gemm_f32_kernel" : columns == BN ? "seg_gemm_bf16_kernel" : columns > BN ? "seg_gemm_bf16_block_kernel" : "seg_gemm_bf16_thin_kernel", rows, p.splits);
    return MOON_OK;
}
