// The tile product as a stream of tiles (gemm_stream.hpp) in tiles of 64 MI (m) x 256 (n) x 64 (k), MI = 3 or 4: eight wavefronts, two per
// SIMD, that all copy and all multiply, 32 MI (m) x 64 (n) each.
// A tile twice as wide as gemm_stream.hpp's needs two thirds (MI = 4) of its copies per product, 512 rows a k-tile where two of those copy 768, and as many operand reads from LDS; what one
// wavefront of a SIMD waits for the other one covers.  A k-tile at MI = 4 takes 1.37 us with every unit busy (1.57 PFLOP/s) where two of gemm_stream.hpp's take 1.59; its copies alone 0.9,
// without copies 1.13.  What bounds it: the products, at the clock that they leave (1.7 to 1.8 of 2.4 GHz), and cycles without one; the matrix cores are busy in 78 % of the cycles at 4096^3 and in 70 % at
// 1920 x 16128 x 2048.  On random operands nothing but 16 x 16 x 32 products reaches 1.99 PFLOP/s in f16 and 2.08 in bf16 (a k-tile in 1.03 to 1.08 us), of 32 x 32 x 16 ones 1.72 and 1.87 (both 2.4 and
// more on zeros; sums are read and written half as often, and come out with the same bits): hence these.
//   1920 x 16128 x 2048 (gated, bf16) among a model's launches, weights from HBM: 136 us in narrow tiles, 117 so (113 with lm_silu's shorter form; other boxes to 107); 768 rows 58, 51 (47); 1301 x 16832 x 2048 by itself 103 -> 88.
// LDS holds two k-tiles, 56 or 64 KiB each, and 4 KiB of each wavefront for its epilogue.  Two whole stages would leave one k-tile's time for a copy (1.2 us at this load); so
// a wavefront's products go by quarters, first half of its rows with the first half of its columns, then first x second, second x second,
// second x first, an operand half stays in registers for the two quarters that it has, and its place in LDS is free for the k-tile after
// next as soon as it has been read:
//   barrier X, before first x second: A's first half and W have been read by all, their copies for k-tile + 2 may start; A's second half has landed.
//   barrier Y, before second x first: A's second half likewise; the next k-tile's first half of A and its W have landed.
// so a copy has one and a half k-tiles, and operand reads run a quarter ahead of their products.
#pragma once
#include "gemm_dma.hpp"

#include <type_traits>

namespace {

template <int MI> struct Block {
    static_assert(MI == 3 || MI == 4, "the second half of a wavefront's rows is not empty, the first has two blocks");
    static constexpr int ROWS = 64 * MI, COLUMNS = 256;
    static constexpr unsigned A_BYTES = ROWS * BK * 2, STAGE_BYTES = A_BYTES + COLUMNS * BK * 2; // [rows of A][rows of W]
    static constexpr int SCRATCH_BYTES = 4096; // per wavefront
    static constexpr size_t LDS_BYTES = 2 * size_t(STAGE_BYTES) + 8 * SCRATCH_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

struct BlockBf16 {
    static __device__ __forceinline__ float4_t mul(const half8_t &a, const half8_t &b, const float4_t &c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    }
};
struct BlockF16 {
    static __device__ __forceinline__ float4_t mul(const half8_t &a, const half8_t &b, const float4_t &c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
struct BlockSource {
    __amdgpu_buffer_rsrc_t a, w;
    int k, n_ktiles; // bytes of the next k-tile, how many are left
};

// What a wavefront does for all of the workgroup's tiles.  next(t, round): the next tile, false behind the last.  open(t, s): its operands as
// buffers that start at its first rows and end behind its last (copies past them bring zeros).  ktiles(t): its k-tiles (>= 1).
// store(t, wm, wn, acc): acc[16 columns][16 rows] of the wavefront's place (wm, wn); lane l, element e is column 4 (l / 16) + e, row l % 16.
template <class Op, int MI, class Tile, class Next, class Open, class KTiles, class Store>
__device__ __forceinline__ void block_stream(half_t *lds, int wave, int lane, int pitch_a, int pitch_w, Next next, Open open, KTiles ktiles, Store store) {
    using S = Block<MI>;
    constexpr int H0 = 2, H1 = MI - 2; // 32-row blocks of the first and the second half of a wavefront's rows
    const int wm = wave >> 2, wn = wave & 3;
    // ---- copies, eight rows each: H0 + H1 of A, 2 + 2 of W.  The first halves of both row groups' rows of A lie in 64 H0 rows
    const int granule = ((lane & 7) ^ ((wave & 1) * 4 + (lane >> 4))) * 16;
    auto row_a = [&](int half, int u) { // of this wavefront's eight
        const int at = 8 * (wave + 8 * u), blocks = half ? H1 : H0, group = at / (32 * blocks);
        return group * 32 * MI + (half ? 32 * H0 : 0) + at % (32 * blocks);
    };
    auto row_w = [&](int half, int u) { return (wave >> 2) * 64 + (wave & 3) * 8 + 128 * u + 32 * half; };
    const int lane_a = (lane >> 3) * pitch_a + granule, lane_w = (lane >> 3) * pitch_w + granule;
    Tile t, ahead;
    BlockSource s;
    int issue_round = 0;
    if (!next(t, issue_round)) return;
    int read_round = issue_round; // (a first slot may be empty: the first tile need not be the first round's)
    ahead = t;
    open(ahead, s);
    unsigned to = 0; // stage of the k-tile being copied
    auto copy_a = [&](int half, int u) {
        const int r = row_a(half, u);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s.a, (__attribute__((address_space(3))) void *)(reinterpret_cast<char *>(lds) + to + r * 128), 16, lane_a + r * pitch_a, s.k, 0, 0);
    };
    auto copy_w = [&](int half, int u) {
        const int r = row_w(half, u);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(s.w, (__attribute__((address_space(3))) void *)(reinterpret_cast<char *>(lds) + S::A_BYTES + to + r * 128), 16, lane_w + r * pitch_w, s.k, 0, 0);
    };
    auto copied = [&] { // the next k-tile to copy
        to = to ? 0 : S::STAGE_BYTES;
        s.k += BK * 2;
        if (--s.n_ktiles == 0) {
            if (next(ahead, issue_round)) open(ahead, s);
            else { // behind the last tile: empty operands, so that the counts of copies in flight stay what they are
                s.a = __builtin_amdgcn_make_buffer_rsrc(nullptr, 0, 0, 0x00020000);
                s.w = s.a;
                s.k = 0;
                s.n_ktiles = 1 << 30;
            }
        }
    };
    // ---- products
    const int frag_row = lane & 15, frag_g = lane >> 4;
    unsigned lane_off[2];
#pragma unroll
    for (int i = 0; i < 2; i++) lane_off[i] = (frag_row * BK + swz(frag_row, 4 * i + frag_g) * 8) * 2;
    const unsigned block_a = wm * 32 * MI * 128, block_w = S::A_BYTES + wn * 64 * 128;
    half8_t fa[2][4], fw0[2][2], fw1[2][2]; // [32-wide slice of k][16 rows]
    float4_t acc[4][2 * MI];
    unsigned at = 0; // stage of the k-tile being read
#define LDS_READ(to, address, offset) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(to) : "v"(address), "n"(offset))
    auto read_a0 = [&](int i) {
#pragma unroll
        for (int j = 0; j < 2 * H0; j++) LDS_READ(fa[i][j], lane_off[i] + (at + block_a), j * 2048);
    };
    auto read_a1 = [&](int i) {
#pragma unroll
        for (int j = 0; j < 2 * H1; j++) LDS_READ(fa[i][j], lane_off[i] + (at + block_a), (2 * H0 + j) * 2048);
    };
    auto read_w0 = [&](int i, int j) { LDS_READ(fw0[i][j], lane_off[i] + (at + block_w), j * 2048); };
    auto read_w1 = [&](int i, int j) { LDS_READ(fw1[i][j], lane_off[i] + (at + block_w), (2 + j) * 2048); };
#undef LDS_READ
    // all but the newest reads have landed, this slice's among them (reads and waits by hand, as in gemm_dma.hpp)
    auto wait_lds = [&](auto newer, half8_t (&a)[4], half8_t (&w)[2]) {
        asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(w[0]), "+v"(w[1]) : "n"(newer.value) : "memory");
    };
#define FENCE() __builtin_amdgcn_sched_barrier(0)
    auto multiply0 = [&](int i, const half8_t &w, float4_t (&c)[2 * MI]) {
#pragma unroll
        for (int j = 0; j < 2 * H0; j++) c[j] = Op::mul(w, fa[i][j], c[j]);
    };
    auto multiply1 = [&](int i, const half8_t &w, float4_t (&c)[2 * MI]) {
#pragma unroll
        for (int j = 0; j < 2 * H1; j++) c[2 * H0 + j] = Op::mul(w, fa[i][j], c[2 * H0 + j]);
    };
    auto copy_first = [&](int n) { // of a k-tile's first half of A and W
        if (n < H0) copy_a(0, n);
        else if (n < H0 + 4) copy_w((n - H0) >> 1, (n - H0) & 1);
    };
    for (int i = 0; i < 2; i++) {
        for (int n = 0; n < H0 + 4; n++) copy_first(n);
        for (int n = 0; n < H1; n++) copy_a(1, n);
        copied();
    }
    wait_vmcnt<H0 + 4 + 2 * H1>();
    lds_barrier();
#pragma unroll
    for (int i = 0; i < 2; i++) { read_w0(i, 0); read_w0(i, 1); read_a0(i); }
    for (bool more = true; more;) {
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
            for (int j = 0; j < 2 * MI; j++) acc[i][j] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        for (int left = ktiles(t); left > 0; left--) {
            // first x first
            wait_lds(std::integral_constant<int, 2 + 2 * H0>(), fa[0], fw0[0]); read_w1(0, 0); read_w1(0, 1); multiply0(0, fw0[0][0], acc[0]); FENCE();
            read_w1(1, 0); read_w1(1, 1); multiply0(0, fw0[0][1], acc[1]); FENCE();
            wait_lds(std::integral_constant<int, 4>(), fa[1], fw0[1]); multiply0(1, fw0[1][0], acc[0]); FENCE();
            multiply0(1, fw0[1][1], acc[1]); FENCE();
            // first x second
            asm volatile("s_waitcnt lgkmcnt(0) vmcnt(%4)" : "+v"(fw1[0][0]), "+v"(fw1[0][1]), "+v"(fw1[1][0]), "+v"(fw1[1][1]) : "n"(H0 + 4 + H1) : "memory");
            __builtin_amdgcn_s_barrier();
            FENCE();
            multiply0(0, fw1[0][0], acc[2]); copy_first(0); FENCE();
            multiply0(0, fw1[0][1], acc[3]); read_a1(0); copy_first(1); FENCE();
            multiply0(1, fw1[1][0], acc[2]); copy_first(2); FENCE();
            multiply0(1, fw1[1][1], acc[3]); read_a1(1); copy_first(3); FENCE();
            // second x second
            wait_lds(std::integral_constant<int, 2 * H1>(), fa[0], fw1[0]); multiply1(0, fw1[0][0], acc[2]); copy_first(4); FENCE();
            multiply1(0, fw1[0][1], acc[3]); copy_first(5); FENCE();
            wait_lds(std::integral_constant<int, 0>(), fa[1], fw1[1]); multiply1(1, fw1[1][0], acc[2]); FENCE();
            multiply1(1, fw1[1][1], acc[3]); FENCE();
            // second x first
            wait_vmcnt<H0 + 4 + H1>();
            __builtin_amdgcn_s_barrier();
            FENCE();
            at = at ? 0 : S::STAGE_BYTES;
            multiply1(0, fw0[0][0], acc[0]); read_w0(0, 0); copy_a(1, 0); FENCE();
            multiply1(0, fw0[0][1], acc[1]); read_w0(0, 1); read_a0(0); if constexpr (H1 == 2) copy_a(1, 1); FENCE();
            multiply1(1, fw0[1][0], acc[0]); read_w0(1, 0); copied(); FENCE();
            multiply1(1, fw0[1][1], acc[1]); read_w0(1, 1); read_a0(1); FENCE();
        }
        wait_lds(std::integral_constant<int, 0>(), fa[0], fw0[0]);
        wait_lds(std::integral_constant<int, 0>(), fa[1], fw0[1]);
        Tile done = t;
        more = next(t, read_round);
        store(done, wm, wn, acc);
    }
#undef FENCE
    wait_vmcnt<0>();
}

} // namespace
