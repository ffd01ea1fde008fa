// The wavefront-specialised tile product (gemm_dma.hpp) as a stream of tiles: a workgroup per compute unit walks its tiles one after
// the other, and its four loader wavefronts go on copying the next tile's k-tiles while the four multiplier wavefronts still work on
// the tile before and write it out.  With a workgroup per tile every tile pays a launch slot, the first k-tile's round trip and an
// epilogue during which nothing is copied: 7 of the 21 us of a 128 x 128 x 2048 tile where a product has more tiles than the chip has
// compute units.
// The tile is 64 MI (m) x 128 (n) x 64 (k), MI = 2, 3 or 4; multipliers in a 2 x 2 grid own 32 MI x 64 (2 MI accumulators of
// 32 x 32, f32).  What bounds the loop, per k-tile at MI = 4 with every unit busy: the products alone take 0.61 us (the clock under
// matrix load), the copies alone 0.58 (1.2 us of latency with two k-tiles, 96 KiB, in flight), the operand reads alone 0.32, all
// together 0.85 with the operands in L2, 0.9 from HBM; MI = 2: 0.30, 0.34, 0.26 and 0.43.  Copies must be whole 128-byte lines: with
// k-tiles of 32 (64-byte rows, four stages) a copy takes twice as long.  Tiles twice as wide are gemm_block.hpp's.
// Stages and the barrier per k-tile are gemm_dma.hpp's, counted on over the tiles.  The epilogue has 16 KiB of LDS of its own, so it
// runs while the loaders fill every stage.  K ranges are whole k-tiles.
#pragma once
#include "gemm_dma.hpp"

namespace {

constexpr int STREAM_SCRATCH_BYTES = 4096; // per multiplier wavefront
template <int MI> struct Stream {
    static constexpr int ROWS = 64 * MI;
    static constexpr int STAGES = MI == 2 ? 4 : 3;
    static constexpr int STAGE_HALFS = (ROWS + BN) * BK;
    static constexpr unsigned STAGE_BYTES = STAGE_HALFS * sizeof(half_t);
    static constexpr int COPIES = 2 * MI + 4; // of a loader wavefront and k-tile: 2 MI of eight activation rows, 4 of eight weight rows
    static constexpr size_t LDS_BYTES = size_t(STAGES) * STAGE_BYTES + 4 * STREAM_SCRATCH_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// A loader wavefront.  next(t): the workgroup's next tile, false behind the last.  open(t, s): its operands, an 8-row group's offset per
// copy (StreamSource).
template <int MI> struct StreamSource {
    __amdgpu_buffer_rsrc_t a, w;
    int off_a[2 * MI], off_w[4]; // bytes at k = 0
    int k, n_ktiles;             // bytes of the first k-tile, their number (>= 1)
    bool once;                   // (with ONCE) no other row tile reads these weights: they are not to push the activations out of the L2 (non-temporal copies)
};
__device__ __forceinline__ int stream_row_a(int mi, int role_wave, int j, int lane) { return 16 * mi * role_wave + 8 * j + (lane >> 3); }

template <int MI, bool ONCE, class Tile, class Next, class Open>
__device__ __forceinline__ void stream_load(half_t *lds, int role_wave, Next next, Open open) {
    using S = Stream<MI>;
    Tile t;
    StreamSource<MI> s;
    bool more = next(t);
    if (more) open(t, s);
    int issued = 0, stage = 0;
    auto issue = [&] {
        half_t *dst = lds + size_t(stage) * S::STAGE_HALFS;
#pragma unroll
        for (int j = 0; j < 2 * MI; j++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(s.a, (__attribute__((address_space(3))) void *)(dst + (16 * MI * role_wave + 8 * j) * BK), 16, s.off_a[j], s.k, 0, 0);
        if (ONCE && s.once) {
#pragma unroll
            for (int j = 0; j < 4; j++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(s.w, (__attribute__((address_space(3))) void *)(dst + S::ROWS * BK + (32 * role_wave + 8 * j) * BK), 16, s.off_w[j], s.k, 0, 2);
        } else {
#pragma unroll
            for (int j = 0; j < 4; j++)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(s.w, (__attribute__((address_space(3))) void *)(dst + S::ROWS * BK + (32 * role_wave + 8 * j) * BK), 16, s.off_w[j], s.k, 0, 0);
        }
        stage = stage + 1 == S::STAGES ? 0 : stage + 1;
        issued++;
        s.k += BK * 2;
        if (--s.n_ktiles == 0 && (more = next(t))) open(t, s);
    };
    while (more && issued < S::STAGES - 1) issue();
    for (int step = 0; step < issued; step++) {
        const int newer = issued - 1 - step; // k-tiles requested behind this one
        if (newer >= 2) wait_vmcnt<2 * S::COPIES>();
        else if (newer == 1) wait_vmcnt<S::COPIES>();
        else wait_vmcnt<0>();
        lds_barrier(); // publishes this step's k-tile; nobody reads the one before any more
        if (more) issue();
    }
}

// A multiplier wavefront.  ktiles(t): k-tiles of a tile; store(t, acc): acc[ni][mi] as in dma_multiply_tiles.
template <class Op, int MI, class Tile, class Next, class KTiles, class Store>
__device__ __forceinline__ void stream_multiply(int wm, int wn, int lane, Next next, KTiles ktiles, Store store) {
    using S = Stream<MI>;
    const int frag_row = lane & 31, frag_g = lane >> 5;
    // Where this lane's part of a 32-row block's 16-wide slice s lies: blocks are 4 KiB apart whatever the lane and enter as the
    // read's offset (gemm_dma.hpp).
    unsigned lane_off[BK / 16];
#pragma unroll
    for (int s = 0; s < BK / 16; s++) lane_off[s] = (frag_row * BK + swz(frag_row, 2 * s + frag_g) * 8) * 2;
    const unsigned block_a = wm * MI * 4096, block_w = (S::ROWS * BK + wn * 64 * BK) * 2;
    struct Frag {
        half8_t fa[MI], fw[2];
    };
    // (reads and waits by hand, as in gemm_dma.hpp: MI + 2 reads per slice, one slice ahead of its 2 MI products)
    auto read = [&](unsigned base, int s, Frag &f) {
        const unsigned at_a = lane_off[s] + (base + block_a), at_w = lane_off[s] + (base + block_w);
#pragma unroll
        for (int i = 0; i < 2; i++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.fw[i]) : "v"(at_w), "n"(i * 4096));
#pragma unroll
        for (int i = 0; i < MI; i++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.fa[i]) : "v"(at_a), "n"(i * 4096));
    };
    auto wait_older = [&](Frag &f) {
        if constexpr (MI == 4)
            asm volatile("s_waitcnt lgkmcnt(6)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fa[2]), "+v"(f.fa[MI - 1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
        else if constexpr (MI == 3)
            asm volatile("s_waitcnt lgkmcnt(5)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fa[MI - 1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
        else
            asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
    };
    auto wait_all = [&](Frag &f) {
        if constexpr (MI == 4)
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fa[2]), "+v"(f.fa[MI - 1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
        else if constexpr (MI == 3)
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fa[MI - 1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
        else
            asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fw[0]), "+v"(f.fw[1])::"memory");
    };
    float16_t acc[2][MI];
    auto multiply = [&](const Frag &f) {
#pragma unroll
        for (int mi = 0; mi < MI; mi++)
#pragma unroll
            for (int ni = 0; ni < 2; ni++) acc[ni][mi] = Op::mul(f.fw[ni], f.fa[mi], acc[ni][mi]);
    };
    Tile t;
    if (!next(t)) return;
    Frag fr[2];
    unsigned base = 0;
    auto advance = [&] { base = base + S::STAGE_BYTES == S::STAGES * S::STAGE_BYTES ? 0 : base + S::STAGE_BYTES; };
    auto first_three = [&] {
        read(base, 1, fr[1]);
        wait_older(fr[0]);
        multiply(fr[0]);
        __builtin_amdgcn_sched_barrier(0);
        read(base, 2, fr[0]);
        wait_older(fr[1]);
        multiply(fr[1]);
        __builtin_amdgcn_sched_barrier(0);
        read(base, 3, fr[1]);
        wait_older(fr[0]);
        multiply(fr[0]);
        __builtin_amdgcn_sched_barrier(0);
    };
    lds_barrier(); // the first k-tile is visible
    for (bool more = true; more;) {
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < MI; j++)
#pragma unroll
                for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
        read(base, 0, fr[0]);
        for (int left = ktiles(t) - 1; left > 0; left--) {
            first_three();
            wait_all(fr[1]);
            __builtin_amdgcn_s_barrier(); // publishes the next k-tile; this wavefront has read all of this one
            advance();
            read(base, 0, fr[0]);
            multiply(fr[1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        first_three();
        wait_all(fr[1]);
        Tile done = t;
        more = next(t);
        if (more) __builtin_amdgcn_s_barrier(); // the same for the next tile's first k-tile: the loaders go on behind it
        advance();
        multiply(fr[1]);
        store(done, acc); // (no operand read is in flight here: the compiler may move those registers)
    }
}

} // namespace
