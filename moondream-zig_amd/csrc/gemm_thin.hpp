// The tile product as a stream of tiles (gemm_stream.hpp) for few rows: tiles of 128 (m) x 64 (n) x 64 (k), five k-tiles in flight.
#pragma once
#include "gemm_dma.hpp"
#include "gemm_block.hpp"

namespace {

struct Thin {
    static constexpr int ROWS = 128, COLUMNS = 64, STAGES = 6, COPIES = 6; // copies of a loader wavefront and k-tile, eight rows each: 4 of A, 2 of W
    static constexpr unsigned A_BYTES = ROWS * BK * 2, STAGE_BYTES = A_BYTES + COLUMNS * BK * 2;
    static constexpr int SCRATCH_BYTES = 4096; // per multiplier wavefront
    static constexpr size_t LDS_BYTES = size_t(STAGES) * STAGE_BYTES + 4 * SCRATCH_BYTES;
    static_assert(LDS_BYTES <= 160 * 1024, "LDS");
};

// A loader wavefront.  next(t): the workgroup's next tile, false behind the last; open(t, s): its operands as block_stream's, and their pitches in bytes.
template <class Tile, class Next, class Open>
__device__ __forceinline__ void thin_load(half_t *lds, int role_wave, int lane, Next next, Open open) {
    using S = Thin;
    Tile t;
    BlockSource s;
    int pitch_a = 0, pitch_w = 0;
    bool more = next(t);
    if (!more) return;
    open(t, s, pitch_a, pitch_w);
    int issued = 0, stage = 0;
    auto issue = [&] {
        char *dst = reinterpret_cast<char *>(lds) + stage * S::STAGE_BYTES;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const int r = 32 * role_wave + 8 * j, row = r + (lane >> 3);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(s.a, (__attribute__((address_space(3))) void *)(dst + r * 128), 16, row * pitch_a + swz(row, lane & 7) * 16, s.k, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const int r = 16 * role_wave + 8 * j, row = r + (lane >> 3);
            __builtin_amdgcn_raw_ptr_buffer_load_lds(s.w, (__attribute__((address_space(3))) void *)(dst + S::A_BYTES + r * 128), 16, row * pitch_w + swz(row, lane & 7) * 16, s.k, 0, 0);
        }
        stage = stage + 1 == S::STAGES ? 0 : stage + 1;
        issued++;
        s.k += BK * 2;
        if (--s.n_ktiles == 0 && (more = next(t))) open(t, s, pitch_a, pitch_w);
    };
    while (more && issued < S::STAGES - 1) issue();
    for (int step = 0; step < issued; step++) {
        const int newer = issued - 1 - step; // k-tiles requested behind this one
        if (newer >= 4) wait_vmcnt<4 * S::COPIES>();
        else if (newer == 3) wait_vmcnt<3 * S::COPIES>();
        else if (newer == 2) wait_vmcnt<2 * S::COPIES>();
        else if (newer == 1) wait_vmcnt<S::COPIES>();
        else wait_vmcnt<0>();
        lds_barrier(); // publishes this step's k-tile; nobody reads the one before any more
        if (more) issue();
    }
}

// A multiplier wavefront: rows 32 wave .. + 31, all 64 columns.  ktiles(t): k-tiles of a tile (>= 1); store(t, acc): acc[16 columns][16 rows], as block_stream's.
template <class Op, class Tile, class Next, class KTiles, class Store>
__device__ __forceinline__ void thin_multiply(int wave, int lane, Next next, KTiles ktiles, Store store) {
    using S = Thin;
    const int frag_row = lane & 15, frag_g = lane >> 4;
    unsigned lane_off[2];
#pragma unroll
    for (int i = 0; i < 2; i++) lane_off[i] = (frag_row * BK + swz(frag_row, 4 * i + frag_g) * 8) * 2;
    const unsigned block_a = wave * 32 * 128;
    struct Frag {
        half8_t fa[2], fw[4];
    };
    // (reads and waits by hand, as in gemm_dma.hpp: six reads per 32-wide slice, one slice ahead of its eight products)
    auto read = [&](unsigned base, int i, Frag &f) {
        const unsigned at_a = lane_off[i] + (base + block_a), at_w = lane_off[i] + (base + S::A_BYTES);
#pragma unroll
        for (int j = 0; j < 2; j++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.fa[j]) : "v"(at_a), "n"(j * 2048));
#pragma unroll
        for (int j = 0; j < 4; j++) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(f.fw[j]) : "v"(at_w), "n"(j * 2048));
    };
    auto wait = [&](auto newer, Frag &f) {
        asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(f.fa[0]), "+v"(f.fa[1]), "+v"(f.fw[0]), "+v"(f.fw[1]), "+v"(f.fw[2]), "+v"(f.fw[3]) : "n"(newer.value) : "memory");
    };
    float4_t acc[4][2];
    auto multiply = [&](const Frag &f) {
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int m = 0; m < 2; m++) acc[n][m] = Op::mul(f.fw[n], f.fa[m], acc[n][m]);
    };
    Tile t;
    if (!next(t)) return;
    Frag fr[2];
    unsigned base = 0;
    auto advance = [&] { base = base + S::STAGE_BYTES == S::STAGES * S::STAGE_BYTES ? 0 : base + S::STAGE_BYTES; };
    using Older = std::integral_constant<int, 6>;
    using All = std::integral_constant<int, 0>;
    lds_barrier(); // the first k-tile is visible
    for (bool more = true; more;) {
#pragma unroll
        for (int n = 0; n < 4; n++)
#pragma unroll
            for (int m = 0; m < 2; m++) acc[n][m] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
        read(base, 0, fr[0]);
        for (int left = ktiles(t) - 1; left > 0; left--) {
            read(base, 1, fr[1]);
            wait(Older(), fr[0]);
            multiply(fr[0]);
            __builtin_amdgcn_sched_barrier(0);
            wait(All(), fr[1]);
            __builtin_amdgcn_s_barrier(); // publishes the next k-tile; this wavefront has read all of this one
            advance();
            read(base, 0, fr[0]);
            multiply(fr[1]);
            __builtin_amdgcn_sched_barrier(0);
        }
        read(base, 1, fr[1]);
        wait(Older(), fr[0]);
        multiply(fr[0]);
        __builtin_amdgcn_sched_barrier(0);
        wait(All(), fr[1]);
        Tile done = t;
        more = next(t);
        if (more) __builtin_amdgcn_s_barrier(); // the same for the next tile's first k-tile: the loaders go on behind it
        advance();
        multiply(fr[1]);
        store(done, acc);
    }
}

} // namespace
