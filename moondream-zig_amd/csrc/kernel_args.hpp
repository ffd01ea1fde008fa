// A launch's arguments, fetched at once.
#pragma once
#include <hip/hip_runtime.h>

namespace {

// The arguments of a launch are new in memory for every launch, so each 64 bytes of them are a miss as far as HBM (about 1 us) for the
// first wavefront of a compute unit that asks.  The compiler loads them where they are needed, as many as there are scalar registers for, and a kernel
// with hundreds of bytes of them waits for that long two or three times in a row before its first load of data.  This reads a word of each
// of their lines ahead of everything else and returns where they are: a kernel that takes them from there finds them in
// the scalar cache.  A token of 24 layers, three launches each: 722 -> 704 us (width 2048, 8 key heads), 550 -> 543 (width 1024, rotated and joined), 12 layers with
// routed experts 382 -> 374; the third launch has two lines only and gains nothing.  (The reads are written as instructions, with their wait, because the compiler puts its own first and in turns; it
// cannot put any ahead of an address that it does not know yet.)
#define MOON_ARGS_LINE(offset) "s_load_dword %0, %1, " #offset "\n\t"
#define MOON_ARGS_1 MOON_ARGS_LINE(0x0)
#define MOON_ARGS_2 MOON_ARGS_1 MOON_ARGS_LINE(0x40)
#define MOON_ARGS_3 MOON_ARGS_2 MOON_ARGS_LINE(0x80)
#define MOON_ARGS_4 MOON_ARGS_3 MOON_ARGS_LINE(0xc0)
#define MOON_ARGS_5 MOON_ARGS_4 MOON_ARGS_LINE(0x100)
#define MOON_ARGS_6 MOON_ARGS_5 MOON_ARGS_LINE(0x140)
#define MOON_ARGS_7 MOON_ARGS_6 MOON_ARGS_LINE(0x180)
#define MOON_ARGS_8 MOON_ARGS_7 MOON_ARGS_LINE(0x1c0)
#define MOON_ARGS_9 MOON_ARGS_8 MOON_ARGS_LINE(0x200)
#define MOON_ARGS_10 MOON_ARGS_9 MOON_ARGS_LINE(0x240)
#define MOON_ARGS_11 MOON_ARGS_10 MOON_ARGS_LINE(0x280)
#define MOON_ARGS_12 MOON_ARGS_11 MOON_ARGS_LINE(0x2c0)
#define MOON_ARGS_13 MOON_ARGS_12 MOON_ARGS_LINE(0x300)
#define MOON_ARGS_14 MOON_ARGS_13 MOON_ARGS_LINE(0x340)
#define MOON_ARGS_15 MOON_ARGS_14 MOON_ARGS_LINE(0x380)
#define MOON_ARGS_16 MOON_ARGS_15 MOON_ARGS_LINE(0x3c0)
#define MOON_ARGS_FETCH(n) if constexpr (LINES == n) asm volatile(MOON_ARGS_##n "s_waitcnt lgkmcnt(0)" : "=&s"(word), "+s"(at))
// Args: the kernel's only parameter
template <class Args> __device__ __forceinline__ const Args &fetch_arguments() {
    constexpr int LINES = (sizeof(Args) + 63) / 64;
    static_assert(LINES <= 16, "more lines");
    auto *at = __builtin_amdgcn_kernarg_segment_ptr();
    unsigned word; // (of no use itself)
    MOON_ARGS_FETCH(1);
    MOON_ARGS_FETCH(2);
    MOON_ARGS_FETCH(3);
    MOON_ARGS_FETCH(4);
    MOON_ARGS_FETCH(5);
    MOON_ARGS_FETCH(6);
    MOON_ARGS_FETCH(7);
    MOON_ARGS_FETCH(8);
    MOON_ARGS_FETCH(9);
    MOON_ARGS_FETCH(10);
    MOON_ARGS_FETCH(11);
    MOON_ARGS_FETCH(12);
    MOON_ARGS_FETCH(13);
    MOON_ARGS_FETCH(14);
    MOON_ARGS_FETCH(15);
    MOON_ARGS_FETCH(16);
    return *(const Args *)(const __attribute__((address_space(4))) Args *)at;
}

} // namespace
