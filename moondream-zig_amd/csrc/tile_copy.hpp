// Copies of whole tiles from memory to LDS that take no registers on the way, for the attention kernels whose tiles serve more than 32 query rows.
#pragma once
#include <hip/hip_runtime.h>

namespace {

typedef unsigned int tile_u32x4 __attribute__((ext_vector_type(4)));

// Rows of 64 16-bit elements, unpadded: granule c (16 bytes) of row s sits at c ^ row64_swizzle(s).  An operand read takes one granule of each
// of 16 consecutive rows, a transposing read 4 granules of each of 4 consecutive rows; 16 granules are all 64 banks.  Of two rows with the
// same parity that follow each other the value differs in bit 2, and over 16 rows each half of the banks sees all eight values.
__device__ __forceinline__ int row64_swizzle(int row) { return (row >> 1 & 1) << 2 | (row >> 2 & 3); }

// The tile whose first row lies at `rows` into the LDS at byte lds: left bytes are what the head's rows still hold from there, what
// lies past them reads as zero.  Written as instructions because the compiler, which cannot tell which of its LDS reads a copy
// in flight touches, would wait for every copy before each of them; tile_landed says what has arrived.  The LDS reads before it
// have returned when the first copy starts.
// (M0 is a register that the compiler keeps for itself and sets anew for each of its own uses: naming it makes it do so behind a copy,
// and clang says that it is not preserved, which is the point)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
template <int COPIES>
__device__ __forceinline__ void tile_copy(const void *rows, int left, unsigned lds, const int (&off)[COPIES]) {
    const unsigned long at = reinterpret_cast<unsigned long>(rows);
    tile_u32x4 rs = {(unsigned)__builtin_amdgcn_readfirstlane((int)at), (unsigned)__builtin_amdgcn_readfirstlane((int)(at >> 32) & 0xffff),
                (unsigned)__builtin_amdgcn_readfirstlane(left), 0x00020000u};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < COPIES; i++)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" // (5 wait states: scalars that the vector unit wrote)
                     ::"s"(lds + i * 1024), "v"(off[i]), "s"(rs) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int NEWER> __device__ __forceinline__ void tile_landed() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NEWER) : "memory"); }
// For tiles that wavefronts share: behind this the tile that all of them copied is whole, and the one before has been read by all, since their reads
// of it have returned (the compiler's own waits for them stand where it needs the values, which may be behind the barrier).
__device__ __forceinline__ void tile_handed_over() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

} // namespace
