// Rows straight from memory into LDS, for kernels that walk over K through a ring of stages: 16 bytes a lane and instruction,
// a wave's instruction filling 1 KB from `lds_base` on, and the wait for all but the youngest of them.
#pragma once
#include "common.h"

__device__ __forceinline__ void row_chunk_into_lds(const void* from, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(lds_base) : "m0", "memory");
}
// the same from a base that all lanes share and a lane's own offset
// ONCE: for what passes once, marked as a stream (nt) that does not push out of the caches what is read again
template <bool ONCE = false> __device__ __forceinline__ void row_chunk_into_lds(const char* base, uint32_t offset, uint32_t lds_base) {
    if constexpr (ONCE)
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1 nt" : : "v"(offset), "s"(base), "s"(lds_base) : "m0", "memory");
    else
        asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(offset), "s"(base), "s"(lds_base) : "m0", "memory");
}
// For a ring that one wave fills and reads without a barrier: its reads of LDS are in registers; reads stay behind a wait.
__device__ __forceinline__ void lds_reads_done() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ __forceinline__ void no_read_before_here() { asm volatile("" ::: "memory"); }
// s_waitcnt vmcnt(N): loads come back in order, so "all but the N youngest" is a stage's rows with the later stages'
// still on their way.  (vmcnt is six bits: the low four in bits 0..3, the high two in bits 14..15.)
template <int N> __device__ __forceinline__ void all_but_the_youngest_have_arrived() {
    static_assert(N >= 0 && N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}
