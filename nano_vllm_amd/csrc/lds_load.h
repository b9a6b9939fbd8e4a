// Loads from global memory straight into LDS, and the waits that go with them (gfx950).
#pragma once
#include "common.h"

// 16 bytes per lane from base + offset (base the same for the whole wave, offset in bytes per lane)
// to LDS at lds + 16 * lane (lds the same for the whole wave).  Written by hand: the compiler would
// make every later read of LDS wait for all such loads; these are waited for by count.
__device__ __forceinline__ void nva_load_to_lds(const void* base, uint32_t offset, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(offset), "s"(base), "s"(lds) : "memory", "m0");
}
// Until at most N of this wave's loads are on their way.  (The counter has six bits.)
template <int N> __device__ __forceinline__ void nva_wait_loads_but() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N < 64 ? N : 63) : "memory"); }
// The workgroup's barrier behind this wave's own reads and writes of LDS; loads on their way stay so.
__device__ __forceinline__ void nva_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
