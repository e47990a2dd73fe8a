// Copies from global memory into LDS that pass no registers.
#pragma once
#include "common.h"

namespace IV2_NS {

__device__ __forceinline__ uint32_t lds_address_of(const void* ptr) {
    return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)ptr));
}
// One wavefront copies 4 KiB from global memory straight into LDS (no registers): lane l moves bytes
// [16 l, 16 l + 16) of each 1 KiB quarter (the instruction offset advances source and destination alike).
// The compiler does not see these loads; callers order them by hand with s_waitcnt vmcnt(n) + barrier.
__device__ __forceinline__ void dma_copy_4k(const void* src_lane, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %1\n\t"
                 "global_load_lds_dwordx4 %0, off\n\t"
                 "global_load_lds_dwordx4 %0, off offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, off offset:2048\n\t"
                 "global_load_lds_dwordx4 %0, off offset:3072\n\t"
                 :
                 : "v"(src_lane), "s"(lds_dst)
                 : "memory", "m0");
}
// The same with the address in two parts: base is uniform over the wavefront, lane l passes 16 l.
__device__ __forceinline__ void dma_copy_4k(const void* base, uint32_t lane_bytes, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\t"
                 "global_load_lds_dwordx4 %0, %1\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:1024\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:2048\n\t"
                 "global_load_lds_dwordx4 %0, %1 offset:3072\n\t"
                 :
                 : "v"(lane_bytes), "s"(base), "s"(lds_dst)
                 : "memory", "m0");
}
// A quarter of it.
__device__ __forceinline__ void dma_copy_1k(const void* base, uint32_t lane_bytes, uint32_t lds_dst) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_bytes), "s"(base), "s"(lds_dst) : "memory", "m0");
}

}  // namespace IV2_NS
