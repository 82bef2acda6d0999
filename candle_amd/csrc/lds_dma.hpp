// Direct global -> LDS loads.
#pragma once
#include "moe_common.hpp"

namespace moe {

__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) void*)p;
}
// Lane i of the wave writes SIZE bytes at lds + SIZE*i; nothing passes through registers, so a whole super-block of
// activations can be in flight while the wave computes.  The compiler does not see these loads: the issuing wave waits for
// them (vmcnt) before the barrier that publishes the buffer.
__device__ __forceinline__ void dma16(const void* gbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(gbase), "s"(lds));
}
__device__ __forceinline__ void dma4(const void* gbase, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dword %0, %1" ::"v"(voff), "s"(gbase), "s"(lds));
}
// waits until at most N of the wave's loads, the newest, are on their way
template <int N>
__device__ __forceinline__ void wait_loads() {
    static_assert(N < 16, "the low field of the count");
    __builtin_amdgcn_s_waitcnt(0x0F70 | N);
}

}  // namespace moe
