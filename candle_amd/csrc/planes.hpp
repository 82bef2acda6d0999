// Weight operands with the block scale inside: products of scales and codes cut into signed byte planes.
#pragma once
#include "moe_common.hpp"

namespace moe {

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
// Q6K: both planes of W = sc * (code - 32).  A word of four codes is spread over two registers of two 16-bit lanes
// (even and odd bytes), each multiplied and offset in one packed multiply-add: W + 128 = code * sc + (128 - 32 sc).
// The high bytes of W + 128 are H = floor((W + 128) / 256); its low bytes, with the top bit flipped, are W - 256 H as a
// signed byte.
__device__ __forceinline__ uint32_t pk_mad_u16(uint32_t a, uint32_t b, uint32_t c) {
    return __builtin_bit_cast(uint32_t, (u16x2)(__builtin_bit_cast(u16x2, a) * __builtin_bit_cast(u16x2, b) + __builtin_bit_cast(u16x2, c)));
}
__device__ __forceinline__ void q6k_planes(uint32_t codes, uint32_t s2, uint32_t add2, int& lo, int& hi) {
    const uint32_t ev = codes & 0x00ff00ffu;
    const uint32_t od = __builtin_amdgcn_perm(0u, codes, 0x0c030c01u);
    const uint32_t we = pk_mad_u16(ev, s2, add2), wo = pk_mad_u16(od, s2, add2);
    lo = (int)(__builtin_amdgcn_perm(wo, we, 0x06020400u) ^ 0x80808080u);
    hi = (int)__builtin_amdgcn_perm(wo, we, 0x07030501u);
}

}  // namespace moe
