// Tiled grouped expert products for large batches (prefill): Q4K (also Q2K, Q3K, Q5K and Q6K) weights x
// Q8K activations on v_mfma_i32_16x16x64_i8, a full-rate int8 MFMA shape of gfx950.
//
// Same integers as BlockQ4K::vec_dot (candle-core/src/quantized/k_quants.rs:1205-1285):
//     sum_j sc_j * (q4_j . q8_j)      and      sum_j m_j * (bsum_2j + bsum_2j+1).
// Applying the 6-bit scale to every block of MFMA results would cost one integer multiply-add per
// result and 32 elements of K -- twice the time of the MFMA itself -- so the scale is moved into the
// weight operand instead: sc = 8*hi + lo with hi, lo <= 7, and the two byte planes hi*q4 and lo*q4
// (<= 105, no carry between bytes) are multiplied by the activations in two MFMAs that accumulate over
// the whole 256-element super-block.  8*acc_hi + acc_lo is then the exact integer the reference
// computes; the mins term is an exact f16 MFMA over the 16 block sums.
//
// Work split: a workgroup (8 or 4 waves) owns one tile of 128 or 64 slots of one expert (from the dispatch
// kernel's tile list, so a skewed routing is balanced by tiles, not by experts) and two 16-row
// weight operands per wave.  The activation rows of a super-block go straight from global
// memory into LDS (double-buffered, no staging registers) and every wave reads them as MFMA A
// operands.  A wave unpacks and pre-scales its 32 weight rows of the super-block once, keeps the
// planes in registers (64 VGPRs) and runs them against the 16-slot operands one after the other.
//
// What bounds it: the issue port of a SIMD, which matrix and vector instructions share (a 16x16x64 MFMA holds it for 8
// cycles, a vector instruction for 4), with the unpacking (95 vector instructions per 16 rows and super-block) and the
// results (5 each), and then waiting: counted over the up launch of 4096 tokens at the Mixtral shape the port is taken 75 % of the
// time, the matrix pipe is busy 50 %, and a wave waits for 30 % of its cycles.  Two weight operands per wave: an LDS read feeds four matrix instructions instead of two.  That
// takes two waves per SIMD (256 registers), too few to cover each other, so a wave overlaps its own work: the results of
// operand o - 1 are added up between the matrix instructions of operand o, and the next super-block's transfers are
// issued a few at a time behind the operands (in one go at the top they held each wave up for 1650 to 4700 of 9000 cycles).
// Up launch, 4096 tokens at the Mixtral shape: one operand per wave, four waves per SIMD 2.23-2.28 ms, this kernel 2.00-2.12 ms;
// the same with 32x32x32 MFMAs and no overlap in the wave 2.3 ms.  Operands beyond a short tile's list are neither
// fetched nor multiplied (the K loop exists for each number of them).
// Down launches of the formats that unpack longest in tiles of 64 slots run one operand per wave at four waves per SIMD
// (launch_gemm).  Registers: 164 to 254 with two operands (Q5K at 128 slots: 256, one to three of them spilled outside the K
// loop, ten with K split, Q4K split one), 122 to 126 with one.
//
// Where a launch would have no more than one workgroup of four waves per CU (a down projection of some hundred tokens, dense products
// of a few hundred rows), a wave alone on its SIMD leaves it idle for two fifths of the time, and nothing else is there to run.
// There the workgroup has eight waves for the same rows, four for each half of K with LDS buffers of their own (KS = 2; KS = 4:
// two waves for each quarter, 64 rows), whose sums meet in LDS at the end.  Down launch, Mixtral shape: Q4_K 200 tokens 112 -> 93 us,
// 301 tokens 128 -> 111; Q6_K 301 tokens 153 -> 135.  The rule and the dense products' times: gemm_plan.hpp.  On a full chip the split
// costs (Q4_K 4096 x 4096 at 4096 rows 161 -> 181).
//
// Q6K weights (the w2 of mixed files) take the same kernel for the down projection.  BlockQ6K::vec_dot
// (k_quants.rs:1613-1671) is d * y.d * sum_j sc_j * ((code_j - 32) . q8_j) with an i8 scale per 16 elements; the
// products W = sc * (code - 32) (|W| <= 4096) are formed in packed 16-bit arithmetic and cut into two signed bytes,
// W = 256 * H + L with L in [-128, 127], which are the two planes: 256 * acc_H + acc_L is the reference's integer, and
// no term over the block sums is left.
//
// Q2K weights (BlockQ2K::vec_dot, k_quants.rs:755-805) need one plane only: a 4-bit scale times a 2-bit code is at most 45,
// so the scaled codes are the weight operand as they are and a super-block takes four int8 MFMAs per operand instead of
// eight; the minimums leave through the sixteen block sums as for Q4K.
#include <type_traits>
#include "act_quant.hpp"
#include "kernels.hpp"
#include "lds_dma.hpp"
#include "planes.hpp"

namespace moe {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef const __attribute__((address_space(1))) uint8_t* gbytes;

template <typename T>
__device__ __forceinline__ T gld(const void* uniform_base, uint32_t off) {
    return *reinterpret_cast<const __attribute__((address_space(1))) T*>((gbytes)uniform_base + off);
}

// four bytes (each <= 15) times a digit (<= 7): no byte overflows, and the packed 16-bit multiply does
// both halves of the register in one full-rate instruction (a 24-bit multiply would drop the top byte)
__device__ __forceinline__ uint32_t scale_bytes(uint32_t q, uint32_t s) {
    const u16x2 a = __builtin_bit_cast(u16x2, q);
    const u16x2 b = {(unsigned short)s, (unsigned short)s};
    return __builtin_bit_cast(uint32_t, (u16x2)(a * b));
}

// A tile is NOP 16-slot MFMA operands: 8 (128 slots) for big batches, 4 (64 slots) when the experts'
// lists are short, so that less of a tile is padding.
// Activations in LDS, laid out so that what one MFMA reads is one contiguous stretch in lane order
// (any other placement of a 16-lane x 4-chunk operand runs into LDS bank conflicts at half the read
// rate), and so that one direct global->LDS load of a wave (lane i lands at byte 16 i) writes exactly
// such a stretch:
//   quants [operand o][pair P][chunk g][row m] 16-byte pieces: 1 KiB per (o, P);
//   block sums [operand o][half h][row m] 16-byte pieces (8 sums): lane (m, g) reads 8 bytes at
//          piece (g/2, m), offset 8 (g%2);
//   scales [slot].
template <int NOP>
struct alignas(16) GemmLds {
    alignas(16) uint8_t q[2][NOP * 16 * 256];
    alignas(16) _Float16 bs[2][NOP][2][16][8];
    alignas(16) float yd[2][NOP * 16];
};

__device__ __forceinline__ void wait_all_loads() { wait_loads<0>(); }

template <int I, int N, class F>
__device__ __forceinline__ void static_for(const F& f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// What a lane fetches for the tile.  Quants: the NOP*4 (operand, pair) stretches of 1 KiB are dealt to
// the NW waves, NB each: lane (m = l%16, g = l/16) fetches piece (P, g) of row 16 o + m.  Block
// sums: one transfer covers two operands: lane fetches half (l/16)%2 of row 32 x + 16 (l/32) + l%16.
// Scales: row 64 x + l.  Waves without a share of the sums and scales repeat another wave's transfer:
// same bytes to the same place, and no branch around a load.
template <int NB>
struct StageRows {
    // byte offsets of the lane's first-super-block bytes; a transfer's super-block and pair are in its (scalar) base address
    uint32_t q[(NB + 3) / 4];   // per operand of the wave's share
    uint32_t bs, yd;
};
// transfer number I of a wave's share: quant stretches 0 .. NB-1, then the block sums, then the scales
template <int I, bool SUMS, int NOP, int NB>
__device__ __forceinline__ void stage_piece(const ActBuf& ab, const StageRows<NB>& r, int sb, GemmLds<NOP>& L, int buf, int wave, int live) {
    if constexpr (I < NB) {
        const int blk = wave * NB + I;      // = 4 o + P
        if ((blk >> 2) < live)              // (operands beyond the list are never read)
            dma16(ab.qs + sb * 256 + (blk & 3) * 64, r.q[I / 4], lds_address(L.q[buf]) + (uint32_t)(blk * 1024));
    } else if constexpr (I == NB) {
        if constexpr (SUMS)
            dma16(static_cast<const uint8_t*>(ab.bsum) + sb * 32, r.bs,
                  lds_address(&L.bs[buf][0][0][0][0]) + (uint32_t)((wave % (NOP / 2)) * 1024));
    } else {
        dma4(ab.d + sb, r.yd, lds_address(&L.yd[buf][0]) + (uint32_t)((wave % (NOP / 4)) * 256));
    }
}

// One wave's weights for one super-block: the 16 rows of one tile of the device layout.  Lane
// (n = l%16, g = l/16) owns row n and k-chunk g of every sub-block: exactly the tile's own lane order.
struct BRegs {
    u32x4 c[2];   // plane pl: (x,y) = 8 bytes of pair 2pl, chunk g; (z,w) = pair 2pl+1 (Q6K: the codes' low nibbles)
    u32x4 hdr;    // Q4K: d, dmin, 12 scale bytes of row n; Q6K: the row's sixteen i8 scales
    u32x4 qh;     // Q6K: the codes' top two bits, word P for pair P
    u32x2 q5;     // Q5K: the lane's fifth bits (pairs 0,1 / 2,3; four bits per byte and pair); Q3K: the codes' third bits, placed alike
    uint32_t d16; // Q6K, Q3K: d (f16 bits); Q2K: d | dmin << 16
};
template <int FMT>
__device__ __forceinline__ BRegs b_load(const uint8_t* tile, int lane) {
    BRegs b;
    b.c[0] = gld<u32x4>(tile, (uint32_t)(lane * 16));
    if (FMT == MOE_GGML_Q3K) {   // the codes' low two bits (placed as Q2K's codes), their high bits, the row's sixteen i8 scales, d
        b.q5 = gld<u32x2>(tile, (uint32_t)(1024 + lane * 8));
        b.hdr = gld<u32x4>(tile, (uint32_t)(1536 + (lane & 15) * 16));
        b.d16 = gld<uint16_t>(tile, (uint32_t)(1792 + (lane & 15) * 2));
        return b;
    }
    if (FMT == MOE_GGML_Q2K) {   // word P of the lane: the 2-bit codes of pair P; then the row's 16 (scale | min << 4) bytes and d | dmin << 16
        b.hdr = gld<u32x4>(tile, (uint32_t)(1024 + (lane & 15) * 16));
        b.d16 = gld<uint32_t>(tile, (uint32_t)(1280 + (lane & 15) * 4));
        return b;
    }
    b.c[1] = gld<u32x4>(tile, (uint32_t)(1024 + lane * 16));
    if (FMT == MOE_GGML_Q6K) {
        b.qh = gld<u32x4>(tile, (uint32_t)(2048 + lane * 16));
        b.hdr = gld<u32x4>(tile, (uint32_t)(3072 + (lane & 15) * 16));
        b.d16 = gld<uint16_t>(tile, (uint32_t)(3328 + (lane & 15) * 2));
    } else {
        b.hdr = gld<u32x4>(tile, (uint32_t)(2048 + (lane & 15) * 16));
        if (FMT == MOE_GGML_Q5K) b.q5 = gld<u32x2>(tile, (uint32_t)(Q4K_TILE_BYTES + lane * 8));
    }
    return b;
}

// The unpacked, pre-scaled operand of one super-block.  MFMA number P multiplies activation piece
// (pair P, chunk g) = [8 values of sub-block 2P | 8 values of sub-block 2P+1] by the low and the high
// nibbles of the same 8 weight bytes, each half scaled by its own sub-block's digit (the planes are
// accumulated over the whole super-block, so an MFMA may mix sub-blocks).
struct BPlanes {
    v4i lo[4], hi[4];
    v4h mB;
    float d, dmin;
};

__device__ __forceinline__ BPlanes b_prepare(const BRegs& b, int lane) {
    const int g = lane >> 4;
    const uint32_t M4 = 0x0f0f0f0fu;
    const uint32_t u0 = b.hdr.y, u1 = b.hdr.z, u2 = b.hdr.w;
    BPlanes o;
    o.d = __half2float(__ushort_as_half((unsigned short)(b.hdr.x & 0xffffu)));
    o.dmin = __half2float(__ushort_as_half((unsigned short)(b.hdr.x >> 16)));
    const uint32_t sc03 = u0 & 0x3f3f3f3fu;
    const uint32_t sc47 = (u2 & M4) | (((u0 >> 6) & 0x03030303u) << 4);
    const uint32_t m03 = u1 & 0x3f3f3f3fu;
    const uint32_t m47 = ((u2 >> 4) & M4) | (((u1 >> 6) & 0x03030303u) << 4);
    // scales split into two 3-bit digits, one per 16-bit lane (which the packed multiply takes for both of its halves): scales 0
    // and 2, 1 and 3, 4 and 6, 5 and 7
    const uint32_t M7 = 0x00070007u;
    const uint32_t dl[4] = {sc03 & M7, (sc03 >> 8) & M7, sc47 & M7, (sc47 >> 8) & M7};
    const uint32_t dh[4] = {(sc03 >> 3) & M7, (sc03 >> 11) & M7, (sc47 >> 3) & M7, (sc47 >> 11) & M7};
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const u32x4 c = b.c[P >> 1];
        const uint32_t w0 = (P & 1) ? c.z : c.x, w1 = (P & 1) ? c.w : c.y;
        const int at = P & 2, up = 16 * (P & 1);
        const uint32_t slo_a = dl[at] >> up, slo_b = dl[at + 1] >> up, shi_a = dh[at] >> up, shi_b = dh[at + 1] >> up;
        const uint32_t a0 = w0 & M4, a1 = w1 & M4, b0 = (w0 >> 4) & M4, b1 = (w1 >> 4) & M4;
        o.lo[P] = v4i{(int)scale_bytes(a0, slo_a), (int)scale_bytes(a1, slo_a), (int)scale_bytes(b0, slo_b), (int)scale_bytes(b1, slo_b)};
        o.hi[P] = v4i{(int)scale_bytes(a0, shi_a), (int)scale_bytes(a1, shi_a), (int)scale_bytes(b0, shi_b), (int)scale_bytes(b1, shi_b)};
    }
    // mins: the f16 MFMA's k = 4g + j is block sum 4g + j, which belongs to sub-block 2g + j/2
    const uint32_t mw = (g < 2) ? m03 : m47;
    const uint32_t ma = (mw >> (16 * (g & 1))) & 0xffu, mb = (mw >> (16 * (g & 1) + 8)) & 0xffu;
    o.mB = v4h{(_Float16)(int)ma, (_Float16)(int)ma, (_Float16)(int)mb, (_Float16)(int)mb};
    return o;
}

// Q6K: both planes of W = sc * (code - 32) (planes.hpp).
__device__ __forceinline__ BPlanes b_prepare_q6k(const BRegs& b, int lane) {
    const int g = lane >> 4;
    const uint32_t M4 = 0x0f0f0f0fu, M2H = 0x30303030u;
    BPlanes o;
    o.d = __half2float(__ushort_as_half((unsigned short)b.d16));
    o.dmin = 0.f;
    o.mB = v4h{0, 0, 0, 0};
    const uint32_t sel = (uint32_t)(g >> 1) * 8u;   // elements 8g .. 8g+7 of a 32-element stretch: its first or second 16
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const u32x4 c = b.c[P >> 1];
        const uint32_t w0 = (P & 1) ? c.z : c.x, w1 = (P & 1) ? c.w : c.y;
        const uint32_t h = b.qh[P], sw = b.hdr[P];
        // i8 scales of sub-blocks 4P + g/2 (first stretch of the pair) and 4P + 2 + g/2 (second), in both 16-bit lanes
        const int sa = __builtin_amdgcn_sbfe(sw, sel, 8), sb = __builtin_amdgcn_sbfe(sw, sel + 16u, 8);
        const uint32_t sa2 = __builtin_amdgcn_perm((uint32_t)sa, (uint32_t)sa, 0x05040100u);
        const uint32_t sb2 = __builtin_amdgcn_perm((uint32_t)sb, (uint32_t)sb, 0x05040100u);
        const uint32_t aa2 = pk_mad_u16(sa2, 0xffe0ffe0u, 0x00800080u), ab2 = pk_mad_u16(sb2, 0xffe0ffe0u, 0x00800080u);
        const uint32_t c0 = (w0 & M4) | ((h << 4) & M2H), c1 = (w1 & M4) | ((h << 2) & M2H);
        const uint32_t c2 = ((w0 >> 4) & M4) | (h & M2H), c3 = ((w1 >> 4) & M4) | ((h >> 2) & M2H);
        int l0, l1, l2, l3, h0, h1, h2, h3;
        q6k_planes(c0, sa2, aa2, l0, h0);
        q6k_planes(c1, sa2, aa2, l1, h1);
        q6k_planes(c2, sb2, ab2, l2, h2);
        q6k_planes(c3, sb2, ab2, l3, h3);
        o.lo[P] = v4i{l0, l1, l2, l3};
        o.hi[P] = v4i{h0, h1, h2, h3};
    }
    return o;
}

// Q5K (BlockQ5K::vec_dot, k_quants.rs:1394-1485): the Q4K sums on 5-bit codes.  A 3-bit digit times a code of up to 31
// no longer fits a signed byte, so the planes are the two bytes of W = sc * code (<= 1953), formed and cut as for Q6K
// (no offset: the minimum leaves through the block sums, as for Q4K).
__device__ __forceinline__ BPlanes b_prepare_q5k(const BRegs& b, int lane) {
    const int g = lane >> 4;
    const uint32_t M4 = 0x0f0f0f0fu, M1H = 0x10101010u;
    const uint32_t u0 = b.hdr.y, u1 = b.hdr.z, u2 = b.hdr.w;
    BPlanes o;
    o.d = __half2float(__ushort_as_half((unsigned short)(b.hdr.x & 0xffffu)));
    o.dmin = __half2float(__ushort_as_half((unsigned short)(b.hdr.x >> 16)));
    const uint32_t sc03 = u0 & 0x3f3f3f3fu;
    const uint32_t sc47 = (u2 & M4) | (((u0 >> 6) & 0x03030303u) << 4);
    const uint32_t m03 = u1 & 0x3f3f3f3fu;
    const uint32_t m47 = ((u2 >> 4) & M4) | (((u1 >> 6) & 0x03030303u) << 4);
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const u32x4 c = b.c[P >> 1];
        const uint32_t w0 = (P & 1) ? c.z : c.x, w1 = (P & 1) ? c.w : c.y;
        const uint32_t h = ((P < 2) ? b.q5.x : b.q5.y) >> (4 * (P & 1));
        const uint32_t scw = (P < 2) ? sc03 : sc47;
        const uint32_t sa = (scw >> (16 * (P & 1))) & 0xffu, sb = (scw >> (16 * (P & 1) + 8)) & 0xffu;
        const uint32_t sa2 = sa | (sa << 16), sb2 = sb | (sb << 16);
        const uint32_t c0 = (w0 & M4) | ((h << 4) & M1H), c1 = (w1 & M4) | ((h << 3) & M1H);
        const uint32_t c2 = ((w0 >> 4) & M4) | ((h << 2) & M1H), c3 = ((w1 >> 4) & M4) | ((h << 1) & M1H);
        int l0, l1, l2, l3, h0, h1, h2, h3;
        q6k_planes(c0, sa2, 0x00800080u, l0, h0);
        q6k_planes(c1, sa2, 0x00800080u, l1, h1);
        q6k_planes(c2, sb2, 0x00800080u, l2, h2);
        q6k_planes(c3, sb2, 0x00800080u, l3, h3);
        o.lo[P] = v4i{l0, l1, l2, l3};
        o.hi[P] = v4i{h0, h1, h2, h3};
    }
    const uint32_t mw = (g < 2) ? m03 : m47;
    const uint32_t ma = (mw >> (16 * (g & 1))) & 0xffu, mb = (mw >> (16 * (g & 1) + 8)) & 0xffu;
    o.mB = v4h{(_Float16)(int)ma, (_Float16)(int)ma, (_Float16)(int)mb, (_Float16)(int)mb};
    return o;
}

// Q3K (BlockQ3K::vec_dot, k_quants.rs:923-1047): d * y.d * sum_j sc_j * ((code_j - 4) . q8_j) with a signed 6-bit scale per
// 16 elements.  W = sc * (code - 4) lies in [-124, 128] -- one too many for a signed byte -- so it is formed and cut into two
// signed bytes exactly as the Q6K products are, W + 128 = code * sc + (128 - 4 sc); the high plane is zero but where W = 128.
__device__ __forceinline__ BPlanes b_prepare_q3k(const BRegs& b, int lane) {
    const int g = lane >> 4;
    const uint32_t M3 = 0x03030303u, M1H = 0x04040404u;
    BPlanes o;
    o.d = __half2float(__ushort_as_half((unsigned short)b.d16));
    o.dmin = 0.f;
    o.mB = v4h{0, 0, 0, 0};
    const uint32_t sel = (uint32_t)(g >> 1) * 8u;   // elements 8g .. 8g+7 of a 32-element stretch: its first or second 16
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const uint32_t q = b.c[0][P], sw = b.hdr[P];
        const uint32_t h = ((P < 2) ? b.q5.x : b.q5.y) >> (4 * (P & 1));
        const int sa = __builtin_amdgcn_sbfe(sw, sel, 8), sb = __builtin_amdgcn_sbfe(sw, sel + 16u, 8);
        const uint32_t sa2 = __builtin_amdgcn_perm((uint32_t)sa, (uint32_t)sa, 0x05040100u);
        const uint32_t sb2 = __builtin_amdgcn_perm((uint32_t)sb, (uint32_t)sb, 0x05040100u);
        const uint32_t aa2 = pk_mad_u16(sa2, 0xfffcfffcu, 0x00800080u), ab2 = pk_mad_u16(sb2, 0xfffcfffcu, 0x00800080u);
        const uint32_t c0 = (q & M3) | ((h << 2) & M1H), c1 = ((q >> 2) & M3) | ((h << 1) & M1H);
        const uint32_t c2 = ((q >> 4) & M3) | (h & M1H), c3 = ((q >> 6) & M3) | ((h >> 1) & M1H);
        int l0, l1, l2, l3, h0, h1, h2, h3;
        q6k_planes(c0, sa2, aa2, l0, h0);
        q6k_planes(c1, sa2, aa2, l1, h1);
        q6k_planes(c2, sb2, ab2, l2, h2);
        q6k_planes(c3, sb2, ab2, l3, h3);
        o.lo[P] = v4i{l0, l1, l2, l3};
        o.hi[P] = v4i{h0, h1, h2, h3};
    }
    return o;
}

// Q2K: the one plane sc * code (<= 45).  A lane's eight elements of a 32-element stretch lie in one 16-element sub-block
// (the first for chunks 0 and 1, the second for chunks 2 and 3), so each half of an MFMA operand takes one scale.
__device__ __forceinline__ BPlanes b_prepare_q2k(const BRegs& b, int lane) {
    const int g = lane >> 4;
    const uint32_t M3 = 0x03030303u;
    BPlanes o;
    o.d = __half2float(__ushort_as_half((unsigned short)(b.d16 & 0xffffu)));
    o.dmin = __half2float(__ushort_as_half((unsigned short)(b.d16 >> 16)));
    const int sel = 8 * (g >> 1);
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const uint32_t q = b.c[0][P], sw = b.hdr[P];
        const uint32_t s_a = (sw >> sel) & 0xFu, s_b = (sw >> (16 + sel)) & 0xFu;
        o.lo[P] = v4i{(int)scale_bytes(q & M3, s_a), (int)scale_bytes((q >> 2) & M3, s_a),
                      (int)scale_bytes((q >> 4) & M3, s_b), (int)scale_bytes((q >> 6) & M3, s_b)};
    }
    // mins: the f16 MFMA's k = 4g + j is block sum 4g + j = sub-block 4g + j
    const uint32_t mg = (b.hdr[g] >> 4) & 0x0f0f0f0fu;
    o.mB = v4h{(_Float16)(int)(mg & 0xffu), (_Float16)(int)((mg >> 8) & 0xffu), (_Float16)(int)((mg >> 16) & 0xffu), (_Float16)(int)(mg >> 24)};
    return o;
}

template <int FMT>
__device__ __forceinline__ BPlanes b_planes(const BRegs& r, int lane) {
    if constexpr (FMT == MOE_GGML_Q6K) return b_prepare_q6k(r, lane);
    else if constexpr (FMT == MOE_GGML_Q2K) return b_prepare_q2k(r, lane);
    else if constexpr (FMT == MOE_GGML_Q3K) return b_prepare_q3k(r, lane);
    else if constexpr (FMT == MOE_GGML_Q5K) return b_prepare_q5k(r, lane);
    else return b_prepare(r, lane);
}

// The matrix results of one 16-slot operand against the wave's J 16-row weight operands, on their way to the sums.
template <int J>
struct OperandAcc {
    v4i lo[J], hi[J];
    v4f dm[J], yd;
};
// Adds result i (slot 16 o + 4 g + i, weight rows n = lane%16 of its operands) of a super-block to the sums.
template <int FMT, int J>
__device__ __forceinline__ void gemm_result(const BPlanes (&B)[J], const OperandAcc<J>& A, int i, v4f (&facc)[J]) {
#pragma unroll
    for (int j = 0; j < J; j++) {
        if constexpr (FMT == MOE_GGML_Q6K || FMT == MOE_GGML_Q3K) {
            const int isum = (A.hi[j][i] << 8) + A.lo[j][i];
            facc[j][i] = __builtin_fmaf(B[j].d * A.yd[i], (float)isum, facc[j][i]);
        } else if constexpr (FMT == MOE_GGML_Q2K) {
            // the reference's own order, every product and the difference rounded (k_quants.rs:772-773, 801): with unsigned
            // 2-bit codes the two terms are large and nearly cancel, and the scalar path's sum has one order only -- a
            // wave walks K in that order, so the up projection repeats vec_dot_unopt bit for bit
            const float dall = A.yd[i] * B[j].d, dminy = A.yd[i] * B[j].dmin;
            facc[j][i] += dall * (float)A.lo[j][i] - dminy * A.dm[j][i];
        } else {
            const int isum = (A.hi[j][i] << (FMT == MOE_GGML_Q5K ? 8 : 3)) + A.lo[j][i];
            const float v = __builtin_fmaf(B[j].d, (float)isum, -(B[j].dmin * A.dm[j][i]));
            facc[j][i] = __builtin_fmaf(A.yd[i], v, facc[j][i]);
        }
        float f = facc[j][i];
        asm volatile("" : "+v"(f));   // the step stays where it is written
        facc[j][i] = f;
    }
}
__device__ __forceinline__ v4i operand_piece(const uint8_t* q, int o, int P, int lane) {
    return *reinterpret_cast<const v4i*>(q + o * 4096 + P * 1024 + lane * 16);
}
// One super-block of the wave's 16 J weight rows against operands O, O + 1, ... of the staged tile.  While the matrix
// instructions of an operand run, the wave's vector instructions add up the results of the operand before it (`prev`).
template <int FMT, int NOP, int LV, int O, int J, class Fill>
__device__ __forceinline__ void gemm_operands(const BPlanes (&B)[J], const GemmLds<NOP>& L, int buf, int lane, v4i (&a)[4], OperandAcc<J>& prev,
                                              v4f (&facc)[NOP][J], const Fill& fill) {
    const int m = lane & 15, g = lane >> 4;
    const v4i zero4 = {0, 0, 0, 0};
    OperandAcc<J> cur;
    v4h mA;
    if constexpr (FMT != MOE_GGML_Q6K && FMT != MOE_GGML_Q3K) mA = *reinterpret_cast<const v4h*>(&L.bs[buf][O][g >> 1][m][(g & 1) * 4]);
    cur.yd = *reinterpret_cast<const v4f*>(&L.yd[buf][O * 16 + g * 4]);
#pragma unroll
    for (int P = 0; P < 4; P++) {
        const v4i x = a[P];
#pragma unroll
        for (int j = 0; j < J; j++) {
            cur.lo[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, B[j].lo[P], P == 0 ? zero4 : cur.lo[j], 0, 0, 0);
            if constexpr (FMT != MOE_GGML_Q2K) cur.hi[j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(x, B[j].hi[P], P == 0 ? zero4 : cur.hi[j], 0, 0, 0);
        }
        if constexpr (O + 1 < LV) a[P] = operand_piece(L.q[buf], O + 1, P, lane);
        if constexpr (O > 0) gemm_result<FMT, J>(B, prev, P, facc[O - 1]);
        // order: a matrix instruction (mask 0x8), three vector instructions (0x2), and so on
        if constexpr (J == 2) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 3, 0);
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 9, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (P == 0) fill(std::integral_constant<int, O>{});
    }
    if constexpr (FMT != MOE_GGML_Q6K && FMT != MOE_GGML_Q3K) {
        const v4f zf = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < J; j++) cur.dm[j] = __builtin_amdgcn_mfma_f32_16x16x16f16(mA, B[j].mB, zf, 0, 0, 0);
    }
    prev = cur;
    if constexpr (O + 1 < LV) {
        gemm_operands<FMT, NOP, LV, O + 1, J>(B, L, buf, lane, a, prev, facc, fill);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; i++) gemm_result<FMT, J>(B, prev, i, facc[O]);
}

__device__ __forceinline__ float silu_gemm(float v) { return v / (1.0f + __expf(-v)); }

// ---------------------------------------------------------------------------------------------
// J 16-row weight operands per wave, NW waves per workgroup, 4 / J waves per SIMD; a tile of NOP*16 slots.
// MODE 0: up   -- a wave carries 16 rows of w1 and the same 16 rows of w3 (J = 2) and writes h = silu(a) * b (f32).
// MODE 1: down -- 16 J rows of w2 per wave; writes yw.
// FMT: the weights' format (Q2K ... Q6K).  KS: parts the waves of a workgroup cut K into.
template <int FMT, int MODE, int NOP, int NW, int J, int KS = 1>
__global__ __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(4 / J, 4 / J))) void q4k_gemm_kernel(ExpertParams p) {
    static_assert(J == 2 || (J == 1 && MODE == 1), "the up projection takes w1 and w3 side by side");
    static_assert(KS == 1 || (MODE == 1 && NW % KS == 0 && NOP % KS == 0), "the up projection's waves walk all of K");
    static_assert(FMT == MOE_GGML_Q2K || FMT == MOE_GGML_Q3K || FMT == MOE_GGML_Q4K || FMT == MOE_GGML_Q5K || FMT == MOE_GGML_Q6K, "formats of the tiled kernel");
    constexpr int NWR = NW / KS;    // waves that share a part of K, each with rows of its own
    constexpr int NB = NOP * 4 / NWR;
    static_assert(NOP / 2 <= NWR, "one transfer of block sums per wave");
    constexpr int TILE_BYTES = FMT == MOE_GGML_Q6K ? Q6K_TILE_BYTES : FMT == MOE_GGML_Q5K ? Q5K_TILE_BYTES : FMT == MOE_GGML_Q2K ? Q2K_TILE_BYTES : FMT == MOE_GGML_Q3K ? Q3K_TILE_BYTES : Q4K_TILE_BYTES;
    constexpr bool kSums = FMT != MOE_GGML_Q6K && FMT != MOE_GGML_Q3K;   // block sums staged (the mins term)
    __shared__ GemmLds<NOP> L_all[KS];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = KS == 1 ? wave_id : wave_id % NWR, kpart = KS == 1 ? 0 : wave_id / NWR;
    GemmLds<NOP>& L = L_all[kpart];
    const int n_tiles = p.rb.tile_tab[0];
    // workgroup -> (row block, slot tile), in patches per XCD (patch_position)
    const int n_rb = MODE == 0 ? p.F / (16 * NW) : p.H / (16 * J * NWR);
    const PatchPos pos = patch_position((int)blockIdx.x, n_rb, p.patch);
    const int rblk = pos.rblk, tile = pos.tile;
    if (tile >= n_tiles || rblk >= n_rb) return;
    const int gi = p.rb.tile_tab[1 + 2 * tile], pos0 = p.rb.tile_tab[2 + 2 * tile];
    if (gi < p.group0 || gi >= p.group0 + p.n_groups) return;
    const int grp = gi - p.group0;
    const int s_begin = p.rb.offsets[gi], n_g = p.rb.offsets[gi + 1] - s_begin;
    const int K = MODE == 0 ? p.H : p.F;        // reduction length
    const int N = MODE == 0 ? p.F : p.H;        // weight rows of the matrix
    const int nsb = K / 256;
    const size_t sb_stride = (size_t)(N / 16) * TILE_BYTES;
    const ActBuf& ab = MODE == 0 ? p.xq : p.hq;

    // activation row behind position r of the tile (positions past the expert's list repeat its last row)
    auto act_row = [&](int r) {
        const int pos = pos0 + r;
        const int slot = s_begin + (pos < n_g ? pos : n_g - 1);
        return MODE == 0 ? p.rb.perm_token[slot] : slot - p.slot_origin;
    };
    StageRows<NB> rows;
#pragma unroll
    for (int c = 0; c < (NB + 3) / 4; c++) rows.q[c] = (uint32_t)act_row(16 * (((wave * NB) >> 2) + c) + (lane & 15)) * (uint32_t)K + (lane >> 4) * 16;
    rows.bs = ((uint32_t)act_row(32 * (wave % (NOP / 2)) + 16 * (lane >> 5) + (lane & 15)) * (uint32_t)nsb * 16 + ((lane >> 4) & 1) * 8) * 2;
    rows.yd = (uint32_t)act_row(64 * (wave % (NOP / 4)) + lane) * (uint32_t)nsb * 4;

    // weight operands of this wave
    const GroupWeights gw = p.groups[grp];
    const int row0 = (rblk * NWR + wave) * (MODE == 0 ? 16 : 16 * J);
    const uint8_t* wp[J];
    if (MODE == 0) {
        wp[0] = gw.w1 + (size_t)(row0 / 16) * TILE_BYTES;
        wp[J - 1] = gw.w3 + (size_t)(row0 / 16) * TILE_BYTES;
    } else {
#pragma unroll
        for (int j = 0; j < J; j++) wp[j] = gw.w2 + (size_t)(row0 / 16 + j) * TILE_BYTES;
    }
    v4f facc[NOP][J];
#pragma unroll
    for (int o = 0; o < NOP; o++)
#pragma unroll
        for (int j = 0; j < J; j++) facc[o][j] = v4f{0.f, 0.f, 0.f, 0.f};

    // operands of the tile that hold slots of the list: a short tile's others are neither fetched nor multiplied
    const int live = __builtin_amdgcn_readfirstlane(min(NOP, (n_g - pos0 + 15) >> 4));
    // the super-blocks of this wave's part of K
    const int sb_lo = KS == 1 ? 0 : kpart * (nsb / KS) + min(kpart, nsb % KS), n_sb = KS == 1 ? nsb : nsb / KS + (kpart < nsb % KS ? 1 : 0);
    const int n_steps = (nsb + KS - 1) / KS;
    const int sb_first = KS == 1 ? 0 : min(sb_lo, nsb - 1);   // (fewer super-blocks than parts: requested, never multiplied)
    auto stage = [&](auto I, int sb, int buf) { stage_piece<decltype(I)::value, kSums, NOP, NB>(ab, rows, sb, L, buf, wave, live); };
    static_for<0, NB + 2>([&](auto I) { stage(I, sb_first, 0); });
    BRegs raw[J];
#pragma unroll
    for (int j = 0; j < J; j++) raw[j] = b_load<FMT>(wp[j] + (size_t)sb_first * sb_stride, lane);
    wait_all_loads();
    __syncthreads();
    // the K loop over LV operands
    auto run = [&](auto lv_tag) {
        constexpr int LV = decltype(lv_tag)::value;
        for (int it = 0; it < n_steps; it++) {
            const int buf = it & 1, nb = buf ^ 1;
            const int sb = sb_lo + it, sbn = it + 1 < n_sb ? sb + 1 : sb;
            if (KS == 1 || it < n_sb) {   // (wave-uniform: a part may be one super-block shorter)
                BPlanes B[J];
#pragma unroll
                for (int j = 0; j < J; j++) B[j] = b_planes<FMT>(raw[j], lane);
                // (for the sake of the registers the next weights are requested after this super-block's are unpacked)
                __builtin_amdgcn_sched_barrier(0);
                v4i a[4];
#pragma unroll
                for (int P = 0; P < 4; P++) a[P] = operand_piece(L.q[buf], 0, P, lane);
                OperandAcc<J> prev;
                // The next super-block's weights and activations are requested while the operands are multiplied, a few requests at a
                // time: issued in one go they fill the CU's memory queue and the wave stands still for a thousand cycles and more.
                gemm_operands<FMT, NOP, LV, 0, J>(B, L, buf, lane, a, prev, facc, [&](auto o_tag) {
                    constexpr int O = decltype(o_tag)::value;
                    // (four waves per SIMD: a format with block sums has registers for the next weights behind its last operand only)
                    if constexpr (O == (J == 1 && kSums ? LV - 1 : 0)) raw[0] = b_load<FMT>(wp[0] + (size_t)sbn * sb_stride, lane);
                    if constexpr (J == 2 && O == (LV > 2 ? 1 : 0)) raw[J - 1] = b_load<FMT>(wp[J - 1] + (size_t)sbn * sb_stride, lane);
                    constexpr int FIRST = LV > 2 ? 1 : 0, SPAN = LV > 4 ? LV - 3 : 1;
                    static_for<0, NB + 2>([&](auto I) {
                        if constexpr (FIRST + decltype(I)::value * SPAN / (NB + 2) == O) stage(I, sbn, nb);
                    });
                });
            }
            wait_all_loads();
            __syncthreads();
        }
    };
    static_for<1, NOP + 1>([&](auto lv_tag) {
        constexpr int LV = decltype(lv_tag)::value;
        if (live == LV) run(lv_tag);
    });

    // epilogue: lane holds weight row n = lane%16 of its operands and slots 16 o + 4 (lane/16) + i
    const int n = lane & 15, g = lane >> 4;
    if constexpr (KS > 1) {
        // the parts' sums meet in LDS (the loop's last barrier has released it); the waves of part q add up, in the order of the
        // parts, and store operands q NOP / KS ...
        float* xch = reinterpret_cast<float*>(L_all);   // [wave][operand][j][i][lane]
        static_assert(NW * NOP * J * 4 * 64 * sizeof(float) <= sizeof(L_all), "exchange area");
#pragma unroll
        for (int o = 0; o < NOP; o++)
#pragma unroll
            for (int j = 0; j < J; j++)
#pragma unroll
                for (int i = 0; i < 4; i++) xch[(((wave_id * NOP + o) * J + j) * 4 + i) * 64 + lane] = facc[o][j][i];
        __syncthreads();
#pragma unroll
        for (int oo = 0; oo < NOP / KS; oo++) {
            const int o = kpart * (NOP / KS) + oo;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int pos = pos0 + o * 16 + g * 4 + i;
                if (pos >= n_g) continue;
                const int slot = s_begin + pos;
                const float w = p.rb.perm_w[slot];
#pragma unroll
                for (int j = 0; j < J; j++) {
                    float sum = 0.f;
#pragma unroll
                    for (int q = 0; q < KS; q++) {
                        const float part = xch[((((q * NWR + wave) * NOP + o) * J + j) * 4 + i) * 64 + lane];
                        sum = q == 0 ? part : sum + part;
                    }
                    p.yw[(int64_t)slot * p.H + row0 + 16 * j + n] = sum * w;
                }
            }
        }
        return;
    }
#pragma unroll
    for (int o = 0; o < NOP; o++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int pos = pos0 + o * 16 + g * 4 + i;
            if (pos >= n_g) continue;
            const int slot = s_begin + pos;
            if (MODE == 0) {
                p.hbuf[(int64_t)(slot - p.slot_origin) * p.F + row0 + n] = silu_gemm(facc[o][0][i]) * facc[o][J - 1][i];
            } else {
                const float w = p.rb.perm_w[slot];
#pragma unroll
                for (int j = 0; j < J; j++) p.yw[(int64_t)slot * p.H + row0 + 16 * j + n] = facc[o][j][i] * w;
            }
        }
}

template <int FMT, int MODE>
static void launch_gemm(ExpertParams& p, hipStream_t s) {
    const int64_t tiles = max_gemm_tiles(p.n_slots, p.n_groups + 1, p.rb.tile_slots);
    const int64_t rows = MODE == 0 ? 2 * (int64_t)p.F : p.H;
    // Down launches in tiles of 64 slots whose weights take long to unpack (Q3K, Q5K, Q6K): one operand per wave, four waves per
    // SIMD.  Their unpacking serves four operands only, and two waves cannot cover each other's: with two operands per
    // wave they were slower at every width (us, best width / this: Q6_K 1024 x 4096 at 2048 rows 48.1 / 45.0, 4096 x 14336 at 512
    // 126 / 115, 14336 x 4096 at 300 82.2 / 78.6, Q3_K 4096 x 4096 at 512 42.9 / 40.4, Q5_K 1024 x 4096 at 2048 50.0 / 48.6).  Q4_K and Q2_K
    // lose by it (4096 x 4096 at 1500 rows 90 / 103 and 79 / 92).
    constexpr bool one_operand = MODE == 1 && (FMT == MOE_GGML_Q3K || FMT == MOE_GGML_Q5K || FMT == MOE_GGML_Q6K);
    const bool tiles64 = p.rb.tile_slots == 64;
    auto launch = [&](auto kernel, int waves, int64_t wg_rows) {
        const int64_t n_rb = rows / wg_rows;
        p.patch = patch_edge(n_rb, tiles);
        hipLaunchKernelGGL(kernel, dim3(patch_grid(n_rb, tiles, p.patch)), dim3(waves * 64), 0, s, p);
    };
    // K split over the waves of a workgroup where the grid would leave SIMDs with one wave or none (gemm_plan)
    if constexpr (MODE == 1) {
        const int parts = p.k_parts ? p.k_parts : gemm_plan(gemm_format(FMT), false, rows, p.F, p.n_slots, p.n_groups, p.rb.tile_slots, tiles).parts;
        if (parts == 4 && tiles64) return launch(q4k_gemm_kernel<FMT, 1, 4, 8, 2, 4>, 8, 64);
        if (parts == 2) return tiles64 ? launch(q4k_gemm_kernel<FMT, 1, 4, 8, 2, 2>, 8, 128) : launch(q4k_gemm_kernel<FMT, 1, 8, 8, 2, 2>, 8, 128);
    }
    const bool wide = !(one_operand && tiles64) && gemm_wide(MODE == 0, rows, p.n_slots, p.n_groups, p.rb.tile_slots, tiles);
    if (!tiles64) {
        if (wide) launch(q4k_gemm_kernel<FMT, MODE, 8, 8, 2>, 8, 256);
        else launch(q4k_gemm_kernel<FMT, MODE, 8, 4, 2>, 4, 128);
    } else if constexpr (one_operand) {
        launch(q4k_gemm_kernel<FMT, MODE, 4, 8, 1>, 8, 128);
    } else if constexpr (MODE == 0) {
        launch(q4k_gemm_kernel<FMT, MODE, 4, 4, 2>, 4, 128);
    } else {
        if (wide) launch(q4k_gemm_kernel<FMT, MODE, 4, 8, 2>, 8, 256);
        else launch(q4k_gemm_kernel<FMT, MODE, 4, 4, 2>, 4, 128);
    }
}
bool q4k_gemm_up_format(int dt) { return dt == MOE_GGML_Q2K || dt == MOE_GGML_Q3K || dt == MOE_GGML_Q4K || dt == MOE_GGML_Q5K || dt == MOE_GGML_Q6K; }
bool q4k_gemm_down_format(int dt) { return q4k_gemm_up_format(dt); }
hipError_t launch_q4k_gemm_up(const ExpertParams& p_in, hipStream_t s) {
    ExpertParams p = p_in;
    if (p.dt == MOE_GGML_Q6K) launch_gemm<MOE_GGML_Q6K, 0>(p, s);
    else if (p.dt == MOE_GGML_Q5K) launch_gemm<MOE_GGML_Q5K, 0>(p, s);
    else if (p.dt == MOE_GGML_Q4K) launch_gemm<MOE_GGML_Q4K, 0>(p, s);
    else if (p.dt == MOE_GGML_Q2K) launch_gemm<MOE_GGML_Q2K, 0>(p, s);
    else if (p.dt == MOE_GGML_Q3K) launch_gemm<MOE_GGML_Q3K, 0>(p, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}
hipError_t launch_q4k_gemm_down(const ExpertParams& p_in, hipStream_t s) {
    ExpertParams p = p_in;
    const int dtd = p.dt_down ? p.dt_down : p.dt;
    if (dtd == MOE_GGML_Q6K) launch_gemm<MOE_GGML_Q6K, 1>(p, s);
    else if (dtd == MOE_GGML_Q5K) launch_gemm<MOE_GGML_Q5K, 1>(p, s);
    else if (dtd == MOE_GGML_Q4K) launch_gemm<MOE_GGML_Q4K, 1>(p, s);
    else if (dtd == MOE_GGML_Q2K) launch_gemm<MOE_GGML_Q2K, 1>(p, s);
    else if (dtd == MOE_GGML_Q3K) launch_gemm<MOE_GGML_Q3K, 1>(p, s);
    else return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace moe
