// The grids of the tiled kernels: how row blocks and slot tiles are dealt to the XCDs, how wide the workgroups of a K-quant
// launch are and whether their waves share K, and which slot tile a product takes.  Plain C++: no HIP types.
#pragma once
#include <algorithm>
#include <cstdint>

#include "../../include/candle_amd_moe.h"

namespace moe {

constexpr int GEMM_MIN_TILE_SLOTS = 64;  // smallest tile of the tiled expert kernels
inline int64_t max_gemm_tiles(int64_t slots, int64_t groups, int tile_slots = GEMM_MIN_TILE_SLOTS) { return slots / tile_slots + groups + 1; }

// Tiled kernels: workgroup id -> (row block, slot tile).  Hardware hands consecutive workgroup ids to the eight XCDs in
// turn, each with its own L2; the ids that land on one XCD are walked in patches of edge x edge (row blocks x tiles), so
// that the workgroups an XCD runs at a time share their weight rows and their activation tiles through that L2.  The
// edge is 8 when that still gives every XCD at least two patches, else 4 or 2: a grid of a few hundred workgroups cut
// into 8 x 8 patches would leave XCDs without work.
struct PatchPos { int rblk, tile; };
// `patch` = rows edge + 256 * tiles edge (a tiles edge of 0: a square patch)
constexpr PatchPos patch_position(int block, int n_rb, int patch) {
    const int er = patch & 255, et = (patch >> 8) ? (patch >> 8) : er;
    const int per = er * et, RG = (n_rb + er - 1) / er;
    const int xcd = block & 7, q = block >> 3;
    const int st = (q / per) * 8 + xcd, within = q % per;
    return PatchPos{(st % RG) * er + within % er, (st / RG) * et + within / er};
}
inline int patch_edge(int64_t n_rb, int64_t tiles) {
    for (int e = 8; e > 2; e >>= 1)
        if (((n_rb + e - 1) / e) * ((tiles + e - 1) / e) >= 16) return e;
    return 2;
}
// One group of a few tiles (the always-on expert, a dense product): a patch holds every tile of its row blocks, so that
// each weight row is fetched into one XCD's L2 only (square patches of 4 x 4 fetched the rows of eight tiles twice).
inline int patch_all_tiles(int64_t n_rb, int64_t tiles) {
    if (tiles < 1 || tiles > 16) return patch_edge(n_rb, tiles);
    int er = 4;
    while (er > 1 && (n_rb + er - 1) / er < 16) er >>= 1;
    return er + 256 * (int)tiles;
}
inline unsigned patch_grid(int64_t n_rb, int64_t tiles, int patch) {
    const int er = patch & 255, et = (patch >> 8) ? (patch >> 8) : er;
    const int64_t RG = (n_rb + er - 1) / er, TG = (tiles + et - 1) / et;
    return (unsigned)((RG * TG + 7) / 8 * 8 * er * et);
}

// Slot tiles of a launch.  One list (a dense product): exact.  Several: the host does not know their lengths; they are taken
// as spread evenly from 7/8 to 9/8 of their mean.  (Half a tile per list beyond the full ones would be right for lists of any
// length, but lists around one mean end at the same place of a tile: eight of about 218 slots fill 16 tiles of 128, not 17.)
inline int64_t gemm_tiles(int64_t slots, int64_t groups, int tile_slots) {
    if (groups <= 1) return (slots + tile_slots - 1) / tile_slots;
    int64_t sum = 0;   // over eight lengths, in units of 1/8 list each
    for (int i = 0; i < 8; i++) {
        const int64_t len = slots * (57 + 2 * i) / (64 * groups);
        sum += (len + tile_slots - 1) / tile_slots;
    }
    return (sum * groups + 4) / 8;
}

// Workgroups that the busiest XCD gets of a grid of n_rb row blocks and `max_tiles` tiles, `tiles` of them live.
inline int64_t busiest_xcd(int64_t n_rb, int64_t tiles, int64_t max_tiles) {
    const int64_t e = patch_edge(n_rb, max_tiles), RG = (n_rb + e - 1) / e, TG = (tiles + e - 1) / e;
    int64_t n[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t st = 0; st < RG * TG; st++)
        n[st % 8] += std::min(e, n_rb - st % RG * e) * std::min(e, tiles - st / RG * e);
    return *std::max_element(n, n + 8);
}

// A workgroup of eight waves (256 weight rows) takes a CU, one of four waves (128 rows) half of one.  The wide ones fetch an
// activation tile half as often: 2 to 7 % on full rounds.  But an XCD's 32 CUs hold 32 of them at a time, and a last
// round that hardly fills takes as long as a full one, where up to 32 narrow workgroups have a CU each and are done in half
// the time of 64.  So both are counted in rounds of the busiest XCD, the narrow ones in halves and at 5 % more a round.
// (In the second round a half holds no more than 24: the dead tiles of the patches leave CUs out while others take two.)
//   Dense products, us wide / narrow: Q4_K 4096 x 4096 at 512 rows, 0.5 rounds 46.5 / 38.6; 576 rows, 0.56: 47.4 / 51.3; 1024, 1.0:
//   52.3 / 55.6; 2800, 1.5 / 1.38: 150 / 130; 3000, 1.5 / 2.0: 152 / 161; 14336 x 4096 at 300, 1.25 / 1.19: 79.6 / 70.4; 1450, 3.0: 221 / 227;
//   1664, 3.12 / 3.25: 282 / 258; 32000 x 4096 at 300, 1.5: 105 / 125; 640, 2.5: 211 / 193; Q6_K 640 238 / 212.
//   Mixtral shape, us per step: down, 450 tokens, 0.5 rounds 523 / 471; 500 tokens 0.69: 589 / 615; 600 tokens, 1.0: 648 / 667; 1000
//   tokens, 1.38: 1032 / 984; 2048 tokens, 2.5: 1701 / 1653; up, 301 tokens, 4.0: 375 / 388; 1000 tokens, 9.5 / 8.5: 1030 / 999.
//   up to 512 rows: always narrow.  One or two wide row blocks leave most of a patch dead, and a CU that is offered a dead wide
//   workgroup takes nothing else (Q4_K 512 x 4096 at 16384 rows 187 / 138, 256 x 256 at 60000 115 / 68; 768 x 4096 191 / 195).
//   up projection in tiles of 64 slots: always narrow.  Its lists are short and uneven, and the finer grid shares them out better
//   (Mixtral shape, 137 / 257 / 287 tokens: Q4_K 280 / 273, 416 / 406, 454 / 433; Q6_K 257 tokens 547 / 521; Q3_K 495 / 470;
//   200 tokens: Q4_K 318 / 323, Q6_K 479 / 457).
// rows: weight rows of the launch (w1 and w3 both counted); groups: expert lists, 1 for a dense product; max_tiles: the grid's tiles.
inline bool gemm_wide(bool up, int64_t rows, int64_t slots, int64_t groups, int tile_slots, int64_t max_tiles) {
    if (rows % 256 || rows <= 512 || (up && tile_slots == 64)) return false;
    const int64_t tiles = std::min(gemm_tiles(slots, groups, tile_slots), max_tiles);
    if (rows / 256 * tiles > 12 * 256) return true;   // a tail is less than 5 % of so many rounds
    const int64_t wide = (busiest_xcd(rows / 256, tiles, max_tiles) + 31) / 32;
    const int64_t narrow = busiest_xcd(rows / 128, tiles, max_tiles), full = narrow / 64, tail = narrow % 64;
    const int64_t halves = 2 * full + (tail == 0 ? 0 : tail <= (full == 1 ? 24 : 32) ? 1 : 2);
    return halves * 21 >= wide * 40;
}

// What a tiled launch takes, in us, for choosing between its variants.  A workgroup of eight waves (two per SIMD) needs
//     0.31 us per super-block and 256 weight rows, times (16-slot operands that hold slots + `unpack`),
// where `unpack` is what the unpacking of a weight costs beside the product with one operand (GemmFormat below), and 3 us
// around its K loop; workgroups come in rounds of 32 on the busiest XCD.  Two workgroups of four waves share a CU at 5 % more; one alone
// takes 0.85 of such a pair's time, which is what makes small grids slow: a wave alone leaves half of its SIMD's cycles
// empty.  So where a launch would have one of them per CU, the four row groups of a workgroup are given to eight waves, four for
// each half of K (or two row groups to eight waves, a quarter of K each), and the sums meet in LDS: half (a quarter of) the K
// steps with every SIMD full, 10 % more per step for the activations fetched per row and 6 us around the loop.
// Against measurements (2043 dense products of 96 to 3000 rows, 3378 layers of 4 to 160 experts with 34 to 500 rows each, the five
// formats, even and skewed lists, every variant timed at each) the choices by this file are 1.7 % off the best variant on average, 5 % of
// the layers and 1.4 % of the products 3 % or more slower than by fixed lines (tiled down projections from 64 rows per expert on, 128
// slots from 72; tiled products from 192 workgroups on, 128 slots from 512; one part), and the mean 7.5 % and 6 % faster.  One part / the
// choice: Q4_K 4096 x 4096 at 384 rows 36.8 / 31.6, at 777 51.2 / 45.4, 4096 x 14336 at 512 rows 107 / 90, 14336 x 4096 at 128
// 47 / 32; Q6_K 4096 x 4096 at 777 58.1 / 49.1; at a full chip it costs: Q4_K 4096 x 4096 at 4096 rows 161 / 181.
struct GemmPlan {
    int parts;    // parts K is cut into: 1 (workgroups as gemm_wide says), 2 (128-row workgroups), 4 (64-row ones, tiles of 64 slots)
    double us;
};
// What a workgroup of 64 rows and a pass of the streaming down kernels takes, in us times the CUs: around its K loop, per super-block, and
// one that finds no slots; dense: of the dense products' rate below.
struct StreamCost { double wg, step, empty, dense; };
// format traits of the tiled kernel: unpack, in operands; one_operand: launches in tiles of 64 slots have one 16-row weight
// operand per wave; crowded: with 128 slots and the two accumulator sets of a split the registers overflow beyond 96 slots
struct GemmFormat {
    double unpack;
    bool one_operand, crowded;
    bool four_tiles;   // the streaming kernels carry 64 slots per pass, not 32
    StreamCost stream;
};
// (the unpacking measured beside the product with one 16-slot operand)
inline GemmFormat gemm_format(int dt) {
    const bool one_operand = dt == MOE_GGML_Q3K || dt == MOE_GGML_Q5K || dt == MOE_GGML_Q6K;
    const StreamCost s = dt == MOE_GGML_Q2K ? StreamCost{2.6, 0.44, 0.18, 0.78} : dt == MOE_GGML_Q3K ? StreamCost{2.0, 0.62, 0.19, 1.0}
                       : dt == MOE_GGML_Q4K ? StreamCost{5.0, 0.78, 0.5, 1.0}  : dt == MOE_GGML_Q5K ? StreamCost{2.4, 0.63, 0.19, 1.0}
                                                                               : StreamCost{2.3, 0.71, 0.185, 1.0};
    return GemmFormat{one_operand ? 5.0 : 2.5, one_operand, dt == MOE_GGML_Q5K, dt == MOE_GGML_Q4K, s};
}
inline GemmPlan gemm_plan(const GemmFormat& f, bool up, int64_t rows, int64_t k, int64_t slots, int64_t groups, int tile_slots, int64_t max_tiles) {
    const int64_t nsb = k / 256, tiles = std::min(gemm_tiles(slots, groups, tile_slots), max_tiles);
    // 16-slot operands of a tile: of the longest of a dense product, on average over lists
    const double ops = groups <= 1 ? (double)std::min<int64_t>(tile_slots / 16, (slots + 15) / 16)
                                   : std::min((double)tile_slots / 16, (double)gemm_tiles(slots, groups, 16) / (double)std::max<int64_t>(1, tiles));
    const double step = 0.155 * (f.unpack + ops);   // 128 rows, one super-block
    auto rounds = [&](int64_t wg_rows) { return (double)((busiest_xcd(rows / wg_rows, tiles, max_tiles) + 31) / 32); };
    if (rows / 256 * tiles > 12 * 256) return GemmPlan{1, (double)(rows / 256 * tiles) / 256.0 * (2 * step * nsb + 3)};   // a tail hardly counts
    GemmPlan best{1, 0};
    const bool one_operand = f.one_operand && !up && tile_slots == 64;
    if (!one_operand && gemm_wide(up, rows, slots, groups, tile_slots, max_tiles)) {
        best.us = rounds(256) * (2 * step * nsb + 3);
    } else {
        const int64_t n = busiest_xcd(rows / 128, tiles, max_tiles), full = n / 64, tail = n % 64;
        const double pair = 2.1 * step * nsb + 3, lone = (one_operand ? 1.5 : 1.7) * step * nsb + 3;
        best.us = full * pair + (tail == 0 ? 0 : tail <= 32 ? lone : pair);
    }
    if (up) return best;
    const double r2 = rounds(128);
    const double two = r2 * ((r2 > 1 ? 1.2 : 1.1) * (f.crowded && ops > 6 ? 1.5 : 1.0) * step * 2 * (double)((nsb + 1) / 2) + 6);
    if (two < best.us) best = GemmPlan{2, two};
    if (tile_slots == 64 && rows % 64 == 0) {
        const double four = rounds(64) * (0.65 * step * 4 * (double)((nsb + 3) / 4) + 6);
        if (four < best.us) best = GemmPlan{4, four};
    }
    return best;
}
// The streaming down kernels, in us.  They give a workgroup 64 rows and a pass of 64 slots (four_tiles: Q4K) or 32.
//   Over expert lists the grid holds a pass for every 64 (32) tokens there could be in a list, most of them empty, and workgroups end at
//   different times: no rounds.  Few super-blocks cost little more than one (F = 256, where tiled and streamed looked alike without the
//   two constants: 3840 -> 256, 34 experts, Q4_K, 3089 tokens, step, tiled / streamed 195 / 511; 768 -> 256, 42 experts, 5591 tokens 82 / 191).
inline double streamed_lists_us(const GemmFormat& f, int64_t rows, int64_t k, int64_t tokens, int64_t slots, int64_t groups) {
    const int64_t nsb = k / 256, pass = f.four_tiles ? 64 : 32;
    const int64_t live = rows / 64 * gemm_tiles(slots, groups, (int)pass), all = rows / 64 * groups * ((tokens + pass - 1) / pass);
    return 4 + std::max(1.0, (double)live / 256) * (f.stream.wg + f.stream.step * (double)nsb) * (live <= 64 ? 0.65 : 1.0) +
           f.stream.empty * (double)std::max<int64_t>(0, all - live) / 256;
}
//   Dense products: rounds of a workgroup per CU, 1.07 us per super-block (Q4K), or only the number of (16 rows x 32 slots) products counts,
//   0.83 ns each (Q2K 0.65: 1024 x 14336 at 480 rows 49, four parts of 64 slots 61).
inline double streamed_us(const GemmFormat& f, int64_t rows, int64_t k, int64_t slots) {
    const int64_t nsb = k / 256, passes = gemm_tiles(slots, 1, f.four_tiles ? 64 : 32);
    if (!f.four_tiles) return 2 + 0.83e-3 * f.stream.dense * (double)(rows / 16 * passes) * (0.95 * (double)nsb + 1);
    const int64_t wgs = rows / 64 * passes;
    return 2 + (double)((wgs + 255) / 256) * (1.07 * (double)nsb + 0.5) * (wgs <= 64 ? 0.65 : 1.0);
}
// A routed layer (w1 and w3 of F rows each over H, w2 of H rows over F): the slots per tile, 64 or 128, by the sum of its two
// launches, and whether the down projection is tiled as well.  (Mixtral shape, us per step, 64 / 128: Q4_K 40 rows per expert
// 282 / 281, 50 rows 308 / 302, 60 rows 388 / 323, 75 rows 437 / 354; a quarter of its width: 75 rows 60 / 69, 125 rows 76 / 92, 250 rows
// 126 / 115.  The down launch alone, streamed / tiled: Q4_K 25 rows 69 / 69, 34 rows 99 / 83, 50 rows 112 / 93; Q6_K 34 rows 145 / 105,
// 50 rows 173 / 118; a quarter of the width Q4_K 35 rows 20 / 17, Q6_K 35 rows 19 / 21, 75 rows 27 / 23.)
// The costs know the mean of the lists only.  What that leaves uncertain goes to the side where the loss is small: 128 slots below 40 rows
// per expert where they promise a tenth (1280 -> 3584, 15 experts, Q5_K, 562 tokens, Zipf loads, 64 / 128 90 / 117), and no streaming
// beyond 200, where the longest list decides (256 -> 7168, 16 experts, top-1, Q4_K, 4857 tokens, Zipf loads, tiled / streamed 199 / 331).
struct LayerPlan {
    int tile_slots;
    bool tiled_down;
};
inline LayerPlan gemm_layer_plan(const GemmFormat& f_up, const GemmFormat& f_down, int64_t H, int64_t F, int64_t tokens, int64_t top_k, int64_t groups) {
    const int64_t slots = tokens * top_k;
    const double streamed = slots > 200 * groups ? 1e30 : streamed_lists_us(f_down, H, F, tokens, slots, groups);
    LayerPlan best{64, false};
    double us = 0;
    for (int tile = 64; tile <= 128; tile *= 2) {
        const int64_t max_tiles = max_gemm_tiles(slots, groups + 1, tile);
        const double down = gemm_plan(f_down, false, H, F, slots, groups, tile, max_tiles).us;
        const double t = gemm_plan(f_up, true, 2 * F, H, slots, groups, tile, max_tiles).us + std::min(down, streamed);
        if (tile == 64 || t <= us * (slots < 40 * groups ? 0.9 : 1.0)) { best = LayerPlan{tile, down <= streamed}; us = t; }
    }
    return best;
}
// Slots per tile of a dense product of m rows with an [n, k] matrix, or 0 where the streaming kernels are faster.  (us, streamed /
// tiled: Q4_K 4096 x 4096 at 256 rows 24.9 / 25.0, 320 36 / 31; 1024 x 4096 at 256 18.8 / 23.1, 512 25.6 / 25.3; 14336 x 4096 at
// 96 38.7 / 29.4; Q6_K 4096 x 4096 at 128 rows 19.7 / 24.4, 192 28.6 / 25.3; 14336 x 4096 at 96 41.4 / 35.8; Q4_K 4096 x 512 at 440 18.3 / 10.7.)
// On a chip that 128-slot tiles fill twice they are the better ones where the costs are close (Q4_K, 64 / 128: 4096 x 4096 at 2059 rows
// 104 / 92, 14336 x 4096 at 572 112 / 98).
inline int gemm_dense_tile(const GemmFormat& f, int64_t n, int64_t k, int64_t m) {
    if (n % 128 || m < 96) return 0;
    const double us64 = gemm_plan(f, false, n, k, m, 1, 64, max_gemm_tiles(m, 2, 64)).us / (n / 128 * ((m + 127) / 128) >= 512 ? 0.95 : 1.0);
    const double us128 = gemm_plan(f, false, n, k, m, 1, 128, max_gemm_tiles(m, 2, 128)).us;
    return streamed_us(f, n, k, m) <= std::min(us64, us128) ? 0 : us128 <= us64 ? 128 : 64;
}

}  // namespace moe
