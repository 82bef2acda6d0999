// How wide the workgroups of a tiled K-quant launch are.  Plain C++: no HIP types.
#pragma once
#include <cstdint>

namespace moe {

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

// A workgroup of eight waves (256 weight rows) takes a CU, one of four waves (128 rows) half of one.  The wide ones fetch an
// activation tile half as often: 2 to 6 % on launches of full rounds.  But a CU holds one of them at a time, and a last
// round that hardly fills takes as long as a full one, where narrow workgroups spread over the CUs.
//   few:   grids up to half of the CUs (4096 x 4096 Q4_K, us wide / narrow: 512 rows, 128 wide workgroups 46.5 / 38.6; 576
//          rows, 144 of them 47.4 / 51.3; Mixtral shape, down, us per step: 450 tokens, 8 tiles of 16 workgroups 523 / 471; 500
//          tokens, 11 tiles: 589 / 615; 600 tokens, 16 tiles: 648 / 667).
//   tails: a last round at most a third full (Q4_K 14336 x 4096 at 300 rows, 1.09 rounds: 80 / 71; 4096 x 4096 at 2500, 1.25
//          rounds: 140 / 118; Mixtral shape, down: 1000 tokens, 1.19 rounds 1032 / 984; 2048 tokens, 2.25: 1701 / 1653) against fuller
//          ones (32000 x 4096 at 300, 1.46 rounds: 104 / 123; 4096 x 4096 at 1500, 1.5: 90 / 96; up, 400 tokens, 3.5: 432 / 446).
//          Below ten rounds: there the tail weighs more than the tile fetches (up: 1000 tokens, 8.3 rounds, 1030 / 999;
//          2048 tokens, 15.75: 1692 / 1722).
//   up projection in tiles of 64 slots: always narrow.  Its lists are short and uneven, and the finer grid shares them out better
//          (Mixtral shape, 137 / 257 / 287 tokens: Q4_K 280 / 273, 416 / 406, 454 / 433; Q6_K 257 tokens 547 / 521; Q3_K 495 / 470;
//          200 tokens: Q4_K 318 / 323, Q6_K 479 / 457).
// rows: weight rows of the launch (w1 and w3 both counted); groups: expert lists, 1 for a dense product.
constexpr int64_t GEMM_CUS = 256;
inline bool gemm_wide(bool up, int64_t rows, int64_t slots, int64_t groups, int tile_slots) {
    if (rows % 256 || (up && tile_slots == 64)) return false;
    const int64_t wide = rows / 256 * gemm_tiles(slots, groups, tile_slots), tail = wide % GEMM_CUS;
    if (wide <= GEMM_CUS / 2) return false;
    return tail == 0 || tail > GEMM_CUS / 3 || wide >= 10 * GEMM_CUS;
}

}  // namespace moe
