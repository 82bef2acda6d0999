// The grids of the tiled kernels: how row blocks and slot tiles are dealt to the XCDs, and how wide the workgroups of a
// K-quant launch are.  Plain C++: no HIP types.
#pragma once
#include <algorithm>
#include <cstdint>

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

}  // namespace moe
