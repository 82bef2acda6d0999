// Which kernels a layer of the 32-element formats takes: tiled or streaming ones, and of the latter workgroups of a quarter of the
// rows ("fine") or whole ones.  Plain C++: no HIP types.
//
// The lines are those of 10962 measured (layer, tokens) pairs: 1160 random layers of 4 to 256 experts (H 256 .. 4096, F 128 .. 8192, top-1
// to top-10, the five formats, with and without an always-on expert), 0.05 to 33 rows per expert, every variant timed at each.
#pragma once
#include <algorithm>
#include <cstdint>

#include "gemm_plan.hpp"

namespace moe {

// Tiled kernels (an expert's weights are read once for up to 64 of its slots) or streaming ones, for layers whose slots a dispatch pass
// has grouped by expert: from 20 rows per expert on, and below as far as the streaming grids hold passes for lists that are not there
// -- one for every 16 tokens and expert, most of them empty: from 17 - passes / 5 rows on.  Experts' number and size alone say little.
//   One tile per pass / tiled, mean time over 4167 random sizes of more than 16 experts: 9 to 13 rows per expert and 8 to 11 passes 0.89,
//   40 to 79 passes 1.08, more 1.38; 16 to 20 rows, 8 to 11 passes 0.96, 12 to 39 1.03, more 1.16 to 1.41.  us, streamed / tiled, Q8_0: Qwen-MoE
//   shape 120 tokens, 8 rows per expert, 191 / 218, 220 tokens 250 / 200; Q5_0, 384 -> 3200, 248 experts, top-1, 2772 tokens, 11 rows, 667 / 377.  (Where
//   it is wrong: 640 -> 2048, 214 experts, top-8, 320 tokens, 12 rows, 243 / 180; 1536 -> 640, 44 experts, 18 rows, 9 passes 80 / 104.)
//   A line at 13 rows for every number of passes was 3 % or more slower than one at 20 in 3.9 % of those sizes, this one is in 2.8 %.
//   (Up to 16 experts no dispatch pass runs below 64 rows per expert.)
inline bool q32_tiled(int64_t T, int64_t k, int64_t E) {
    const int64_t slots = T * k, passes = (T + 15) / 16;
    return slots > 20 * E || (slots > 6 * E && 5 * slots + passes * E >= 85 * E);
}

// What a streaming launch's grid holds, in passes of 16 slots.
struct Q32Grid {
    enum Kind { ROWS, DIRECT, LISTS, ALWAYS_ON } kind;   // one list alone; lists found by scanning the assignments; lists measured by a dispatch pass; the always-on expert, beside the routed launches
    int64_t live, first;   // passes that find slots, and those among them that are their list's first
    int64_t empty;         // passes that find none, in the grid of a fine launch: the host knows no list's length
};
// groups: lists (one for a dense product); direct: no dispatch pass ran
inline Q32Grid q32_grid(int64_t T, int64_t k, int64_t groups, bool direct, bool always_on) {
    const int64_t z = (T + 15) / 16;
    if (always_on || groups == 1) return Q32Grid{always_on ? Q32Grid::ALWAYS_ON : Q32Grid::ROWS, z, 1, 0};
    const int64_t slots = T * k, first = std::min(groups, slots);
    const int64_t live = std::max(gemm_tiles(slots, groups, 16), first);   // (lists as evenly filled as gemm_tiles takes them)
    const int64_t rows = direct ? first : groups;
    return Q32Grid{direct ? Q32Grid::DIRECT : Q32Grid::LISTS, live, first, std::max<int64_t>(0, rows * z - live)};
}
// The fine kernels fill the chip where the coarse ones (128 rows of F, 64 of H per workgroup) leave CUs without work.  Counted in coarse
// workgroups of passes that find slots; the empty ones of a fine launch at a 40th (up), a 20th (down) of a coarse one each where lists
// are found by scanning the assignments, at a 30th where a dispatch pass has measured them.
//   Up: to 800, a list's second and later passes counted 1.3 times (they read its weights again).  us, coarse / fine: a quarter of
//   Mixtral's width, Q4_0, 224 workgroups (up to 40 tokens) 16.8 / 14.6, 448 (100 tokens, two passes) 31.4 / 28.0; Qwen-MoE shape, Q8_0, 44
//   (one token) 31 / 15, 176 47 / 21, 660 (16 tokens) 54 / 43; Mixtral, Q4_0, 448 (two tokens) 85 / 56, 896 93 / 97.
//   Down: to 400.  Dense, Q8_0 4096 x 4096, 64 (16 rows) 21.4 / 11.4, 256 27.8 / 18.6, 448 28.4 / 27.7, 512 28.9 / 30.8.
//   The always-on expert: beside the routed launches its passes compete for the chip, and the lines lie at 350 and 300 (4096 -> 1408, 48
//   experts with one of 5632, Q8_0: 89 tokens 263 / 279, 113 tokens 272 / 329).
//   Against coarse kernels alone, all four choices measured at 10935 random sizes (0.05 to 24 rows per expert): mean 0.813, 0.9 % are 3 % or
//   more slower, 0.1 % by 10 %; with lines that count no empty workgroup 0.817, 2.1 % and 0.5 % (256 -> 512, 128 experts, top-1, Q4_0, layer, 640
//   tokens 40.8 / 67.1).  Empty ones at a tenth, for a while, cost too much at sizes the fine kernels are made for (1024 -> 3584, eight experts,
//   top-2, Q4_1, 65 tokens 60.5 / 37.7).
inline bool q32_up_fine(int64_t F, const Q32Grid& g) {
    const int64_t passes10 = 10 * g.live + 3 * (g.live - g.first), weight = g.kind == Q32Grid::LISTS ? 30 : 40;
    return (F / 32 + 3) / 4 * passes10 / 10 + F / 32 * g.empty / weight <= (g.kind == Q32Grid::ALWAYS_ON ? 350 : 800);
}
inline bool q32_down_fine(int64_t H, const Q32Grid& g) {
    const int64_t weight = g.kind == Q32Grid::LISTS ? 30 : 20;
    return (H / 16 + 3) / 4 * g.live + H / 16 * g.empty / weight <= (g.kind == Q32Grid::ALWAYS_ON ? 300 : 400);
}

}  // namespace moe
