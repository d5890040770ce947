// moe_internal.hpp -- the many-token expert path (moe_grouped.hip) as the
// layer entry point (moe_packed.hip) calls it.
#pragma once

#include <algorithm>

#include "internal.hpp"

namespace qmla {

// Pairs from which a call takes the grouped path: eight per expert, and with
// fewer than 32 experts 320 in all (384 with fewer than 4).  Its six launches
// cost 38-60 us where a few experts' bins keep the GEMV's blocks within one round
// of the device.  GEMV / grouped us at the reference widths 2048 x 1408, random
// routing: 32 experts top 4, 192 pairs 61 / 67, 256 74 / 68, 320 80 / 69; 64 top
// 6, 384 pairs 87 / 91, 516 114 / 91; 24 top 4, 256 pairs 62 / 66, 320 73 / 67; 8
// top 2, 256 pairs 61 / 69, 320 77 / 63; 4 top 2, 256 pairs 61 / 62, 320 76 / 63; 1
// expert, 256 pairs 52 / 61, 384 64 / 64, 512 82 / 66.  256 top 8 of 1024 x 512
// would gain from four per expert (1024 pairs 118 / 113).  Routing that prefers
// some experts moves the line down (8 top 2, 96 tokens of like content: 111 / 61),
// which the call cannot know.
constexpr int kGroupedMinPairs = 8;
inline int64_t moe_grouped_min_pairs(int32_t experts) {
  const int64_t total = experts < 4 ? 384 : experts < 32 ? 320 : 0;
  return std::max<int64_t>(total, (int64_t)kGroupedMinPairs * experts);
}

struct MoeGrouped {
  qmla_moe_config cfg;
  int P;  // (token, expert) pairs
  const uint8_t *gate_packed, *up_packed, *down_packed;
  const float *gate_scales, *up_scales, *down_scales;
  const int4 *tiles;      // {expert, first bin position, tokens, 0}
  const int32_t *ntiles;
  const int32_t *slots;   // bin position -> slot (pair)
  float *h;               // [P][I] f32, then digit rows
  float *y;               // [P][H] f32; before that the tokens' digit rows
};

// Sizes the grouped path takes (the caller has checked that both widths are
// multiples of 128 and the alignment).
bool moe_grouped_supported(const qmla_moe_config &c, int32_t T);
// Tiles of 32 pairs that P pairs over E experts make at most.
int moe_grouped_max_tiles(int P, int E);
// Routing of every token and its digit row (4 H bytes apart) in xdig.
qmla_status launch_moe_grouped_route(const qmla_moe_config &c, const float *xs, int T, const float *gw,
                                     int32_t *sel, float *selw, int32_t *user_idx, float *user_w,
                                     uint8_t *xdig, hipStream_t s);
// y[pair] from the digit rows in y, over the tiles.
qmla_status launch_moe_grouped_experts(const MoeGrouped &m, hipStream_t s);

}  // namespace qmla
