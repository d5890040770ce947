// moe_internal.hpp -- the many-token expert path (moe_grouped.hip) as the
// layer entry point (moe_packed.hip) calls it.
#pragma once

#include <algorithm>

#include "internal.hpp"

namespace qmla {

// Pairs per expert from which a call takes the grouped path.
constexpr int kGroupedMinPairs = 8;

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
