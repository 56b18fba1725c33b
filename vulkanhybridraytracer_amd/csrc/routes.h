// routes.h - the rules by which calls choose between kernels and launch shapes:
// plain functions of sizes, for the host, the kernels and a host compiler. The
// measured times on both sides of each line stand beside the rule.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define HR_RULE __host__ __device__ inline constexpr
#else
#define HR_RULE inline constexpr
#endif

namespace hr {

// Ray queues (consume_queue). Lanes of a wave stay in the inner node loop until
// fewer than this many of them walk; the others wait with a leaf or, in a queue
// that hands out rays as lanes finish, without a ray. `live`: lanes of the wave
// that hold a ray. A dealt queue (a ray per lane, none to take afterwards) has
// waves of 16 to 64 lanes, and a fixed 16 there made a wave of 16 to 26 lanes
// leave the loop at every step: us of the shading pass, 8 bounces at 1 sample
// (before the queues were dealt / 16 lanes / three quarters of the live ones;
// seven eighths, half and none: within 2%, within 2%, 25% slower):
//   97 x 64, 262k triangles    1130 / 1230 / 1156, 1M triangles 1399 / 1497 / 1417
//   160 x 100, 1M triangles    1690 / 1800 / 1692
//   256 x 256, 1M triangles    2358 / 2373 / 2242
//   1280 x 720, 1M triangles   4448 / 3467 / 3303
HR_RULE uint32_t queue_leave_below(bool dealt, uint32_t live) { return dealt ? live * 3u / 4u : 16u; }

}  // namespace hr
