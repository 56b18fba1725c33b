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

// Triangles from which a scene's rays are long: they visit many nodes and their
// data leaves the caches, so idle lanes and single launches cost less than walks
// that wait for one another.
constexpr uint32_t LARGE_SCENE = 100000u;

// Adaptive shadow passes in stages over the listed groups (powers of two up to
// 64), or a lane per group? With 1 or 2 samples there is one stage and nothing to
// adapt, so the probes over all groups, 4 items each, and the lists are overhead:
// us in stages and a lane per group, 2 lights in 20k triangles (spheres): 1
// sample 256 x 256 218, 72, 1280 x 720 667, 198, 2 samples 667, 198; 4 lights in
// 1M triangles: 1 sample 960 x 540 772, 573, but 2 samples 640 x 360 507, 791
// and 1920 x 1080 1660, 2453 (262k: 480, 581 and 1372, 1817; 16k: 432, 412 and
// 950, 1068).
HR_RULE bool adaptive_stages(uint32_t samples, uint32_t tris) {
    return samples >= 1u && samples <= 64u && (samples & (samples - 1u)) == 0u &&
           (samples >= 4u || (samples == 2u && tris >= LARGE_SCENE));
}

}  // namespace hr
