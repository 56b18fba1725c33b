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

HR_RULE uint32_t div_up(uint32_t a, uint32_t b) { return a / b + (a % b != 0u ? 1u : 0u); }

// Triangles from which a scene's rays are long: they visit many nodes and their
// data leaves the caches, so idle lanes and single launches cost less than walks
// that wait for one another.
constexpr uint32_t LARGE_SCENE = 100000u;

// Ray queues (consume_queue). A queue that the grid's lanes hold at once is dealt
// out without take counters (finding all 8 bands empty costs every wave 8 round
// trips to memory): so many rays to each of `waves` waves, 16 at least, the rest
// of the lanes idle, since a wave takes as long as the nodes its rays visit
// together. (640 x 360, depth 8: the 16 trace launches 985 -> 325 us; 853 x 479:
// 1000 -> 817 us. 8 or 64 lanes a wave are no better.) In small scenes, whose rays
// are short, over at most 4096 waves: 960 x 540, 20k triangles, us of the shading
// pass (2 samples, 3 bounces) and of pure ray tracing (1 sample, 2 depths) over
// all 8192 waves and 4096: 488, 448 and 719, 682 (657 with a ray per lane), 16k
// triangles 998, 994 and 1274, 1228; but 1M triangles 1678, 1686 and 1719, 1776.
HR_RULE uint32_t dealt_lanes(uint32_t rays, uint32_t waves, uint32_t tris) {
    const uint32_t lanes = div_up(rays, tris < LARGE_SCENE && waves > 4096u ? 4096u : waves);
    return lanes < 16u ? 16u : (lanes > 64u ? 64u : lanes);
}
// Lanes of a wave stay in the inner node loop until
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

// Adaptive shadow passes in stages over the listed groups (powers of two up to
// 64), or a lane per group? With 1 or 2 samples there is one stage and nothing to
// adapt, so the probes over all groups, 4 items each, and the lists are overhead:
// us in stages and a lane per group, 2 lights in 20k triangles (spheres): 1
// sample 256 x 256 218, 72, 1280 x 720 667, 198, 2 samples 667, 198; 4 lights in
// 1M triangles: 1 sample 960 x 540 772, 573, but 2 samples 640 x 360 507, 791
// and 1920 x 1080 1660, 2453 (262k: 480, 581 and 1372, 1817; 16k: 432, 412 and
// 950, 1068). The line by size gives up what the stages won in small terrains
// (16k: 97 x 64 135, 200, 1280 x 720 535, 688, but 853 x 479 580, 490) for the
// two- to threefold in scenes of spheres.
HR_RULE bool adaptive_stages(uint32_t samples, uint32_t tris) {
    return samples >= 1u && samples <= 64u && (samples & (samples - 1u)) == 0u &&
           (samples >= 4u || (samples == 2u && tris >= LARGE_SCENE));
}

// A launch of `packets` waves that walk the tree once per wave (packet_walk)
// waits for its nodes one after another and hides that only behind other
// waves: at 640 x 360 (3,600 packets) the primary rays took 127 us as packets
// and 88 us with a walk per lane, at 1280 x 720 and above (14,400) packets win.
constexpr uint32_t PACKETS_MIN = 8192u;
HR_RULE bool packets_fill(uint64_t packets) { return packets >= PACKETS_MIN; }

// How a shadow pass of 1 to 64 samples runs. Items: one per group (pixel and
// light) and sample, 2^lg2s >= samples to a group, 64 to a wave.
enum class ShadowRoute : uint32_t {
    Group,   // a lane per group, its samples one after the other (k_shadows)
    Once,    // a lane per item and walk, all groups (k_shadows_once)
    Direct,  // packets of items, all groups (k_shadows_direct)
    Listed,  // the groups that need rays listed, their items traced (k_shadows_spl)
};
HR_RULE uint32_t log2_up(uint32_t n) {
    uint32_t l = 0u;
    while ((1u << l) < n) ++l;
    return l;
}
// Listing the groups costs about 30 us of launches, and drops 57% of the items of
// the terrain scenes' 1080p frames. Without adaptive sampling, us of Group, Once,
// Direct, Listed (Direct was taken from 8192 waves of items on, Once below):
//                                  waves
//   20k triangles (spheres, 2 lights)
//     256 x 256, 3 samples          8,192    129   92  149  165
//     640 x 360, 2 samples         14,400    188  145  186  190
//     960 x 540, 1 sample          16,320    187  171  198  201
//     1280 x 720, 1 sample         28,800    209  243  222  222
//     1920 x 1080, 2 samples      129,600    387  883  420  363
//   16k triangles (terrain, 4 lights)
//     160 x 100, 4 samples          4,160    392  144  132  176
//     400 x 300, 2 samples         15,200    376  253  282  246
//     1920 x 1080, 1 sample       129,600    706  990  496  564
//     1920 x 1080, 2 samples      259,200   1053 1885  766  670
//   262k triangles
//     97 x 64, 1 sample               416    163  172  340  134
//     640 x 360, 1 sample          14,400    332  346  373  275
//     1280 x 720, 1 sample         57,600    629  760  456  475
//     1920 x 1080, 2 samples      259,200   1840 2390 1035 1190
//   1M triangles
//     256 x 256, 1 sample           4,096    352  312  604  230
//     640 x 360, 1 sample          14,400    434  428  584  292
//     1920 x 1080, 1 sample       129,600   1358 1644 1020  939
// scratch: is there memory for the lists?
HR_RULE ShadowRoute shadow_route(uint32_t samples, bool adaptive, uint32_t groups, uint32_t tris, bool scratch) {
    const uint64_t waves = ((uint64_t)groups << log2_up(samples)) >> 6;
    if (!adaptive && samples <= 4u && tris < LARGE_SCENE && waves < 16384u) return ShadowRoute::Once;
    if (!adaptive && samples == 1u && tris < 500000u && waves >= 49152u) return ShadowRoute::Direct;
    if (!adaptive && samples == 2u && tris >= LARGE_SCENE && tris < 500000u && waves >= 98304u)
        return ShadowRoute::Direct;
    if (scratch) return ShadowRoute::Listed;
    if (adaptive || samples > 2u) return ShadowRoute::Group;
    return packets_fill(waves) ? ShadowRoute::Direct : ShadowRoute::Once;
}

// The number of waves of listed items, `samples` per (surface point, light), from
// which they are traced as packets (packet_loop) and not with a walk per lane
// (item_loop). Packets need waves to hide their serial node loads behind, and
// rays that stay together: rays of one point do, those of neighbouring points
// less the more triangles lie between them, and less to a disk light (random
// directions: scattered) than to an area light (stratified). us per lane and as packets
// (waves with rays), area lights:
//   262k triangles  640 x 360  4 samples 411, 405 (28,700), 8 samples 575, 509
//                              (57,400), 16 samples 878, 674 (115,000)
//   1M              256 x 256  16 samples 452, 390 (29,600); 640 x 360 4 samples
//                              498, 540 (22,500), 8 samples 671, 589 (45,100)
//   4M              256 x 256  16 samples 608, 517 (33,100); 640 x 360 8 samples
//                              854, 891 (49,900); 1280 x 720 4 samples 1596, 1622
//                              (99,800); 1920 x 1080 4 samples 3134, 2768 (224,000);
//                              the adaptive passes' 12 to 32 samples of 1920 x 1080
//                              (some 35,000) 160 of 3470 us faster as packets
// disk lights:
//   262k            640 x 360  8 samples 586, 538 (57,400)
//   1M              640 x 360  8 samples 752, 812 (45,100), 16 samples 1118, 1052
//                              (90,200); 853 x 479 8 samples 1098, 1088 (80,000)
//   4M              640 x 360  8 samples 985, 1260 (49,900); 960 x 540 8 samples
//                              1873, 2024 (112,000); 1280 x 720 4 samples 1839,
//                              2169 (99,800), 16 samples 5409, 4424 (399,000)
// tris: the scene's, 0 for several scenes.
HR_RULE uint32_t packets_from(uint32_t samples, uint32_t tris, bool scattered) {
    const uint32_t per = samples < 16u ? samples : 16u;
    const uint32_t grain = scattered ? tris >> 19 : (samples < 12u ? tris >> 21 : 0u);
    return ((grain > 1u ? grain : 1u) * (1u << 18) + per - 1u) / per;
}

// Bare ray queries (us before and now; closest hits). As a queue, whose lanes take
// new rays, or a ray per lane? 4.1M rays, 1M triangles: 2415 -> 1641, any hit 1458
// -> 1090; in small scenes a ray is over before its lane's next one is fetched
// (80k triangles, 1M rays: 245 -> 275, 20k: 135 -> 211).
HR_RULE bool ray_queue(uint32_t rays, uint32_t tris) { return rays >= 262144u && tris >= LARGE_SCENE; }
// With a ray per lane, the lanes of a wave in use: the rays go over about 4096
// waves, 2 a wave at least, since a wave takes as long as the nodes its rays visit
// together (4,096 random pixels of a 20k-triangle scene 42 -> 28, of a 1M-triangle
// one 207 -> 84; 16 lanes at least: 36 and 142). From 120,000 rays to 262,144 full
// waves are as good within 10% either way (131,072 rays, full and partly used: 20k
// triangles 44, 47, 16k 142, 128; 200,000 rays: 46, 49 and 145, 142, 1M any hit
// 218, 199).
HR_RULE uint32_t ray_lanes(uint32_t rays) {
    const uint32_t lanes = div_up(rays, 4096u);
    return lanes > 64u ? 64u : (lanes > 2u ? lanes : 2u);
}

}  // namespace hr
