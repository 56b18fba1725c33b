"""CPU: the rules that choose between kernels and launch shapes (csrc/routes.h),
compiled by the host compiler, at the sizes where the measured lines lie."""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vulkanhybridraytracer_amd", "csrc")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """rule("expression") -> the values of C++ expressions over namespace hr"""
    tmp = tmp_path_factory.mktemp("routes")

    def run(*exprs):
        src = tmp / "t.cpp"
        src.write_text('#include <cstdio>\n#include "routes.h"\nusing namespace hr;\nint main() {\n'
                       + "".join('  printf("%%llu\\n", (unsigned long long)(%s));\n' % e for e in exprs)
                       + "  return 0;\n}\n")
        subprocess.check_call(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(tmp / "t")])
        return [int(v) for v in subprocess.check_output([str(tmp / "t")]).split()]
    return run


def test_dealt_queue_covers_every_ray(rule):
    """any queue that the grid's lanes hold, on small and large grids; short rays over fewer waves"""
    cases = [(n, w, t) for w in (1, 4, 100, 4095, 4096, 4097, 8192) for t in (20_000, 1_000_000)
             for n in sorted({1, 15, 16 * w, 17 * w + 1, 64 * w - 1, 64 * w, min(64 * w, 262_145)}) if 1 <= n <= 64 * w]
    got = rule(*["dealt_lanes(%du, %du, %du)" % c for c in cases])
    for (n, w, t), per in zip(cases, got):
        assert 16 <= per <= 64 and w * per >= n, (n, w, t, per)
    assert rule("dealt_lanes(200000u, 8192u, 20000u)", "dealt_lanes(200000u, 8192u, 1000000u)",
                "dealt_lanes(500000u, 8192u, 20000u)", "dealt_lanes(1u, 8192u, 20000u)") == [49, 25, 64, 16]


def test_dealt_queue_walks_with_part_of_its_own_lanes(rule):
    """a wave leaves the node loop for its leaves only when a share of the lanes
    it holds has one, also where it holds few"""
    lanes = list(range(1, 65))
    below = rule(*["queue_leave_below(true, %du)" % n for n in lanes])
    for n, b in zip(lanes, below):
        assert b <= n - n // 4 and (n < 4 or b >= n // 2), (n, b)
    assert rule("queue_leave_below(false, 64u)", "queue_leave_below(false, 20u)") == [16, 16]


def test_adaptive_frames_of_few_samples_take_a_lane_per_group(rule):
    """1 sample always, 2 in small scenes; other counts that are no power of two never go in stages"""
    cases = [(1, 20_000, 0), (1, 4_000_000, 0), (2, 20_000, 0), (2, 99_999, 0), (2, 262_144, 1), (2, 4_000_000, 1),
             (3, 4_000_000, 0), (4, 100, 1), (16, 20_000, 1), (48, 20_000, 0), (64, 1_000_000, 1), (65, 1_000_000, 0),
             (128, 1_000_000, 0), (0, 1_000_000, 0)]
    assert rule(*["adaptive_stages(%du, %du)" % (s, t) for s, t, _ in cases]) == [e for _, _, e in cases]


def test_shadow_routes_of_few_samples(rule):
    """the measured fastest route of frames (samples, groups, triangles) at both sides of every line, and
    the routes without memory for lists"""
    def groups(w, h, lights):
        return -(-w // 8) * -(-h // 8) * 64 * lights
    group, once, direct, listed = 0, 1, 2, 3
    cases = [((3, 0, groups(256, 256, 2), 20_482, 1), once), ((4, 0, groups(160, 100, 4), 16_384, 1), once),
             ((2, 0, groups(640, 360, 2), 20_482, 1), once), ((1, 0, groups(960, 540, 2), 20_482, 1), once),
             ((1, 0, groups(1280, 720, 2), 20_482, 1), listed), ((2, 0, groups(1920, 1080, 2), 20_482, 1), listed),
             ((5, 0, groups(97, 64, 2), 20_482, 1), listed), ((1, 0, groups(97, 64, 4), 262_144, 1), listed),
             ((1, 0, groups(1280, 720, 4), 262_144, 1), direct), ((2, 0, groups(1920, 1080, 4), 262_144, 1), direct),
             ((2, 0, groups(1920, 1080, 4), 16_384, 1), listed), ((1, 0, groups(1920, 1080, 4), 16_384, 1), direct),
             ((1, 0, groups(640, 360, 4), 1_048_576, 1), listed), ((1, 0, groups(1920, 1080, 4), 1_048_576, 1), listed),
             ((2, 1, groups(1920, 1080, 4), 1_048_576, 1), listed), ((64, 1, groups(97, 64, 4), 20_482, 1), listed),
             ((1, 0, groups(640, 360, 4), 1_048_576, 0), direct), ((2, 0, groups(97, 64, 4), 1_048_576, 0), once),
             ((3, 0, groups(640, 360, 4), 1_048_576, 0), group), ((2, 1, groups(640, 360, 4), 1_048_576, 0), group),
             ((3, 0, groups(97, 64, 4), 16_384, 0), once)]
    got = rule(*["(unsigned)shadow_route(%du, %d, %du, %du, %d)" % a for a, _ in cases])
    assert got == [e for _, e in cases]


def test_packets_ask_for_more_waves_in_fine_scenes(rule):
    """waves of items (samples, triangles, scattered lights) measured at both sides of the line: as packets or not"""
    cases = [(16, 262_144, 0, 18_800, 1), (8, 262_144, 1, 57_400, 1), (4, 262_144, 0, 28_700, 0),
             (16, 1_048_576, 0, 29_600, 1), (8, 1_048_576, 0, 45_100, 1), (8, 1_048_576, 1, 45_100, 0),
             (8, 1_048_576, 1, 80_000, 1), (16, 1_048_576, 1, 90_200, 1), (16, 4_194_304, 0, 33_100, 1), (12, 4_194_304, 0, 35_000, 1), (12, 4_194_304, 0, 21_845, 0), (32, 4_194_304, 0, 16_384, 1),
             (8, 4_194_304, 0, 49_900, 0), (4, 4_194_304, 0, 99_800, 0), (4, 4_194_304, 0, 224_000, 1),
             (8, 4_194_304, 1, 112_000, 0), (4, 4_194_304, 1, 99_800, 0), (16, 4_194_304, 1, 399_000, 1),
             (3, 0, 0, 87_381, 0), (3, 0, 0, 87_382, 1), (64, 0, 0, 16_384, 1), (64, 0, 1, 16_383, 0)]
    got = rule(*["%du >= packets_from(%du, %du, %d)" % (w, s, t, d) for s, t, d, w, _ in cases])
    assert got == [e for *_, e in cases]


def test_lanes_of_bare_ray_queries(rule):
    """few rays over many waves, and counts near 2^32 as any other: their sums would wrap"""
    cases = [(1, 2), (4_096, 2), (40_960, 10), (98_305, 25), (262_143, 64), (2 ** 32 - 4_096, 64), (2 ** 32 - 4_095, 64),
             (2 ** 32 - 1, 64)]
    assert rule(*["ray_lanes(%du)" % n for n, _ in cases]) == [e for _, e in cases]
    assert rule("ray_queue(262143u, 1000000u)", "ray_queue(262144u, 100000u)", "ray_queue(4000000u, 99999u)") == [0, 1, 0]
    assert rule("div_up(4294967295u, 256u)", "div_up(256u, 256u)", "div_up(0u, 8u)") == [2 ** 24, 1, 0]


def test_bench_names_the_routes(rule):
    """bench.py's kernel names against the library's rules, over sample counts, sizes and scenes"""
    import bench
    frames = [(n, ad, w, h, nl, t) for n in (1, 2, 3, 4, 5, 16, 48, 64, 65) for ad in (0, 1)
              for w, h, nl, t in ((97, 64, 2, 20_482), (640, 360, 2, 20_482), (1280, 720, 4, 262_144),
                                  (1920, 1080, 4, 262_144), (1920, 1080, 4, 1_048_576), (16384, 16384, 4, 4_194_304))]
    exprs = []
    for n, ad, w, h, nl, t in frames:
        groups = -(-w // 8) * -(-h // 8) * 64 * nl
        exprs.append("%du > 64u || (%d && !adaptive_stages(%du, %du)) || ((uint64_t)%du << log2_up(%du)) >= (1ull << 32)"
                     " ? 0u : (unsigned)shadow_route(%du, %d, %du, %du, true)"
                     % (n, ad, n, t, groups, n, n, ad, groups, t))
    names = ["k_shadows", "k_shadows_once", "k_shadows_direct", "k_shadows_spl"]
    for (n, ad, w, h, nl, t), route in zip(frames, rule(*exprs)):
        got = bench.shadow_kernel_name(dict(shadow_samples=n, flags=4 * ad), w, h, nl, t)
        assert got.split()[0] == names[route], (n, ad, w, h, nl, t)


def test_bench_binds_by_the_nearer_peak():
    """no fraction of a bound above 1; packets by VALU issue, the walk per lane of the closest hits by vector loads;
    no bound without a profile"""
    import bench
    shadows = bench.roofline_of("k_shadows_spl", "hybrid_1080p_1m", 4.2, 57_000_000, 2_000_000_000, 300_000_000)
    assert shadows["bound"] == "valu_issue" and 0.3 < shadows["frac"] < 1
    trace = bench.roofline_of("k_wf_trace", "hybrid_1080p_4m", 13.2, 57_000_000, 2_000_000_000, 300_000_000)
    assert trace["bound"] == "vmem" and trace["valu"]["issue_frac"] < trace["frac"] < 1
    unprofiled = bench.roofline_of("k_shadows_spl", "hybrid_1080p_4m", 4.7, 22_000_000, 1_100_000_000, 170_000_000)
    assert unprofiled["hbm_algorithmic"]["frac"] > 1 and unprofiled["bound"] is unprofiled["frac"] is None
