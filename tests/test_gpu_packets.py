"""GPU: packet walks (one tree walk per wave) against the counting kernels,
which walk the binary nodes ray by ray in the oracle's order.

Bar: bit-exact shadow factors and equal ray counts for every sample count
class (one launch over all groups, listed groups, counts that are no power of
two, adaptive stages), at frame sizes that take packets and at ones below,
with edges that cut the pixel tiles; a batch whose waves straddle frames;
primary rays of a camera inside the scene, whose tiles mix ray octants.
"""
import numpy as np
import pytest

from vulkanhybridraytracer_amd import abi, scenes

pytestmark = pytest.mark.gpu


def _scene(kind, w, h, samples, adaptive, seed=3):
    if kind == "terrain":
        return scenes.make_terrain_scene(seed=seed, width=w, height=h, quads=64, instances=12, soup_tris=256,
                                         samples=samples, spp=1, adaptive=adaptive)
    sc = scenes.make_small(seed=seed, width=w, height=h, spheres=40)
    sc.params = dict(sc.params, shadow_samples=samples, flags=abi.HR_FLAG_ADAPTIVE if adaptive else 0)
    sc.lights = sc.lights.copy()
    sc.lights[:, 8] = 0.05  # disks: rays of one point differ
    return sc


def _shadows(rd, flags):
    st = abi.hr_stats()
    base = rd.params.flags
    rd.shadow.zero()
    rd.params.flags = base | flags
    rd.trace_shadows(st)
    rd.params.flags = base
    return rd.download_shadow(), int(st.shadow_rays), int(st.occluded_rays)


# sizes: below every line for packets; packets from 8 or 16 samples on; packets
# for 3 to 32 samples and the adaptive stages (979 and 603: the right and bottom
# tiles are cut). 33 and 64 samples keep the walk per lane at every size.
@pytest.mark.parametrize("kind", ["terrain", "spheres"])
@pytest.mark.parametrize("w,h", [(45, 27), (322, 181), (979, 603)])
@pytest.mark.parametrize("samples,adaptive", [(1, False), (2, False), (3, False), (4, False), (7, False), (16, False),
                                              (33, False), (64, False), (1, True), (2, True), (4, True), (16, True)])
def test_shadows_equal_counting_walk(gpu_ctx, kind, w, h, samples, adaptive):
    from vulkanhybridraytracer_amd import hr
    print("case", kind, w, h, samples, adaptive, flush=True)
    rd = hr.HybridRenderer(gpu_ctx, hr.HybridScene(gpu_ctx, _scene(kind, w, h, samples, adaptive)))
    rd.gbuffer_primary()
    got = _shadows(rd, 0)
    ref = _shadows(rd, abi.HR_FLAG_COUNT_VISITS)
    assert np.array_equal(got[0].view(np.uint32), ref[0].view(np.uint32))
    assert got[1:] == ref[1:]


@pytest.mark.parametrize("samples", [(16, 16, 16), (1, 2, 1), (8, 32, 4)])
def test_batch_packets_straddle_frames(gpu_ctx, samples):
    """sizes whose listed groups are no multiple of a wave's 64 items"""
    from vulkanhybridraytracer_amd import hr
    rds = []
    for k, (s, (w, h)) in enumerate(zip(samples, ((731, 411), (402, 655), (517, 389)))):
        rd = hr.HybridRenderer(gpu_ctx, hr.HybridScene(gpu_ctx, _scene("terrain", w, h, s, False, seed=5 + k)))
        rd.gbuffer_primary()
        rds.append(rd)
    ref = [_shadows(rd, abi.HR_FLAG_COUNT_VISITS)[0] for rd in rds]
    for rd in rds:
        rd.shadow.zero()
    hr.BatchRenderer(gpu_ctx, rds).trace_shadows()
    for rd, r in zip(rds, ref):
        assert np.array_equal(rd.download_shadow().view(np.uint32), r.view(np.uint32))


@pytest.mark.parametrize("w,h", [(979, 603), (322, 181)])
def test_primary_rays_inside_the_scene(gpu_ctx, oracle_lib, w, h):
    """the G-buffer against the oracle's, and the pure ray tracing mode against
    its counting kernel"""
    from oracle import pyoracle
    from vulkanhybridraytracer_amd import hr
    sc = _scene("spheres", w, h, 4, False)
    sc.camera = scenes.rt_camera((0.0, 6.0, 0.0), (10.0, 5.0, 9.0), w, h)  # between the spheres
    rd = hr.HybridRenderer(gpu_ctx, hr.HybridScene(gpu_ctx, sc))
    rd.gbuffer_primary()
    gb = rd.gb.download()
    ogb, _ = pyoracle.OracleScene(sc).gbuffer()
    for k in ("position", "normal"):
        assert np.array_equal(gb[k], ogb[k]), k
    d = gb["position"][..., :3][gb["normal"][..., 3] != 0] - np.float32((0.0, 6.0, 0.0))
    assert len(d) > 0.2 * w * h
    assert len({tuple(x) for x in (d < 0)[::97]}) >= 3  # several octants
    accum = gpu_ctx.alloc(w * h * 16)
    base = rd.params.flags
    out = []
    for flags in (0, abi.HR_FLAG_COUNT_VISITS):
        rd.params.flags = base | flags
        accum.zero()
        rd.render_rt(accum)
        out.append(accum.download((h, w, 4)))
    rd.params.flags = base
    assert np.allclose(out[0], out[1], rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("n", [1, 63, 4097, 8193, 40001, 262144, 300001])
@pytest.mark.parametrize("any_hit", [False, True])
def test_ray_queries_of_every_size(gpu_ctx, n, any_hit):
    """rays spread over waves and rays as a queue (large scene, 262144 rays on)
    against the counting walk; an unaligned end and rays that miss"""
    from vulkanhybridraytracer_amd import hr
    sc = scenes.make_terrain_scene(seed=2, width=64, height=36, quads=230, instances=4, soup_tris=512)
    hs = hr.HybridScene(gpu_ctx, sc)
    assert hs.info()["tri_count"] > 100000
    r = np.random.default_rng(n)
    rays = np.zeros(n, dtype=abi.RAY_DTYPE)
    rays["org"] = r.uniform([-80, 2, -80], [80, 60, 80], size=(n, 3))
    d = r.normal(size=(n, 3))
    rays["dir"] = d / np.linalg.norm(d, axis=1, keepdims=True)
    rays["tmin"], rays["tmax"] = 1e-3, r.choice([5.0, 1e4], size=n)
    fast = hs.trace_rays(rays, any_hit=any_hit, count=False)
    slow = hs.trace_rays(rays, any_hit=any_hit, count=True)
    assert np.array_equal(fast["tri"] != 0xFFFFFFFF, slow["tri"] != 0xFFFFFFFF)
    if not any_hit:
        assert np.array_equal(fast.view(np.uint32), slow.view(np.uint32))
