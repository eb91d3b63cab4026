"""The form a pass takes when it has too few paths to fill the chip (one
kernel, four lanes per path) against the separate per-bounce kernels: closest
hits and images are the same bits."""
import numpy as np
import pytest

from ratbite_amd import _lib as L
from ratbite_amd import scenes
from ratbite_amd.renderer import Renderer

pytestmark = pytest.mark.gpu


def _trace(ctx, rays, mode):
    hits = np.zeros((len(rays), 4), np.float32)
    ctx.check(L.lib().rbh_test_trace(ctx.h, L.ptr(rays), L.ptr(hits), len(rays), mode))
    return hits.view(np.uint32)


@pytest.mark.parametrize("ntri,nrays", [(1, 3), (2, 64), (3, 1), (37, 1021), (5000, 20000)])
def test_four_lanes_per_ray_walk_matches_one_lane(ctx, ntri, nrays):
    # every third triangle twice (exact ties), rays along the axes (infinite
    # reciprocal directions) among random ones
    rng = np.random.default_rng(ntri)
    c = rng.uniform(-5, 5, (ntri, 3))
    v = (c[:, None, :] + rng.normal(scale=0.7, size=(ntri, 3, 3))).astype(np.float32)
    v = np.concatenate([v, v[::3]]).reshape(-1, 3)
    n = len(v) // 3
    ctx.upload_textures(np.zeros(0, L.TEXTURE_DTYPE), np.zeros(0, np.uint8))
    mats = np.zeros(1, L.MATERIAL_DTYPE)
    mats["bxdf"] = 2
    ctx.upload_materials(mats)
    ctx.upload_geometry(v, np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), np.zeros(16, np.uint8),
                        np.zeros(n, np.uint32), np.full(n, 0xFFFFFFFF, np.uint32))
    ctx.build_accel()
    rays = np.zeros((nrays, 8), np.float32)
    rays[:, 0:3] = rng.uniform(-6, 6, (nrays, 3))
    rays[:, 4:7] = rng.normal(size=(nrays, 3))
    rays[::5, 4:7] = np.eye(3, dtype=np.float32)[rng.integers(0, 3, len(rays[::5]))]
    rays[:, 7] = 3.4e38
    one = _trace(ctx, rays, 0)
    assert np.array_equal(one, _trace(ctx, rays, 16))
    assert np.array_equal(one, _trace(ctx, rays, 16 | 2))      # a 2-entry LDS stack: the rest spills
    rays[:, 7] = rng.uniform(0.1, 10, nrays)
    miss = _trace(ctx, rays, 1)[:, 1] == 0xFFFFFFFF
    assert np.array_equal(miss, _trace(ctx, rays, 16 | 1)[:, 1] == 0xFFFFFFFF)
    assert np.array_equal(miss, _trace(ctx, rays, 16 | 1 | 2)[:, 1] == 0xFFFFFFFF)


@pytest.mark.parametrize("make,no_drop", [
    (lambda: scenes.features(width=37, height=23), False),
    (lambda: scenes.features(width=37, height=23), True),
    (lambda: scenes.cornell(width=64, height=64, shapes="mixed"), False),
    (lambda: scenes.spheres(n_spheres=12, level=2, n_lights=40, n_light_tex=2, env_size=(64, 32), width=33, height=9,
                            depth=12), False),
])
def test_pass_size_leaves_the_image_bits(ctx, make, no_drop):
    # one sample per pass (at most 4096 paths), a launch in one small pass,
    # and per-kernel timing (always the separate kernels); then enough
    # samples that the pass starts in the separate kernels and ends in the one
    sc = make()
    r = Renderer(sc, ctx=ctx)
    px = sc.width * sc.height
    images, stats = [], []
    for slots, flags in ((px, 0), (0, 0), (0, L.RBH_RENDER_TIMING)):
        ctx.set_path_slots(slots)
        st = r.render(spp=3, offset=0, no_drop=no_drop, flags=flags)
        images.append(r.accum())
        stats.append([st[k] for k in ("closestRays", "shadowRays", "pathVertices", "nonFiniteSamples")])
    ctx.set_path_slots(0)
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
    assert stats[0] == stats[1] == stats[2] and stats[0][0] >= 3 * px
    spp = -(-300000 // px)
    a = r.render(spp=spp, offset=0, no_drop=no_drop)
    big = r.accum()
    b = r.render(spp=spp, offset=0, no_drop=no_drop, flags=L.RBH_RENDER_TIMING)
    assert np.array_equal(big, r.accum())
    assert [a[k] for k in ("closestRays", "shadowRays", "pathVertices")] == \
        [b[k] for k in ("closestRays", "shadowRays", "pathVertices")]


@pytest.mark.parametrize("width,height", [(256, 128), (257, 128), (256, 256), (257, 256)])
def test_pass_sizes_where_the_register_budget_changes(ctx, width, height):
    # 32768 paths are the last that run with the larger register budget, 65536
    # the last that are one kernel from the start
    r = Renderer(scenes.features(width=width, height=height), ctx=ctx)
    r.render(spp=1, offset=0)
    a = r.accum()
    r.render(spp=1, offset=0, flags=L.RBH_RENDER_TIMING)
    assert np.array_equal(a, r.accum())


def _soup(rng, n):
    c = rng.uniform(-5, 5, (n, 3))
    return (c[:, None, :] + rng.normal(scale=0.7, size=(n, 3, 3))).astype(np.float32)


def _lattice(rng, n):
    """Right triangles with two unit edges along the axes: boxes share planes."""
    c = rng.integers(-6, 7, (n, 3)).astype(np.float32)
    e = np.eye(3, dtype=np.float32)[rng.permuted(np.tile([0, 1, 2], (n, 1)), axis=1)]
    return np.stack([c, c + e[:, 0], c + e[:, 1]], 1)


def _axis_rays(rng, n):
    """Along the axes (either zero beside the direction), from points whose
    coordinates are mostly those of box planes and shared edges."""
    r = np.zeros((n, 8), np.float32)
    r[:, 0:3] = rng.integers(-14, 15, (n, 3)) / 2.0
    r[:, 4:7] = np.where(rng.random((n, 3)) < 0.5, np.float32(0.0), np.float32(-0.0))
    r[np.arange(n), 4 + rng.integers(0, 3, n)] = rng.choice([-1.0, 1.0], n)
    r[:, 7] = 3.4e38
    return r


@pytest.mark.parametrize("quant", [False, True], ids=["full-boxes", "grid"])
@pytest.mark.parametrize("which", ["nine-times", "one-plane", "lattice"])
def test_walks_agree_where_hits_tie_and_rays_lie_in_faces(ctx, which, quant):
    # the two forms that one image mixes, over the same nodes: distances,
    # triangles, misses and occlusion are the same bits
    rng = np.random.default_rng(17)
    if which == "nine-times":        # more coincident triangles than a node holds
        v = np.repeat(_soup(rng, 600), 9, axis=0)
    elif which == "one-plane":       # overlapping triangles of one tilted plane: distances a few ulp apart, or equal
        p = rng.uniform(-4, 4, (4000, 1, 2)) + rng.normal(scale=0.5, size=(4000, 3, 2))
        v = np.stack([p[..., 0], 0.3 * p[..., 0] - 0.7 * p[..., 1], p[..., 1]], -1).astype(np.float32)
    else:
        v = _lattice(rng, 4000)
    n = len(v)
    ctx.upload_textures(np.zeros(0, L.TEXTURE_DTYPE), np.zeros(0, np.uint8))
    mats = np.zeros(1, L.MATERIAL_DTYPE)
    mats["bxdf"] = 2
    ctx.upload_materials(mats)
    ctx.upload_geometry(v.reshape(-1, 3), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3), np.zeros(16, np.uint8),
                        np.zeros(n, np.uint32), np.full(n, 0xFFFFFFFF, np.uint32))
    ctx.build_accel()
    rays = _axis_rays(rng, 20000)
    if which != "lattice":
        rays[:, 0:3] = rng.uniform(-6, 6, (20000, 3))
        rays[:, 4:7] = rng.normal(size=(20000, 3))
    form = 8 if quant else 0
    one = _trace(ctx, rays, form)
    hit = one[:, 1] != 0xFFFFFFFF
    assert hit.sum() > 2000
    assert np.array_equal(one, _trace(ctx, rays, form | 16))
    assert np.array_equal(_trace(ctx, rays, form | 2), _trace(ctx, rays, form | 16 | 2))
    # any hit: the range ends at the closest hit, just before and just behind it
    rays[:, 7] = np.where(hit, one[:, 0].view(np.float32) * rng.choice(np.float32([0.999, 1.0, 1.001]), len(rays)),
                          np.float32(3e38))
    miss = _trace(ctx, rays, form | 1)[:, 1] == 0xFFFFFFFF
    assert np.array_equal(miss, _trace(ctx, rays, form | 16 | 1)[:, 1] == 0xFFFFFFFF)
    assert np.array_equal(miss, _trace(ctx, rays, form | 16 | 1 | 2)[:, 1] == 0xFFFFFFFF)


@pytest.mark.parametrize("tuning", [dict(), dict(quant_nodes=False), dict(trace_fetch=1, quant_nodes=False)],
                         ids=["grid", "full-boxes", "work-fetch"])
def test_coincident_surfaces_whatever_the_pass_size(ctx, tuning):
    # every surface of the box three times, each with another material: which
    # one a ray meets must not depend on the kernel that walked it
    sc = scenes.cornell(width=48, height=40, depth=6)
    solid = np.flatnonzero(sc.tri_light == 0xFFFFFFFF)
    plain = np.unique(sc.tri_material[solid])
    rng = np.random.default_rng(3)
    idx, tm, tl = [sc.indices], [sc.tri_material], [sc.tri_light]
    for _ in range(2):
        idx.append(sc.indices[solid])
        tm.append(rng.choice(plain, len(solid)).astype(np.uint32))
        tl.append(np.full(len(solid), 0xFFFFFFFF, np.uint32))
    sc.indices, sc.tri_material, sc.tri_light = (np.ascontiguousarray(np.concatenate(a)) for a in (idx, tm, tl))
    r = Renderer(sc, ctx=ctx)
    defaults = r.tuning()
    r.set_tuning(**dict(dict(quant_nodes=bool(defaults["quantNodes"])), **tuning))
    try:
        # 96000 paths: separate kernels, then one; a few passes of one kernel only; separate kernels only
        r.render(spp=50, offset=0)
        mixed = r.accum()
        r.render(spp=50, offset=0, flags=L.RBH_RENDER_TIMING)
        assert np.array_equal(mixed, r.accum())
        ctx.set_path_slots(30000)
        r.render(spp=50, offset=0)
        assert np.array_equal(mixed, r.accum())
    finally:
        ctx.set_path_slots(0)
        r.set_tuning(path_slots=0, trace_blocks=defaults["traceBlocksPerCU"], shade_blocks=defaults["shadeBlocksPerCU"],
                     use_graph=bool(defaults["useGraph"]), shade_waves=defaults["shadeWaves"],
                     trace_fetch=defaults["traceFetch"], trace_waves=defaults["traceWaves"],
                     quant_nodes=bool(defaults["quantNodes"]), sort_hits=bool(defaults["sortHits"]))
