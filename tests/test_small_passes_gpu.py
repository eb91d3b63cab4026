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
