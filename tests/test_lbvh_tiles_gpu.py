"""The LBVH's bottom-up boxes and four-wide collapse at the edges of their
workgroups (2048 leaves a tile, 32 tiles a group), on even and on very uneven
trees: node invariants over all nodes, the reported depth, and four-wide hits
against the binary tree's, after a build and after a refit."""
import numpy as np
import pytest

from ratbite_amd import _lib as L
from test_lbvh_gpu import _brute, _rays, _read_lbvh, _trace, _upload

pytestmark = pytest.mark.gpu


def _triangles(n, spread, seed):
    rng = np.random.default_rng(seed)
    if spread == "even":
        c = rng.uniform(-5, 5, (n, 3))
    elif spread == "geometric":      # a cluster at every scale: the tree is deep on one side
        c = np.exp2(-rng.uniform(0, 40, (n, 1))) * rng.uniform(0.5, 1.0, (n, 3)) * 10.0
    else:                            # one centroid: the keys differ in the triangle index only
        return np.tile(rng.normal(size=(3, 3)), (n, 1)).astype(np.float32)
    return (c[:, None, :] + rng.normal(scale=0.05, size=(n, 3, 3))).reshape(-1, 3).astype(np.float32)


def _check_tree(nodes, tris, n, depth):
    lo = np.stack([nodes["lminx"], nodes["lminy"], nodes["lminz"]], 1), np.stack([nodes["rminx"], nodes["rminy"], nodes["rminz"]], 1)
    hi = np.stack([nodes["lmaxx"], nodes["lmaxy"], nodes["lmaxz"]], 1), np.stack([nodes["rmaxx"], nodes["rmaxy"], nodes["rmaxz"]], 1)
    ref = nodes["left"], nodes["right"]
    tv = np.stack([tris["v0"], tris["v1"], tris["v2"]], 1)
    for side in (0, 1):
        inner = ref[side] >= 0
        c = ref[side][inner]
        assert np.array_equal(lo[side][inner], np.minimum(lo[0][c], lo[1][c]))
        assert np.array_equal(hi[side][inner], np.maximum(hi[0][c], hi[1][c]))
        t = ~ref[side][~inner]
        assert np.array_equal(lo[side][~inner], tv[t].min(axis=1)) and np.array_equal(hi[side][~inner], tv[t].max(axis=1))
    ch = np.concatenate(ref)
    assert np.array_equal(np.sort(ch[ch >= 0]), np.arange(1, n - 1)) and np.array_equal(np.sort(~ch[ch < 0]), np.arange(n))
    # levels from the root down; the last one with inner nodes is the leaves' depth
    level, d = np.array([0]), 0
    while len(level):
        d += 1
        level = np.concatenate([nodes["left"][level], nodes["right"][level]])
        level = level[level >= 0]
    assert d == depth


@pytest.mark.parametrize("spread", ["even", "geometric", "one-centroid"])
@pytest.mark.parametrize("n", [2, 3, 5, 2047, 2048, 2049, 2 * 2048 + 1, 65535, 65537, 3 * 65536 + 77])
def test_tiles_and_groups(ctx, n, spread):
    v = _triangles(n, spread, n)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    st = _upload(ctx, v, idx)
    rays = _rays(np.random.default_rng(5), 500, -6, 6)
    for refit in (False, True):
        if refit:
            v = (v * np.float32([1.0, -1.5, 0.75]) + np.float32(0.125)).astype(np.float32)
            ctx.update_vertices(0, v)
            ctx.refit_accel()
        _, nodes, tris = _read_lbvh(ctx, n)
        _check_tree(nodes, tris, n, st["bvhDepth"])
        a, b = _trace(ctx, rays, False), _trace(ctx, rays, False, binary=True)
        # the same closest distances; equal distances may name either triangle
        assert np.array_equal(a[:, 0], b[:, 0])
        q = _trace(ctx, rays, False, quant=True)
        assert np.array_equal(a[:, 0], q[:, 0])


@pytest.mark.parametrize("which", ["axis-parallel", "far", "tiny", "huge"])
def test_grid_nodes_at_the_ends_of_their_range(ctx, which):
    # child boxes on the node's 11-bit grid only ever grow: the closest hit is
    # the brute-force one for rays along box faces, origins far outside and
    # scales far from one (the triangle test itself holds third powers)
    rng = np.random.default_rng(7)
    n = 3000
    c = rng.integers(-6, 7, (n, 3)).astype(np.float64)
    e = np.eye(3)[rng.permuted(np.tile([0, 1, 2], (n, 1)), axis=1)]   # two axis-aligned edges each
    v = np.stack([c, c + e[:, 0], c + e[:, 1]], 1).reshape(-1, 3)
    scale = {"tiny": 2.0 ** -30, "huge": 2.0 ** 30}.get(which, 1.0)
    rays = _rays(rng, 4000, -7, 7)
    if which == "axis-parallel":
        d = np.zeros((4000, 3))
        d[np.arange(4000), rng.integers(0, 3, 4000)] = rng.choice([-1.0, 1.0], 4000)
        rays[:, 4:7] = d
        rays[:, 0:3] = rng.integers(-28, 29, (4000, 3)) / 4.0
        rays[2000:, 4:7] = np.where(rays[2000:, 4:7] == 0, np.float32(-0.0), rays[2000:, 4:7])
    elif which == "far":
        o = rays[:, 0:3] - 1e5 * rays[:, 4:7]
        rays[:, 0:3] = o
    rays[:, 0:3] *= np.float32(scale)
    v = (v * scale).astype(np.float32)
    idx = np.arange(3 * n, dtype=np.uint32).reshape(-1, 3)
    _upload(ctx, v, idx)
    g, b = _trace(ctx, rays, False, quant=True), _brute(v, idx, rays, False)
    hit = b[:, 1].view(np.uint32) != 0xFFFFFFFF
    assert hit.sum() > 500
    assert np.array_equal(g[:, 1].view(np.uint32) != 0xFFFFFFFF, hit)
    # the same triangle test on both sides: a few ulp
    np.testing.assert_allclose(g[hit, 0], b[hit, 0], rtol=1e-6)
    if which != "axis-parallel":   # rays in a face pass the boxes of the other nodes by
        f = _trace(ctx, rays, False)
        assert np.array_equal(f[:, 0], g[:, 0])
    # any hit: occluded exactly where there is a closest hit within the range
    rays[:, 7] = np.where(hit, b[:, 0] * np.float32(1.001), np.float32(3e38))
    a = _trace(ctx, rays, True, quant=True)
    assert np.array_equal(a[:, 1].view(np.uint32) != 0xFFFFFFFF, hit)


def _with_bad_triangles(n, bad, kind, seed):
    """Valid triangles around the origin and then bad ones, whose x is not
    finite (or spans more than a float holds) and whose y and z are near 100."""
    rng = np.random.default_rng(seed)
    v = (rng.uniform(-5, 5, (n, 1, 3)) + rng.normal(scale=0.3, size=(n, 3, 3))).astype(np.float32)
    b = (100.0 + rng.random((bad, 3, 3))).astype(np.float32)
    if kind == "nan":
        b[..., 0] = np.nan
    elif kind == "infinity":
        b[..., 0] = np.inf
    elif kind == "infinite-flat":
        b[:, 0, 0], b[:, 1, 0], b[..., 1] = -np.inf, np.inf, 100.0
    else:
        b[:, 0, 0], b[:, 1, 0], b[..., 1] = -3e38, 3e38, 100.0
    return np.concatenate([v, b]).reshape(-1, 3)


def _rays_past(rng, n):
    """Rays that stay clear of the bad triangles' y and z."""
    r = _rays(rng, n, -6, 6)
    lo, hi = (98.0 - r[:, 1:3]) / r[:, 5:7], (103.0 - r[:, 1:3]) / r[:, 5:7]
    near, far = np.minimum(lo, hi).max(axis=1), np.maximum(lo, hi).min(axis=1)
    return np.ascontiguousarray(r[(near > far) | (far < 0)])


# the walks rbh_test_trace has (its mode bits)
WALKS = {"four-wide": 0, "binary": 4, "grid": 8, "four lanes": 16}


@pytest.mark.parametrize("kind", ["nan", "infinity", "infinite-flat", "overflow"])
@pytest.mark.parametrize("n,bad", [(1, 2), (3, 61), (200, 40), (4000, 3000), (40000, 30000)])
def test_vertices_that_are_not_finite(ctx, n, bad, kind):
    # the other triangles are hit as if they were alone, after a build and
    # after a refit
    v = _with_bad_triangles(n, bad, kind, n + bad)
    idx = np.arange(len(v), dtype=np.uint32).reshape(-1, 3)
    rays = _rays_past(np.random.default_rng(11), 2000)
    for refit in (False, True):
        if refit:
            v = np.roll(v.reshape(-1, 3, 3), 1, axis=1).reshape(-1, 3) + np.float32([0.0, 0.125, 0.0])
            ctx.update_vertices(0, v)
            ctx.refit_accel()
        else:
            _upload(ctx, v, idx)
        b = _brute(v[:3 * n], idx[:n], rays, False)
        hit = b[:, 1].view(np.uint32) != 0xFFFFFFFF
        for name, mode in WALKS.items():
            g = _trace_mode(ctx, rays, mode)
            assert np.array_equal(g[:, 1].view(np.uint32) != 0xFFFFFFFF, hit), name
            np.testing.assert_allclose(g[hit, 0], b[hit, 0], rtol=1e-5, atol=1e-5, err_msg=name)


def _trace_mode(ctx, rays, mode):
    hits = np.zeros((len(rays), 4), np.float32)
    ctx.check(L.lib().rbh_test_trace(ctx.h, L.ptr(rays), L.ptr(hits), len(rays), mode))
    return hits
