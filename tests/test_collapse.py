"""The collapse of the binary tree into four-wide nodes, on the CPU: every
subtree's nodes stay within the indices that are its own, whatever the boxes
hold (vertices may be infinite or NaN), and every triangle keeps one place."""
import ctypes
import os
import sys

import numpy as np
import pytest

from test_lbvh_gpu import NODE_DTYPE

HB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "hostbuild")
sys.path.insert(0, HB)
import host_wavefront as H  # noqa: E402

EMPTY = -2 ** 31
NODE4_DTYPE = np.dtype([(k, "f4", 4) for k in ("lox", "hix", "loy", "hiy", "loz", "hiz")] + [("child", "i4", 4), ("pad", "i4", 4)])
NODE4H_DTYPE = np.dtype([("o", "f4", 3), ("meta", "u4"), ("plane", "f2", (4, 3, 2)), ("child", "i4", 4), ("pad", "i4", 12)])


@pytest.fixture(scope="module")
def lib():
    H.build()
    lib = H.lib()
    lib.host_collapse.restype = ctypes.c_int64
    lib.host_max_nodes4.restype = ctypes.c_uint32
    return lib


def binary_tree(tri, rng):
    """Two-child nodes over triangles in their order, split at random; boxes
    are the merged corner minima and maxima as fminf / fmaxf give them."""
    n = len(tri)
    lo, hi = np.fmin.reduce(tri, axis=1), np.fmax.reduce(tri, axis=1)
    nodes = np.zeros(n - 1, NODE_DTYPE)
    todo, made = [(0, 0, n)], 1
    while todo:
        i, a, b = todo.pop()
        mid = int(rng.integers(a + 1, b)) if rng.random() < 0.5 else (a + b) // 2
        for side, (x, y) in (("l", (a, mid)), ("r", (mid, b))):
            mn, mx = np.fmin.reduce(lo[x:y], axis=0), np.fmax.reduce(hi[x:y], axis=0)
            for k, axis in enumerate("xyz"):
                nodes[i][side + "min" + axis], nodes[i][side + "max" + axis] = mn[k], mx[k]
            nodes[i][side + "cnt"] = y - x
            ref = ~x
            if y - x > 1:
                ref, made = made, made + 1
                todo.append((ref, x, y))
            nodes[i]["left" if side == "l" else "right"] = ref
    return nodes


def collapse(lib, nodes):
    n = len(nodes) + 1
    cap = lib.host_max_nodes4(n)
    n4, n4h = np.zeros(cap, NODE4_DTYPE), np.zeros(cap, NODE4H_DTYPE)
    writes = np.zeros(cap, np.uint32)
    p = [a.ctypes.data_as(ctypes.c_void_p) for a in (nodes, n4, n4h, writes)]
    count = lib.host_collapse(p[0], n, p[1], p[2], p[3])
    assert count > 0, "index %d of %d" % (~count, cap)
    return n4, n4h, writes, count


def triangles(kind, n, rng):
    c = rng.uniform(-5, 5, (n, 1, 3))
    t = (c + rng.normal(scale=0.2, size=(n, 3, 3))).astype(np.float32)
    some = rng.random(n) < 0.4
    if kind == "all-nan":
        t[:] = np.nan
    elif kind == "some-nan":
        t[some] = np.nan
    elif kind == "nan-axis":
        t[some, :, 1] = np.nan
    elif kind == "infinite-flat":      # inf * 0 in the box's surface
        t[:, :, 1] = 0.25
        t[some, 0, 0] = np.inf
        t[some, 1, 0] = -np.inf
    elif kind == "overflow-flat":      # finite corners whose extent is not
        t[:, :, 1] = 0.25
        t[some, 0, 0] = 3e38
        t[some, 1, 0] = -3e38
    elif kind == "one-infinity":       # inf - inf
        t[some, :, 2] = np.inf
    return t


@pytest.mark.parametrize("kind", ["finite", "all-nan", "some-nan", "nan-axis", "infinite-flat", "overflow-flat", "one-infinity"])
@pytest.mark.parametrize("n", [2, 3, 4, 5, 17, 64, 300])
def test_indices(lib, kind, n):
    for seed in range(8):
        rng = np.random.default_rng(1000 * n + seed)
        n4, n4h, writes, count = collapse(lib, binary_tree(triangles(kind, n, rng), rng))
        assert writes.max() == 1 and writes.sum() == count
        used = writes == 1
        child = n4["child"][used]
        assert np.array_equal(child, n4h["child"][used])
        inner, leaves = child[child >= 0], child[(child < 0) & (child != EMPTY)]
        assert np.array_equal(np.sort(inner), np.flatnonzero(used)[1:])
        assert np.array_equal(np.sort(~leaves), np.arange(n))
        # a node is short of children only if none of them could be opened
        short = (child == EMPTY).any(axis=1)
        assert not (child[short] >= 0).any()


@pytest.mark.parametrize("kind", ["finite", "all-nan", "some-nan", "nan-axis", "infinite-flat", "overflow-flat", "one-infinity"])
def test_grid_boxes_hold_the_full_ones(lib, kind):
    # the 11-bit planes lie outside the full ones, the node's corner is finite
    # and a box without a position on an axis is open there
    for n in (2, 5, 64, 300):
        rng = np.random.default_rng(n)
        n4, n4h, writes, _ = collapse(lib, binary_tree(triangles(kind, n, rng), rng))
        n4, n4h = n4[writes == 1], n4h[writes == 1]
        assert np.isfinite(n4h["o"]).all()
        full = n4["child"] != EMPTY
        for a, (lo, hi) in enumerate((("lox", "hix"), ("loy", "hiy"), ("loz", "hiz"))):
            e = ((n4h["meta"] >> np.uint32(8 * a)) & np.uint32(0xFF)).astype(np.int8).astype(np.float64)
            with np.errstate(invalid="ignore"):
                plane = n4h["o"][:, a, None, None].astype(np.float64) + \
                    n4h["plane"][:, :, a].astype(np.float64) * np.exp2(e)[:, None, None]
            below, above = plane[..., 0][full], plane[..., 1][full]
            l, h = n4[lo][full].astype(np.float64), n4[hi][full].astype(np.float64)
            none = np.isnan(l)
            assert np.array_equal(none, np.isnan(h))
            assert np.all(below[none] == -np.inf) and np.all(above[none] == np.inf)
            assert np.all(below[~none] <= l[~none]) and np.all(above[~none] >= h[~none])
            # and within one step of them where they are finite
            step = np.broadcast_to(np.exp2(e)[:, None], full.shape)[full]
            for p, q in ((below, l), (above, h)):
                f = np.isfinite(q)
                assert np.all(np.abs(p[f] - q[f]) <= step[f])
