// Nodes of the LBVH's last stages: the halves of a two-child node, and the
// collapse of the binary tree into four-wide nodes (kernels/lbvh.hip runs it
// level by level; the bodies are per node).
#pragma once
#include <hip/hip_runtime.h>
#include "types.hpp"

namespace rbh {
namespace lbvh {

struct Box { float lo[3], hi[3]; };

__device__ __forceinline__ Box merge(const Box& a, const Box& b) {
    Box r;
    for (int k = 0; k < 3; ++k) {
        r.lo[k] = fminf(a.lo[k], b.lo[k]);
        r.hi[k] = fmaxf(a.hi[k], b.hi[k]);
    }
    return r;
}

// Box and reference of one side of a two-child node.
__device__ __forceinline__ Box node_half(const BvhNode& nd, uint32_t side) {
    return side ? Box{{nd.rminx, nd.rminy, nd.rminz}, {nd.rmaxx, nd.rmaxy, nd.rmaxz}}
                : Box{{nd.lminx, nd.lminy, nd.lminz}, {nd.lmaxx, nd.lmaxy, nd.lmaxz}};
}
__device__ __forceinline__ void put_half(BvhNode* __restrict__ nd, uint32_t side, const Box& b, int ref, uint32_t tris) {
    if (side) {
        nd->rminx = b.lo[0]; nd->rmaxx = b.hi[0]; nd->rminy = b.lo[1]; nd->rmaxy = b.hi[1];
        nd->rminz = b.lo[2]; nd->rmaxz = b.hi[2];
        nd->right = ref;
        nd->rcnt = tris;
    } else {
        nd->lminx = b.lo[0]; nd->lmaxx = b.hi[0]; nd->lminy = b.lo[1]; nd->lmaxy = b.hi[1];
        nd->lminz = b.lo[2]; nd->lmaxz = b.hi[2];
        nd->left = ref;
        nd->lcnt = tris;
    }
}

__device__ __forceinline__ float half_area(const Box& b) {
    const float x = b.hi[0] - b.lo[0], y = b.hi[1] - b.lo[1], z = b.hi[2] - b.lo[2];
    return x * y + y * z + z * x;
}

// A plane on the grid, rounded outwards (towards -inf for the lower ones). An
// infinite one stays infinite (half floats have both), and a box without a
// position on the axis (all vertices NaN) is open to that side.
template <bool UPPER>
__device__ __forceinline__ uint16_t grid_plane(float p, float o, int e) {
    const double x = ldexp((double)p - (double)o, -e);
    const float q = (float)(UPPER ? ceil(x) : floor(x));
    return __builtin_bit_cast(uint16_t, (_Float16)(q == q ? q : UPPER ? INFINITY : -INFINITY));
}

// The 11-bit form of a four-wide node whose inner children come first. Grid
// steps are powers of two and the arithmetic is in double precision, where a
// difference of two floats divided by one is exact (or rounded by 2^-53, far
// below the traversal's margin), so floor and ceil give planes outside. The
// grid spans the finite planes: beside an infinite vertex the other boxes
// keep their resolution.
__device__ __forceinline__ Bvh4HNode grid_node(const Bvh4Node& nd) {
    Bvh4HNode q;
    uint32_t tris = 0u, inner = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        q.child[k] = nd.child[k];
        tris |= nd.child[k] < 0 && nd.child[k] != kBvh4Empty ? 1u << k : 0u;
        inner += nd.child[k] >= 0 ? 1u : 0u;
    }
    q.meta = tris << 24 | inner << 28;
    auto axis = [&](int a, const float (&lo)[4], const float (&hi)[4]) {
        float o = INFINITY, top = -INFINITY;
#pragma unroll
        for (int k = 0; k < 4; ++k) {   // (empty boxes are (+inf, -inf))
            const bool l = fabsf(lo[k]) < INFINITY, h = fabsf(hi[k]) < INFINITY;
            o = fminf(o, fminf(l ? lo[k] : INFINITY, h ? hi[k] : INFINITY));
            top = fmaxf(top, fmaxf(l ? lo[k] : -INFINITY, h ? hi[k] : -INFINITY));
        }
        if (o > top) o = top = 0.0f;   // none
        int e = 0;
        (void)frexp(((double)top - (double)o) / (double)kGridMax, &e);   // extent / 2047 < 2^e
        e = min(max(e, -126), 127);
        q.o[a] = o;
        q.meta |= ((uint32_t)e & 0xFFu) << (8 * a);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            q.plane[k][a][0] = grid_plane<false>(lo[k], o, e);
            q.plane[k][a][1] = grid_plane<true>(hi[k], o, e);
        }
    };
    axis(0, nd.lox, nd.hix);
    axis(1, nd.loy, nd.hiy);
    axis(2, nd.loz, nd.hiz);
#pragma unroll
    for (int k = 0; k < 12; ++k) q.pad[k] = 0;
    return q;
}

// The most four-wide nodes a subtree of n >= 1 triangles collapses into: a
// node has four children unless all of them are triangles, so with the bound
// for its children 1 + sum (2 n_i - 1) / 3 = (2 n - 1) / 3.
__host__ __device__ __forceinline__ uint32_t max_nodes4(uint32_t n) { return (uint32_t)((2ull * n - 1ull) / 3ull); }

// A four-wide node to write: its index, the binary node it starts at and the
// first of the max_nodes4(triangles) - 1 indices that are its subtree's. With
// indices that no other subtree can take, nodes need no shared counter (one
// atomic per wave step on it made the step 17 us) and a subtree's nodes lie
// together.
struct Open {
    uint32_t id;
    int node;
    uint32_t room;
};

// Writes the four-wide node of t: the two children of its binary node, then
// again and again the inner child with the largest box surface replaced by
// its own two, until there are four. Its inner children go to t.room,
// t.room + 1, ... in slot order, their subtrees' indices follow. Returns the
// number of inner children, next[0..] the nodes to write for them.
__device__ __forceinline__ uint32_t collapse_node(const Open& t, const BvhNode* nodes, Bvh4Node* __restrict__ nodes4,
                                                  Bvh4HNode* __restrict__ nodes4h, Open (&next)[4]) {
    Box box[4];
    int ref[4];
    uint32_t tris[4];
    {
        const BvhNode nd = nodes[t.node];
        box[0] = node_half(nd, 0u);
        box[1] = node_half(nd, 1u);
        ref[0] = nd.left;
        ref[1] = nd.right;
        tris[0] = nd.lcnt;
        tris[1] = nd.rcnt;
    }
#pragma unroll
    for (int k = 2; k < 4; ++k) {
        box[k] = Box{{INFINITY, INFINITY, INFINITY}, {-INFINITY, -INFINITY, -INFINITY}};
        ref[k] = kBvh4Empty;
        tris[k] = 0u;
    }
#pragma unroll
    for (int ns = 2; ns < 4; ++ns) {
        int best = -1, open = 0;
        float area = 0.0f;
#pragma unroll
        for (int k = 0; k < ns; ++k)
            if (ref[k] >= 0) {
                // (the first one whatever its surface, which is NaN beside vertices
                // that are not finite: max_nodes4 counts on every opening)
                const float a = half_area(box[k]);
                if (best < 0 || a > area) { area = fmaxf(a, 0.0f); best = k; open = ref[k]; }
            }
        if (best < 0) break;
        const BvhNode nd = nodes[open];
#pragma unroll
        for (int k = 0; k < ns; ++k)
            if (k == best) {
                box[k] = node_half(nd, 0u);
                ref[k] = nd.left;
                tris[k] = nd.lcnt;
            }
        box[ns] = node_half(nd, 1u);
        ref[ns] = nd.right;
        tris[ns] = nd.rcnt;
    }
    // inner children first, either kind in its order
#pragma unroll
    for (int pass = 0; pass < 3; ++pass)
#pragma unroll
        for (int k = 0; k < 3 - pass; ++k)
            if (ref[k] < 0 && ref[k + 1] >= 0) {
                const Box b = box[k];
                box[k] = box[k + 1];
                box[k + 1] = b;
                const int rf = ref[k];
                ref[k] = ref[k + 1];
                ref[k + 1] = rf;
                const uint32_t tr = tris[k];
                tris[k] = tris[k + 1];
                tris[k + 1] = tr;
            }
    uint32_t inner = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) inner += ref[k] >= 0 ? 1u : 0u;
    Bvh4Node out;
    uint32_t id = t.room, room = t.room + inner;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        out.lox[k] = box[k].lo[0]; out.loy[k] = box[k].lo[1]; out.loz[k] = box[k].lo[2];
        out.hix[k] = box[k].hi[0]; out.hiy[k] = box[k].hi[1]; out.hiz[k] = box[k].hi[2];
        out.child[k] = ref[k];
        if (ref[k] >= 0) {
            next[k] = Open{id, ref[k], room};
            out.child[k] = (int)id++;
            room += max_nodes4(tris[k]) - 1u;
        }
    }
    out.pad[0] = out.pad[1] = out.pad[2] = out.pad[3] = 0;
    nodes4[t.id] = out;
    nodes4h[t.id] = grid_node(out);
    return inner;
}

}  // namespace lbvh
}  // namespace rbh
