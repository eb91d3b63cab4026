// LBVH traversal: closest-hit and any-hit queries replacing optixTrace /
// optixTraverse(TERMINATE_ON_FIRST_HIT) (src/kernels/pathtrace.cu:1162-1177,
// 1704-1720). Stack in LDS (one column per lane, so consecutive lanes hit
// consecutive banks); ray/box slabs with a conservative far bound; the
// watertight ray/triangle test of Woop, Benthin and Wald (JCGT 2013) with
// per-ray shear constants.
#pragma once
#include "vec.hpp"
#include "types.hpp"

namespace rbh {
namespace dev {

// The ray's dominant axis and the shear that maps its direction to it. The
// other two axes follow cyclically for either sign of the direction: swapping
// them for a negative one, as published, negates U, V, W, the determinant and
// T exactly, and the test makes the determinant positive anyway.
struct RayShear {
    int kz;
    float Sx, Sy, Sz;
};
__device__ __forceinline__ V3 to_ray_axes(V3 v, int kz) {
    const bool z = kz == 2, x = kz == 0;
    return V3{z ? v.x : x ? v.y : v.z, z ? v.y : x ? v.z : v.x, z ? v.z : x ? v.x : v.y};
}
__device__ __forceinline__ RayShear make_shear(V3 d) {
    RayShear s;
    const float ax = fabsf(d.x), ay = fabsf(d.y), az = fabsf(d.z);
    s.kz = ax > ay ? (ax > az ? 0 : 2) : (ay > az ? 1 : 2);
    const V3 r = to_ray_axes(d, s.kz);
    s.Sx = r.x / r.z;
    s.Sy = r.y / r.z;
    s.Sz = 1.0f / r.z;
    return s;
}

struct Hit {
    float t, b1, b2;
    uint32_t leaf;   // leaf-order triangle record of the hit; 0xFFFFFFFF: miss
};

// A hit at or before tmax; T and det give its distance as the unrounded
// quotient t = T / det.
__device__ __forceinline__ bool tri_candidate(const RayShear& s, V3 o, const TriRecord& tr, float tmax, float& T,
                                              float& det, float& t, float& b1, float& b2) {
    // No FMA contraction: the 2D edge functions of a shared edge must round
    // identically from both triangles for the test to stay watertight.
#pragma clang fp contract(off)
    const V3 A = to_ray_axes(V3{tr.v0x - o.x, tr.v0y - o.y, tr.v0z - o.z}, s.kz);
    const V3 B = to_ray_axes(V3{tr.v1x - o.x, tr.v1y - o.y, tr.v1z - o.z}, s.kz);
    const V3 C = to_ray_axes(V3{tr.v2x - o.x, tr.v2y - o.y, tr.v2z - o.z}, s.kz);
    const float Akz = A.z, Bkz = B.z, Ckz = C.z;
    const float Ax = A.x - s.Sx * Akz, Ay = A.y - s.Sy * Akz;
    const float Bx = B.x - s.Sx * Bkz, By = B.y - s.Sy * Bkz;
    const float Cx = C.x - s.Sx * Ckz, Cy = C.y - s.Sy * Ckz;
    float U = Cx * By - Cy * Bx, V = Ax * Cy - Ay * Cx, W = Bx * Ay - By * Ax;
    if (U == 0.0f || V == 0.0f || W == 0.0f) {
        U = (float)((double)Cx * By - (double)Cy * Bx);
        V = (float)((double)Ax * Cy - (double)Ay * Cx);
        W = (float)((double)Bx * Ay - (double)By * Ax);
    }
    if ((U < 0.0f || V < 0.0f || W < 0.0f) && (U > 0.0f || V > 0.0f || W > 0.0f)) return false;
    det = U + V + W;
    if (det == 0.0f) return false;
    T = U * (s.Sz * Akz) + V * (s.Sz * Bkz) + W * (s.Sz * Ckz);
    if (det < 0.0f) { T = -T; det = -det; V = -V; W = -W; }
    if (T < 0.0f || T > tmax * det) return false;
    const float r = 1.0f / det;
    t = T * r;
    b1 = V * r;
    b2 = W * r;
    return true;
}
__device__ __forceinline__ bool tri_hit(const RayShear& s, V3 o, const TriRecord& tr, float tmax, float& t, float& b1,
                                        float& b2) {
    float T, det;
    return tri_candidate(s, o, tr, tmax, T, det, t, b1, b2);
}

// Traversal stack of at most kMaxStack entries (the LBVH builder rejects
// trees deeper than that). The LDS_DEPTH entries nearest the bottom live in
// LDS, one column per lane (stride = lanes per block), so consecutive lanes
// hit consecutive banks; deeper entries go to a per-lane spill column in
// global memory (entry k of lane t at spill[k * spillStride + t]), which only
// rays with many deferred subtrees touch. A small LDS part keeps more waves
// resident per CU than a full 64-entry LDS stack would.
constexpr int kMaxStack = 64;     // binary tree: depth <= 64
constexpr int kMaxStack4 = 192;   // four-wide tree: at most 3 deferred children per level, <= 64 levels
// Entries of the closest-hit walks with a distance (DistStack): six bytes each
// in LDS, as many as leave room for seven waves per SIMD of the trace kernel,
// which the registers allow. Every closest-hit walk keeps as many, so that
// they drop the same entries.
constexpr int kDistLds = 12;

template <int LDS_DEPTH>
struct TravStack {
    int* __restrict__ lds;
    int stride;
    int* __restrict__ spill;
    uint32_t spillStride;
    __device__ __forceinline__ void put(int sp, int v) const {
        if (sp < LDS_DEPTH) lds[sp * stride] = v;
        else spill[(size_t)(sp - LDS_DEPTH) * spillStride] = v;
    }
    __device__ __forceinline__ int get(int sp) const {
        if (sp < LDS_DEPTH) return lds[sp * stride];
        return spill[(size_t)(sp - LDS_DEPTH) * spillStride];
    }
    // Pushes the children of the keys that are not ~0, the last one first.
    // With room in the LDS part every child is written, a missing one where
    // the next push overwrites it: no branch per child.
    template <typename CHILD>
    __device__ __forceinline__ void push3(int& sp, uint32_t k1, uint32_t k2, uint32_t k3, CHILD child) const {
        if (sp + 3 <= LDS_DEPTH) {
            lds[sp * stride] = child(k3);
            sp += k3 != ~0u ? 1 : 0;
            lds[sp * stride] = child(k2);
            sp += k2 != ~0u ? 1 : 0;
            lds[sp * stride] = child(k1);
            sp += k1 != ~0u ? 1 : 0;
        } else {
            if (k3 != ~0u) put(sp++, child(k3));
            if (k2 != ~0u) put(sp++, child(k2));
            if (k1 != ~0u) put(sp++, child(k1));
        }
    }
    __device__ __forceinline__ bool beyond(int, float) const { return false; }
};

// The same stack with the entry distance of each deferred subtree, its upper
// 16 bits (rounded towards the ray's origin): a closest-hit walk drops the
// entries that lie beyond the hit found since, instead of visiting them and
// missing all their boxes. (Spilled entries have no distance and are visited.)
template <int LDS_DEPTH>
struct DistStack {
    int* __restrict__ lds;
    uint16_t* __restrict__ dist;
    int stride;
    int* __restrict__ spill;
    uint32_t spillStride;
    template <typename CHILD>
    __device__ __forceinline__ void push3(int& sp, uint32_t k1, uint32_t k2, uint32_t k3, CHILD child) const {
        if (sp + 3 <= LDS_DEPTH) {
            lds[sp * stride] = child(k3);
            dist[sp * stride] = (uint16_t)(k3 >> 16);
            sp += k3 != ~0u ? 1 : 0;
            lds[sp * stride] = child(k2);
            dist[sp * stride] = (uint16_t)(k2 >> 16);
            sp += k2 != ~0u ? 1 : 0;
            lds[sp * stride] = child(k1);
            dist[sp * stride] = (uint16_t)(k1 >> 16);
            sp += k1 != ~0u ? 1 : 0;
        } else {
            if (k3 != ~0u) put(sp++, child(k3), k3);
            if (k2 != ~0u) put(sp++, child(k2), k2);
            if (k1 != ~0u) put(sp++, child(k1), k1);
        }
    }
    __device__ __forceinline__ void put(int sp, int v, uint32_t key) const {
        if (sp < LDS_DEPTH) {
            lds[sp * stride] = v;
            dist[sp * stride] = (uint16_t)(key >> 16);
        } else {
            spill[(size_t)(sp - LDS_DEPTH) * spillStride] = v;
        }
    }
    __device__ __forceinline__ int get(int sp) const {
        if (sp < LDS_DEPTH) return lds[sp * stride];
        return spill[(size_t)(sp - LDS_DEPTH) * spillStride];
    }
    // the subtree of entry sp starts after distance `limit`
    __device__ __forceinline__ bool beyond(int sp, float limit) const {
        return sp < LDS_DEPTH && __uint_as_float((uint32_t)dist[sp * stride] << 16) > limit;
    }
};

// Traverses the LBVH. Returns the closest hit below tmax or, with ANY, the
// first one found.
template <bool ANY, int LDS_DEPTH>
__device__ __forceinline__ Hit traverse(const BvhNode* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                        uint32_t nnodes, V3 o, V3 d, float tmax, const TravStack<LDS_DEPTH>& stack) {
    Hit h;
    h.t = tmax;
    h.leaf = 0xFFFFFFFFu;
    h.b1 = h.b2 = 0.0f;
    const RayShear sh = make_shear(d);
    const float ix = 1.0f / d.x, iy = 1.0f / d.y, iz = 1.0f / d.z;
    int node = nnodes ? 0 : ~0;
    int sp = 0;
    while (true) {
        if (node >= 0) {
            const float4* q = reinterpret_cast<const float4*>(nodes + node);
            const float4 a = q[0], b = q[1], c = q[2];
            const int4 e = reinterpret_cast<const int4*>(q)[3];
            const float best = h.t * 1.00000024f;
            // left child
            const float l0x = (a.x - o.x) * ix, l1x = (a.y - o.x) * ix;
            const float l0y = (a.z - o.y) * iy, l1y = (a.w - o.y) * iy;
            const float l0z = (c.x - o.z) * iz, l1z = (c.y - o.z) * iz;
            const float lnear = fmaxf(fmaxf(fminf(l0x, l1x), fminf(l0y, l1y)), fmaxf(fminf(l0z, l1z), 0.0f));
            const float lfar = fminf(fminf(fmaxf(l0x, l1x), fmaxf(l0y, l1y)), fminf(fmaxf(l0z, l1z), best));
            // right child
            const float r0x = (b.x - o.x) * ix, r1x = (b.y - o.x) * ix;
            const float r0y = (b.z - o.y) * iy, r1y = (b.w - o.y) * iy;
            const float r0z = (c.z - o.z) * iz, r1z = (c.w - o.z) * iz;
            const float rnear = fmaxf(fmaxf(fminf(r0x, r1x), fminf(r0y, r1y)), fmaxf(fminf(r0z, r1z), 0.0f));
            const float rfar = fminf(fminf(fmaxf(r0x, r1x), fmaxf(r0y, r1y)), fminf(fmaxf(r0z, r1z), best));
            const bool hl = lnear <= lfar * 1.00000024f, hr = rnear <= rfar * 1.00000024f;
            if (hl && hr) {
                const bool lfirst = lnear <= rnear;
                stack.put(sp, lfirst ? e.y : e.x);
                ++sp;
                node = lfirst ? e.x : e.y;
                continue;
            }
            if (hl) { node = e.x; continue; }
            if (hr) { node = e.y; continue; }
        } else {
            const TriRecord& tr = tris[~node];
            float t, b1, b2;
            if (tri_hit(sh, o, tr, h.t, t, b1, b2)) {
                h.t = t;
                h.b1 = b1;
                h.b2 = b2;
                h.leaf = (uint32_t)~node;
                if (ANY) return h;
            }
        }
        if (sp == 0) break;
        --sp;
        node = stack.get(sp);
    }
    return h;
}

// Four-wide traversal: a node fetch tests four child boxes; leaf children
// (single triangles) are intersected on the spot, inner children that
// survive the updated distance are visited nearest first, the others pushed.
// Four-wide traversal as a resumable state machine, so that a persistent
// kernel can give a lane a new ray as soon as its previous one finishes
// while the other lanes of the wave keep traversing.
struct TravRay {
    V3 o, d;
    float ix, iy, iz;
    // per axis: byte offset in a Bvh4Node of the row of near planes; modulo 32
    // the rotation that brings the near plane of a Bvh4HNode's pair down
    uint32_t ox, oy, oz;
    RayShear sh;
    Hit h;
    int node;   // next node to visit (~i: the root is triangle i)
    int sp;     // entries on the traversal stack
};

// 1 / d, or 1e30 if that is larger in size: a slab parallel to the ray is then
// entered and left far away on either side, or never, without infinities times
// zero. (Positive, so that a ray in a face meets the box on the grid: the
// lower plane at exactly 0, the upper one at its margin of 2^-22.)
__device__ __forceinline__ float finite_inverse(float d) {
    const float i = 1.0f / d;
    return fabsf(i) > 1e30f ? 1e30f : i;
}

__device__ __forceinline__ void trav_init(TravRay& r, V3 o, V3 d, float tmax, uint32_t nnodes) {
    r.o = o;
    r.d = d;
    r.ix = finite_inverse(d.x);
    r.iy = finite_inverse(d.y);
    r.iz = finite_inverse(d.z);
    r.ox = r.ix < 0.0f ? 16u : 0u;
    r.oy = r.iy < 0.0f ? 48u : 32u;
    r.oz = r.iz < 0.0f ? 80u : 64u;
    r.sh = make_shear(d);
    r.h.t = tmax;
    r.h.leaf = 0xFFFFFFFFu;
    r.h.b1 = r.h.b2 = 0.0f;
    r.node = nnodes ? 0 : ~0;
    r.sp = 0;
}

// A four-wide node as a ray meets it: where it enters and leaves the children's
// boxes (not yet bounded by the ray's ends), and the child references.
struct Visit4 {
    float tn[4], tf[4];
    uint32_t first;      // index of the first inner child
    uint32_t order[4];   // inner children: their number among them; others: 4
    uint32_t tris;       // slots with a triangle
};
// Of the two planes a box has on an axis the ray reaches the lower one first
// if its direction is positive. Which row is the near one is an address here,
// so the choice costs no instruction per child.
__device__ __forceinline__ void visit_node(const Bvh4Node* __restrict__ nodes, const TravRay& r, Visit4& v) {
    const char* base = reinterpret_cast<const char*>(nodes);
    const uint32_t at = (uint32_t)r.node << 7;
    auto row = [&](uint32_t off, float (&w)[4]) {
        const float4 q = *reinterpret_cast<const float4*>(base + off);
        w[0] = q.x; w[1] = q.y; w[2] = q.z; w[3] = q.w;
    };
    float nx[4], fx[4], ny[4], fy[4], nz[4], fz[4];
    row(at + r.ox, nx);
    row((at + r.ox) ^ 16u, fx);
    row(at + r.oy, ny);
    row((at + r.oy) ^ 16u, fy);
    row(at + r.oz, nz);
    row((at + r.oz) ^ 16u, fz);
    const int4 c4 = *reinterpret_cast<const int4*>(base + (at + 96u));
    const uint32_t c[4] = {(uint32_t)c4.x, (uint32_t)c4.y, (uint32_t)c4.z, (uint32_t)c4.w};
    // the inner children's indices are consecutive and the others have the sign bit
    const uint32_t c01 = c[0] < c[1] ? c[0] : c[1], c23 = c[2] < c[3] ? c[2] : c[3];
    v.first = c01 < c23 ? c01 : c23;
    v.tris = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        v.tn[k] = fmaxf(fmaxf((nx[k] - r.o.x) * r.ix, (ny[k] - r.o.y) * r.iy), (nz[k] - r.o.z) * r.iz);
        v.tf[k] = fminf(fminf((fx[k] - r.o.x) * r.ix, (fy[k] - r.o.y) * r.iy), (fz[k] - r.o.z) * r.iz);
        v.order[k] = (int32_t)c[k] >= 0 ? c[k] - v.first : 4u;
        v.tris |= c[k] > (uint32_t)kBvh4Empty ? 1u << k : 0u;
    }
}
// On the grid plane q is met at q * (2^e / d) + (o - origin) / d: one fused
// multiply-add per plane. The second term, computed with two roundings, is
// moved outwards by four units of its own size (2^-22), which covers them and
// the rounding of the product's factor; the relative error of the sum is the
// caller's margin.
struct GridAxis {
    float a, bn, bf;   // distance to near plane q: q a + bn, to far plane q: q a + bf
};
__device__ __forceinline__ GridAxis grid_axis(uint32_t meta, int sh, uint32_t corner, float o, float i) {
    const float b = (__uint_as_float(corner) - o) * i;
    return GridAxis{ldexpf(i, (int)(meta << (24 - sh)) >> 24), fmaf(fabsf(b), -2.3841858e-7f, b),
                    fmaf(fabsf(b), 2.3841858e-7f, b)};
}
__device__ __forceinline__ float half_bits(uint32_t u) { return (float)__builtin_bit_cast(_Float16, (uint16_t)u); }
// The pair of planes w of one slot and axis: near in tn, far in tf.
__device__ __forceinline__ void grid_planes(const GridAxis& g, uint32_t w, uint32_t rotation, float& tn, float& tf) {
    const uint32_t r = __builtin_rotateright32(w, rotation);
    tn = fmaf(half_bits(r), g.a, g.bn);
    tf = fmaf(half_bits(r >> 16), g.a, g.bf);
}

__device__ __forceinline__ void visit_node(const Bvh4HNode* __restrict__ nodes, const TravRay& r, Visit4& v) {
    const Bvh4HNode* __restrict__ nd = nodes + r.node;
    const uint4* q = reinterpret_cast<const uint4*>(nd);
    const uint4 h = q[0], p0 = q[1], p1 = q[2], p2 = q[3];
    v.first = (uint32_t)nd->child[0];
    const uint32_t w[4][3] = {{p0.x, p0.y, p0.z}, {p0.w, p1.x, p1.y}, {p1.z, p1.w, p2.x}, {p2.y, p2.z, p2.w}};
    const GridAxis x = grid_axis(h.w, 0, h.x, r.o.x, r.ix), y = grid_axis(h.w, 8, h.y, r.o.y, r.iy),
                   z = grid_axis(h.w, 16, h.z, r.o.z, r.iz);
    v.tris = (h.w >> 24) & 15u;
    const uint32_t inner = h.w >> 28;
#pragma unroll
    for (uint32_t k = 0; k < 4u; ++k) {
        float nx, fx, ny, fy, nz, fz;
        grid_planes(x, w[k][0], r.ox, nx, fx);
        grid_planes(y, w[k][1], r.oy, ny, fy);
        grid_planes(z, w[k][2], r.oz, nz, fz);
        v.tn[k] = fmaxf(fmaxf(nx, ny), nz);
        v.tf[k] = fminf(fminf(fx, fy), fz);
        v.order[k] = k < inner ? k : 4u;
    }
}

// The same for child k alone, by the same arithmetic: where the ray enters and
// leaves its box (an empty slot has no meaningful distances), and the child's
// reference.
__device__ __forceinline__ int visit_child(const Bvh4Node* __restrict__ nodes, const TravRay& r, uint32_t k, float& tn,
                                           float& tf) {
    const Bvh4Node* __restrict__ nd = nodes + r.node;
    const float* rows = reinterpret_cast<const float*>(nd) + k;
    auto row = [&](uint32_t off) { return rows[off >> 2]; };
    const float nx = row(r.ox), fx = row(r.ox ^ 16u), ny = row(r.oy), fy = row(r.oy ^ 16u), nz = row(r.oz), fz = row(r.oz ^ 16u);
    tn = fmaxf(fmaxf((nx - r.o.x) * r.ix, (ny - r.o.y) * r.iy), (nz - r.o.z) * r.iz);
    tf = fminf(fminf((fx - r.o.x) * r.ix, (fy - r.o.y) * r.iy), (fz - r.o.z) * r.iz);
    return nd->child[k];
}
__device__ __forceinline__ int visit_child(const Bvh4HNode* __restrict__ nodes, const TravRay& r, uint32_t k, float& tn,
                                           float& tf) {
    const Bvh4HNode* __restrict__ nd = nodes + r.node;
    const uint4 h = *reinterpret_cast<const uint4*>(nd);
    const uint32_t* w = reinterpret_cast<const uint32_t*>(nd->plane[k]);
    float nx, fx, ny, fy, nz, fz;
    grid_planes(grid_axis(h.w, 0, h.x, r.o.x, r.ix), w[0], r.ox, nx, fx);
    grid_planes(grid_axis(h.w, 8, h.y, r.o.y, r.iy), w[1], r.oy, ny, fy);
    grid_planes(grid_axis(h.w, 16, h.z, r.o.z, r.iz), w[2], r.oz, nz, fz);
    tn = fmaxf(fmaxf(nx, ny), nz);
    tf = fminf(fminf(fx, fy), fz);
    return nd->child[k];
}

// The margins of a step: a box is met if it is entered before it is left and
// before the hit so far, and visited if that hit, after the node's triangles,
// still lies behind its entry.
__device__ __forceinline__ bool box_met(float tn, float tf, float hit) {
    return tn <= fminf(tf, hit * 1.00000024f) * 1.0000005f;
}
__device__ __forceinline__ float visit_limit(float hit) { return hit * 1.00000024f * 1.0000005f; }

__device__ __forceinline__ uint32_t min_u(uint32_t a, uint32_t b) { return a < b ? a : b; }
__device__ __forceinline__ uint32_t max_u(uint32_t a, uint32_t b) { return a < b ? b : a; }
__device__ __forceinline__ uint32_t med3_u(uint32_t a, uint32_t b, uint32_t c) {
    return max_u(min_u(a, b), min_u(max_u(a, b), c));
}

// Visits r.node: tests its triangle children (nearest hit so far shortens
// the ray), descends into the nearest box hit and defers the others,
// nearest last on the stack. Returns true when the query is complete.
// NODE: Bvh4Node or Bvh4HNode.
// The kernels that walk are bound by the latency of a step: waves wait for
// memory in 60% of their cycles at 25 waves a CU, and a CU issues 0.85 vector
// instructions a cycle (1.4 in k_accumulate). So a step loads little (68 bytes
// instead of 112), its pushes and its sorting network have no branches, and
// entries beyond the hit are dropped when they are popped. 1080p frame of 4.1M
// triangles at 64 samples, against four rows a box, a branch per push and no
// dropping: bounce rays 31.3 -> 25.8 ms, shadow rays 21.1 -> 16.6 ms, camera
// rays 25.3 -> 25.0 ms.
template <bool ANY, typename STACK, typename NODE>
__device__ __forceinline__ bool trav_step(const NODE* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                          TravRay& r, const STACK& stack) {
    if (r.node < 0) {
        // a single-triangle scene: the root is the leaf
        const TriRecord& tr = tris[~r.node];
        float t, b1, b2;
        if (tri_hit(r.sh, r.o, tr, r.h.t, t, b1, b2)) {
            r.h.t = t;
            r.h.b1 = b1;
            r.h.b2 = b2;
            r.h.leaf = (uint32_t)~r.node;
        }
        return true;
    }
    Visit4 v;
    visit_node(nodes, r, v);
    float tn[4];
    bool in[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        tn[k] = fmaxf(v.tn[k], 0.0f);
        in[k] = box_met(tn[k], v.tf[k], r.h.t);
    }
    // Triangle children first (a hit shortens the ray for the boxes), in
    // slot order. One loop over each lane's own triangle slots: a wave runs
    // it as often as its lane with the most triangle children needs, instead
    // of once for every slot in which some lane has one.
    uint32_t triMask = 0;
#pragma unroll
    for (int k = 0; k < 4; ++k) triMask |= in[k] ? (1u << k) : 0u;
    triMask &= v.tris;
    while (triMask) {
        const uint32_t k = (uint32_t)__builtin_ctz(triMask);
        triMask &= triMask - 1u;
        const int c = nodes[r.node].child[k];
        const TriRecord& tr = tris[~c];
        float t, b1, b2;
        if (tri_hit(r.sh, r.o, tr, r.h.t, t, b1, b2)) {
            r.h.t = t;
            r.h.b1 = b1;
            r.h.b2 = b2;
            r.h.leaf = (uint32_t)~c;
            if (ANY) return true;
        }
    }
    // Surviving inner children nearest first. A child's key is the bit
    // pattern of its entry distance (>= 0, so ordered as an unsigned
    // integer; the sign bit cleared for -0) with its number among the node's
    // inner children in the two low bits: their indices are consecutive, and
    // children within 4 ulp of each other go in slot order. Culled and empty
    // slots sort last as ~0.
    const float limit = visit_limit(r.h.t);
    uint32_t key[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
        key[k] = (in[k] && v.order[k] < 4u && (ANY || tn[k] <= limit)) ? ((__float_as_uint(tn[k]) & 0x7FFFFFFCu) | v.order[k])
                                                                       : ~0u;
    // three keys by minimum, median and maximum, the fourth inserted the same way
    const uint32_t lo = min_u(min_u(key[0], key[1]), key[2]), mid = med3_u(key[0], key[1], key[2]),
                   hi = max_u(max_u(key[0], key[1]), key[2]);
    const uint32_t k0 = min_u(lo, key[3]), k1 = med3_u(lo, mid, key[3]), k2 = med3_u(mid, hi, key[3]), k3 = max_u(hi, key[3]);
    auto child = [&](uint32_t kk) { return (int)(v.first + (kk & 3u)); };
    if (k0 != ~0u) {
        // farthest pushed first, so the nearer ones are popped first
        stack.push3(r.sp, k1, k2, k3, child);
        r.node = child(k0);
        return false;
    }
    while (r.sp > 0) {
        --r.sp;
        if (!ANY && stack.beyond(r.sp, limit)) continue;
        r.node = stack.get(r.sp);
        return false;
    }
    return true;
}

// Whole query in one call: the closest hit below tmax or, with ANY, the
// first one found.
template <bool ANY, typename STACK, typename NODE>
__device__ __forceinline__ Hit traverse4(const NODE* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                         uint32_t nnodes, V3 o, V3 d, float tmax, const STACK& stack) {
    TravRay r;
    trav_init(r, o, d, tmax, nnodes);
    while (!trav_step<ANY>(nodes, tris, r, stack)) {
    }
    return r.h;
}

}  // namespace dev
}  // namespace rbh
