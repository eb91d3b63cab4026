// Four lanes per ray: the four-wide traversal of traverse.hpp with one child
// of the node per lane of a quad, for launches with too few rays to fill the
// chip. A wave then walks 16 rays instead of 64, each step tests one box and
// at most one triangle per lane, and a lane's chain of dependent instructions
// per step is less than half as long, which is what bounds a launch of a few
// waves per SIMD. (With the chip full it is slower: the same boxes cost four
// times the lanes and the ordering work is repeated by every lane.)
//
// The walk is the per-lane one exactly: children in the same order, triangle
// tests folded in slot order with the same comparisons, so closest hits are
// the same bits whichever form ran, ties included.
#pragma once
#include "traverse.hpp"

namespace rbh {
namespace dev {

constexpr int kQuadRays = 16;      // rays of a wave
constexpr int kQuadStackLds = 64;  // stack entries per ray in LDS (4 KB per wave); deeper ones spill

// The value of lane J of the quad / of the quad's lane xor X, on all four lanes.
template <int J>
__device__ __forceinline__ uint32_t quad_lane(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, J * 0x55, 0xF, 0xF, true);
}
template <int J>
__device__ __forceinline__ float quad_lane(float v) { return __uint_as_float(quad_lane<J>(__float_as_uint(v))); }
template <int X>
__device__ __forceinline__ uint32_t quad_xor(uint32_t v) {
    constexpr int ctrl = X == 1 ? 0xB1 : X == 2 ? 0x4E : 0x1B;
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, ctrl, 0xF, 0xF, true);
}

// Row r (lo x, hi x, lo y, hi y, lo z, hi z, child) of child j of a node.
__device__ __forceinline__ float node_row(const Bvh4Node* __restrict__ n, int r, uint32_t j) {
    return reinterpret_cast<const float*>(n)[4 * r + (int)j];
}

// One fold step of the closest hit: lane K's candidate against the ray's
// distance so far, as tri_hit compares it.
template <int K>
__device__ __forceinline__ void quad_fold(bool cand, float T, float det, float t, float& best, uint32_t& owner) {
    const bool hit = cand && !(T > best * det);
    const uint32_t h = quad_lane<K>(hit ? 1u : 0u);
    const float tk = quad_lane<K>(t);
    if (h) {
        best = tk;
        owner = (uint32_t)K;
    }
}

// The closest hit below tmax or, with ANY, whether there is one (leaf other
// than ~0). All four lanes of a quad pass the same ray and receive the same
// hit; quads of a wave may be inactive as a whole.
template <bool ANY, int LDS_DEPTH>
__device__ __forceinline__ Hit traverse4_quad(const Bvh4Node* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                              uint32_t nnodes, V3 o, V3 d, float tmax,
                                              const TravStack<LDS_DEPTH>& stack) {
    const uint32_t j = (uint32_t)__lane_id() & 3u;
    Hit h;
    h.t = tmax;
    h.leaf = 0xFFFFFFFFu;
    h.b1 = h.b2 = 0.0f;
    const RayShear sh = make_shear(d);
    if (nnodes == 0u) {
        // a single-triangle scene
        float t, b1, b2;
        if (tri_hit(sh, o, tris[0], tmax, t, b1, b2)) h = Hit{t, b1, b2, 0u};
        return h;
    }
    const float ix = 1.0f / d.x, iy = 1.0f / d.y, iz = 1.0f / d.z;
    // this lane's last accepted triangle; owner: the quad lane holding the closest hit (4: none)
    float mb1 = 0.0f, mb2 = 0.0f;
    uint32_t mleaf = 0u, owner = 4u;
    int node = 0, sp = 0;
    while (true) {
        const Bvh4Node* __restrict__ n = nodes + node;
        const float lx = node_row(n, 0, j), hx = node_row(n, 1, j), ly = node_row(n, 2, j), hy = node_row(n, 3, j),
                    lz = node_row(n, 4, j), hz = node_row(n, 5, j);
        const int ch = (int)__float_as_uint(node_row(n, 6, j));
        const float best = h.t * 1.00000024f;
        const float x0 = (lx - o.x) * ix, x1 = (hx - o.x) * ix;
        const float y0 = (ly - o.y) * iy, y1 = (hy - o.y) * iy;
        const float z0 = (lz - o.z) * iz, z1 = (hz - o.z) * iz;
        const float tnear = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fmaxf(fminf(z0, z1), 0.0f));
        const float tfar = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fminf(fmaxf(z0, z1), best));
        const bool in = ch != kBvh4Empty && tnear <= tfar * 1.00000024f;
        bool cand = false;
        float T = 0.0f, det = 0.0f, t = 0.0f, b1 = 0.0f, b2 = 0.0f;
        if (in && ch < 0) cand = tri_candidate(sh, o, tris[~ch], h.t, T, det, t, b1, b2);
        if (__ballot(cand) != 0ull) {
            if (ANY) {
                const uint32_t c = cand ? 1u : 0u;
                uint32_t a = c | quad_xor<1>(c);
                a |= quad_xor<2>(a);
                if (a) {
                    h.leaf = 0u;
                    return h;
                }
            } else {
                uint32_t win = 4u;
                quad_fold<0>(cand, T, det, t, h.t, win);
                quad_fold<1>(cand, T, det, t, h.t, win);
                quad_fold<2>(cand, T, det, t, h.t, win);
                quad_fold<3>(cand, T, det, t, h.t, win);
                if (win != 4u) owner = win;
                if (win == j) {
                    mb1 = b1;
                    mb2 = b2;
                    mleaf = (uint32_t)~ch;
                }
            }
        }
        // surviving inner children nearest first, ordered by the keys of the per-lane walk
        const float limit = h.t * 1.00000024f * 1.00000024f;
        const uint32_t key = (in && ch >= 0 && tnear <= limit) ? ((__float_as_uint(tnear) & 0x7FFFFFFCu) | j) : ~0u;
        const uint32_t k1 = quad_xor<1>(key), k2 = quad_xor<2>(key), k3 = quad_xor<3>(key);
        const uint32_t rank = (k1 < key ? 1u : 0u) + (k2 < key ? 1u : 0u) + (k3 < key ? 1u : 0u);
        const uint32_t cnt = (key != ~0u ? 1u : 0u) + (k1 != ~0u ? 1u : 0u) + (k2 != ~0u ? 1u : 0u) + (k3 != ~0u ? 1u : 0u);
        if (cnt != 0u) {
            // the nearest next, the others farthest first on the stack
            if (key != ~0u && rank != 0u) stack.put(sp + (int)(cnt - 1u - rank), ch);
            uint32_t next = key != ~0u && rank == 0u ? (uint32_t)ch : 0u;
            next |= quad_xor<1>(next);
            next |= quad_xor<2>(next);
            node = (int)next;
            sp += (int)cnt - 1;
            continue;
        }
        if (sp == 0) break;
        --sp;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // the entry may be another lane's
        node = stack.get(sp);
    }
    if (!ANY && owner != 4u) {
        const int src = (__lane_id() & ~3) | (int)owner;
        h.b1 = __shfl(mb1, src);
        h.b2 = __shfl(mb2, src);
        h.leaf = (uint32_t)__shfl((int)mleaf, src);
    }
    return h;
}

}  // namespace dev
}  // namespace rbh
