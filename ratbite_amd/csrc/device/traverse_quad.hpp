// Four lanes per ray: the four-wide traversal of traverse.hpp with one child
// of the node per lane of a quad, for launches with too few rays to fill the
// chip. A wave then walks 16 rays instead of 64, each step tests one box and
// at most one triangle per lane, and a lane's chain of dependent instructions
// per step is less than half as long, which is what bounds a launch of a few
// waves per SIMD. (With the chip full it is slower: the same boxes cost four
// times the lanes and the ordering work is repeated by every lane.)
//
// The walk is trav_step's: the same node form, the same arithmetic per box and
// margins, triangle tests folded in slot order with the same comparisons,
// children visited in the same order and deferred ones dropped by the same
// distances. So hits are the same bits whichever form ran over the same nodes,
// ties included.
#pragma once
#include "traverse.hpp"

namespace rbh {
namespace dev {

constexpr int kQuadRays = 16;      // rays of a wave
constexpr int kQuadStackLds = 64;  // stack entries per ray in LDS (8 KB per wave); deeper ones spill

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

// The stack of a ray's quad: LDS_DEPTH entries in LDS with the key they were
// deferred under, read together, and deeper ones in the spill column. Entries
// from DIST_DEPTH on are visited whatever their distance, as DistStack's are.
template <int LDS_DEPTH, int DIST_DEPTH>
struct QuadStack {
    uint2* __restrict__ lds;
    int stride;
    int* __restrict__ spill;
    uint32_t spillStride;
    __device__ __forceinline__ void put(int sp, int v, uint32_t key) const {
        if (sp < LDS_DEPTH) lds[sp * stride] = make_uint2((uint32_t)v, key);
        else spill[(size_t)(sp - LDS_DEPTH) * spillStride] = v;
    }
    // Entry sp; beyond: it starts after distance `limit` (its distance cut to
    // the 16 bits that DistStack keeps).
    __device__ __forceinline__ int get(int sp, float limit, bool& beyond) const {
        beyond = false;
        if (sp >= LDS_DEPTH) return spill[(size_t)(sp - LDS_DEPTH) * spillStride];
        const uint2 e = lds[sp * stride];
        beyond = sp < DIST_DEPTH && __uint_as_float(e.y & 0xFFFF0000u) > limit;
        return (int)e.x;
    }
};

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
template <bool ANY, typename STACK, typename NODE>
__device__ __forceinline__ Hit traverse4_quad(const NODE* __restrict__ nodes, const TriRecord* __restrict__ tris,
                                              uint32_t nnodes, V3 o, V3 d, float tmax, const STACK& stack) {
    const uint32_t j = (uint32_t)__lane_id() & 3u;
    TravRay r;
    trav_init(r, o, d, tmax, nnodes);
    Hit& h = r.h;
    if (nnodes == 0u) {
        // a single-triangle scene
        float t, b1, b2;
        if (tri_hit(r.sh, o, tris[0], tmax, t, b1, b2)) h = Hit{t, b1, b2, 0u};
        return h;
    }
    // this lane's last accepted triangle; owner: the quad lane holding the closest hit (4: none)
    float mb1 = 0.0f, mb2 = 0.0f;
    uint32_t mleaf = 0u, owner = 4u;
    while (true) {
        float tn, tf;
        const int ch = visit_child(nodes, r, j, tn, tf);
        tn = fmaxf(tn, 0.0f);
        const bool in = ch != kBvh4Empty && box_met(tn, tf, h.t);
        bool cand = false;
        float T = 0.0f, det = 0.0f, t = 0.0f, b1 = 0.0f, b2 = 0.0f;
        // (closest hit: the distance is compared in the fold alone, as an accepted
        // hit may lie a rounding behind the one before it)
        if (in && ch < 0) cand = tri_candidate(r.sh, o, tris[~ch], ANY ? h.t : INFINITY, T, det, t, b1, b2);
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
        const float limit = visit_limit(h.t);
        const uint32_t key = (in && ch >= 0 && (ANY || tn <= limit)) ? ((__float_as_uint(tn) & 0x7FFFFFFCu) | j) : ~0u;
        const uint32_t k1 = quad_xor<1>(key), k2 = quad_xor<2>(key), k3 = quad_xor<3>(key);
        const uint32_t rank = (k1 < key ? 1u : 0u) + (k2 < key ? 1u : 0u) + (k3 < key ? 1u : 0u);
        const uint32_t cnt = (key != ~0u ? 1u : 0u) + (k1 != ~0u ? 1u : 0u) + (k2 != ~0u ? 1u : 0u) + (k3 != ~0u ? 1u : 0u);
        if (cnt != 0u) {
            // the nearest next, the others farthest first on the stack
            if (key != ~0u && rank != 0u) stack.put(r.sp + (int)(cnt - 1u - rank), ch, key);
            uint32_t next = key != ~0u && rank == 0u ? (uint32_t)ch : 0u;
            next |= quad_xor<1>(next);
            next |= quad_xor<2>(next);
            r.node = (int)next;
            r.sp += (int)cnt - 1;
            continue;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // the entries may be another lane's
        bool beyond = true;
        while (beyond && r.sp > 0) {
            r.node = stack.get(--r.sp, limit, beyond);
            if (ANY) beyond = false;
        }
        if (beyond) break;
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
