// Linear BVH build on gfx950, replacing optixAccelBuild
// (src/core/rendering_interface.cpp:733-1064):
//   1. triangle centroid bounds (block reduction + ordered-int atomics)
//   2. Morton codes on the centroid grid, made unique with the triangle
//      index in the low bits of a 64-bit key: the index takes the bits n
//      needs, the Morton code as many of the rest as fit three axes (at most
//      21 per axis; 14 for 4.1M triangles, where 10 bits per axis would put
//      84% of the triangles in cells shared with others)
//   3. stable LSD radix sort of the keys (radix.hpp: ballot-ranked 8-bit digits)
//   4. Karras (HPG 2012) hierarchy: internal node i covers a key range and
//      splits at the highest differing bit
//   5. boxes bottom up: a workgroup takes 2048 consecutive leaves, writes their
//      triangle records and climbs the hierarchy in LDS (of a node's two
//      children the second to arrive merges them) as far as the nodes' leaf
//      ranges stay within the workgroup's; above them a workgroup climbs for
//      every group of 32 such tiles, and one for the few nodes above the
//      groups (no cross-XCD fences: only kernel boundaries order the three). A node is emitted where its children meet, as the 64-byte
//      two-child node with both child boxes
//   6. collapse into 128-byte four-wide nodes (with full boxes and on an
//      11-bit grid), top down: a four-wide node
//      takes its binary node's children and keeps opening the inner child
//      with the largest box surface until it has four (device/collapse.hpp).
//      The same workgroup runs the upper levels, then waves take the subtrees
//      below, in rounds that spread what is left over all of them again. The inner
//      children of a four-wide node have consecutive indices in slot order,
//      from a range of indices that belongs to the node alone
// Every root-to-leaf path strictly lengthens the common key prefix, so the
// depth is at most 64 and a 64-entry traversal stack never overflows.
#include "../context.hpp"
#include "../device/collapse.hpp"
#include "radix.hpp"

namespace rbh {

using namespace lbvh;

namespace {

constexpr int kBuildBlock = 256;

__device__ __forceinline__ uint32_t f2ord(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float ord2f(uint32_t u) {
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7fffffffu) : ~u);
}

__global__ void k_bounds_init(uint32_t* __restrict__ b) {
    if (threadIdx.x < 3) b[threadIdx.x] = 0xFFFFFFFFu;           // min (ordered)
    else if (threadIdx.x < 6) b[threadIdx.x] = 0u;               // max (ordered)
}

// One set of six atomics per workgroup, all on one line (2048 workgroups
// waited 140 us for them, 512 do not)
constexpr int kBoundsBlocks = 512;
__global__ __launch_bounds__(kBuildBlock) void k_centroid_bounds(const float* __restrict__ v, const uint32_t* __restrict__ idx,
                                                                 uint32_t n, uint32_t* __restrict__ b) {
    __shared__ float smin[3][kBuildBlock], smax[3][kBuildBlock];
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    float mn[3] = {INFINITY, INFINITY, INFINITY}, mx[3] = {-INFINITY, -INFINITY, -INFINITY};
    for (uint32_t i = t; i < n; i += gridDim.x * blockDim.x) {
        const uint32_t a = idx[3 * i], bb = idx[3 * i + 1], c = idx[3 * i + 2];
        for (int k = 0; k < 3; ++k) {
            const float lo = fminf(fminf(v[3 * a + k], v[3 * bb + k]), v[3 * c + k]);
            const float hi = fmaxf(fmaxf(v[3 * a + k], v[3 * bb + k]), v[3 * c + k]);
            const float ce = 0.5f * (lo + hi);
            mn[k] = fminf(mn[k], ce);
            mx[k] = fmaxf(mx[k], ce);
        }
    }
    for (int k = 0; k < 3; ++k) { smin[k][threadIdx.x] = mn[k]; smax[k][threadIdx.x] = mx[k]; }
    __syncthreads();
    for (int s = kBuildBlock / 2; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s)
            for (int k = 0; k < 3; ++k) {
                smin[k][threadIdx.x] = fminf(smin[k][threadIdx.x], smin[k][threadIdx.x + s]);
                smax[k][threadIdx.x] = fmaxf(smax[k][threadIdx.x], smax[k][threadIdx.x + s]);
            }
        __syncthreads();
    }
    if (threadIdx.x == 0)
        for (int k = 0; k < 3; ++k) {
            atomicMin(&b[k], f2ord(smin[k][0]));
            atomicMax(&b[3 + k], f2ord(smax[k][0]));
        }
}

// bits 0..20 of x to bits 0, 3, 6, ..., 60
__device__ __forceinline__ unsigned long long spread21(uint32_t x) {
    unsigned long long y = x & 0x1FFFFFu;
    y = (y | (y << 32)) & 0x001F00000000FFFFull;
    y = (y | (y << 16)) & 0x001F0000FF0000FFull;
    y = (y | (y << 8)) & 0x100F00F00F00F00Full;
    y = (y | (y << 4)) & 0x10C30C30C30C30C3ull;
    y = (y | (y << 2)) & 0x1249249249249249ull;
    return y;
}

__global__ __launch_bounds__(kBuildBlock) void k_morton(const float* __restrict__ v, const uint32_t* __restrict__ idx,
                                                        uint32_t n, const uint32_t* __restrict__ b, int axisBits,
                                                        int idxBits, unsigned long long* __restrict__ keys) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float lo[3], ext[3];
    for (int k = 0; k < 3; ++k) {
        lo[k] = ord2f(b[k]);
        ext[k] = ord2f(b[3 + k]) - lo[k];
    }
    const float cells = (float)(1u << axisBits);          // exact: a power of two
    const uint32_t a = idx[3 * i], bb = idx[3 * i + 1], c = idx[3 * i + 2];
    uint32_t q[3];
    for (int k = 0; k < 3; ++k) {
        const float l = fminf(fminf(v[3 * a + k], v[3 * bb + k]), v[3 * c + k]);
        const float h = fmaxf(fmaxf(v[3 * a + k], v[3 * bb + k]), v[3 * c + k]);
        const float ce = 0.5f * (l + h);
        const float u = ext[k] > 0.0f ? (ce - lo[k]) / ext[k] : 0.5f;
        q[k] = (uint32_t)fminf(fmaxf(u * cells, 0.0f), cells - 1.0f);
    }
    const unsigned long long m = (spread21(q[0]) << 2) | (spread21(q[1]) << 1) | spread21(q[2]);
    keys[i] = (m << idxBits) | i;
}

__device__ __forceinline__ int common_prefix(const unsigned long long* __restrict__ k, int n, int i, int j) {
    if (j < 0 || j >= n) return -1;
    return __clzll(k[i] ^ k[j]);
}

// Parent link of a binary subtree: the parent's index and the side of the
// child (1: right); kNoParent for the root.
constexpr uint32_t kNoParent = 0xFFFFFFFFu;

// Karras 2012, Figure 4. Internal nodes 0..n-2; child ids >= 0 internal,
// < 0 leaf ~sortedIndex. parent[] holds the parent links of internal nodes
// (slot i) and of leaves (slot n-1+j).
__global__ __launch_bounds__(kBuildBlock) void k_karras(const unsigned long long* __restrict__ k, int n,
                                                        uint32_t* __restrict__ parent) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n - 1) return;
    const int d = (common_prefix(k, n, i, i + 1) - common_prefix(k, n, i, i - 1)) >= 0 ? 1 : -1;
    const int dmin = common_prefix(k, n, i, i - d);
    int lmax = 2;
    while (common_prefix(k, n, i, i + lmax * d) > dmin) lmax <<= 1;
    int l = 0;
    for (int t = lmax >> 1; t >= 1; t >>= 1)
        if (common_prefix(k, n, i, i + (l + t) * d) > dmin) l += t;
    const int j = i + l * d;
    const int dnode = common_prefix(k, n, i, j);
    int s = 0;
    int t = l;
    do {
        t = (t + 1) >> 1;
        if (common_prefix(k, n, i, i + (s + t) * d) > dnode) s += t;
    } while (t > 1);
    const int split = i + s * d + min(d, 0);
    const int first = min(i, j), last = max(i, j);
    parent[first == split ? n - 1 + split : split] = (uint32_t)i << 1;
    parent[last == split + 1 ? n - 1 + split + 1 : split + 1] = ((uint32_t)i << 1) | 1u;
    if (i == 0) parent[0] = kNoParent;
}

// A finished subtree that a workgroup hands on: its parent is not one of the
// nodes with the workgroup's own indices. Lists of them are kept per group of
// kGroupTiles leaf tiles. A workgroup hands on at most one subtree per level
// on either side of its leaves (the parents' ranges are nested), or the root.
struct Pending {
    Box box;
    int ref;            // node, or ~leaf
    uint32_t parent;    // parent link
    uint32_t height;    // inner nodes on its longest path down
    uint32_t tris;
};
// counters of the build's last stages
constexpr int kCollapseRounds = 4;
enum : int { BC_DEPTH = 0, BC_TOP = 1, BC_QUEUE = 2, BC_COUNT = BC_QUEUE + kCollapseRounds + 1 };
constexpr int kLeafTile = 2048;
constexpr int kGroupTiles = 32;
constexpr int kGroupLeaves = kGroupTiles * kLeafTile;
constexpr int kHandedOn = 130;   // most subtrees one workgroup hands on (trees of at most 64 levels)

// cnt: the counters above, then the length of every group's list
__global__ __launch_bounds__(kBuildBlock) void k_build_counters(uint32_t* __restrict__ cnt, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) cnt[i] = 0u;
}

// Triangle records in leaf (Morton) order and the boxes of the hierarchy as
// far as they lie within the workgroup's leaves [first, first + kLeafTile).
// Every thread starts at its leaves and climbs: at a node the first child to
// arrive leaves its box in LDS and stops, the second merges the two, emits
// the node and goes on. An internal node's index is an end of its leaf
// range, so the nodes a workgroup can finish are the ones with its leaves'
// indices; a subtree whose parent lies elsewhere is handed on, and of the
// workgroup's own nodes that stay incomplete the arrived half is stored for
// the climb above. Bound by the records' and nodes' 64-byte writes and
// the vertex gathers.
constexpr int kLeafBlock = 1024;
constexpr uint32_t kArrivedLeft = 1u, kArrivedRight = 0x100u;
__global__ __launch_bounds__(kLeafBlock) void k_leaves(const float* __restrict__ v, const uint32_t* __restrict__ idx,
                                                       const uint32_t* __restrict__ triMaterial,
                                                       const uint32_t* __restrict__ triLight,
                                                       const Material* __restrict__ mats, uint32_t nmats,
                                                       const unsigned long long* __restrict__ keys, int n, int idxBits,
                                                       const uint32_t* __restrict__ parent, TriRecord* __restrict__ tris,
                                                       BvhNode* __restrict__ nodes, uint32_t* __restrict__ arrived,
                                                       uint32_t* __restrict__ height, Pending* __restrict__ pending,
                                                       uint32_t* __restrict__ cnt) {
    __shared__ float sbox[2][6][kLeafTile];
    __shared__ int sref[2][kLeafTile];
    __shared__ uint32_t smeta[2][kLeafTile];   // height << 16 | triangles (at most a tile's)
    __shared__ uint32_t sarrived[kLeafTile], sparent[kLeafTile];
    const int first = blockIdx.x * kLeafTile;
    const uint32_t group = blockIdx.x / kGroupTiles;
    const int own = min(kLeafTile, n - 1 - first);   // internal nodes with the tile's indices
    for (int k = threadIdx.x; k < kLeafTile; k += kLeafBlock) {
        sarrived[k] = 0u;
        sparent[k] = k < own ? parent[first + k] : kNoParent;
    }
    __syncthreads();
    for (int q = threadIdx.x; q < kLeafTile && first + q < n; q += kLeafBlock) {
        const int j = first + q;
        const uint32_t tri = (uint32_t)(keys[j] & ((1ull << idxBits) - 1ull));
        const uint32_t a = idx[3 * (size_t)tri], b = idx[3 * (size_t)tri + 1], c = idx[3 * (size_t)tri + 2];
        TriRecord r;
        r.v0x = v[3 * a]; r.v0y = v[3 * a + 1]; r.v0z = v[3 * a + 2]; r.prim = tri;
        r.v1x = v[3 * b]; r.v1y = v[3 * b + 1]; r.v1z = v[3 * b + 2]; r.material = triMaterial[tri];
        r.v2x = v[3 * c]; r.v2y = v[3 * c + 1]; r.v2z = v[3 * c + 2]; r.light = triLight[tri];
        r.i0 = a; r.i1 = b; r.i2 = c;
        r.shadeClass = r.material < nmats ? shade_class(mats[r.material]) : (uint32_t)SC_SURFACE;
        tris[j] = r;
        if (n == 1) break;
        Pending t;
        t.box = Box{{fminf(fminf(r.v0x, r.v1x), r.v2x), fminf(fminf(r.v0y, r.v1y), r.v2y), fminf(fminf(r.v0z, r.v1z), r.v2z)},
                    {fmaxf(fmaxf(r.v0x, r.v1x), r.v2x), fmaxf(fmaxf(r.v0y, r.v1y), r.v2y), fmaxf(fmaxf(r.v0z, r.v1z), r.v2z)}};
        t.ref = ~j;
        t.parent = parent[n - 1 + j];
        t.height = 0u;
        t.tris = 1u;
        while (true) {
            const int p = (int)(t.parent >> 1), k = p - first;
            const uint32_t side = t.parent & 1u, other = side ^ 1u;
            if (t.parent == kNoParent || k < 0 || k >= own) {
                pending[(size_t)group * kGroupTiles * kHandedOn + atomicAdd(cnt + BC_COUNT + group, 1u)] = t;
                break;
            }
            for (int e = 0; e < 3; ++e) {
                sbox[side][e][k] = t.box.lo[e];
                sbox[side][3 + e][k] = t.box.hi[e];
            }
            sref[side][k] = t.ref;
            smeta[side][k] = t.height << 16 | t.tris;
            const uint32_t old = __hip_atomic_fetch_add(&sarrived[k], side ? kArrivedRight : kArrivedLeft, __ATOMIC_ACQ_REL,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
            if (old == 0u) break;
            const Box ob{{sbox[other][0][k], sbox[other][1][k], sbox[other][2][k]},
                         {sbox[other][3][k], sbox[other][4][k], sbox[other][5][k]}};
            const int oref = sref[other][k];
            const uint32_t om = smeta[other][k], otris = om & 0xFFFFu;
            const Box lb = side ? ob : t.box, rb = side ? t.box : ob;
            BvhNode nd;
            put_half(&nd, 0u, lb, side ? oref : t.ref, side ? otris : t.tris);
            put_half(&nd, 1u, rb, side ? t.ref : oref, side ? t.tris : otris);
            nodes[p] = nd;
            t.box = merge(lb, rb);
            t.ref = p;
            t.height = max(t.height, om >> 16) + 1u;
            t.tris += otris;
            t.parent = sparent[k];
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < own; k += kLeafBlock) {
        const uint32_t got = sarrived[k];
        if (got == (kArrivedLeft | kArrivedRight)) continue;
        arrived[first + k] = got ? 1u : 0u;
        if (!got) continue;
        const uint32_t side = got == kArrivedRight ? 1u : 0u;
        put_half(nodes + first + k, side,
                 Box{{sbox[side][0][k], sbox[side][1][k], sbox[side][2][k]},
                     {sbox[side][3][k], sbox[side][4][k], sbox[side][5][k]}}, sref[side][k], smeta[side][k] & 0xFFFFu);
        height[2 * (size_t)(first + k) + side] = smeta[side][k] >> 16;
    }
}

// Sum of v over the lanes below (v <= 4) and over the wave.
__device__ __forceinline__ uint32_t wave_prefix4(uint32_t v, uint32_t& sum) {
    const unsigned long long b0 = __ballot(v & 1u), b1 = __ballot(v & 2u), b2 = __ballot(v & 4u);
    const unsigned long long lt = (1ull << __lane_id()) - 1ull;
    sum = (uint32_t)(__popcll(b0) + 2 * __popcll(b1) + 4 * __popcll(b2));
    return (uint32_t)(__popcll(b0 & lt) + 2 * __popcll(b1 & lt) + 4 * __popcll(b2 & lt));
}

// One thread's climb from a handed-on subtree over the internal nodes
// [first, last), whose halves, arrival counts and heights lie in global
// memory, which one workgroup sees in order. Returns true with t the subtree
// whose parent lies outside (or the root), false when the other child of a
// node is still to come.
__device__ __forceinline__ bool climb(Pending& t, uint32_t first, uint32_t last, const uint32_t* __restrict__ parent,
                                      BvhNode* nodes, uint32_t* arrived, uint32_t* height) {
    while (true) {
        const uint32_t p = t.parent >> 1, side = t.parent & 1u;
        if (t.parent == kNoParent || p < first || p >= last) return true;
        const uint32_t up = parent[p];
        put_half(nodes + p, side, t.box, t.ref, t.tris);
        height[2 * (size_t)p + side] = t.height;
        if (__hip_atomic_fetch_add(arrived + p, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) == 0u) return false;
        const BvhNode nd = nodes[p];
        t.box = merge(node_half(nd, 0u), node_half(nd, 1u));
        t.ref = (int)p;
        t.height = max(t.height, height[2 * (size_t)p + (side ^ 1u)]) + 1u;
        t.tris = nd.lcnt + nd.rcnt;
        t.parent = up;
    }
}

// The nodes above the leaf tiles: a workgroup per group of 32 tiles, as far
// as the nodes' indices are the group's (about ten subtrees a tile, one a
// thread; one workgroup for all of them took 200 us at 1M triangles).
constexpr int kTopBlock = 1024;
__global__ __launch_bounds__(kTopBlock) void k_tree_groups(const uint32_t* __restrict__ parent, uint32_t ninner,
                                                           BvhNode* nodes, uint32_t* arrived, uint32_t* height,
                                                           const Pending* __restrict__ pending,
                                                           Pending* __restrict__ top, uint32_t* __restrict__ cnt) {
    const uint32_t first = blockIdx.x * (uint32_t)kGroupLeaves, last = min(first + (uint32_t)kGroupLeaves, ninner);
    const uint32_t items = cnt[BC_COUNT + blockIdx.x];
    const Pending* __restrict__ mine = pending + (size_t)blockIdx.x * kGroupTiles * kHandedOn;
    for (uint32_t i = threadIdx.x; i < items; i += kTopBlock) {
        Pending t = mine[i];
        if (climb(t, first, last, parent, nodes, arrived, height)) top[atomicAdd(cnt + BC_TOP, 1u)] = t;
    }
}

// The upper part of the tree in one workgroup: the binary nodes above the
// groups, then the four-wide levels from the root down to the first with
// kSubtrees nodes, which k_collapse takes over (or to the last). The levels'
// lists alternate between the two queues; the final one is left in queue 0.
constexpr uint32_t kSubtrees = 256;
__global__ __launch_bounds__(kTopBlock) void k_tree_top(const uint32_t* __restrict__ parent, uint32_t ninner,
                                                        BvhNode* nodes, uint32_t* arrived, uint32_t* height,
                                                        const Pending* __restrict__ top, const uint32_t* __restrict__ ntop,
                                                        Bvh4Node* __restrict__ nodes4,
                                                        Bvh4HNode* __restrict__ nodes4h, Open* __restrict__ queue,
                                                        uint32_t* __restrict__ cnt) {
    __shared__ Open level[2][4 * kSubtrees];
    __shared__ uint32_t count[2];
    const uint32_t items = *ntop;
    for (uint32_t i = threadIdx.x; i < items; i += kTopBlock) {
        Pending t = top[i];
        if (climb(t, 0u, ninner, parent, nodes, arrived, height)) cnt[BC_DEPTH] = t.height;   // the root: one thread
    }
    if (threadIdx.x == 0) {
        level[0][0] = Open{0u, 0, 1u};   // the binary root becomes four-wide node 0
        count[0] = 1u;
        count[1] = 0u;
    }
    __syncthreads();
    int cur = 0;
    uint32_t n = 1;
    while (n > 0u && n < kSubtrees) {
        const bool live = threadIdx.x < n;
        Open next[4];
        const uint32_t inner = live ? collapse_node(level[cur][live ? threadIdx.x : 0u], nodes, nodes4, nodes4h, next) : 0u;
        uint32_t sum;
        const uint32_t below = wave_prefix4(inner, sum);
        uint32_t base = 0;
        if (__lane_id() == 0 && sum) base = atomicAdd(&count[cur ^ 1], sum);
        base = __shfl(base, 0) + below;
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e)
            if (e < inner) level[cur ^ 1][base + e] = next[e];
        __syncthreads();
        n = count[cur ^ 1];
        __syncthreads();
        if (threadIdx.x == 0) count[cur] = 0u;
        cur ^= 1;
        __syncthreads();
    }
    for (uint32_t i = threadIdx.x; i < n; i += kTopBlock) queue[i] = level[cur][i];
    if (threadIdx.x == 0) cnt[BC_QUEUE] = n;
}

// The subtrees of the nodes in `in`: every wave takes a run of them and works
// through its own stack in LDS, up to 64 nodes at a time from the top.
// Subtrees of one level differ in size by orders of magnitude, so a wave
// stops after `budget` steps (0: none) and leaves what it still has in `out`,
// which the next launch spreads over all waves again (1M triangles, 200
// spheres: 860 us in one launch without a budget).
// The stack: a step takes n nodes and pushes at most 4 n. Above kStackWide
// entries a step takes a single node, so that the walk of the node on top
// adds at most 3 entries per level (64) until it is done: with the 3 x 64 of
// the last wide step never more than kStackSize.
constexpr int kStackWide = 640, kStackSize = kStackWide + 2 * 3 * 64;
constexpr int kCollapseWaves = 2048;
constexpr int kCollapseBudget[kCollapseRounds] = {4, 8, 8, 0};
__global__ __launch_bounds__(64) void k_collapse(const BvhNode* __restrict__ nodes, Bvh4Node* __restrict__ nodes4,
                                                 Bvh4HNode* __restrict__ nodes4h, uint32_t* __restrict__ cnt, int round,
                                                 int budget, const Open* __restrict__ in, Open* __restrict__ out) {
    __shared__ Open stack[kStackSize];
    const uint32_t total = cnt[BC_QUEUE + round];
    const uint32_t per = (total + gridDim.x - 1u) / gridDim.x;
    uint32_t b = min(blockIdx.x * per, total);
    const uint32_t e = min(b + per, total);
    const int lane = __lane_id();
    int sp = 0;
    for (int step = 0; (sp > 0 || b < e) && (budget == 0 || step < budget); ++step) {
        // lanes take nodes from the top of the stack, then from the wave's run
        const int popped = sp > kStackWide ? 1 : min(sp, 64);
        const int fresh = sp > kStackWide ? 0 : (int)min(e - b, (uint32_t)(64 - popped));
        Open t{0u, 0, 0u};
        if (lane < popped) t = stack[sp - 1 - lane];
        else if (lane < popped + fresh) t = in[b + (uint32_t)(lane - popped)];
        __syncthreads();   // one wave: its own order
        Open next[4];
        const uint32_t inner = lane < popped + fresh ? collapse_node(t, nodes, nodes4, nodes4h, next) : 0u;
        sp -= popped;
        b += (uint32_t)fresh;
        uint32_t sum;
        const uint32_t below = wave_prefix4(inner, sum);
#pragma unroll
        for (uint32_t q = 0; q < 4u; ++q)
            if (q < inner) stack[sp + (int)(below + q)] = next[q];
        sp += (int)sum;
        __syncthreads();
    }
    if (sp == 0 && b >= e) return;
    uint32_t o = 0;
    if (lane == 0) o = atomicAdd(cnt + BC_QUEUE + round + 1, (uint32_t)sp + (e - b));
    o = __shfl(o, 0);
    for (int i = lane; i < sp; i += 64) out[o + (uint32_t)i] = stack[i];
    o += (uint32_t)sp;
    for (uint32_t i = b + (uint32_t)lane; i < e; i += 64u) out[o + (i - b)] = in[i];
}

inline size_t align_up(size_t x) { return (x + 255) & ~(size_t)255; }

}  // namespace

// p[i * stride + a] -= delta[a] for npoints points (stride 3: packed float3;
// stride 0: the 9 corner floats of 68-byte emissive records, 3 points each)
__global__ __launch_bounds__(kBuildBlock) void k_translate(float* __restrict__ p, size_t npoints, uint32_t stride,
                                                           float dx, float dy, float dz) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= npoints) return;
    float* q = stride ? p + i * stride : p + (i / 3) * 17 + (i % 3) * 3;
    q[0] -= dx;
    q[1] -= dy;
    q[2] -= dz;
}

// Scratch layout of a build over n triangles (kept after the build: the
// sorted keys and the parent links are what a refit reuses).
struct BuildLayout {
    size_t groups, oBounds, oKeys, oKeys2, oParent, oArrived, oHeight, oPending, oTop, oQueue0, oQueue1, oCounts,
        oSort, total;
};

hipError_t build_layout(rbh_ctx c, int n, BuildLayout& L) {
    const size_t nInt = n > 1 ? (size_t)n - 1 : 1;
    L.groups = ((size_t)n + kGroupLeaves - 1) / kGroupLeaves;
    const size_t tiles = ((size_t)n + kLeafTile - 1) / kLeafTile;
    size_t off = 0;
    L.oBounds = off; off = align_up(off + 64);
    L.oKeys = off; off = align_up(off + (size_t)n * 8);
    L.oKeys2 = off; off = align_up(off + (size_t)n * 8);
    L.oParent = off; off = align_up(off + ((size_t)n + nInt) * 4);
    L.oArrived = off; off = align_up(off + nInt * 4);
    L.oHeight = off; off = align_up(off + nInt * 8);
    L.oPending = off; off = align_up(off + tiles * kHandedOn * sizeof(Pending));
    L.oTop = off; off = align_up(off + L.groups * kHandedOn * sizeof(Pending));
    // nodes still to write: disjoint subtrees of at least two triangles
    L.oQueue0 = off; off = align_up(off + ((size_t)n / 2 + 1) * sizeof(Open));
    L.oQueue1 = off; off = align_up(off + ((size_t)n / 2 + 1) * sizeof(Open));
    L.oCounts = off; off = align_up(off + (BC_COUNT + L.groups) * 4);
    L.oSort = off; off = align_up(off + radix::sort_scratch_bytes(n, 8, 0));
    L.total = off;
    return hipSuccess;
}

// The build's last stages, which a refit repeats over the kept topology:
// triangle records and boxes from the current vertices, the two-child nodes
// and the four-wide collapse.
int build_boxes_and_nodes(rbh_ctx c, const BuildLayout& L) {
    Geometry& g = c->geom;
    Accel& acc = c->accel;
    const int n = (int)g.ntris;
    char* s = acc.scratch.as<char>();
    auto* keys2 = reinterpret_cast<unsigned long long*>(s + L.oKeys2);
    auto* parent = reinterpret_cast<uint32_t*>(s + L.oParent);
    auto* arrived = reinterpret_cast<uint32_t*>(s + L.oArrived);
    auto* height = reinterpret_cast<uint32_t*>(s + L.oHeight);
    auto* pending = reinterpret_cast<Pending*>(s + L.oPending);
    auto* top = reinterpret_cast<Pending*>(s + L.oTop);
    Open* queue[2] = {reinterpret_cast<Open*>(s + L.oQueue0), reinterpret_cast<Open*>(s + L.oQueue1)};
    auto* cnt = reinterpret_cast<uint32_t*>(s + L.oCounts);
    BvhNode* nodes = acc.nodes.as<BvhNode>();
    Bvh4Node* nodes4 = acc.nodes4.as<Bvh4Node>();
    Bvh4HNode* nodes4h = acc.nodes4h.as<Bvh4HNode>();
    const uint32_t ncnt = (uint32_t)(BC_COUNT + L.groups), ninner = (uint32_t)(n - 1);
    hipLaunchKernelGGL(k_build_counters, dim3((ncnt + kBuildBlock - 1) / kBuildBlock), dim3(kBuildBlock), 0, c->stream, cnt,
                       ncnt);
    hipLaunchKernelGGL(k_leaves, dim3((n + kLeafTile - 1) / kLeafTile), dim3(kLeafBlock), 0, c->stream, g.verts.as<float>(),
                       g.indices.as<uint32_t>(), g.triMaterial.as<uint32_t>(), g.triLight.as<uint32_t>(),
                       c->materials.as<Material>(), c->nmaterials, keys2, n, acc.keyIndexBits, parent,
                       acc.tris.as<TriRecord>(), nodes, arrived, height, pending, cnt);
    if (n > 1) {
        // a single group's list is the top list
        const bool one = L.groups == 1;
        if (!one)
            hipLaunchKernelGGL(k_tree_groups, dim3((unsigned)L.groups), dim3(kTopBlock), 0, c->stream, parent, ninner, nodes,
                               arrived, height, pending, top, cnt);
        hipLaunchKernelGGL(k_tree_top, dim3(1), dim3(kTopBlock), 0, c->stream, parent, ninner, nodes, arrived, height,
                           one ? pending : top, cnt + (one ? (int)BC_COUNT : (int)BC_TOP), nodes4, nodes4h, queue[0], cnt);
        for (int r = 0; r < kCollapseRounds; ++r)
            hipLaunchKernelGGL(k_collapse, dim3(kCollapseWaves), dim3(64), 0, c->stream, nodes, nodes4, nodes4h, cnt, r,
                               kCollapseBudget[r], queue[r & 1], queue[(r & 1) ^ 1]);
    }
    RBH_HIP(c, hipGetLastError());
    return RBH_OK;
}

// Synchronises, times the stages since ev0 and reads the depth.
int finish_build(rbh_ctx c, const BuildLayout& L, float* ms, uint32_t* depth) {
    Accel& acc = c->accel;
    const int n = (int)c->geom.ntris;
    char* s = acc.scratch.as<char>();
    RBH_HIP(c, hipEventRecord(c->ev1, c->stream));
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    RBH_HIP(c, hipEventElapsedTime(ms, c->ev0, c->ev1));
    uint32_t cnt[BC_COUNT] = {};
    if (n > 1) RBH_HIP(c, hipMemcpy(cnt, s + L.oCounts, sizeof(cnt), hipMemcpyDeviceToHost));
    if (cnt[BC_QUEUE + kCollapseRounds] != 0u)
        return fail(c, RBH_ERR_RANGE, "four-wide collapse left %u subtrees unwritten", cnt[BC_QUEUE + kCollapseRounds]);
    acc.nnodes4 = n > 1 ? max_nodes4((uint32_t)n) : 0u;   // indices in use are below, with gaps
    *depth = cnt[BC_DEPTH];
    return RBH_OK;
}

int lbvh_build(rbh_ctx c) {
    Geometry& g = c->geom;
    Accel& acc = c->accel;
    const int n = (int)g.ntris;
    if (n <= 0) return fail(c, RBH_ERR_STATE, "no geometry uploaded");
    const size_t nInt = n > 1 ? (size_t)n - 1 : 1;
    BuildLayout L;
    RBH_HIP(c, build_layout(c, n, L));
    acc.built = false;
    RBH_ALLOC(c, acc.scratch, L.total);
    RBH_ALLOC(c, acc.nodes, nInt * sizeof(BvhNode));
    RBH_ALLOC(c, acc.tris, (size_t)n * sizeof(TriRecord));
    const size_t n4 = std::max<size_t>(1, max_nodes4((uint32_t)n));
    RBH_ALLOC(c, acc.nodes4, n4 * sizeof(Bvh4Node));
    RBH_ALLOC(c, acc.nodes4h, n4 * sizeof(Bvh4HNode));
    char* s = acc.scratch.as<char>();
    acc.keysOffset = L.oKeys2;
    uint32_t* bounds = reinterpret_cast<uint32_t*>(s + L.oBounds);
    auto* keys = reinterpret_cast<unsigned long long*>(s + L.oKeys);
    auto* keys2 = reinterpret_cast<unsigned long long*>(s + L.oKeys2);

    const float* v = g.verts.as<float>();
    const uint32_t* idx = g.indices.as<uint32_t>();
    const int nb = (n + kBuildBlock - 1) / kBuildBlock;
    RBH_HIP(c, hipEventRecord(c->ev0, c->stream));
    hipLaunchKernelGGL(k_bounds_init, dim3(1), dim3(64), 0, c->stream, bounds);
    hipLaunchKernelGGL(k_centroid_bounds, dim3(std::min(nb, kBoundsBlocks)), dim3(kBuildBlock), 0, c->stream, v, idx,
                       (uint32_t)n, bounds);
    // key bits: the triangle index below, the Morton code above
    int idxBits = 1;
    while (idxBits < 32 && ((uint64_t)1 << idxBits) < (uint64_t)n) ++idxBits;
    const int axisBits = std::min(21, (64 - idxBits) / 3);
    acc.keyIndexBits = idxBits;
    hipLaunchKernelGGL(k_morton, dim3(nb), dim3(kBuildBlock), 0, c->stream, v, idx, (uint32_t)n, bounds, axisBits,
                       idxBits, keys);
    // stable, and the keys start in index order: sorting by the Morton bits sorts the keys
    RBH_HIP(c, (radix::sort<unsigned long long, uint32_t>(s + L.oSort, keys, keys2, nullptr, nullptr, (uint32_t)n, idxBits,
                                                          idxBits + 3 * axisBits, c->stream)));
    if (n > 1)
        hipLaunchKernelGGL(k_karras, dim3(((int)nInt + kBuildBlock - 1) / kBuildBlock), dim3(kBuildBlock), 0, c->stream,
                           keys2, n, reinterpret_cast<uint32_t*>(s + L.oParent));
    const int rc = build_boxes_and_nodes(c, L);
    if (rc) return rc;
    float ms = 0.0f;
    uint32_t depth = 0;
    const int fr = finish_build(c, L, &ms, &depth);
    if (fr) return fr;
    c->stats.bvhMs = ms;
    c->stats.bvhDepth = depth;
    acc.nnodes = n > 1 ? (uint32_t)(n - 1) : 0u;
    acc.depth = depth;
    acc.ntris = (uint32_t)n;
    if (depth > 64) return fail(c, RBH_ERR_RANGE, "LBVH depth %u exceeds the 64-entry traversal stack", depth);
    acc.built = true;
    acc.stale = false;
    return RBH_OK;
}

__global__ __launch_bounds__(kBuildBlock) void k_tri_classes(TriRecord* __restrict__ tris, int n,
                                                             const Material* __restrict__ mats, uint32_t nmats) {
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t m = tris[j].material;
    tris[j].shadeClass = m < nmats ? shade_class(mats[m]) : (uint32_t)SC_SURFACE;
}

// Re-derives the triangle records' shading classes after the materials
// changed (the classes only order the shade kernel's queue).
hipError_t refresh_tri_classes(rbh_ctx c) {
    const Accel& acc = c->accel;
    if (!acc.built || acc.ntris == 0) return hipSuccess;
    const int n = (int)acc.ntris;
    hipLaunchKernelGGL(k_tri_classes, dim3((n + kBuildBlock - 1) / kBuildBlock), dim3(kBuildBlock), 0, c->stream,
                       acc.tris.as<TriRecord>(), n, c->materials.as<Material>(), c->nmaterials);
    return hipGetLastError();
}

hipError_t translate_points(rbh_ctx c, float* p, size_t npoints, uint32_t strideFloats, const float* delta) {
    if (!npoints) return hipSuccess;
    const size_t blocks = (npoints + kBuildBlock - 1) / kBuildBlock;
    hipLaunchKernelGGL(k_translate, dim3((unsigned)blocks), dim3(kBuildBlock), 0, c->stream, p, npoints, strideFloats,
                       delta[0], delta[1], delta[2]);
    return hipGetLastError();
}

// Refit: new vertex positions under the kept topology (the triangles' leaf
// order and the binary hierarchy stay; every box, the
// triangle records and the four-wide nodes are recomputed). The traversal
// stays exact for any positions; its cost grows as the positions drift from
// the ones the hierarchy was built for.
int lbvh_refit(rbh_ctx c) {
    Accel& acc = c->accel;
    const int n = (int)c->geom.ntris;
    if (!acc.built || acc.ntris != (uint32_t)n || n <= 0)
        return fail(c, RBH_ERR_STATE, "refit needs an acceleration structure built over the same triangles");
    BuildLayout L;
    RBH_HIP(c, build_layout(c, n, L));
    if (acc.scratch.bytes < L.total) return fail(c, RBH_ERR_STATE, "build scratch was released");
    RBH_HIP(c, hipEventRecord(c->ev0, c->stream));
    const int rc = build_boxes_and_nodes(c, L);
    if (rc) return rc;
    float ms = 0.0f;
    uint32_t depth = 0;
    const int fr = finish_build(c, L, &ms, &depth);
    if (fr) return fr;
    c->stats.bvhMs = ms;
    acc.stale = false;
    return RBH_OK;
}

}  // namespace rbh
