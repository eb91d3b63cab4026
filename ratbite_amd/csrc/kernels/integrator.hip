// Wavefront spectral path tracer replacing the OptiX megakernel
// __raygen__main (src/kernels/pathtrace.cu:1114-1813). The per-path bodies
// live in device/wavefront.hpp; the kernels here run them over persistent
// grids and compact the queues.
//
// One pass renders S consecutive samples of every pixel at once (S*W*H path
// slots, slot = sample-major pixel index) so that the long tail of a few deep
// paths is paid once per pass rather than once per sample; path state lives in
// structure-of-arrays buffers in HBM. Per bounce:
//   k_trace    closest hit for the queued paths           (pathtrace.cu:1162-1177),
//              sorting them into a hit queue (by shading class) and a miss
//              queue; at the first bounce it generates the camera rays
//              (pathtrace.cu:1114-1160)
//   k_miss     sky emission + MIS for the misses; the path ends
//              (pathtrace.cu:1185-1274, sky branch)
//   k_shade    emission + MIS, surface attributes, light-tree NEE, BxDF,
//              Russian roulette, next origin, depth caps   (pathtrace.cu:1179-1785)
//   k_shadow   any-hit test of the deferred NEE rays; adds the NEE term of
//              the bounce when the light is visible        (pathtrace.cu:1704-1720)
// and after the last bounce k_accumulate adds each sample's XYZ to the FP64
// accumulation buffer (pathtrace.cu:1789-1812). Queues are compacted with
// wave ballots; the trace and shade kernels stage finished paths in per-wave
// LDS lists and write them 64 or more at a time (one atomic per run). Queue lengths stay on the device; every
// kernel reads its count and exits early, so the host issues a fixed launch
// sequence per pass.
#include "../context.hpp"
#include "../device/mlp_wave.hpp"
#include "../device/traverse.hpp"
#include "../device/traverse_quad.hpp"
#include "../device/wavefront.hpp"
#include "../integrator.hpp"

namespace rbh {

using namespace dev;
using namespace wf;

namespace {

// Traversal stack entries of the any-hit walk kept in LDS per lane
constexpr int kStackLds = 16;

__device__ __forceinline__ uint32_t wave_push(uint32_t* __restrict__ counter, bool pred) {
    // one atomic per wave: ballot, leader adds the popcount, lanes take
    // consecutive slots by their rank among the active lanes
    const unsigned long long mask = __ballot(pred);
    const uint32_t n = (uint32_t)__popcll(mask);
    if (n == 0) return 0xFFFFFFFFu;
    const int lane = __lane_id();
    const int leader = __ffsll((long long)mask) - 1;
    uint32_t base = 0;
    if (lane == leader) base = atomicAdd(counter, n);
    base = __shfl(base, leader);
    const uint32_t rank = (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
    return pred ? base + rank : 0xFFFFFFFFu;
}

__device__ __forceinline__ void wave_count(unsigned long long* __restrict__ counter, uint32_t v) {
    // sum v over the wave with one atomic
    uint32_t s = v;
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (__lane_id() == 0 && s) atomicAdd(counter, (unsigned long long)s);
}

// The queue counters at the start of a pass: every bounce has its own block
// of CNT_COUNT counters, all cleared here (n of them), and every slot traces
// its camera ray (the first closest-hit pass generates it). Clearing one block
// between bounces instead took two one-wave launches a bounce, 5 us each
// (256x256, 16 samples, depth 8: 4.16 -> 3.79 ms; eight scenes in a batch:
// 66.7 -> 63.8 ms).
__global__ __launch_bounds__(256) void k_pass_start(Frame1 f, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) f.counters[i] = i == CNT_QUEUE0 ? f.NP : 0u;
}

// The ray a closest-hit pass traces for path slot pid: at the first bounce
// the camera ray, generated here and stored for the shading kernels (with a
// fresh training-record chain when collecting), afterwards the stored ray.
template <bool BATCH>
__device__ __forceinline__ void pass_ray(const Frame1& f, const SceneView& S, uint32_t pid, bool first, V3& o, V3& d) {
    if (first) {
        camera_ray(S, pid, o, d);
        f.p.od[pid] = make_float4(o.x, o.y, o.z, 1.0f);   // bxdfPdf = 1
        f.p.dr[pid] = make_float4(d.x, d.y, d.z, 1.0f);   // refractionScale = 1
        if (f.collect) f.p.prec[pid] = kNoRec;
    } else {
        const float4 od = f.p.od[pid], dr = f.p.dr[pid];
        o = V3{od.x, od.y, od.z};
        d = V3{dr.x, dr.y, dr.z};
    }
}

// Hit-queue entries in shading order: the segments of the shading classes
// one after the other (class c's entries at hq[c * NP ...]).
struct HitQueue {
    uint32_t start[kShadeClasses + 1];   // first shading-order index of each class, then the total
    __device__ __forceinline__ explicit HitQueue(const Frame1& f) {
        start[0] = 0u;
#pragma unroll
        for (uint32_t c = 0; c < kShadeClasses; ++c) start[c + 1] = start[c] + f.counters[hit_counter(c)];
    }
    __device__ __forceinline__ uint32_t count() const { return start[kShadeClasses]; }
    __device__ __forceinline__ uint32_t entry(const Frame1& f, uint32_t i) const {
        uint32_t c = 0;
#pragma unroll
        for (uint32_t k = 1; k < kShadeClasses; ++k) c += i >= start[k] ? 1u : 0u;
        return f.p.hq[(size_t)c * f.NP + (i - start[c])];
    }
};

// Work fetch of the persistent trace and shadow kernels. A wave claims
// chunks of kChunk consecutive queue entries with one atomic on *head and
// hands them to its idle lanes whenever at least kRefill lanes are idle (or
// all of them), so a lane takes a new ray as soon as its query completes
// while the wave's rays stay a contiguous, coherent stretch of the queue.
constexpr int kRefill = 16;
constexpr uint32_t kChunk = 256;
struct WaveChunk {
    uint32_t next = 0, end = 0;   // wave-uniform: unclaimed entries [next, end) of the wave's chunk
    bool drained = false;         // the queue has no further chunk
    // Returns this lane's new entry or ~0. Every lane of the wave calls it.
    __device__ __forceinline__ uint32_t fetch(uint32_t* __restrict__ head, uint32_t count, bool idle, bool anyBusy) {
        const unsigned long long mask = __ballot(idle);
        const uint32_t n = (uint32_t)__popcll(mask);
        if (n == 0 || (anyBusy && n < (uint32_t)kRefill)) return 0xFFFFFFFFu;
        if (next >= end && !drained) {
            const int lane = __lane_id();
            const int leader = __ffsll((long long)mask) - 1;
            uint32_t base = 0;
            if (lane == leader) base = atomicAdd(head, kChunk);
            base = __shfl(base, leader);
            if (base >= count) {
                drained = true;
            } else {
                next = base;
                end = min(base + kChunk, count);
            }
        }
        if (next >= end) return 0xFFFFFFFFu;
        const uint32_t idx = next + (uint32_t)__popcll(mask & ((1ull << __lane_id()) - 1ull));
        next = min(next + n, end);
        return idle && idx < end ? idx : 0xFFFFFFFFu;
    }
    // no lane active, nothing left to hand out
    __device__ __forceinline__ bool done(bool anyActive) const { return !anyActive && drained && next >= end; }
};

// ------------------------------------------------------------- closest hit
__device__ __forceinline__ TravStack<kStackLds> lane_stack(const Frame1& f, int* lds) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    return TravStack<kStackLds>{lds + threadIdx.x, (int)blockDim.x, f.spill + t, f.spillStride};
}
__device__ __forceinline__ DistStack<kDistLds> lane_stack(const Frame1& f, int* lds, uint16_t* dist) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    return DistStack<kDistLds>{lds + threadIdx.x, dist + threadIdx.x, (int)blockDim.x, f.spill + t, f.spillStride};
}

// Wave-private staging of queue pushes: finished rays are appended to an
// LDS list of the wave and written out 64 or more at a time with one atomic,
// instead of one atomic per wave for every traversal step in which some lane
// finished.
struct WaveList {
    uint32_t* buf;   // 128 entries of this wave
    uint32_t n;      // entries held (wave-uniform)
    __device__ __forceinline__ void add(bool pred, uint32_t v) {
        const unsigned long long mask = __ballot(pred);
        const uint32_t rank = (uint32_t)__popcll(mask & ((1ull << __lane_id()) - 1ull));
        if (pred) buf[n + rank] = v;
        n += (uint32_t)__popcll(mask);
    }
    // writes the held entries to queue[*counter ...] when at least `min` are held
    __device__ __forceinline__ void flush(uint32_t* __restrict__ counter, uint32_t* __restrict__ queue, uint32_t min) {
        if (n == 0 || n < min) return;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // the lanes' LDS writes are visible
        const int lane = __lane_id();
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(counter, n);
        base = __shfl(base, 0);
        for (uint32_t k = (uint32_t)lane; k < n; k += 64u) queue[base + k] = buf[k];
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");   // reads done before the list is refilled
        n = 0;
    }
};

// The same staging for the hit queue, with each entry's shading class: a
// flush writes every class present in the list as one run of that class's
// queue segment, with one atomic on the class's counter.
struct ClassList {
    uint32_t* buf;   // 128 path slots of this wave
    uint8_t* cls;    // their shading classes
    uint32_t n;      // entries held (wave-uniform)
    __device__ __forceinline__ void add(bool pred, uint32_t v, uint32_t c) {
        const unsigned long long mask = __ballot(pred);
        const uint32_t rank = (uint32_t)__popcll(mask & ((1ull << __lane_id()) - 1ull));
        if (pred) {
            buf[n + rank] = v;
            cls[n + rank] = (uint8_t)c;
        }
        n += (uint32_t)__popcll(mask);
    }
    // at most 127 entries are held (64 added at a time, flushed from 64 on)
    __device__ __forceinline__ void flush(const Frame1& f, uint32_t min) {
        if (n == 0 || n < min) return;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const uint32_t lane = (uint32_t)__lane_id();
        const bool v0 = lane < n, v1 = lane + 64u < n;
        const uint32_t p0 = v0 ? buf[lane] : 0u, p1 = v1 ? buf[lane + 64u] : 0u;
        const uint32_t c0 = v0 ? cls[lane] : (uint32_t)kShadeClasses, c1 = v1 ? cls[lane + 64u] : (uint32_t)kShadeClasses;
        const unsigned long long lt = (1ull << lane) - 1ull;
        for (uint32_t c = 0; c < kShadeClasses; ++c) {
            const unsigned long long m0 = __ballot(c0 == c), m1 = __ballot(c1 == c);
            const uint32_t k0 = (uint32_t)__popcll(m0), k = k0 + (uint32_t)__popcll(m1);
            if (k == 0u) continue;
            uint32_t base = 0;
            if (lane == 0u) base = atomicAdd(f.counters + hit_counter(c), k);
            base = __shfl(base, 0);
            uint32_t* __restrict__ q = f.p.hq + (size_t)c * f.NP + base;
            if (c0 == c) q[__popcll(m0 & lt)] = p0;
            if (c1 == c) q[k0 + (uint32_t)__popcll(m1 & lt)] = p1;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        n = 0;
    }
};

// The four-wide nodes a kernel traverses: full boxes or on an 11-bit grid
template <bool QN>
__device__ __forceinline__ auto scene_nodes(const SceneView& S) {
    if constexpr (QN) return S.nodes4h;
    else return S.nodes4;
}

// WAVES: minimum resident waves per SIMD the register allocation must allow
// (1 = unconstrained), traded by the launch shape against spills; QN: the
// nodes on an 11-bit grid
// CAM0: the first bounce of a pass without depth of field, whose camera
// rays all start at the camera position, the origin of the camera-relative
// scene: the origin is the constant 0 there, which removes the origin
// subtractions of every box and triangle test (x - 0 is x exactly, so the
// walk is the same).
template <bool BATCH, bool FETCH, int WAVES, bool QN, bool CAM0>
__global__ __launch_bounds__(kTraceBlock, WAVES) void k_trace(Frame1 f, uint32_t qsel) {
    __shared__ int stack[kDistLds * kTraceBlock];
    __shared__ uint16_t dist[kDistLds * kTraceBlock];
    __shared__ uint32_t staged[2 * kTraceBlock * 2];   // per wave: 128 hits, 128 misses
    __shared__ uint8_t stagedCls[2 * kTraceBlock];     // per wave: the hits' shading classes
    const DistStack<kDistLds> st = lane_stack(f, stack, dist);
    const uint32_t count = f.counters[qsel ? CNT_QUEUE1 : CNT_QUEUE0];
    if (f.bounce > 0u && count <= f.tail) return;   // k_paths ran these paths to their end
    const uint32_t* __restrict__ queue = qsel ? f.p.q1 : f.p.q0;
    const bool identity = f.bounce == 0;
    uint32_t nrays = 0;
    // finished rays are staged per wave and queued 64 or more at a time;
    // hits in their shading class's segment when sorting by material
    const uint32_t wave = threadIdx.x >> 6;
    ClassList hits{staged + wave * 256u, stagedCls + wave * 128u, 0u};
    WaveList misses{staged + wave * 256u + 128u, 0u};
    if (FETCH) {
        // lanes take a new ray as soon as theirs completes
        TravRay ray;
        const Bvh4Node* nodes = nullptr;
        const TriRecord* tris = nullptr;
        uint32_t pid = 0;
        bool active = false;
        WaveChunk chunk;
        while (true) {
            const bool anyBusy = __ballot(active) != 0ull;
            const uint32_t idx = chunk.fetch(f.counters + CNT_TRACE_HEAD, count, !active, anyBusy);
            if (idx != 0xFFFFFFFFu) {
                pid = identity ? idx : queue[idx];
                const SceneView& S = scene_of<BATCH>(f, pid);
                nodes = S.nodes4;
                tris = S.tris;
                V3 o, d;
                pass_ray<BATCH>(f, S, pid, identity, o, d);
                if constexpr (CAM0) o = V3{0.0f, 0.0f, 0.0f};
                trav_init(ray, o, d, 3.402823466e+38f, S.nnodes4);
                // the nearest shape light bounds the walk; a nearer triangle replaces it
                if (S.nshapes) shape_closest(S.shapes, S.nshapes, ray.o, ray.d, 3.402823466e+38f, ray.h.t, ray.h.leaf);
                active = true;
                ++nrays;
            }
            if (chunk.done(__ballot(active) != 0ull)) break;
            bool done = false;
            if (active) done = trav_step<false>(nodes, tris, ray, st);
            const bool hit = done && ray.h.leaf != 0xFFFFFFFFu;
            uint32_t cls = 0;
            if (hit) {
                f.p.hit[pid] = make_float4(ray.h.t, ray.h.b1, ray.h.b2, __uint_as_float(ray.h.leaf));
                if (f.sortHits) cls = (ray.h.leaf & kShapeHit) ? (uint32_t)SC_SHAPE : tris[ray.h.leaf].shadeClass;
            }
            hits.add(hit, pid, cls);
            misses.add(done && !hit, pid);
            hits.flush(f, 64u);
            misses.flush(f.counters + CNT_MISS, f.p.mq, 64u);
            if (done) active = false;
        }
    } else {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i - threadIdx.x < count; i += gridDim.x * blockDim.x) {
            bool hit = false;
            uint32_t cls = 0;
            uint32_t pid = 0;
            if (i < count) {
                pid = identity ? i : queue[i];
                const SceneView& S = scene_of<BATCH>(f, pid);
                V3 o, d;
                pass_ray<BATCH>(f, S, pid, identity, o, d);
                if constexpr (CAM0) o = V3{0.0f, 0.0f, 0.0f};
                // the nearest shape light bounds the walk; a nearer triangle replaces it
                float ts = 3.402823466e+38f;
                uint32_t shape = 0xFFFFFFFFu;
                if (S.nshapes) shape_closest(S.shapes, S.nshapes, o, d, ts, ts, shape);
                Hit h = traverse4<false>(scene_nodes<QN>(S), S.tris, S.nnodes4, o, d, ts, st);
                if (h.leaf == 0xFFFFFFFFu && shape != 0xFFFFFFFFu) h = Hit{ts, 0.0f, 0.0f, shape};
                hit = h.leaf != 0xFFFFFFFFu;
                if (hit) {
                    f.p.hit[pid] = make_float4(h.t, h.b1, h.b2, __uint_as_float(h.leaf));
                    // material-sorted shading: the hit joins its shading class's segment
                    if (f.sortHits) cls = (h.leaf & kShapeHit) ? (uint32_t)SC_SHAPE : S.tris[h.leaf].shadeClass;
                }
                ++nrays;
            }
            const bool live = i < count;
            hits.add(live && hit, pid, cls);
            misses.add(live && !hit, pid);
            hits.flush(f, 64u);
            misses.flush(f.counters + CNT_MISS, f.p.mq, 64u);
        }
    }
    hits.flush(f, 1u);
    misses.flush(f.counters + CNT_MISS, f.p.mq, 1u);
    wave_count(f.stats + STAT_CLOSEST, nrays);
}

// Network input of every queued hit, one thread per hit (the gathers run
// fully parallel), kept for the training records of the vertex.
__global__ __launch_bounds__(256) void k_guide_features(Frame1 f) {
    const HitQueue hq(f);
    const uint32_t count = hq.count();
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x)
        guide_input(f, f.sc, hq.entry(f, i), f.gfeat + (size_t)i * guide::kRec);
}

// Mixture of every queued hit: wave-resident MLP inference over the
// feature records (BF16 or FP8 E4M3 weights).
template <bool FP8>
__global__ __launch_bounds__(256, 2) void k_guide_mlp(Frame1 f) {
    __shared__ mlp::WaveLds L[4];
    mlp::wave_infer<FP8, true>(L[threadIdx.x >> 6], f.gfeat, HitQueue(f).count(), f.gwf, f.gwq, f.gws, f.gbias, f.gmix);
}

template <bool BATCH>
__global__ __launch_bounds__(256) void k_miss(Frame1 f) {
    const uint32_t count = f.counters[CNT_MISS];
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < count; i += gridDim.x * blockDim.x) {
        const uint32_t pid = f.p.mq[i];
        shade_miss(f, scene_of<BATCH>(f, pid), pid);
    }
}

template <bool BATCH, bool FETCH, int WAVES, bool QN>
__global__ __launch_bounds__(kTraceBlock, WAVES) void k_shadow(Frame1 f) {
    __shared__ int stack[kStackLds * kTraceBlock];
    const TravStack<kStackLds> st = lane_stack(f, stack);
    const uint32_t count = f.counters[CNT_SHADOW];
    uint32_t nrays = 0;
    if (FETCH) {
        TravRay ray;
        const Bvh4Node* nodes = nullptr;
        const TriRecord* tris = nullptr;
        uint32_t pid = 0;
        bool active = false;
        WaveChunk chunk;
        while (true) {
            const bool anyBusy = __ballot(active) != 0ull;
            const uint32_t idx = chunk.fetch(f.counters + CNT_SHADOW_HEAD, count, !active, anyBusy);
            if (idx != 0xFFFFFFFFu) {
                pid = f.p.sq[idx];
                const SceneView& S = scene_of<BATCH>(f, pid);
                nodes = S.nodes4;
                tris = S.tris;
                const float4 so = f.p.sro[pid], sd = f.p.srd[pid];
                const V3 o{so.x, so.y, so.z}, d{sd.x, sd.y, sd.z};
                // a shape light in the way settles the ray without a walk
                if (!(S.nshapes && shape_any(S.shapes, S.nshapes, o, d, so.w))) {
                    trav_init(ray, o, d, so.w, S.nnodes4);
                    active = true;
                }
                ++nrays;
            }
            if (chunk.done(__ballot(active) != 0ull)) break;
            if (active && trav_step<true>(nodes, tris, ray, st)) {
                if (ray.h.leaf == 0xFFFFFFFFu) add_nee(f, pid);
                active = false;
            }
        }
    } else {
        for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i - threadIdx.x < count; i += gridDim.x * blockDim.x) {
            if (i < count) {
                const uint32_t pid = f.p.sq[i];
                const SceneView& S = scene_of<BATCH>(f, pid);
                const float4 so = f.p.sro[pid], sd = f.p.srd[pid];
                const V3 o{so.x, so.y, so.z}, d{sd.x, sd.y, sd.z};
                if (!(S.nshapes && shape_any(S.shapes, S.nshapes, o, d, so.w))) {
                    const Hit h = traverse4<true>(scene_nodes<QN>(S), S.tris, S.nnodes4, o, d, so.w, st);
                    if (h.leaf == 0xFFFFFFFFu) add_nee(f, pid);
                }
                ++nrays;
            }
        }
    }
    wave_count(f.stats + STAT_SHADOW, nrays);
}

// WAVES: minimum resident waves per SIMD the register allocation must allow
// (1 = unconstrained); the autotuner picks between fewer spills and more
// latency hiding.
template <bool GUIDED, bool BATCH, int WAVES>
__global__ __launch_bounds__(kShadeBlock, WAVES) void k_shade(Frame1 f, uint32_t qsel) {
    // shades the paths whose ray hit a surface or a shape light (misses were finished by k_trace)
    const HitQueue hq(f);
    const uint32_t count = hq.count();
    uint32_t* __restrict__ qout = qsel ? f.p.q0 : f.p.q1;
    uint32_t* __restrict__ cout = f.counters + CNT_COUNT + (qsel ? CNT_QUEUE0 : CNT_QUEUE1);   // the next bounce's block
    uint32_t nvert = 0;
    // continuing paths and shadow rays are staged per wave and queued 64 or more at a time
    __shared__ uint32_t staged[2 * kShadeBlock * 2];
    const uint32_t wave = threadIdx.x >> 6;
    WaveList next{staged + wave * 256u, 0u}, shadows{staged + wave * 256u + 128u, 0u};
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i - threadIdx.x < count; i += gridDim.x * blockDim.x) {
        bool alive = false, shadow = false;
        bool recordSlot = false;      // guided + collecting: record this vertex's direction
        V3 recDir{0.0f, 0.0f, 0.0f};
        float recPb = 0.0f;           // BSDF sampler's density of the recorded direction
        S4 recT = s4(0.0f);           // throughput before the recorded vertex
        uint32_t pid = 0;
        if (i < count) {
            pid = hq.entry(f, i);
            ++nvert;
            const SceneView& S = scene_of<BATCH>(f, pid);
            shade_hit<GUIDED>(f, S, pid, i, alive, shadow, recordSlot, recDir, recPb, recT);
        }
        next.add(alive, pid);
        shadows.add(shadow, pid);
        next.flush(cout, qout, 64u);
        shadows.flush(f.counters + CNT_SHADOW, f.p.sq, 64u);
        if (GUIDED && f.collect) {
            // a recorded direction needs the path to go on (its radiance is measured later)
            const bool rec = recordSlot && alive;
            const uint32_t r = wave_push(f.grecCount, rec);
            if (rec && r < f.grecCap) {
                float* d = f.grec + (size_t)r * kPendingRec;
                const float* in = f.gfeat + (size_t)i * guide::kRec;
                for (int k = 0; k < 11; ++k) d[k] = in[k];
                d[11] = recDir.x;
                d[12] = recDir.y;
                d[13] = recDir.z;
                d[14] = recPb;
                d[15] = __uint_as_float(f.p.prec[pid]);
                d[16] = recT.v[0]; d[17] = recT.v[1]; d[18] = recT.v[2]; d[19] = recT.v[3];
                f.p.prec[pid] = r | kRecPending;
            }
        }
    }
    next.flush(cout, qout, 1u);
    shadows.flush(f.counters + CNT_SHADOW, f.p.sq, 1u);
    wave_count(f.stats + STAT_VERTICES, nvert);
}

// ------------------------------------------------------ few paths: one kernel
// All remaining bounces of the queued paths in one launch, from closest hit
// to shadow ray, four lanes per path, for queues too short to fill the chip: a
// bounce of the separate kernels then takes as long as the slowest wave of
// each of them (about 200 us however few the paths); here a wave only waits
// for its own 16 paths, and their walks take one box and one triangle per
// lane (traverse_quad.hpp). The four lanes shade their path redundantly, with
// the same values, and only the first one counts. State, per-path bodies, node
// form and walk are those of the separate kernels, so a path's values do not
// depend on which form ran it. Bound by the latency of a path's chain of bounces: one
// sample of a 64x64 Cornell box at depth 8 takes 0.42 ms against 1.27 ms in
// the separate kernels (0.68 ms with one lane per path), 640x360 over 1M
// triangles with a refit 3.9 against 5.3 ms. bounce: the bounce the queue
// belongs to (0: every slot starts with its camera ray).
// kTailPaths: 4096 waves. Measured at 16k / 64k / 128k / 256k paths: 256x256x16 Cornell 3.68 /
// 3.61 / 3.72 / 4.10 ms, feature scene 333x187x8 2.40 / 2.36 / 2.53 / 2.92 ms,
// 1080p x 64 spp of 4.1M triangles 114.3 / 114.1 / 116.3 / 122.3 ms.
constexpr uint32_t kTailPaths = 65536u;
// Waves per SIMD: a tail is up to 4096 waves, two rounds at two waves per SIMD
// (231 registers) and better off with a few spills and three: feature scene
// 333x187x8 2.27 -> 2.17 ms, edit of 1M triangles with a 640x360 preview 2.85 ->
// 2.62 ms (four waves: 2.24 / 2.85 ms). Up to kFewPaths are resident at once
// either way, and the registers shorten their chain: 64x64 preview 0.485 against
// 0.502 ms.
constexpr int kTailWaves = 3;
constexpr uint32_t kFewPaths = 32768u;
template <bool BATCH, int WAVES>
__global__ __launch_bounds__(kPathBlock, WAVES) void k_paths(Frame1 f, uint32_t bounce, uint32_t depthMax) {
    __shared__ uint2 stack[kQuadStackLds * kQuadRays];
    const uint32_t t = (blockIdx.x * kPathBlock + threadIdx.x) >> 2;
    const QuadStack<kQuadStackLds, kDistLds> st{stack + (threadIdx.x >> 2), kQuadRays, f.spill + t, f.spillStride};
    const uint32_t qsel = bounce & 1u;
    const uint32_t count = f.counters[qsel ? CNT_QUEUE1 : CNT_QUEUE0];
    if (count > f.tail) return;   // long enough for the separate kernels
    const uint32_t* __restrict__ queue = qsel ? f.p.q1 : f.p.q0;
    uint32_t nclosest = 0, nshadow = 0, nvert = 0;
    for (uint32_t i = t; i < count; i += gridDim.x * kQuadRays) {
        const uint32_t pid = bounce == 0u ? i : queue[i];
        const SceneView& S = scene_of<BATCH>(f, pid);
        bool alive = true;
        for (uint32_t b = bounce; alive && b < depthMax; ++b) {
            V3 o, d;
            pass_ray<BATCH>(f, S, pid, b == 0u, o, d);
            float ts = 3.402823466e+38f;
            uint32_t shape = 0xFFFFFFFFu;
            if (S.nshapes) shape_closest(S.shapes, S.nshapes, o, d, ts, ts, shape);
            Hit h = f.gridNodes ? traverse4_quad<false>(S.nodes4h, S.tris, S.nnodes4, o, d, ts, st)
                                 : traverse4_quad<false>(S.nodes4, S.tris, S.nnodes4, o, d, ts, st);
            if (h.leaf == 0xFFFFFFFFu && shape != 0xFFFFFFFFu) h = Hit{ts, 0.0f, 0.0f, shape};
            ++nclosest;
            alive = false;
            if (h.leaf == 0xFFFFFFFFu) {
                shade_miss(f, S, pid, b == 0u);
                continue;
            }
            f.p.hit[pid] = make_float4(h.t, h.b1, h.b2, __uint_as_float(h.leaf));
            ++nvert;
            bool shadow = false, rec = false;
            V3 recDir{0.0f, 0.0f, 0.0f};
            float recPb = 0.0f;
            S4 recT = s4(0.0f);
            shade_hit<false>(f, S, pid, i, b == 0u, alive, shadow, rec, recDir, recPb, recT);
            if (shadow) {
                const float4 so = f.p.sro[pid], sd = f.p.srd[pid];
                const V3 so3{so.x, so.y, so.z}, sd3{sd.x, sd.y, sd.z};
                if (!(S.nshapes && shape_any(S.shapes, S.nshapes, so3, sd3, so.w))) {
                    const Hit q = f.gridNodes ? traverse4_quad<true>(S.nodes4h, S.tris, S.nnodes4, so3, sd3, so.w, st)
                                              : traverse4_quad<true>(S.nodes4, S.tris, S.nnodes4, so3, sd3, so.w, st);
                    if (q.leaf == 0xFFFFFFFFu) add_nee(f, pid);
                }
                ++nshadow;
            }
        }
    }
    const bool first = (threadIdx.x & 3u) == 0u;
    wave_count(f.stats + STAT_CLOSEST, first ? nclosest : 0u);
    wave_count(f.stats + STAT_SHADOW, first ? nshadow : 0u);
    wave_count(f.stats + STAT_VERTICES, first ? nvert : 0u);
}

// ----------------------------------------------------------- accumulation
template <bool BATCH>
__global__ __launch_bounds__(256) void k_accumulate(Frame1 f) {
    // per pixel, the S samples of the pass are added one at a time in sample
    // order, so any split of a sample range into passes gives the same sums
    const SceneView& S = BATCH ? f.scenes[blockIdx.y] : f.sc;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;   // scene-local slot of sample 0
    if (i >= S.P) return;
    accumulate_slot(f, S, i);
}

}  // namespace

// Expanded light-tree nodes: the packed nodes decoded once.
__global__ __launch_bounds__(256) void k_expand_tree(const PackedNode* __restrict__ in, TreeNodeX* __restrict__ out,
                                                     uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) out[i] = expand_node(load_node(in, i));
}

// sRGB decode of the 256 8-bit channel values
__global__ void k_srgb_lut(float* __restrict__ out) {
    const uint32_t k = threadIdx.x;
    if (k < 256u) out[k] = srgb_decode((float)k / 255.0f);
}

// ------------------------------------------------------------------ host
hipError_t srgb_lut_fill(rbh_ctx c) {
    hipLaunchKernelGGL(k_srgb_lut, dim3(1), dim3(256), 0, c->stream, c->srgbLut.as<float>());
    return hipGetLastError();
}

hipError_t light_tree_expand(rbh_ctx c) {
    const uint32_t n = c->tree.nnodes;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_expand_tree, dim3((n + 255) / 256), dim3(256), 0, c->stream, c->tree.nodes.as<PackedNode>(),
                       c->tree.nodesX.as<TreeNodeX>(), n);
    return hipGetLastError();
}

// Spill entries per lane of the traversal stack beyond the LDS part.
size_t trace_spill_words(size_t lanes) { return lanes * (size_t)(kMaxStack4 - kDistLds); }

template <bool BATCH, bool FETCH, bool QN>
static void launch_trace_q(rbh_ctx c, const Frame1& f, uint32_t qsel, const LaunchShape& ls) {
    const dim3 g(ls.traceGrid), b(kTraceBlock);
    if (f.bounce == 0u && f.camOrigin0) {
        if (ls.traceWaves >= 8) hipLaunchKernelGGL((k_trace<BATCH, FETCH, 8, QN, true>), g, b, 0, c->stream, f, qsel);
        else if (ls.traceWaves == 7) hipLaunchKernelGGL((k_trace<BATCH, FETCH, 7, QN, true>), g, b, 0, c->stream, f, qsel);
        else hipLaunchKernelGGL((k_trace<BATCH, FETCH, 1, QN, true>), g, b, 0, c->stream, f, qsel);
        return;
    }
    if (ls.traceWaves >= 8) hipLaunchKernelGGL((k_trace<BATCH, FETCH, 8, QN, false>), g, b, 0, c->stream, f, qsel);
    else if (ls.traceWaves == 7) hipLaunchKernelGGL((k_trace<BATCH, FETCH, 7, QN, false>), g, b, 0, c->stream, f, qsel);
    else hipLaunchKernelGGL((k_trace<BATCH, FETCH, 1, QN, false>), g, b, 0, c->stream, f, qsel);
}

// The work-fetch variants read the nodes with full boxes, which are indexed
// up to 4 GiB; larger trees run the nodes on the grid. All kernels of a pass
// read the same form.
static bool work_fetch(const LaunchShape& ls) { return ls.traceFetch && !ls.quantOnly; }
static bool grid_nodes(const LaunchShape& ls) { return ls.quantOnly || (ls.quantNodes && !ls.traceFetch); }

template <bool BATCH>
static void launch_trace(rbh_ctx c, const Frame1& f, uint32_t qsel, const LaunchShape& ls) {
    if (work_fetch(ls)) launch_trace_q<BATCH, true, false>(c, f, qsel, ls);
    else if (grid_nodes(ls)) launch_trace_q<BATCH, false, true>(c, f, qsel, ls);
    else launch_trace_q<BATCH, false, false>(c, f, qsel, ls);
}

template <bool BATCH, bool FETCH, bool QN>
static void launch_shadow_q(rbh_ctx c, const Frame1& f, const LaunchShape& ls) {
    const dim3 g(ls.traceGrid), b(kTraceBlock);
    if (ls.traceWaves >= 8) hipLaunchKernelGGL((k_shadow<BATCH, FETCH, 8, QN>), g, b, 0, c->stream, f);
    else if (ls.traceWaves == 7) hipLaunchKernelGGL((k_shadow<BATCH, FETCH, 7, QN>), g, b, 0, c->stream, f);
    else hipLaunchKernelGGL((k_shadow<BATCH, FETCH, 1, QN>), g, b, 0, c->stream, f);
}

template <bool BATCH>
static void launch_shadow(rbh_ctx c, const Frame1& f, const LaunchShape& ls) {
    if (work_fetch(ls)) launch_shadow_q<BATCH, true, false>(c, f, ls);
    else if (grid_nodes(ls)) launch_shadow_q<BATCH, false, true>(c, f, ls);
    else launch_shadow_q<BATCH, false, false>(c, f, ls);
}

// One wavefront pass: camera rays for every slot, depthMax bounces of
// trace / miss / (guide) / shade / shadow, then accumulation. f.sc (single
// scene) or f.scenes (batched) must describe the pass's samples and slots.
template <bool BATCH>
static hipError_t launch_pass_t(rbh_ctx c, Frame1 f, uint32_t depthMax, const LaunchShape& ls, KernelTimer* kt) {
    // guiding: feature gather over all hit slots, then resident blocks of four
    // MLP waves, as many per CU as the register budget allows (weights and
    // the prefetched next records in registers: 2 waves per SIMD)
    const int nbGuide = (int)std::min<uint32_t>((f.NP + 255) / 256, 65535u * 16u);
    int cus = 256;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess || cus <= 0) cus = 256;
    const int mlpGrid = 2 * cus;
    const dim3 accGrid((f.maxP + 255) / 256, BATCH ? f.nscenes : 1u);
    hipError_t e = hipSuccess;
#define RBH_TIMED(cls, launch)                                       \
    do {                                                             \
        if (kt && (e = kt->begin(c->stream, cls)) != hipSuccess) return e; \
        launch;                                                      \
        if (kt && (e = kt->end(c->stream)) != hipSuccess) return e;  \
    } while (0)
    f.bounce = 0;
    f.sortHits = ls.sortHits ? 1u : 0u;
    f.gridNodes = grid_nodes(ls) ? 1u : 0u;
    uint32_t* const counters = f.counters;
    const uint32_t ncount = (depthMax + 1u) * CNT_COUNT;
    hipLaunchKernelGGL(k_pass_start, dim3((ncount + 255u) / 256u), dim3(256), 0, c->stream, f, ncount);
    // k_paths: launched before each later bounce of an unguided pass, it leaves
    // at once unless the queue has become short; a pass short from the start
    // is that one launch. Per-kernel timing keeps the kernels apart, and so
    // does the tuning of their shapes.
    f.tail = f.guided || kt || !ls.tail ? 0u : kTailPaths;
    // (no more lanes than the trace grid's spill columns)
    const dim3 pathGrid(std::min<uint32_t>((std::min(std::max(f.tail, 1u), f.NP) + kQuadRays - 1) / kQuadRays,
                                           (uint32_t)ls.traceGrid * kTraceBlock / kQuadRays));
    const bool allPaths = f.NP <= f.tail;
    const auto paths = [&](uint32_t b) {
        const bool few = b == 0u && f.NP <= kFewPaths;
        auto k = few ? k_paths<BATCH, 2> : k_paths<BATCH, kTailWaves>;
        hipLaunchKernelGGL(k, pathGrid, dim3(kPathBlock), 0, c->stream, f, b, depthMax);
    };
    if (allPaths) paths(0u);
    for (uint32_t b = 0; b < depthMax && !allPaths; ++b) {
        const uint32_t qsel = b & 1u;
        f.bounce = b;
        f.counters = counters + b * CNT_COUNT;
        if (f.tail && b > 0) paths(b);
        RBH_TIMED(KernelTimer::TRACE, launch_trace<BATCH>(c, f, qsel, ls));
        RBH_TIMED(KernelTimer::SHADE,
                  hipLaunchKernelGGL(k_miss<BATCH>, dim3(ls.shadeGrid), dim3(256), 0, c->stream, f));
        if (!BATCH && f.guided) {
            RBH_TIMED(KernelTimer::GUIDE,
                      hipLaunchKernelGGL(k_guide_features, dim3(nbGuide), dim3(256), 0, c->stream, f));
            RBH_TIMED(KernelTimer::GUIDE,
                      if (f.gwq) hipLaunchKernelGGL((k_guide_mlp<true>), dim3(mlpGrid), dim3(256), 0, c->stream, f);
                      else hipLaunchKernelGGL((k_guide_mlp<false>), dim3(mlpGrid), dim3(256), 0, c->stream, f));
        }
        if (!BATCH && f.guided && ls.shadeWaves >= 3)
            RBH_TIMED(KernelTimer::SHADE, hipLaunchKernelGGL((k_shade<true, false, 3>), dim3(ls.shadeGrid),
                                                             dim3(kShadeBlock), 0, c->stream, f, qsel));
        else if (!BATCH && f.guided)
            RBH_TIMED(KernelTimer::SHADE, hipLaunchKernelGGL((k_shade<true, false, 1>), dim3(ls.shadeGrid),
                                                             dim3(kShadeBlock), 0, c->stream, f, qsel));
        else if (ls.shadeWaves >= 4)
            RBH_TIMED(KernelTimer::SHADE, hipLaunchKernelGGL((k_shade<false, BATCH, 4>), dim3(ls.shadeGrid),
                                                             dim3(kShadeBlock), 0, c->stream, f, qsel));
        else if (ls.shadeWaves == 3)
            RBH_TIMED(KernelTimer::SHADE, hipLaunchKernelGGL((k_shade<false, BATCH, 3>), dim3(ls.shadeGrid),
                                                             dim3(kShadeBlock), 0, c->stream, f, qsel));
        else
            RBH_TIMED(KernelTimer::SHADE, hipLaunchKernelGGL((k_shade<false, BATCH, 1>), dim3(ls.shadeGrid),
                                                             dim3(kShadeBlock), 0, c->stream, f, qsel));
        RBH_TIMED(KernelTimer::SHADOW, launch_shadow<BATCH>(c, f, ls));
    }
#undef RBH_TIMED
    hipLaunchKernelGGL(k_accumulate<BATCH>, accGrid, dim3(256), 0, c->stream, f);
    return hipGetLastError();
}

hipError_t launch_pass(rbh_ctx c, const Frame1& f, uint32_t depthMax, const LaunchShape& ls, KernelTimer* kt) {
    return f.scenes ? launch_pass_t<true>(c, f, depthMax, ls, kt) : launch_pass_t<false>(c, f, depthMax, ls, kt);
}

}  // namespace rbh
