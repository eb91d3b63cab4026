// Path-guiding network on CDNA4 matrix cores: BF16 MFMA forward, fused
// loss + backward with per-block weight-gradient accumulation, reduction +
// Adam, and inference (BF16 or FP8 E4M3 with per-tensor scales).
//
// The training kernel's work layout stands at k_guide_train.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "radix.hpp"

#include "../context.hpp"
#include "../guide.hpp"
#include "../device/mlp_wave.hpp"

// the sizes the public header documents
static_assert(RBH_GUIDE_RECORD == rbh::guide::kRec, "record size");
static_assert(RBH_GUIDE_OUTPUTS == rbh::guide::kOut, "output row size");
static_assert(RBH_GUIDE_PARAMS == rbh::guide::kParams, "parameter count");

namespace rbh {

using namespace guide;
using namespace mlp;

namespace {

// ------------------------------------------------------------- mixture
// log of kappa / (2 pi (1 - exp(-2 kappa)))
__device__ __forceinline__ float vmf_log_norm(float kappa) {
    return logf(kappa) - 1.8378770664093453f - logf(-expm1f(-2.0f * kappa));
}

// Largest value and sum over the eight lanes of a record.
__device__ __forceinline__ float max8(float v) {
    for (int o = 1; o < 8; o <<= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}
__device__ __forceinline__ float sum8(float v) {
    for (int o = 1; o < 8; o <<= 1) v += __shfl_xor(v, o);
    return v;
}

// Training: forward, loss and backward of tiles of 64 records by one
// workgroup of eight waves per CU; weight gradients stay in registers over
// all tiles of the workgroup.
//
// In the layers a wave owns 16 output (backward: input) features of 32
// records: its weights are the same for every tile and stay in registers, and
// the layers hand over through LDS, one barrier each. A product is formed
// twice, with its operands swapped: the matrix instruction gives a lane four
// consecutive rows of one column, so one order yields four features of a
// record, the next layer's operand, and the other four records of a feature,
// the operand of the weight gradients' contraction over records; both are
// stored with 8-byte writes and read with 16-byte ones. ReLU masks stay in
// registers: the wave that produced a value also masks its gradient. The loss
// runs one vMF lobe per thread.
// Bound by the latency of the tile's twelve phases (two waves per SIMD). One
// pass over 262,144 records on 256 CUs: 194 us; the matrix products alone
// would take 13 us. With four waves of 16 records, each walking all columns
// with weights re-read from the cache, a record's eight lobes in one lane and
// 2-byte reads for the weight gradients it took 607 us.
constexpr int kTrainBlock = 512;
constexpr int kTrainTile = 64;      // records per tile
constexpr int kST = kTrainTile + 8; // row stride of [feature][record] arrays, in bf16
constexpr int kSOT = 52;            // row stride of the outputs, in floats
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;

struct TrainLds {
    bf16 x0[kTrainTile * kSX0];          // encoded inputs [record][feature]
    bf16 x0t[kIn * kST];                 // ... [feature][record]
    bf16 ht[4][kWidth * kST];            // inputs of layers 1..4 [feature][record]
    bf16 row[2][kTrainTile * kSH];       // activations, then gradients [record][feature], alternating
    bf16 dy4[kTrainTile * kSH];          // gradient of the outputs [record][feature], zero past them
    bf16 dy4t[48 * kST];                 // ... [feature][record]
    union {
        float out[kTrainTile * kSOT];    // raw outputs, read before the first gradient is written
        bf16 dyt[2][kWidth * kST];       // gradients [feature][record], alternating
    };
    float bias[kBiasPad];
    float red[kTrainBlock / 64];
};

// The lane index, anew in every phase: addresses of the dozen LDS arrays kept
// over the tile loop instead would spill the weights.
__device__ __forceinline__ int phase_lane() {
    int lane = __lane_id();
    asm volatile("" : "+v"(lane));
    return lane;
}
__device__ __forceinline__ bf16x8 frag(const bf16* p) { return *reinterpret_cast<const bf16x8*>(p); }

// Four values as bf16 in one 8-byte store; with a mask, its bits decide which
// pass; returns which are positive.
__device__ __forceinline__ uint32_t put4(bf16* dst, f32x4 v) {
    bf16x4 b;
    uint32_t m = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        b[i] = (bf16)v[i];
        m |= (float)b[i] > 0.0f ? 1u << i : 0u;
    }
    *reinterpret_cast<bf16x4*>(dst) = b;
    return m;
}
__device__ __forceinline__ f32x4 masked(f32x4 v, uint32_t m) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = (m >> i) & 1u ? v[i] : 0.0f;
    return v;
}

// One hidden layer for the wave's 32 records and 16 features: y and yt from
// x. Returns the ReLU mask, per 16 records 4 bits in either operand order.
template <int KB>
__device__ __forceinline__ uint32_t train_hidden(const bf16* x, int sx, const bf16x8 (&w)[KB], const float* bias, bf16* y,
                                                 bf16* yt, int ct, int half) {
    const int lane = phase_lane(), r = lane & 15, g = lane >> 4;
    const f32x4 b1 = *reinterpret_cast<const f32x4*>(bias + ct * 16 + 4 * g);
    const float b2 = bias[ct * 16 + r];
    uint32_t mask = 0;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int R = half * 32 + q * 16;
        f32x4 c1 = {0.0f, 0.0f, 0.0f, 0.0f}, c2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            const bf16x8 a = frag(x + (R + r) * sx + kb * 32 + 8 * g);
            c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kb], a, c1, 0, 0, 0);
            c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[kb], c2, 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            c1[i] = fmaxf(c1[i] + b1[i], 0.0f);
            c2[i] = fmaxf(c2[i] + b2, 0.0f);
        }
        mask |= put4(y + (R + r) * kSH + ct * 16 + 4 * g, c1) << (8 * q);
        mask |= put4(yt + (ct * 16 + r) * kST + R + 4 * g, c2) << (8 * q + 4);
    }
    return mask;
}

// The gradient of a layer's inputs, masked by their ReLU, from the gradient
// dy of its outputs; ROWS: also the [record][feature] form for the layer below.
template <bool ROWS>
__device__ __forceinline__ void train_back(const bf16* dy, const bf16x8 (&w)[2], uint32_t mask, bf16* dx, bf16* dxt, int ct,
                                           int half) {
    const int lane = phase_lane(), r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const int R = half * 32 + q * 16;
        f32x4 c1 = {0.0f, 0.0f, 0.0f, 0.0f}, c2 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const bf16x8 a = frag(dy + (R + r) * kSH + kb * 32 + 8 * g);
            if (ROWS) c1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[kb], a, c1, 0, 0, 0);
            c2 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w[kb], c2, 0, 0, 0);
        }
        if (ROWS) put4(dx + (R + r) * kSH + ct * 16 + 4 * g, masked(c1, mask >> (8 * q)));
        put4(dxt + (ct * 16 + r) * kST + R + 4 * g, masked(c2, mask >> (8 * q + 4)));
    }
}

// Adds the tile's weight gradients of one layer: output features 16 rt ..,
// input features 16 (c0 + 2 j) ..; waves with c0 = 0 also the bias gradients.
template <int NJ>
__device__ __forceinline__ void train_grads(const bf16* dyt, const bf16* xt, int rt, int c0, int ncols, f32x4 (&acc)[NJ],
                                            f32x4& accb) {
    const int lane = phase_lane(), r = lane & 15, g = lane >> 4;
    bf16x8 ones;
#pragma unroll
    for (int q = 0; q < 8; ++q) ones[q] = (bf16)1.0f;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        const bf16x8 a = frag(dyt + (rt * 16 + r) * kST + kb * 32 + 8 * g);
#pragma unroll
        for (int j = 0; j < NJ; ++j)
            if (c0 + 2 * j < ncols)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, frag(xt + ((c0 + 2 * j) * 16 + r) * kST + kb * 32 + 8 * g),
                                                                 acc[j], 0, 0, 0);
        if (c0 == 0) accb = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, ones, accb, 0, 0, 0);
    }
}

// Writes one layer's share of the workgroup's gradient in the master layout.
template <int NJ>
__device__ __forceinline__ void store_grads(float* __restrict__ part, int l, int rt, int c0, const f32x4 (&acc)[NJ],
                                            const f32x4& accb) {
    const int lane = __lane_id(), r = lane & 15, g = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int out = rt * 16 + 4 * g + i;
        if (out >= fan_out(l)) continue;
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int in = (c0 + 2 * j) * 16 + r;
            if (in < fan_in(l)) part[w_off(l) + out * fan_in(l) + in] = acc[j][i];
        }
        if (c0 == 0 && r == 0) part[b_off(l) + out] = accb[i];
    }
}

// floats ahead of the partial sums in GuideState::scalars
enum : int { GS_LOSS = 0, GS_COLLECTED = 1, kScalars = 4 };   // the loss; the weight sum of a collected set
constexpr int kSumBlocks = 256;     // partial weight sums, then as many partial losses

__global__ __launch_bounds__(kTrainBlock) void k_guide_train(const float* __restrict__ recs, uint32_t n,
                                                             const float* __restrict__ weightPart,
                                                             const bf16* __restrict__ wf, const bf16* __restrict__ wt,
                                                             const float* __restrict__ bias, float* __restrict__ partials,
                                                             float* __restrict__ lossPart, uint32_t fixedSel) {
    __shared__ TrainLds L;
    const int t = (int)threadIdx.x, wave = t >> 6, lane = __lane_id(), r = lane & 15, g = lane >> 4;
    const int ct = wave & 3, half = wave >> 2;
    float wsum;
    {
        float v = t < kSumBlocks ? weightPart[t] : 0.0f;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (lane == 0) L.red[wave] = v;
        if (t < kBiasPad) L.bias[t] = bias[t];
        // the columns that no phase writes
        for (int q = t; q < kTrainTile * (96 - kIn); q += kTrainBlock) L.x0[(q / (96 - kIn)) * kSX0 + kIn + q % (96 - kIn)] = (bf16)0.0f;
        for (int q = t; q < kTrainTile * kSH; q += kTrainBlock) L.dy4[q] = (bf16)0.0f;
        for (int q = t; q < 48 * kST; q += kTrainBlock) L.dy4t[q] = (bf16)0.0f;
        __syncthreads();
        wsum = ((L.red[0] + L.red[1]) + (L.red[2] + L.red[3])) + ((L.red[4] + L.red[5]) + (L.red[6] + L.red[7]));
    }
    const float invW = wsum > 0.0f ? 1.0f / wsum : 0.0f;
    // this wave's weights: output features 16 ct .. of every layer, and input features 16 ct .. going back
    bf16x8 w0[3], w1[2], w2[2], w3[2], w4[2], v1[2], v2[2], v3[2], v4[2];
    {
        const int row = ct * 16 + r;
#pragma unroll
        for (int kb = 0; kb < 3; ++kb) w0[kb] = frag(wf + wf_off(0) + row * 96 + kb * 32 + 8 * g);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const int o = row * 64 + kb * 32 + 8 * g;
            w1[kb] = frag(wf + wf_off(1) + o); w2[kb] = frag(wf + wf_off(2) + o);
            w3[kb] = frag(wf + wf_off(3) + o); w4[kb] = frag(wf + wf_off(4) + o);
            v1[kb] = frag(wt + wf_off(1) + o); v2[kb] = frag(wt + wf_off(2) + o);
            v3[kb] = frag(wt + wf_off(3) + o); v4[kb] = frag(wt + wf_off(4) + o);
        }
    }
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 g0[3] = {zero, zero, zero}, g1[2] = {zero, zero}, g2[2] = {zero, zero}, g3[2] = {zero, zero}, g4[2] = {zero, zero};
    f32x4 gb0 = zero, gb1 = zero, gb2 = zero, gb3 = zero, gb4 = zero;
    float lossAcc = 0.0f;

    for (uint32_t tile = blockIdx.x; (size_t)tile * kTrainTile < n; tile += gridDim.x) {
        const uint32_t base = tile * kTrainTile;
        // the loss's inputs of record t / 8, needed after the forward pass
        const uint32_t ls = base + (uint32_t)(t >> 3);
        float lr[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
        if (ls < n) {
#pragma unroll
            for (int k = 0; k < 5; ++k) lr[k] = recs[(size_t)ls * kRec + 11 + k];
        }
        // ---- encode: record t % 64, sin/cos pairs wave, wave + 8, ... and feature 72 + wave
        {
            const int lane = phase_lane();
            const uint32_t s = base + (uint32_t)lane;
            const bool live = s < n;
            const float* rec = recs + (size_t)(live ? s : 0u) * kRec;
            const float px = rec[0], py = rec[1], pz = rec[2], ft = live ? rec[3 + wave] : 0.0f;
            __syncthreads();   // the previous tile's gradients are done with the inputs
#pragma unroll
            for (int j = 0; j < 5; ++j) {
                const int p = wave + 8 * j;
                if (p >= 36) break;
                const int axis = p / 12, k = p % 12;
                float sn = 0.0f, cs = 0.0f;
                if (live) {
                    const float x = (axis == 0 ? px : axis == 1 ? py : pz) * (float)(1 << k);   // exact power-of-two scaling
                    const float rr = x - 2.0f * floorf(x * 0.5f);                                // exact reduction modulo 2
                    sincospif(rr, &sn, &cs);
                }
                const bf16 bs = (bf16)sn, bc = (bf16)cs;
                L.x0[lane * kSX0 + 2 * p] = bs;
                L.x0[lane * kSX0 + 2 * p + 1] = bc;
                L.x0t[(2 * p) * kST + lane] = bs;
                L.x0t[(2 * p + 1) * kST + lane] = bc;
            }
            const bf16 bf = (bf16)ft;
            L.x0[lane * kSX0 + 72 + wave] = bf;
            L.x0t[(72 + wave) * kST + lane] = bf;
        }
        // ---- forward
        __syncthreads();
        const uint32_t m0 = train_hidden<3>(L.x0, kSX0, w0, L.bias + bp_off(0), L.row[0], L.ht[0], ct, half);
        __syncthreads();
        const uint32_t m1 = train_hidden<2>(L.row[0], kSH, w1, L.bias + bp_off(1), L.row[1], L.ht[1], ct, half);
        __syncthreads();
        const uint32_t m2 = train_hidden<2>(L.row[1], kSH, w2, L.bias + bp_off(2), L.row[0], L.ht[2], ct, half);
        __syncthreads();
        const uint32_t m3 = train_hidden<2>(L.row[0], kSH, w3, L.bias + bp_off(3), L.row[1], L.ht[3], ct, half);
        __syncthreads();
        if (ct < 3) {
            const int lane = phase_lane(), r = lane & 15, g = lane >> 4;
            const f32x4 b = *reinterpret_cast<const f32x4*>(L.bias + bp_off(4) + ct * 16 + 4 * g);
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int R = half * 32 + q * 16;
                f32x4 c = zero;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
                    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w4[kb], frag(L.row[1] + (R + r) * kSH + kb * 32 + 8 * g), c, 0, 0, 0);
                *reinterpret_cast<f32x4*>(L.out + (R + r) * kSOT + ct * 16 + 4 * g) = c + b;
            }
        }
        __syncthreads();
        // ---- loss: lobe t % 8 of record t / 8. Loss of a record is
        // weight * -log(a q(d) + (1 - a) p_bsdf(d)) with q the lobe mixture and a
        // the selection probability; its gradient * 1 / weight sum goes to dy4
        {
            const int rec = wave * 8 + (phase_lane() >> 3), j = t & 7;
            float dv[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f}, dsel = 0.0f;
            if (ls < n) {   // all eight lanes of a record or none
                const float dx = lr[0], dy = lr[1], dz = lr[2], wgt = lr[3], pb = lr[4];
                const float* o = L.out + rec * kSOT;
                const float q0 = o[5 * j], q1 = o[5 * j + 1], q2 = o[5 * j + 2], lk = o[5 * j + 3], logit = o[5 * j + 4];
                const float c = o[kMix];
                const float nrm = fmaxf(sqrtf(q0 * q0 + q1 * q1 + q2 * q2), 1e-6f);
                const float mx = q0 / nrm, my = q1 / nrm, mz = q2 / nrm;
                const float kappa = expf(fminf(fmaxf(lk, kLogKappaMin), kLogKappaMax));
                const float lmax = max8(logit);
                const float lw = logit - (lmax + logf(sum8(expf(logit - lmax))));   // log of the softmax weight
                const float dot = mx * dx + my * dy + mz * dz;
                const float lc = lw + vmf_log_norm(kappa) + kappa * (dot - 1.0f);
                const float cmax = max8(lc);
                const float lse = cmax + logf(sum8(expf(lc - cmax)));               // log q
                const float q = expf(lse);
                const float sig = 1.0f / (1.0f + expf(-c));
                const float a = kSelMin + (kSelMax - kSelMin) * sig;
                const float P = fmaxf(a * q + (1.0f - a) * pb, 1e-30f);
                const float s0 = wgt * invW;
                const float s = s0 * (a * q / P);               // the lobes' share of the combined density
                const float w = expf(lw), gj = expf(lc - lse);
                const float dlnorm = 1.0f / kappa - 2.0f / expm1f(2.0f * kappa);
                const float dk = -s * gj * (dlnorm + dot - 1.0f);
                const bool inside = lk > kLogKappaMin && lk < kLogKappaMax;
                const float cc = -s * gj * kappa;
                const float gx = cc * dx, gy = cc * dy, gz = cc * dz;
                const float pr = gx * mx + gy * my + gz * mz;
                dv[0] = (gx - mx * pr) / nrm;
                dv[1] = (gy - my * pr) / nrm;
                dv[2] = (gz - mz * pr) / nrm;
                dv[3] = inside ? dk * kappa : 0.0f;
                dv[4] = -s * (gj - w);
                // selection: d(-log P)/da = -(q - p_bsdf) / P, da/dc = (kSelMax - kSelMin) sig (1 - sig)
                // (with a fixed selection the selection output stays zero, a = 0.5)
                dsel = fixedSel ? 0.0f : -s0 * (q - pb) / P * (kSelMax - kSelMin) * sig * (1.0f - sig);
                if (j == 0) lossAcc += wgt * -logf(P);
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                const bf16 b = (bf16)dv[k];
                L.dy4[rec * kSH + 5 * j + k] = b;
                L.dy4t[(5 * j + k) * kST + rec] = b;
            }
            if (j == 0) {
                const bf16 b = (bf16)dsel;
                L.dy4[rec * kSH + kMix] = b;
                L.dy4t[kMix * kST + rec] = b;
            }
        }
        // ---- backward: the next gradient, and the weight gradients of the layer it came from
        __syncthreads();
        train_back<true>(L.dy4, v4, m3, L.row[0], L.dyt[0], ct, half);
        if (ct < 3) train_grads(L.dy4t, L.ht[3], ct, half, 4, g4, gb4);
        __syncthreads();
        train_back<true>(L.row[0], v3, m2, L.row[1], L.dyt[1], ct, half);
        train_grads(L.dyt[0], L.ht[2], ct, half, 4, g3, gb3);
        __syncthreads();
        train_back<true>(L.row[1], v2, m1, L.row[0], L.dyt[0], ct, half);
        train_grads(L.dyt[1], L.ht[1], ct, half, 4, g2, gb2);
        __syncthreads();
        train_back<false>(L.row[0], v1, m0, nullptr, L.dyt[1], ct, half);
        train_grads(L.dyt[0], L.ht[0], ct, half, 4, g1, gb1);
        __syncthreads();
        train_grads(L.dyt[1], L.x0t, ct, half, 5, g0, gb0);
    }

    float* part = partials + (size_t)blockIdx.x * kParams;
    store_grads(part, 0, ct, half, g0, gb0);
    store_grads(part, 1, ct, half, g1, gb1);
    store_grads(part, 2, ct, half, g2, gb2);
    store_grads(part, 3, ct, half, g3, gb3);
    if (ct < 3) store_grads(part, 4, ct, half, g4, gb4);
    float v = lossAcc;
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    __syncthreads();
    if (lane == 0) L.red[wave] = v;
    __syncthreads();
    if (t == 0) {
        float sum = 0.0f;
        for (int k = 0; k < kTrainBlock / 64; ++k) sum += L.red[k];
        lossPart[blockIdx.x] = sum * invW;
    }
}

__global__ void k_zero_f32(float* p, int n) {
    if ((int)threadIdx.x < n) p[threadIdx.x] = 0.0f;
}

__global__ __launch_bounds__(256) void k_weight_sum(const float* __restrict__ recs, uint32_t n, float* out) {
    float s = 0.0f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) s += recs[(size_t)i * kRec + 14];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (__lane_id() == 0) atomicAdd(out, s);
}

// Partial sums of the weights: block b's at out[b], the rest of out cleared
// by the last block. (One 4-byte value of a 64-byte record, so all lines are
// read; partial sums instead of atomics on one address, which took most of
// 16 us for 262,144 records, and the training kernel adds them in order.)
__global__ __launch_bounds__(1024) void k_weight_partials(const float* __restrict__ recs, uint32_t n, float* __restrict__ out) {
    __shared__ float red[16];
    float s = 0.0f;
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) s += recs[(size_t)i * kRec + 14];
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (__lane_id() == 0) red[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) {
        float v = 0.0f;
        for (int k = 0; k < 16; ++k) v += red[k];
        out[blockIdx.x] = v;
    }
    if (blockIdx.x + 1 == gridDim.x && gridDim.x + threadIdx.x < kSumBlocks) out[gridDim.x + threadIdx.x] = 0.0f;
}

// ------------------------------------------------- collected training set
struct PositiveWeight {
    const float* recs;
    __device__ __forceinline__ bool operator()(uint32_t i) const { return recs[(size_t)i * kRec + 14] > 0.0f; }
};

// out[j] = recs[idx[(j * stride) mod m]]: a fixed permutation (stride is
// coprime with m) so that consecutive batches mix all regions of the image
__global__ __launch_bounds__(256) void k_gather_records(const float* __restrict__ recs, const uint32_t* __restrict__ idx,
                                                        uint32_t m, uint32_t stride, float* __restrict__ out) {
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < m; j += gridDim.x * blockDim.x) {
        const uint32_t s = idx[(uint32_t)(((uint64_t)j * stride) % m)];
        const float4* src = reinterpret_cast<const float4*>(recs + (size_t)s * kRec);
        float4* dst = reinterpret_cast<float4*>(out + (size_t)j * kRec);
#pragma unroll
        for (int k = 0; k < kRec / 4; ++k) dst[k] = src[k];
    }
}

// w = min(w, mult * mean w), the mean read from *sum
__global__ __launch_bounds__(256) void k_clamp_weights(float* __restrict__ recs, uint32_t m, const float* __restrict__ sum,
                                                       float mult) {
    const float cap = mult * (*sum / (float)m);
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < m; j += gridDim.x * blockDim.x)
        recs[(size_t)j * kRec + 14] = fminf(recs[(size_t)j * kRec + 14], cap);
}

// parameter p of the master layout -> (layer, out, in) or bias (in = -1)
__device__ __forceinline__ void param_index(int p, int& l, int& out, int& in) {
    l = 0;
    while (l + 1 < kLayers && p >= w_off(l + 1)) ++l;
    const int q = p - w_off(l);
    if (q < fan_in(l) * fan_out(l)) { out = q / fan_in(l); in = q % fan_in(l); }
    else { out = q - fan_in(l) * fan_out(l); in = -1; }
}

__device__ __forceinline__ void publish(int p, float w, bf16* wf, bf16* wt, float* bias) {
    int l, out, in;
    param_index(p, l, out, in);
    if (in < 0) { bias[bp_off(l) + out] = w; return; }
    wf[wf_off(l) + out * k_pad(l) + in] = (bf16)w;
    wt[wf_off(l) + in * 64 + out] = (bf16)w;
}

// Sums the block partials; mode 0: Adam step and publish, mode 1: write the
// gradient. 32 parameters per workgroup, eight lanes each over every eighth
// partial (one lane per parameter over all 256: 64 us, 80 workgroups).
constexpr int kReduceParams = 32;
__global__ __launch_bounds__(256) void k_guide_reduce(const float* __restrict__ partials, int nblocks, int mode,
                                                      float* __restrict__ master, float* __restrict__ m,
                                                      float* __restrict__ v, float lr, float b1, float b2, float eps,
                                                      float bc1, float bc2, bf16* wf, bf16* wt, float* bias,
                                                      float* __restrict__ gradOut, const float* __restrict__ lossPart,
                                                      float* __restrict__ lossOut) {
    __shared__ float red[8][kReduceParams];
    const int c = threadIdx.x & (kReduceParams - 1), k = threadIdx.x / kReduceParams;
    const int p = blockIdx.x * kReduceParams + c;
    float part = 0.0f;
    if (p < kParams) {
#pragma unroll 8
        for (int b = k; b < nblocks; b += 8) part += partials[(size_t)b * kParams + p];
    }
    red[k][c] = part;
    __syncthreads();
    if (blockIdx.x == 0 && threadIdx.x == 64) {
        float l = 0.0f;
        for (int b = 0; b < nblocks; ++b) l += lossPart[b];
        *lossOut = l;
    }
    if (k != 0 || p >= kParams) return;
    float gsum = 0.0f;
#pragma unroll
    for (int q = 0; q < 8; ++q) gsum += red[q][c];
    if (mode == 1) { gradOut[p] = gsum; return; }
    const float mm = b1 * m[p] + (1.0f - b1) * gsum;
    const float vv = b2 * v[p] + (1.0f - b2) * gsum * gsum;
    m[p] = mm;
    v[p] = vv;
    const float w = master[p] - lr * (mm / bc1) / (sqrtf(vv / bc2) + eps);
    master[p] = w;
    publish(p, w, wf, wt, bias);
}

__global__ __launch_bounds__(256) void k_guide_publish(const float* __restrict__ master, bf16* wf, bf16* wt, float* bias) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p < kParams) publish(p, master[p], wf, wt, bias);
}

// inference of staged records (raw outputs), the renderer's wave-resident
// kernel body; FP8: E4M3 weights with per-layer scales
template <bool FP8>
__global__ __launch_bounds__(256, 2) void k_guide_infer(const float* __restrict__ recs, uint32_t n,
                                                        const bf16* __restrict__ wf, const uint8_t* __restrict__ wq,
                                                        const float* __restrict__ wqs, const float* __restrict__ bias,
                                                        float* __restrict__ out) {
    __shared__ WaveLds L[4];
    wave_infer<FP8, false>(L[threadIdx.x >> 6], recs, n, wf, wq, wqs, bias, out);
}

// FP8 copy of the weights: one block per layer finds the largest magnitude,
// then writes E4M3 bytes of W / scale into the [n_pad][k_pad] layout.
__global__ __launch_bounds__(256) void k_fp8_quant(const float* __restrict__ master, uint8_t* __restrict__ wq,
                                                   float* __restrict__ scales) {
    __shared__ float red[4];
    const int l = blockIdx.x;
    const float* W = master + w_off(l);
    const int nw = fan_in(l) * fan_out(l);
    float m = 0.0f;
    for (int i = threadIdx.x; i < nw; i += blockDim.x) m = fmaxf(m, fabsf(W[i]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    if (__lane_id() == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    const float amax = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float sc = amax > 0.0f ? amax / kFp8Max : 1.0f;
    if (threadIdx.x == 0) scales[l] = sc;
    const float inv = 1.0f / sc;
    uint8_t* q = wq + wf_off(l);
    for (int i = threadIdx.x; i < n_pad(l) * k_pad(l); i += blockDim.x) {
        const int out = i / k_pad(l), in = i % k_pad(l);
        const float v = (out < fan_out(l) && in < fan_in(l)) ? W[out * fan_in(l) + in] * inv : 0.0f;
        q[i] = (uint8_t)(__builtin_amdgcn_cvt_pk_fp8_f32(v, 0.0f, 0, false) & 0xFF);
    }
}

int train_blocks(rbh_ctx c) {
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device) != hipSuccess || cus <= 0) cus = 256;
    return cus;
}

template <typename T> T* dptr(void* p) { return static_cast<T*>(p); }

}  // namespace

// ------------------------------------------------------------------ host
void guide_release(GuideState& g) {
    void* ptrs[] = {g.master, g.adamM, g.adamV, g.wf, g.wt, g.bias, g.partials, g.scalars, g.records, g.trainRecs, g.recCount, g.fp8w, g.fp8s};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    g = GuideState{};
}

}  // namespace rbh

using namespace rbh;

namespace {

GuideState& gs(rbh_ctx c) {
    if (!c->guide) c->guide = new GuideState();
    return *static_cast<GuideState*>(c->guide);
}

hipError_t alloc(void** p, size_t bytes) {
    if (*p) return hipSuccess;
    return hipMalloc(p, bytes);
}

// deterministic He-uniform initialisation (SplitMix64 stream)
void init_params(uint32_t seed, std::vector<float>& p) {
    p.assign(kParams, 0.0f);
    uint64_t st = 0x9E3779B97F4A7C15ull * (seed + 1);
    auto next = [&]() {
        uint64_t z = (st += 0x9E3779B97F4A7C15ull);
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        z ^= z >> 31;
        return (double)(z >> 11) * (1.0 / 9007199254740992.0);
    };
    for (int l = 0; l < kLayers; ++l) {
        const double lim = std::sqrt(6.0 / fan_in(l));
        for (int i = 0; i < fan_in(l) * fan_out(l); ++i) p[w_off(l) + i] = (float)((2.0 * next() - 1.0) * lim);
    }
}

// The selection output's weights and bias (output kMix of the last layer):
// zero and never trained when the selection is fixed at 0.5, which makes the
// network the 40-output mixture network.
void clear_selection_row(std::vector<float>& p) {
    const int l = kLayers - 1;
    for (int i = 0; i < fan_in(l); ++i) p[w_off(l) + kMix * fan_in(l) + i] = 0.0f;
    p[b_off(l) + kMix] = 0.0f;
}

// FP8 copy of the current weights
void quantise_fp8(rbh_ctx c) {
    GuideState& g = gs(c);
    hipLaunchKernelGGL(k_fp8_quant, dim3(kLayers), dim3(256), 0, c->stream, dptr<float>(g.master), dptr<uint8_t>(g.fp8w),
                       dptr<float>(g.fp8s));
}

int upload_master(rbh_ctx c, const float* params) {
    GuideState& g = gs(c);
    std::vector<float> fixedParams;
    if (g.fixedSel) {
        fixedParams.assign(params, params + kParams);
        clear_selection_row(fixedParams);
        params = fixedParams.data();
    }
    RBH_HIP(c, hipMemcpyAsync(g.master, params, kParams * 4, hipMemcpyHostToDevice, c->stream));
    RBH_HIP(c, hipMemsetAsync(g.adamM, 0, kParams * 4, c->stream));
    RBH_HIP(c, hipMemsetAsync(g.adamV, 0, kParams * 4, c->stream));
    hipLaunchKernelGGL(k_guide_publish, dim3((kParams + 255) / 256), dim3(256), 0, c->stream, dptr<float>(g.master),
                       dptr<bf16>(g.wf), dptr<bf16>(g.wt), dptr<float>(g.bias));
    quantise_fp8(c);
    RBH_HIP(c, hipGetLastError());
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    g.step = 0;
    return RBH_OK;
}

// gradient pass over n device records; mode 0 = Adam step, 1 = gradient to gradOut
int run_train(rbh_ctx c, const float* drecs, uint32_t n, int mode, float* gradOut, float* lossOut) {
    GuideState& g = gs(c);
    const int blocks = (int)std::min<size_t>(std::min(train_blocks(c), kSumBlocks), (n + kTrainTile - 1) / (size_t)kTrainTile);
    if (blocks <= 0) return fail(c, RBH_ERR_INVALID, "no training records");
    if ((size_t)blocks > g.partialBlocks) {
        if (g.partials) (void)hipFree(g.partials);
        g.partials = nullptr;
        RBH_HIP(c, hipMalloc(&g.partials, (size_t)blocks * kParams * 4));
        g.partialBlocks = blocks;
    }
    float* sc = dptr<float>(g.scalars);
    float* wpart = sc + kScalars;
    float* lpart = wpart + kSumBlocks;
    hipLaunchKernelGGL(k_weight_partials, dim3((unsigned)std::min<size_t>(kSumBlocks, (n + 1023) / (size_t)1024)), dim3(1024), 0,
                       c->stream, drecs, n, wpart);
    hipLaunchKernelGGL(k_guide_train, dim3(blocks), dim3(kTrainBlock), 0, c->stream, drecs, n, wpart, dptr<bf16>(g.wf),
                       dptr<bf16>(g.wt), dptr<float>(g.bias), dptr<float>(g.partials), lpart, g.fixedSel ? 1u : 0u);
    if (mode == 0) ++g.step;
    const float bc1 = 1.0f - std::pow(g.beta1, (float)std::max<uint32_t>(1, g.step));
    const float bc2 = 1.0f - std::pow(g.beta2, (float)std::max<uint32_t>(1, g.step));
    hipLaunchKernelGGL(k_guide_reduce, dim3((kParams + kReduceParams - 1) / kReduceParams), dim3(256), 0, c->stream,
                       dptr<float>(g.partials), blocks, mode, dptr<float>(g.master), dptr<float>(g.adamM),
                       dptr<float>(g.adamV), g.lr, g.beta1, g.beta2, g.eps, bc1, bc2, dptr<bf16>(g.wf), dptr<bf16>(g.wt),
                       dptr<float>(g.bias), gradOut, lpart, sc + GS_LOSS);
    RBH_HIP(c, hipGetLastError());
    if (lossOut) {
        float l = 0.0f;
        RBH_HIP(c, hipMemcpyAsync(&l, sc + GS_LOSS, sizeof(l), hipMemcpyDeviceToHost, c->stream));
        RBH_HIP(c, hipStreamSynchronize(c->stream));
        *lossOut = l;
    }
    return RBH_OK;
}

// `steps` Adam steps over consecutive batches of n device records, wrapping
// around; the FP8 copy follows the last.
int run_steps(rbh_ctx c, const float* drecs, uint32_t n, uint32_t batch, uint32_t steps, float* loss) {
    for (uint32_t s = 0; s < steps; ++s) {
        const uint32_t off = (uint32_t)(((uint64_t)s * batch) % n);
        const uint32_t len = std::min(batch, n - off);
        const int rc = run_train(c, drecs + (size_t)off * kRec, len, 0, nullptr, s + 1 == steps ? loss : nullptr);
        if (rc) return rc;
    }
    if (steps) quantise_fp8(c);
    RBH_HIP(c, hipGetLastError());
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    return RBH_OK;
}

}  // namespace

extern "C" {

int rbh_guide_configure(rbh_ctx c, const rbh_guide_config* cfg) {
    if (!c || !cfg) return RBH_ERR_INVALID;
    if (!(cfg->lr > 0.0f) || !(cfg->beta1 >= 0.0f && cfg->beta1 < 1.0f) || !(cfg->beta2 >= 0.0f && cfg->beta2 < 1.0f) ||
        !(cfg->eps > 0.0f))
        return fail(c, RBH_ERR_INVALID, "Adam parameters out of range");
    if (cfg->fixedSelection > 1u) return fail(c, RBH_ERR_INVALID, "fixedSelection must be 0 or 1");
    GuideState& g = gs(c);
    RBH_HIP(c, hipSetDevice(c->device));
    RBH_HIP(c, alloc(&g.master, kParams * 4));
    RBH_HIP(c, alloc(&g.adamM, kParams * 4));
    RBH_HIP(c, alloc(&g.adamV, kParams * 4));
    RBH_HIP(c, alloc(&g.wf, kWfTotal * 2));
    RBH_HIP(c, alloc(&g.wt, kWfTotal * 2));
    RBH_HIP(c, alloc(&g.bias, kBiasPad * 4));
    RBH_HIP(c, alloc(&g.scalars, (kScalars + 2 * kSumBlocks) * 4));
    RBH_HIP(c, alloc(&g.fp8w, kWfTotal));
    RBH_HIP(c, alloc(&g.fp8s, 64));
    RBH_HIP(c, hipMemsetAsync(g.fp8w, 0, kWfTotal, c->stream));
    RBH_HIP(c, hipMemsetAsync(g.wf, 0, kWfTotal * 2, c->stream));
    RBH_HIP(c, hipMemsetAsync(g.wt, 0, kWfTotal * 2, c->stream));
    RBH_HIP(c, hipMemsetAsync(g.bias, 0, kBiasPad * 4, c->stream));
    g.recCapacity = cfg->recordCapacity ? cfg->recordCapacity : (1u << 22);
    if (g.records) { (void)hipFree(g.records); g.records = nullptr; }
    if (g.trainRecs) { (void)hipFree(g.trainRecs); g.trainRecs = nullptr; }
    RBH_HIP(c, hipMalloc(&g.records, (size_t)g.recCapacity * 24 * 4));
    RBH_HIP(c, hipMalloc(&g.trainRecs, (size_t)g.recCapacity * kRec * 4));
    RBH_HIP(c, alloc(&g.recCount, 16));
    RBH_HIP(c, hipMemsetAsync(g.recCount, 0, 16, c->stream));
    g.lr = cfg->lr;
    g.beta1 = cfg->beta1;
    g.beta2 = cfg->beta2;
    g.eps = cfg->eps;
    g.fixedSel = cfg->fixedSelection != 0u;
    for (int a = 0; a < 3; ++a) {
        const float e = cfg->sceneMax[a] - cfg->sceneMin[a];
        if (!(e > 0.0f)) return fail(c, RBH_ERR_INVALID, "scene bounds must have positive extent");
        g.sceneMin[a] = cfg->sceneMin[a];
        g.sceneInvExtent[a] = 1.0f / e;
    }
    std::vector<float> p;
    init_params(cfg->seed, p);
    const int rc = upload_master(c, p.data());
    if (rc) return rc;
    g.configured = true;
    return RBH_OK;
}

int rbh_guide_set_params(rbh_ctx c, const float* params, uint32_t n) {
    if (!c || !params) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    if (n != (uint32_t)kParams) return fail(c, RBH_ERR_INVALID, "expected %d parameters, got %u", kParams, n);
    return upload_master(c, params);
}

int rbh_guide_get_params(rbh_ctx c, float* params, uint32_t n) {
    if (!c || !params) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    if (n != (uint32_t)kParams) return fail(c, RBH_ERR_INVALID, "expected %d parameters, got %u", kParams, n);
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    RBH_HIP(c, hipMemcpy(params, gs(c).master, kParams * 4, hipMemcpyDeviceToHost));
    return RBH_OK;
}

// The record and output buffers of a call stay on the context, up to this size
// each (2M records in, 800k records' outputs); larger ones go with the call.
constexpr size_t kKeptBytes = (size_t)128 << 20;
struct KeptBuffers {
    rbh_ctx c;
    ~KeptBuffers() {
        for (DevBuf* b : {&c->guideRecords, &c->guideOutputs})
            if (b->bytes > kKeptBytes) b->release();
    }
};

static int stage_records(rbh_ctx c, const float* recs, uint32_t n) {
    DevBuf& buf = c->guideRecords;
    RBH_ALLOC(c, buf, (size_t)std::max<uint32_t>(n, 1) * kRec * 4);
    RBH_HIP(c, copy_in(c, buf.p, recs, (size_t)n * kRec * 4));
    return RBH_OK;
}

int rbh_guide_gradient(rbh_ctx c, const float* recs, uint32_t n, float* grad, float* loss) {
    if (!c || !recs || !grad || n == 0) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    const KeptBuffers kept{c};
    DevBuf gbuf;
    int rc = stage_records(c, recs, n);
    if (rc) return rc;
    RBH_ALLOC(c, gbuf, kParams * 4);
    float l = 0.0f;
    rc = run_train(c, c->guideRecords.as<float>(), n, 1, gbuf.as<float>(), &l);
    if (rc) return rc;
    RBH_HIP(c, hipMemcpy(grad, gbuf.p, kParams * 4, hipMemcpyDeviceToHost));
    if (loss) *loss = l;
    return RBH_OK;
}

int rbh_guide_train(rbh_ctx c, const float* recs, uint32_t n, uint32_t batch, uint32_t steps, float* lastLoss) {
    if (!c || !recs || n == 0 || batch == 0) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    const KeptBuffers kept{c};
    int rc = stage_records(c, recs, n);
    if (rc) return rc;
    float l = 0.0f;
    rc = run_steps(c, c->guideRecords.as<float>(), n, batch, steps, &l);
    if (rc) return rc;
    if (lastLoss) *lastLoss = l;
    return RBH_OK;
}

static int collected(rbh_ctx c, uint32_t* n) {
    GuideState& g = gs(c);
    uint32_t cnt = 0;
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    RBH_HIP(c, hipMemcpy(&cnt, g.recCount, 4, hipMemcpyDeviceToHost));
    *n = std::min(cnt, g.recCapacity);
    return RBH_OK;
}

int rbh_guide_records(rbh_ctx c, float* out, uint32_t max, uint32_t* n) {
    if (!c || !n) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    uint32_t k = 0;
    int rc = collected(c, &k);
    if (rc) return rc;
    *n = k;
    if (out && max) RBH_HIP(c, copy_out(c, out, gs(c).trainRecs, (size_t)std::min(k, max) * kRec * 4));
    return RBH_OK;
}

// Training set of a collecting render, in the pending-record buffer (free
// between renders): the records with a positive weight, in a fixed
// pseudo-random order, weights clamped twice at kClampMean times their mean.
// Clamping only changes what the network is fitted to, never the render's
// estimator; it keeps a few one-sample radiance outliers from dominating
// every batch.
constexpr float kClampMean = 10.0f;

static int prepare_collected(rbh_ctx c, uint32_t n, uint32_t* m) {
    GuideState& g = gs(c);
    const float* recs = static_cast<const float*>(g.trainRecs);
    DevBuf idx, tmp;
    RBH_ALLOC(c, idx, (size_t)n * 4 + 16);
    uint32_t* cnt = idx.as<uint32_t>() + n + (4 - n % 4) % 4;
    RBH_ALLOC(c, tmp, radix::select_scratch_bytes(n));
    RBH_HIP(c, radix::select_indices(tmp.p, n, PositiveWeight{recs}, idx.as<uint32_t>(), cnt, c->stream));
    uint32_t k = 0;
    RBH_HIP(c, hipMemcpyAsync(&k, cnt, 4, hipMemcpyDeviceToHost, c->stream));
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    if (k == 0) return fail(c, RBH_ERR_STATE, "no collected training record has a positive weight");
    static const uint32_t primes[] = {1000003u, 999983u, 104729u, 7919u};
    uint32_t stride = 1u;
    for (uint32_t p : primes)
        if (k % p != 0u) { stride = p % k == 0u ? 1u : p; break; }
    float* out = static_cast<float*>(g.records);
    const int blocks = (int)std::min<uint32_t>(4096u, (k + 255u) / 256u);
    hipLaunchKernelGGL(k_gather_records, dim3(blocks), dim3(256), 0, c->stream, recs, idx.as<uint32_t>(), k, stride, out);
    float* sum = dptr<float>(g.scalars) + GS_COLLECTED;
    for (int pass = 0; pass < 2; ++pass) {
        hipLaunchKernelGGL(k_zero_f32, dim3(1), dim3(64), 0, c->stream, sum, 1);
        hipLaunchKernelGGL(k_weight_sum, dim3(256), dim3(256), 0, c->stream, out, k, sum);
        hipLaunchKernelGGL(k_clamp_weights, dim3(blocks), dim3(256), 0, c->stream, out, k, sum, kClampMean);
    }
    RBH_HIP(c, hipGetLastError());
    RBH_HIP(c, hipStreamSynchronize(c->stream));
    *m = k;
    return RBH_OK;
}

int rbh_guide_train_collected(rbh_ctx c, uint32_t batch, uint32_t steps, float* lastLoss) {
    if (!c || batch == 0) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    uint32_t n0 = 0, n = 0;
    int rc = collected(c, &n0);
    if (rc) return rc;
    if (n0 == 0) return fail(c, RBH_ERR_STATE, "no training records collected");
    rc = prepare_collected(c, n0, &n);
    if (rc) return rc;
    float l = 0.0f;
    rc = run_steps(c, static_cast<const float*>(gs(c).records), n, batch, steps, &l);
    if (rc) return rc;
    if (lastLoss) *lastLoss = l;
    return RBH_OK;
}

static int infer(rbh_ctx c, const float* recs, uint32_t n, float* out, bool fp8) {
    if (!c || !recs || !out) return RBH_ERR_INVALID;
    if (!gs(c).configured) return fail(c, RBH_ERR_STATE, "rbh_guide_configure first");
    if (n == 0) return RBH_OK;
    GuideState& g = gs(c);
    const KeptBuffers kept{c};
    int rc = stage_records(c, recs, n);
    if (rc) return rc;
    DevBuf &d = c->guideRecords, &o = c->guideOutputs;
    RBH_ALLOC(c, o, (size_t)n * kOut * 4);
    // four waves of 16 records per block
    const int blocks = (int)std::min<size_t>((size_t)train_blocks(c) * 2, (n + 4 * kRows - 1) / (4 * kRows));
    if (fp8)
        hipLaunchKernelGGL((k_guide_infer<true>), dim3(blocks), dim3(256), 0, c->stream, d.as<float>(), n,
                           dptr<bf16>(g.wf), dptr<uint8_t>(g.fp8w), dptr<float>(g.fp8s), dptr<float>(g.bias), o.as<float>());
    else
        hipLaunchKernelGGL((k_guide_infer<false>), dim3(blocks), dim3(256), 0, c->stream, d.as<float>(), n,
                           dptr<bf16>(g.wf), nullptr, dptr<float>(g.fp8s), dptr<float>(g.bias), o.as<float>());
    RBH_HIP(c, hipGetLastError());
    RBH_HIP(c, copy_out(c, out, o.p, (size_t)n * kOut * 4));
    return RBH_OK;
}

int rbh_guide_infer(rbh_ctx c, const float* recs, uint32_t n, float* out) { return infer(c, recs, n, out, false); }

int rbh_guide_infer_fp8(rbh_ctx c, const float* recs, uint32_t n, float* out) { return infer(c, recs, n, out, true); }

}  // extern "C"
