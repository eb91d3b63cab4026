// Shared constants and types of the guiding MLP's device code, and the FP8
// activation scale. Inference runs the wave-resident form in mlp_wave.hpp,
// training k_guide_train (kernels/guide.hip).
#pragma once
#include <hip/hip_runtime.h>
#include "../guide.hpp"

namespace rbh {
namespace mlp {

using namespace guide;

typedef __bf16 bf16;
typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kRows = 16;                  // records per wave per tile of the inference
constexpr int kSX0 = 96 + 8;               // LDS row strides in bf16 (16 B multiples, staggered banks)
constexpr int kSH = 64 + 8;
constexpr int kSO = kOut + 1;              // f32 output rows
// ----------------------------------------------------------------- FP8
// E4M3 inference with per-tensor scales: weights carry one scale per layer,
// activations one scale per layer and 16-record tile (the largest magnitude
// of the tile's rows maps to kFp8Max). kFp8Max stays within the finite range
// of both E4M3 encodings (240 and 448).
constexpr float kFp8Max = 240.0f;

__device__ __forceinline__ float wave_amax(const bf16* X, int sx, int K, int row0) {
    const int lane = __lane_id();
    float m = 0.0f;
    for (int q = lane; q < kRows * K; q += 64) m = fmaxf(m, fabsf((float)X[(row0 + q / K) * sx + q % K]));
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
    return m;
}

}  // namespace mlp
}  // namespace rbh
