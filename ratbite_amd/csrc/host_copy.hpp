// Copies between pageable host memory and the device.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>

struct rbh_context;

namespace rbh {

// Copies `bytes` from host memory into a device buffer, behind the work on the
// context's stream; returns when the source may be reused. (Small copies are
// left on the stream: the caller synchronises it as before.)
hipError_t copy_in(rbh_context* c, void* dst, const void* src, size_t bytes);

// Copies a device buffer to host memory once the context's stream is done.
hipError_t copy_out(rbh_context* c, void* dst, const void* src, size_t bytes);

}  // namespace rbh
