// The 32-bit matrix product (see linear_f32.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace psamd {

// Whether the kernels take these operands: rows of whole 16-byte pieces.
bool linear_f32_takes(const void* x, const void* w, int64_t M, int N, int K);
int launch_linear_f32(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K);

}  // namespace psamd
