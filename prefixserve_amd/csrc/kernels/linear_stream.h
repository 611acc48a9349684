// bfloat16 products of 17 to 128 tokens through LDS (linear_stream.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace psamd {

// What a q/k/v projection needs behind its product, as in qkv_rope_append_kernel.
struct QkvOut {
  int hq, hkv, d;
  const int32_t* positions;
  const float2* table;
  bf16_t* kv;
  const int32_t* write_slot;
};

bool linear_stream_takes(const void* x, const void* w, const void* out, int M, int n_out, int K, bool gated);
// The number of K-slices of a product that it takes, if somebody adds them up.
int linear_stream_ksplit(int n_out, int K);
// gate_act < 0: out [M, n_out] in float32 ([ksplit] slices of it) or bfloat16; else act(gate) * up in bfloat16.
int launch_linear_stream(hipStream_t s, const void* x, const void* w, void* out, bool out_f32, int M, int n_out, int K, int gate_act,
                         int ksplit);
int launch_qkv_stream(hipStream_t s, const void* x, const void* w, void* out, int M, int K, const QkvOut& q);

}  // namespace psamd
