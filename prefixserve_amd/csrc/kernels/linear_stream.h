// bfloat16 products of 17 to 128 tokens through LDS (linear_stream.hip), and of up to 16 that are normalized on the way in (linear_normed.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace psamd {

// Where the tokens of a small step come from: bfloat16 rows x[M][K], or (x == nullptr) rows of the
// float32 residual stream that the kernel normalizes itself on the way in (RMS norm: statistics
// in 32-bit, eps inside the root, times the norm's weight), row rows[m] for token m (rows ==
// nullptr: row m). A kernel that reads its tokens this way needs no norm kernel in front of it.
struct Tokens {
  const bf16_t* x;
  const float* resid;
  const void* norm_w;
  const int32_t* rows;
  float eps;
  int norm_w_bf16;      // the norm's weight is bfloat16 (else float32)
};

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


// out[M, n_out] = norm(the residual stream's rows) * w^T, in one of the forms of stream_operands.h; whether that
// kernel takes it and is the faster.
bool linear_normed_takes(const void* w, const void* out, int form, int M, int n_out, int K);
int launch_linear_normed(hipStream_t s, const Tokens& tk, const void* w, void* out, int form, int M, int n_out, int K, int gate_act,
                         const QkvOut& q = {});

}  // namespace psamd
