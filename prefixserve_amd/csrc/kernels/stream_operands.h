// Operands of the small bfloat16 products from LDS, 64 k at a time, and the waits for the copies that brought them there
// (linear_stream.hip, linear_normed.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "common.h"
#include "linear_stream.h"

namespace psamd {

constexpr int kSlices = 0, kPlain = 1, kGated = 2, kQkv = 3;                   // what becomes of the sums: float32, bfloat16, act(gate) * up, q/k/v


typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(1))) const void* global_ptr;
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(3))) const unsigned char* lds_bytes;

// RT row tiles of w (TN rows apart) and RM tiles of tokens for 64 k, from LDS. The wait is in the same block as the reads, and
// they are written this way because the compiler waits for every copy under way in front of a read of LDS that it sees.
template <int TN, int RT, int RM>
struct Operands;
template <int TN>
struct Operands<TN, 1, 1> {
  bf16x8 w[2][1], x[2][1];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %4\n\tds_read_b128 %1, %6\n\tds_read_b128 %2, %5\n\tds_read_b128 %3, %7\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(w[1][0]), "=&v"(x[1][0])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 1, 2> {
  bf16x8 w[2][1], x[2][2];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %6\n\tds_read_b128 %1, %8\n\tds_read_b128 %2, %8 offset:2048\n\tds_read_b128 %3, %7\n\t"
      "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[1][0]), "=&v"(x[1][0]), "=&v"(x[1][1])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 1, 3> {
  bf16x8 w[2][1], x[2][3];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %10\n\tds_read_b128 %2, %10 offset:2048\n\tds_read_b128 %3, %10 offset:4096\n\t"
      "ds_read_b128 %4, %9\n\tds_read_b128 %5, %11\n\tds_read_b128 %6, %11 offset:2048\n\tds_read_b128 %7, %11 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(w[1][0]), "=&v"(x[1][0]),
        "=&v"(x[1][1]), "=&v"(x[1][2])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 1, 4> {
  bf16x8 w[2][1], x[2][4];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %10\n\tds_read_b128 %1, %12\n\tds_read_b128 %2, %12 offset:2048\n\tds_read_b128 %3, %12 offset:4096\n\t"
      "ds_read_b128 %4, %12 offset:6144\n\tds_read_b128 %5, %11\n\tds_read_b128 %6, %13\n\tds_read_b128 %7, %13 offset:2048\n\t"
      "ds_read_b128 %8, %13 offset:4096\n\tds_read_b128 %9, %13 offset:6144\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(w[1][0]),
        "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 1, 6> {
  bf16x8 w[2][1], x[2][6];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %14\n\tds_read_b128 %1, %16\n\tds_read_b128 %2, %16 offset:2048\n\tds_read_b128 %3, %16 offset:4096\n\t"
      "ds_read_b128 %4, %16 offset:6144\n\tds_read_b128 %5, %16 offset:8192\n\tds_read_b128 %6, %16 offset:10240\n\tds_read_b128 %7, %15\n\t"
      "ds_read_b128 %8, %17\n\tds_read_b128 %9, %17 offset:2048\n\tds_read_b128 %10, %17 offset:4096\n\tds_read_b128 %11, %17 offset:6144\n\t"
      "ds_read_b128 %12, %17 offset:8192\n\tds_read_b128 %13, %17 offset:10240\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]), "=&v"(x[0][4]),
        "=&v"(x[0][5]), "=&v"(w[1][0]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3]),
        "=&v"(x[1][4]), "=&v"(x[1][5])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 2, 1> {
  bf16x8 w[2][2], x[2][1];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:%10\n\tds_read_b128 %2, %8\n\tds_read_b128 %3, %7\n\t"
      "ds_read_b128 %4, %7 offset:%10\n\tds_read_b128 %5, %9\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(x[1][0])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u), "i"(TN * 128) : "memory");
  }
};
template <int TN>
struct Operands<TN, 2, 2> {
  bf16x8 w[2][2], x[2][2];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %8\n\tds_read_b128 %1, %8 offset:%12\n\tds_read_b128 %2, %10\n\tds_read_b128 %3, %10 offset:2048\n\t"
      "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:%12\n\tds_read_b128 %6, %11\n\tds_read_b128 %7, %11 offset:2048\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[1][0]), "=&v"(w[1][1]),
        "=&v"(x[1][0]), "=&v"(x[1][1])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u), "i"(TN * 128) : "memory");
  }
};
template <int TN>
struct Operands<TN, 2, 3> {
  bf16x8 w[2][2], x[2][3];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %10\n\tds_read_b128 %1, %10 offset:%14\n\tds_read_b128 %2, %12\n\tds_read_b128 %3, %12 offset:2048\n\t"
      "ds_read_b128 %4, %12 offset:4096\n\tds_read_b128 %5, %11\n\tds_read_b128 %6, %11 offset:%14\n\tds_read_b128 %7, %13\n\t"
      "ds_read_b128 %8, %13 offset:2048\n\tds_read_b128 %9, %13 offset:4096\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(w[1][0]),
        "=&v"(w[1][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u), "i"(TN * 128) : "memory");
  }
};
template <int TN>
struct Operands<TN, 2, 4> {
  bf16x8 w[2][2], x[2][4];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %12\n\tds_read_b128 %1, %12 offset:%16\n\tds_read_b128 %2, %14\n\tds_read_b128 %3, %14 offset:2048\n\t"
      "ds_read_b128 %4, %14 offset:4096\n\tds_read_b128 %5, %14 offset:6144\n\tds_read_b128 %6, %13\n\tds_read_b128 %7, %13 offset:%16\n\t"
      "ds_read_b128 %8, %15\n\tds_read_b128 %9, %15 offset:2048\n\tds_read_b128 %10, %15 offset:4096\n\tds_read_b128 %11, %15 offset:6144\n\t"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]),
        "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u), "i"(TN * 128) : "memory");
  }
};

constexpr int stream_wait(int vmcnt) { return (vmcnt & 15) | ((vmcnt >> 4) << 14) | (7 << 4) | (15 << 8); }   // s_waitcnt vmcnt(n) alone

// Waits until of `left` steps of COPIES copies, asked for last, no more than MOST are under way. Where they are fewer, half of MOST or none:
// a wait for every number of them cost short loops more than it gave (17 steps 0.6 us).
template <int COPIES, int MOST>
__device__ __forceinline__ void wait_for_step(int left) {
  if (left >= MOST) __builtin_amdgcn_s_waitcnt(stream_wait(MOST * COPIES));
  else if (MOST > 2 && left >= MOST / 2) __builtin_amdgcn_s_waitcnt(stream_wait(MOST / 2 * COPIES));
  else __builtin_amdgcn_s_waitcnt(stream_wait(0));
}

// Four elements of one head of token m behind the rotation, from element e0 on: into the row of qkv, keys and values also into their slot.
__device__ __forceinline__ void put_qkv(bf16_t* qkv, int N, int m, int head, int e0, ushort4 pk, int slot, const QkvOut& q) {
  *reinterpret_cast<ushort4*>(qkv + static_cast<int64_t>(m) * N + head * q.d + e0) = pk;
  if (q.kv == nullptr || head < q.hq) return;
  const int off = slot % kPage;
  bf16_t* page = q.kv + static_cast<int64_t>(slot / kPage) * (2LL * q.hkv * kPage * q.d);
  if (head < q.hq + q.hkv) {                                                   // key row [16][D]
    *reinterpret_cast<ushort4*>(page + (static_cast<int64_t>(head - q.hq) * kPage + off) * q.d + e0) = pk;
  } else {                                                                     // value, transposed [D][16], behind the keys
    bf16_t* vp = page + (static_cast<int64_t>(head - q.hq) * q.d + e0) * kPage + off;
    vp[0] = pk.x;
    vp[kPage] = pk.y;
    vp[2 * kPage] = pk.z;
    vp[3 * kPage] = pk.w;
  }
}

}  // namespace psamd
