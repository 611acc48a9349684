// bfloat16 products of 17 to 128 tokens, out[M,N] = x[M,K] * w[N,K]^T, with both operands through LDS.
//
// They are bound by reading w once, but the kernels of linear.hip read the tokens from L2 beside it, in pieces of 64 bytes
// of 16 rows: as many bytes as w at 64 tokens, through the path that carries w. Here a workgroup copies whole lines of both into
// LDS (global_load_lds, 16 bytes a lane, nothing through registers), several steps ahead, for up to 64 rows of w at a time, and the
// matrix instructions read them there. Microseconds of a product whose weights are not in any cache (from 65 tokens on the other
// side is the library, with the rotation or the activation in a kernel behind it):
//   rows x K            17 tokens      32             64             77             128
//   2,048 x 2,048       4.9 -> 4.3     5.3 -> 4.5     7.1 -> 5.0     8.5 -> 5.3     8.8 -> 6.0
//   2,048 x 8,192      11.7 -> 9.3    13.5 -> 9.5    15.6 -> 10.4   21.0 -> 12.7   21.8 -> 14.1
//   4,096 x 14,336     35.1 -> 23.6   40.2 -> 24.1   41.2 -> 29.3   49.5 -> 37.3   75.9 -> 38.7
//   2 x 8,192 x 2,048  20.3 -> 17.7   21.4 -> 17.7   22.0 -> 18.5   23.3 -> 22.0   25.7 -> 22.9   (gated)
//   2 x 14,336 x 4,096 58.4 -> 50     62.0 -> 52     58.3 -> 53     60   -> 58     62.7 -> 60     (gated)
//   6,144 x 4,096      19.6 -> 15.8   22.4 -> 16.5   30.5 -> 20.4   28.9 -> 25.5   31.4 -> 28.4   (q/k/v)
//   128,256 x 2,048     131 -> 107     138 -> 108     159 -> 125    (float32 out; above 64 tokens the library's product is as fast)
// So do the bfloat16 products above 64 tokens (16,384 x 2,048 at 77: 18.4 there, 19.1 here), which stay with the library.

#include <algorithm>

#include "api.h"
#include "common.h"
#include "linear_stream.h"

namespace psamd {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((address_space(1))) const void* global_ptr;
typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(3))) const unsigned char* lds_bytes;

constexpr int kSlices = 0, kPlain = 1, kGated = 2, kQkv = 3;

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
      "ds_read_b128 %4, %9\n\tds_read_b128 %5, %9 offset:2048\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[1][0]), "=&v"(x[1][0]),
        "=&v"(x[1][1])
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
      "ds_read_b128 %8, %13 offset:4096\n\tds_read_b128 %9, %13 offset:6144\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]), "=&v"(x[0][3]),
        "=&v"(w[1][0]), "=&v"(x[1][0]), "=&v"(x[1][1]), "=&v"(x[1][2]), "=&v"(x[1][3])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u) : "memory");
  }
};
template <int TN>
struct Operands<TN, 2, 1> {
  bf16x8 w[2][2], x[2][1];
  __device__ __forceinline__ void read(uint32_t w_at, uint32_t x_at) {
    asm volatile(
      "ds_read_b128 %0, %6\n\tds_read_b128 %1, %6 offset:%10\n\tds_read_b128 %2, %8\n\tds_read_b128 %3, %7\n\t"
      "ds_read_b128 %4, %7 offset:%10\n\tds_read_b128 %5, %9\n\ts_waitcnt lgkmcnt(0)"
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(w[1][0]), "=&v"(w[1][1]),
        "=&v"(x[1][0])
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
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(w[1][0]),
        "=&v"(w[1][1]), "=&v"(x[1][0]), "=&v"(x[1][1])
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
      : "=&v"(w[0][0]), "=&v"(w[0][1]), "=&v"(x[0][0]), "=&v"(x[0][1]), "=&v"(x[0][2]),
        "=&v"(x[0][3]), "=&v"(w[1][0]), "=&v"(w[1][1]), "=&v"(x[1][0]), "=&v"(x[1][1]),
        "=&v"(x[1][2]), "=&v"(x[1][3])
      : "v"(w_at), "v"(w_at ^ 64u), "v"(x_at), "v"(x_at ^ 64u), "i"(TN * 128) : "memory");
  }
};

constexpr int stream_wait(int vmcnt) { return (vmcnt & 15) | ((vmcnt >> 4) << 14) | (7 << 4) | (15 << 8); }   // s_waitcnt vmcnt(n) alone

// grid (ceil(rows of w / TN), K-slices), W waves: TN rows of w for all of up to TM tokens; the gated form takes TN gate rows and
// the TN up rows of the same columns, the q/k/v form lays 8 rotation pairs of a head into each tile of 16 rows: 8 rows of its
// first half and their partners in the second, whose sums then lie two lane groups apart. A wave makes 16 columns for
// TM / (W / (TN / 16)) tokens. A step is 64 k: rows of 128 bytes whose 16-byte pieces are exchanged by row / 2, so that 16 rows'
// reads meet every bank once. Buffer t % STAGES holds step t, which is asked for STAGES - 1 steps ahead, into the buffer that
// everybody has read when the barrier in front of its asking has been passed.
template <int TM, int TN, int W, int FORM, int STAGES>
__global__ __launch_bounds__(64 * W) void stream_tiles_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                              void* __restrict__ out, int M, int N, int K, int slice_steps, int act,
                                                              QkvOut q) {
  constexpr int CT = TN / 16, RM = TM / 16 / (W / CT), RT = FORM == kGated ? 2 : 1, ROWS = TN * RT, STAGE = (ROWS + TM) * 128;
  constexpr int LW = ROWS / 8 / W, LX = TM / 8 / W, COPIES = LW + LX;           // copies of 8 rows per wave and step
  static_assert(W % CT == 0 && RM * 16 * (W / CT) == TM && LW * 8 * W == ROWS && LX * 8 * W == TM, "whole copies per wave");
  extern __shared__ __align__(16) unsigned char stream_smem[];                 // STAGES x [ROWS rows of w, TM of x][128]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN;
  const int first = blockIdx.y * slice_steps, steps = min(slice_steps, K / 64 - first);
  const char* xb = reinterpret_cast<const char*>(x) + static_cast<int64_t>(first) * 128;
  const char* wb = reinterpret_cast<const char*>(w) + static_cast<int64_t>(first) * 128;
  const int half = FORM == kQkv ? q.d >> 1 : 0;
  uint32_t w_off[LW], x_off[LX];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (wave * LW + i) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    int col = min(n0 + row % TN, N - 1);
    if (FORM == kQkv) {                                                        // N is a multiple of 16: whole tiles of 8 pairs
      const int pair = col / 16 * 8 + col % 8, head = pair / half;
      col = head * q.d + (pair - head * half) + (col % 16 < 8 ? 0 : half);
    }
    w_off[i] = static_cast<uint32_t>(row >= TN ? N + col : col) * (2u * K) + 16u * piece;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (wave * LX + i) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    x_off[i] = static_cast<uint32_t>(min(row, M - 1)) * (2u * K) + 16u * piece;
  }
  auto copy = [&](int t) {
    unsigned char* to = stream_smem + t % STAGES * STAGE;
#pragma unroll
    for (int i = 0; i < LW; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr)(wb + w_off[i] + t * 128), (lds_ptr)(to + (wave * LW + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < LX; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr)(xb + x_off[i] + t * 128), (lds_ptr)(to + ROWS * 128 + (wave * LX + i) * 1024), 16, 0, 0);
  };
  // For sums that leave in 32 bits two steps (one where there are few) are summed from zero and then added to the rest: one long
  // chain through the matrix instructions has up to three times the error of the kernels that split K over waves (against 64 bits,
  // 128,256 columns of K = 2,048 at 64 tokens: 2.7e-7 in one chain, 1.3e-7 there, 1.0e-7 here; 2,048 x 8,192 in eight slices:
  // 1.9e-7, 0.82e-7, 0.82e-7). In sums that are rounded to 16 bits it makes no difference (1.66e-3 each way) and costs up to 1.5 us.
  constexpr bool RUNS = FORM == kSlices;
  f32x4 acc[RT][RM], part[RT][RM];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int j = 0; j < RM; ++j) acc[rt][j] = part[rt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tile = wave % CT, tokens = wave / CT * (16 * RM);                  // this wave's column tile and first token
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes)stream_smem));
  const uint32_t piece0 = 16u * (g ^ ((r >> 1) & 7));
  const uint32_t w_at = base + (16 * tile + r) * 128 + piece0, x_at = base + (ROWS + tokens + r) * 128 + piece0;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < steps) copy(t);
  int buf = 0;
  for (int t = 0; t < steps; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    // Of what has been asked for, only the steps behind t may still be under way; near the end they are fewer.
    if (t + STAGES - 2 < steps) __builtin_amdgcn_s_waitcnt(stream_wait((STAGES - 2) * COPIES));
    else __builtin_amdgcn_s_waitcnt(stream_wait(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + STAGES - 1 < steps) copy(t + STAGES - 1);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t at = static_cast<uint32_t>(buf) * STAGE;
    buf = buf + 1 == STAGES ? 0 : buf + 1;
    Operands<TN, RT, RM> ops;
    ops.read(w_at + at, x_at + at);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < RM; ++j) {
          f32x4& sum = RUNS ? part[rt][j] : acc[rt][j];
          sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ops.w[h][rt], ops.x[h][j], sum, 0, 0, 0);
        }
    if (!RUNS) continue;
    if ((t & 1) != 0 || t + 1 == steps || steps < 8) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < RM; ++j) {
          acc[rt][j] += part[rt][j];
          part[rt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  const int n = n0 + 16 * tile + 4 * g;                                        // this lane's four columns of token tokens + 16 j + r
  auto pack = [](f32x4 v) { return ushort4{float_to_bf16(v[0]), float_to_bf16(v[1]), float_to_bf16(v[2]), float_to_bf16(v[3])}; };
#pragma unroll
  for (int j = 0; j < RM; ++j) {
    const int m = tokens + 16 * j + r;
    if constexpr (FORM == kQkv) {
      const bool second = g >= 2;
      const int pair = (n0 + 16 * tile) / 2 + 4 * (g & 1), head = pair / half, p = pair - head * half;
      f32x4 v = acc[0][j];
      const bool here = m < M && n < N;                                        // N is a multiple of 16: both halves of a pair or none
      const bool rotate = here && q.table != nullptr && head < q.hq + q.hkv;
      const float2* cs = rotate ? q.table + static_cast<int64_t>(q.positions[m]) * half + p : nullptr;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float other = __shfl_xor(v[i], 32, kWave);                       // the pair's other half
        const float2 c = rotate ? cs[i] : float2{1.f, 0.f};
        v[i] = second ? v[i] * c.x + other * c.y : v[i] * c.x - other * c.y;
      }
      if (!here) continue;
      const ushort4 pk = pack(v);
      const int e0 = (second ? half : 0) + p;                                  // element of the head, 4 consecutive
      *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + head * q.d + e0) = pk;
      if (q.kv == nullptr || head < q.hq) continue;
      const int slot = q.write_slot[m], off = slot % kPage;
      bf16_t* page = q.kv + static_cast<int64_t>(slot / kPage) * (2LL * q.hkv * kPage * q.d);
      if (head < q.hq + q.hkv) {                                               // key row [16][D]
        *reinterpret_cast<ushort4*>(page + (static_cast<int64_t>(head - q.hq) * kPage + off) * q.d + e0) = pk;
      } else {                                                                 // value, transposed [D][16], behind the keys
        bf16_t* vp = page + (static_cast<int64_t>(head - q.hq) * q.d + e0) * kPage + off;
        vp[0] = pk.x;
        vp[kPage] = pk.y;
        vp[2 * kPage] = pk.z;
        vp[3 * kPage] = pk.w;
      }
      continue;
    }
    if (m >= M || n >= N) continue;                                            // N is a multiple of 4
    if constexpr (FORM == kSlices) {
      float* o = static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n;
      *reinterpret_cast<f32x4*>(o) = acc[0][j];
    } else {
      f32x4 v = acc[0][j];
      if constexpr (FORM == kGated) {
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gate_act(v[i], act) * acc[RT - 1][j][i];
      }
      *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + n) = pack(v);
    }
  }
}

// The most rows of w per workgroup, which read the tokens least often, that still leave most of the 256 compute units one
// (64, 32 and 16 rows at 64 tokens: 2 x 14,336 x 4,096 49.5, 50.5 and 62 us; 2 x 8,192 x 2,048 24.1, 18.6 and 20.1;
// 2 x 4,096 x 2,048 20.3, 13.9 and 12.0; 16,384 x 2,048 16.8, 18.6 and 26.0; 4,096 x 2,048 12.6, 10.1 and 9.2). With K-slices,
// which linear_stream_ksplit chooses for 64 rows, fewer only where even eight slices leave units idle (1,024 x 1,024: 3.5, 3.2, 3.2).
static int stream_columns(int N, int ksplit) {
  constexpr int kEnough = 192;
  return ceil_div(N, 64) * ksplit >= kEnough ? 64 : (ceil_div(N, 32) * ksplit >= kEnough ? 32 : 16);
}

// 80 KB of buffers, so that two workgroups share a compute unit; at least three, which for 128 tokens and 64 rows of gate and up are
// 96 KB: one.
constexpr int stream_stages(int stage) { return std::min(8, std::max(3, 80 * 1024 / stage)); }

template <int TM, int TN, int W, int FORM>
static int launch_stream_tiles(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                               const QkvOut& q) {
  constexpr int STAGE = ((FORM == kGated ? 2 : 1) * TN + TM) * 128, STAGES = stream_stages(STAGE);
  constexpr size_t smem = static_cast<size_t>(STAGES) * STAGE;
  auto kernel = stream_tiles_kernel<TM, TN, W, FORM, STAGES>;
  if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("linear_stream: " + std::to_string(smem) + " bytes of LDS were refused");
  const int slice_steps = static_cast<int>(ceil_div(K / 64, ksplit));
  kernel<<<dim3(static_cast<unsigned>(ceil_div(N, TN)), static_cast<unsigned>(ksplit)), dim3(64 * W), smem, s>>>(
      static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), out, M, N, K, slice_steps, act, q);
  return check_launch("linear_stream");
}

template <int FORM>
static int launch_stream_form(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                              const QkvOut& q = {}) {
  const int tn = stream_columns(N, ksplit);
#define PSAMD_STREAM(TM_, W64_, W32_, W16_)                                                              \
  if (tn == 64) return launch_stream_tiles<TM_, 64, W64_, FORM>(s, x, w, out, M, N, K, ksplit, act, q);  \
  if (tn == 32) return launch_stream_tiles<TM_, 32, W32_, FORM>(s, x, w, out, M, N, K, ksplit, act, q);  \
  return launch_stream_tiles<TM_, 16, W16_, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  if (M <= 32) { PSAMD_STREAM(32, 4, 4, 2) }
  if (M <= 64) { PSAMD_STREAM(64, 4, 4, 2) }
  PSAMD_STREAM(128, 8, 4, 2)
#undef PSAMD_STREAM
}

bool linear_stream_takes(const void* x, const void* w, const void* out, int M, int n_out, int K, bool gated) {
  return M > 16 && M <= 128 && n_out > 0 && n_out % 4 == 0 && K >= 64 && K % 64 == 0 &&
         (gated ? 4LL : 2LL) * n_out * K < (1LL << 32) &&                      // offsets of 32 bits
         (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
}

// As many slices as give every compute unit a workgroup of 64 rows, up to the eight that the buffers of their consumers hold
// (at 64 tokens, with 2, 4 and 8 slices: 2,048 x 2,048 6.5, 4.8 and 4.5 us; 4,096 x 4,096 13.5, 9.3 and 10.7; 4,096 x 14,336 41, 25
// and 27; 5,120 x 5,120 20.0, 18.9 with 4, 16.1 with 3).
int linear_stream_ksplit(int n_out, int K) {
  const int64_t blocks = ceil_div(n_out, 64), steps = K / 64;
  const int64_t wanted = std::min<int64_t>({8, (256 + blocks / 2) / blocks, std::max<int64_t>(steps / 2, 1)});
  const int64_t slice = ceil_div(steps, std::max<int64_t>(wanted, 1));
  return static_cast<int>(ceil_div(steps, slice));                             // no slice is empty
}

int launch_linear_stream(hipStream_t s, const void* x, const void* w, void* out, bool out_f32, int M, int n_out, int K, int gate_act,
                         int ksplit) {
  if (gate_act >= 0) return launch_stream_form<kGated>(s, x, w, out, M, n_out, K, 1, gate_act);
  if (out_f32) return launch_stream_form<kSlices>(s, x, w, out, M, n_out, K, ksplit, 0);
  return launch_stream_form<kPlain>(s, x, w, out, M, n_out, K, 1, 0);
}

int launch_qkv_stream(hipStream_t s, const void* x, const void* w, void* out, int M, int K, const QkvOut& q) {
  return launch_stream_form<kQkv>(s, x, w, out, M, (q.hq + 2 * q.hkv) * q.d, K, 1, 0, q);
}

}  // namespace psamd
