// The 32-bit matrix product out[M,N] = x[M,K] * w[N,K]^T on the float32 matrix instructions
// (v_mfma_f32_16x16x4_f32: products and sums in float32, nothing rounded below it).
//
// Both kernels here sum every output in one order, whatever M is and whichever of them runs, so that a position's 32-bit
// result is the same bit for bit whether its step had 1 token or 1,000 (tests of the 32-bit path demand equality between
// different ways of cutting a sequence):
//   * kChain k are one chain of matrix instructions from zero, 16 k at a time, the i-th of four instructions taking
//     k = 4 g + i for the lane groups g = 0..3 (so a lane reads four neighbours at once);
//   * the chains of a segment (kSegment k) are added in ascending order, and then the segments.
// The chains are short because the matrix instruction rounds more than a fused multiply-add does: at K = 252 one chain is
// 4.5e-7 off the product in 64 bits where a chain of fused multiply-adds is 2.8e-7 off.

#include "api.h"
#include "common.h"
#include "linear_f32.h"

namespace psamd {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kChain = 64;
constexpr int kSegment = 256;

// 16 k of one tile: lane (r = l % 16, g = l / 16) holds k = 4 g .. 4 g + 3 of row r of both operands.
__device__ __forceinline__ f32x4 mma16(float4 a, float4 b, f32x4 acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.x, b.x, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.y, b.y, acc, 0, 0, 0);
  acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a.z, b.z, acc, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a.w, b.w, acc, 0, 0, 0);
}

// Lane (r, g) of a finished tile holds columns n .. n + 3 of token m.
__device__ __forceinline__ void put_columns(float* __restrict__ out, int64_t m, int n, int N, f32x4 v) {
  float* dst = out + m * N + n;
  if (n + 3 < N && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
    *reinterpret_cast<float4*>(dst) = float4{v[0], v[1], v[2], v[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) dst[i] = v[i];
  }
}

// ------------------------------------------------------------------ many tokens

// A workgroup of four waves makes 64 columns x BM tokens (a wave 32 x 32, or 16 x 32), both operands through LDS 64 k at a
// time, the next ones on their way in registers. Bound by the matrix instructions: 2,048 cycles of them per step and wave
// at 64 x 64 against 16 LDS reads of 16 bytes; 64 k a step because 32 k's instructions are over before the next step's
// rows arrive (one workgroup on a compute unit, K = 2,048: 57 -> 46 us). Rows of LDS are 68 floats apart: the 16 rows a read
// touches lie on 16 different groups of four banks. Tiles that share rows of w run on one die (its L2 serves them): die d
// takes the d-th eighth of the tiles, tokens fastest.
// 600 tokens x 16,384 columns x 2,048: 404 us, 100 TFLOP/s, where tiles of 64 x 64 by fused multiply-adds took 1,034.
constexpr int kColumns = 64;

template <int BM>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       float* __restrict__ out, int M, int N, int K, int m_tiles, int tiles,
                                                       int per_die) {
  constexpr int BN = kColumns, BK = 64, LD = BK + 4, RT = BN * BM / 2048, MT = 2;
  constexpr int CH = BK / 4, ROWS = 256 / CH;                          // 16-byte pieces per row, rows the workgroup brings at once
  constexpr int PW = BN / ROWS, PX = BM / ROWS;                        // pieces per thread
  static_assert(BM == 64 || BM == 32, "a wave takes 32 tokens");
  __shared__ __align__(16) float ws[2][BN * LD];
  __shared__ __align__(16) float xs[2][BM * LD];
  const int local = static_cast<int>(blockIdx.x >> 3), tile = static_cast<int>(blockIdx.x & 7) * per_die + local;
  if (local >= per_die || tile >= tiles) return;
  const int n0 = tile / m_tiles * BN, m0 = tile % m_tiles * BM;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int wn = (BM == 64 ? wave >> 1 : wave) * (RT * 16), wm = BM == 64 ? (wave & 1) * 32 : 0;   // this wave's part of the tile

  const float* wsrc[PW];
  const float* xsrc[PX];
  const int c4 = 4 * (tid % CH), row0 = tid / CH;                                        // first k of this thread's pieces
#pragma unroll
  for (int p = 0; p < PW; ++p) wsrc[p] = w + static_cast<int64_t>(min(n0 + row0 + ROWS * p, N - 1)) * K + c4;
#pragma unroll
  for (int p = 0; p < PX; ++p) xsrc[p] = x + static_cast<int64_t>(min(m0 + row0 + ROWS * p, M - 1)) * K + c4;
  float4 wr[PW], xr[PX];
  auto ask = [&](int k0) {
    const bool in = k0 + c4 < K;                                       // K is a multiple of 4
#pragma unroll
    for (int p = 0; p < PW; ++p) wr[p] = in ? *reinterpret_cast<const float4*>(wsrc[p] + k0) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < PX; ++p) xr[p] = in ? *reinterpret_cast<const float4*>(xsrc[p] + k0) : float4{0.f, 0.f, 0.f, 0.f};
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int p = 0; p < PW; ++p) *reinterpret_cast<float4*>(ws[buf] + (row0 + ROWS * p) * LD + c4) = wr[p];
#pragma unroll
    for (int p = 0; p < PX; ++p) *reinterpret_cast<float4*>(xs[buf] + (row0 + ROWS * p) * LD + c4) = xr[p];
  };
  f32x4 acc[RT][MT], part[RT][MT], total[RT][MT];                      // of the chain, the segment, all of K
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = part[rt][mt] = total[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  ask(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
    const bool more = k0 + BK < K;
    if (more) ask(k0 + BK);
    const float* wl = ws[buf] + (wn + r) * LD + 4 * g;
    const float* xl = xs[buf] + (wm + r) * LD + 4 * g;
#pragma unroll
    for (int kk = 0; kk < BK; kk += 16) {
      f32x4 a[RT], b[MT];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) a[rt] = *reinterpret_cast<const f32x4*>(wl + rt * 16 * LD + kk);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[mt] = *reinterpret_cast<const f32x4*>(xl + mt * 16 * LD + kk);
      // One k of every tile after the other: neighbouring instructions do not wait for each other's sums.
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][i], b[mt][i], acc[rt][mt], 0, 0, 0);
    }
    if (((k0 + BK) & (kChain - 1)) == 0 || !more) {                    // a chain is complete
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          part[rt][mt] += acc[rt][mt];
          acc[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (((k0 + BK) & (kSegment - 1)) == 0 || !more) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          total[rt][mt] += part[rt][mt];
          part[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (more) stage(buf ^ 1);                                          // last read before the barrier in front of this step
    __syncthreads();
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = m0 + wm + mt * 16 + r;
    if (m >= M) continue;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) put_columns(out, m, n0 + wn + rt * 16 + 4 * g, N, total[rt][mt]);
  }
}

// ------------------------------------------------------------------ a few tokens

// 16 MT tokens (blockIdx.y: which) by 16 rows of w per workgroup of eight waves: for a few tokens, where reading w once bounds
// it, and for products with too few tiles of the kernel above to fill the chip. The waves take the segments of K in turn,
// one each per round; a chain's rows of both operands are asked for while the chain before is multiplied; the round's sums
// are added in ascending order through LDS.
template <int MT>
__global__ __launch_bounds__(512) void rows_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                       float* __restrict__ out, int M, int N, int K) {
  constexpr int WV = 8, U = kChain / 16, kChains = kSegment / kChain;
  __shared__ f32x4 red[2][WV][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT;
  const float* wrow = w + static_cast<int64_t>(min(n0 + r, N - 1)) * K + 4 * g;
  const float* xrow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) xrow[mt] = x + static_cast<int64_t>(min(m0 + mt * 16 + r, M - 1)) * K + 4 * g;
  const int segments = (K + kSegment - 1) / kSegment;
  float4 a[2][U], b[2][MT][U];
  auto ask = [&](int which, int k0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = k0 + 16 * u;
      const bool in = k + 4 * g < K;                                   // K is a multiple of 4
      a[which][u] = in ? *reinterpret_cast<const float4*>(wrow + k) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[which][mt][u] = in ? *reinterpret_cast<const float4*>(xrow[mt] + k) : float4{0.f, 0.f, 0.f, 0.f};
    }
  };
  f32x4 total = {0.f, 0.f, 0.f, 0.f};                                  // of token tile `wave`, in waves below MT
  int buf = 0;
  ask(0, wave * kSegment);
  for (int s0 = 0; s0 < segments; s0 += WV, buf ^= 1) {
    const int k_seg = (s0 + wave) * kSegment;
    f32x4 part[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) part[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < kChains; ++c) {
      ask((c + 1) & 1, c + 1 < kChains ? k_seg + (c + 1) * kChain : k_seg + WV * kSegment);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < U; ++u) acc = mma16(a[c & 1][u], b[c & 1][mt][u], acc);
        part[mt] += acc;
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[buf][wave][mt][lane] = part[mt];
    __syncthreads();                                                   // the other buffer is written before the next barrier
    if (wave < MT) {
      const int n_seg = min(WV, segments - s0);
      for (int i = 0; i < n_seg; ++i) total += red[buf][i][wave][lane];
    }
  }
  const int m = m0 + wave * 16 + r;
  if (wave < MT && m < M) put_columns(out, m, n0 + 4 * g, N, total);
}

// The same where K is one segment: 16 rows of w per workgroup, a wave for each of its chains, which one wave then adds in
// ascending order. Of the eight waves above one had all the work (a chain is 0.2 us of matrix instructions). us at 1 token, by
// fused multiply-adds / above / here: 16,384 columns of K = 64 4.2 / 12.4 / 4.0, of 256 8.5 / 13.1 / 6.5, 1,024 of 256 4.5 / 5.2 / 4.7; at
// 64 tokens 34.8 / 7.9 / 4.9.
template <int MT>
__global__ __launch_bounds__(kSegment) void rows_short_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                  float* __restrict__ out, int M, int N, int K) {
  constexpr int U = kChain / 16;
  __shared__ f32x4 red[kSegment / kChain][MT][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, chains = blockDim.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16 * MT, k0 = wave * kChain + 4 * g;
  const float* wrow = w + static_cast<int64_t>(min(n0 + r, N - 1)) * K + k0;
  float4 a[U], b[MT][U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const bool in = k0 + 16 * u < K;                                   // K is a multiple of 4
    a[u] = in ? *reinterpret_cast<const float4*>(wrow + 16 * u) : float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const float* xrow = x + static_cast<int64_t>(min(m0 + mt * 16 + r, M - 1)) * K + k0;
      b[mt][u] = in ? *reinterpret_cast<const float4*>(xrow + 16 * u) : float4{0.f, 0.f, 0.f, 0.f};
    }
  }
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < U; ++u) acc = mma16(a[u], b[mt][u], acc);
    red[wave][mt][lane] = acc;
  }
  __syncthreads();
  for (int mt = wave; mt < MT; mt += chains) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    for (int i = 0; i < chains; ++i) total += red[i][mt][lane];
    const int m = m0 + mt * 16 + r;
    if (m < M) put_columns(out, m, n0 + 4 * g, N, total);
  }
}

template <int MT>
static void launch_rows_short(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const dim3 grid(static_cast<unsigned>(ceil_div(N, 16)), static_cast<unsigned>(ceil_div(M, 16 * MT)));
  rows_short_f32_kernel<MT><<<grid, dim3(64 * static_cast<unsigned>(ceil_div(K, kChain))), 0, s>>>(x, w, out, M, N, K);
}

template <int MT>
static void launch_rows(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const dim3 grid(static_cast<unsigned>(ceil_div(N, 16)), static_cast<unsigned>(ceil_div(M, 16 * MT)));
  rows_f32_kernel<MT><<<grid, dim3(512), 0, s>>>(x, w, out, M, N, K);
}

template <int BM>
static void launch_tiles(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const int m_tiles = static_cast<int>(ceil_div(M, BM)), tiles = static_cast<int>(ceil_div(N, kColumns)) * m_tiles;
  const int per_die = static_cast<int>(ceil_div(tiles, 8));
  gemm_f32_kernel<BM><<<dim3(static_cast<unsigned>(8 * per_die)), dim3(256), 0, s>>>(x, w, out, M, N, K, m_tiles, tiles, per_die);
}

bool linear_f32_takes(const void* x, const void* w, int64_t M, int N, int K) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w);
  return K % 4 == 0 && bits % 16 == 0 && M <= (1 << 24) && ceil_div(M, 64) * ceil_div(N, 64) < (1LL << 31) - 8;
}

// Which kernel, us at one MI355X (K = 2,048 unless given; every one gives the same bits):
//  * K of one segment, and up to 16 tokens or so few tiles as below: a wave per chain.
//  * up to 8 tokens, or 16 where the columns are fewer than 16,384: 16 rows of w per workgroup. 2,048 columns at 8 tokens 13
//    (tiles of 32 tokens 36), 128,256 at 1 token 187 (234); at 16 tokens 282 (224).
//  * fewer tiles of 32 tokens than half the compute units: the same kernel with 32 tokens. 64 tokens x 2,048 columns 16
//    (35), K = 8,192 54 (128); 200 tokens 50 (35).
//  * tiles of 32 tokens while those of 64 are so few that their last round is mostly empty: 600 x 2,048 71 (84), K = 8,192
//    267 (319); 600 x 3,072 97 (85); from there on tiles of 64: 600 x 16,384 404 (422), 100 TFLOP/s.
int launch_linear_f32(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const int64_t tiles64 = ceil_div(M, 64) * ceil_div(N, 64), tiles32 = ceil_div(M, 32) * ceil_div(N, 64);
  if (K <= kSegment && M <= 16) launch_rows_short<1>(s, x, w, out, M, N, K);
  else if (K <= kSegment && tiles32 <= 128) launch_rows_short<2>(s, x, w, out, M, N, K);
  else if (M <= 8 || (M <= 16 && N < 16384)) launch_rows<1>(s, x, w, out, M, N, K);
  else if (tiles32 <= 128) launch_rows<2>(s, x, w, out, M, N, K);
  else if (tiles64 <= 384) launch_tiles<32>(s, x, w, out, M, N, K);
  else launch_tiles<64>(s, x, w, out, M, N, K);
  return check_launch("psamd_linear");
}

}  // namespace psamd
