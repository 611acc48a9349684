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

#include <algorithm>

#include "api.h"
#include "common.h"
#include "linear_f32.h"
#include "tile_product.h"

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

// A workgroup of WM x WN waves makes BN columns x BM tokens, both operands through LDS 64 k, a chain, at a time: the next chain's rows are copied
// there while this one is multiplied (copy_to_lds: no register holds them), a wave's operands are read 32 k ahead of the matrix
// instructions, and a chain's first instruction takes zero for its sums. A row of LDS is 256 bytes, its sixteen 16-byte pieces exchanged by
// the row's number, so that the 16 rows a read touches lie on all banks. Tiles that share rows of w run on one die (its L2 serves
// them): die d takes the d-th eighth of the tiles, tokens fastest. Bound by the matrix instructions, whose rate on this card is 150 TFLOP/s (a loop of
// them and nothing else); what is left of it goes to the wait for a chain's first operands behind the barrier, which the other
// workgroups of the compute unit fill. us with weights that are in no cache, with rows on their way in registers and operands read as they are needed / so, both
// on a card that copies 1 GiB at 5.16 TB/s: 600 tokens x 16,384 columns x 2,048 411 / 346 (116 TFLOP/s), 600 x 3,072 86 / 73, 600 x 2,048 71 / 56, 600 x 2,048 x
// 8,192 266 / 209, 300 x 2,048 50 / 34, 150 x 2,048 x 8,192 127 / 90, 2,048 x 16,384 1,301 / 1,093 (126). A third buffer costs workgroups and is slower everywhere
// (600 x 2,048 65).
template <int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_f32_kernel(const float* __restrict__ x, const float* __restrict__ w,
                                                                float* __restrict__ out, int M, int N, int K, int m_tiles, int tiles,
                                                                int per_die) {
  constexpr int W = WM * WN, RT = BN / 16 / WN, MT = BM / 16 / WM, LW = BN / 4 / W, LX = BM / 4 / W, STAGE = (BM + BN) * 256;
  static_assert(LW * 4 * W == BN && LX * 4 * W == BM && RT * 16 * WN == BN && MT * 16 * WM == BM, "whole copies and tiles per wave");
  __shared__ __align__(16) unsigned char buffers[2 * STAGE];           // 2 x [BN rows of w, BM of x][64 k]
  const int local = static_cast<int>(blockIdx.x >> 3), tile = static_cast<int>(blockIdx.x & 7) * per_die + local;
  if (local >= per_die || tile >= tiles) return;
  const int n0 = tile / m_tiles * BN, m0 = tile % m_tiles * BM;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int wn = wave % WN * (RT * 16), wm = wave / WN * (MT * 16);    // this wave's part of the tile
  const char* wb = reinterpret_cast<const char*>(w + static_cast<int64_t>(n0) * K);
  const char* xb = reinterpret_cast<const char*>(x + static_cast<int64_t>(m0) * K);
  uint32_t w_off[LW], x_off[LX];                                       // copy i of this wave brings four rows; a lane its 16 bytes of them
  const int row0 = lane >> 4, last_w = N - 1 - n0, last_x = M - 1 - m0;
  auto piece = [&](int row) { return (lane & 15) ^ (row & 15); };
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (wave * LW + i) * 4 + row0;
    w_off[i] = static_cast<uint32_t>(min(row, last_w)) * (4u * K) + 16u * piece(row);
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int row = (wave * LX + i) * 4 + row0;
    x_off[i] = static_cast<uint32_t>(min(row, last_x)) * (4u * K) + 16u * piece(row);
  }
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)buffers));
  auto copy = [&](int t, int to) {
#pragma unroll
    for (int i = 0; i < LW; ++i) copy_to_lds(base + to + (wave * LW + i) * 1024, w_off[i], wb + static_cast<int64_t>(t) * 256);
#pragma unroll
    for (int i = 0; i < LX; ++i) copy_to_lds(base + to + BN * 256 + (wave * LX + i) * 1024, x_off[i], xb + static_cast<int64_t>(t) * 256);
  };
  f32x4 part[RT][MT], total[RT][MT];                                   // of the segment, of all of K
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) part[rt][mt] = total[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int whole = K / kChain, chains = (K + kChain - 1) / kChain;
  auto multiply = [&](int t, int at) {
    f32x4 a[4][RT], b[4][MT], acc[RT][MT];
    auto operands = [&](int q) {                                       // of k = 16 q .. 16 q + 15
      const unsigned char* from = buffers + at + r * 256 + 16 * ((4 * q + g) ^ r);
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) a[q][rt] = *reinterpret_cast<const f32x4*>(from + (wn + 16 * rt) * 256);
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) b[q][mt] = *reinterpret_cast<const f32x4*>(from + (BN + wm + 16 * mt) * 256);
    };
    operands(0);
    operands(1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      if (q < 2) operands(q + 2);
      __builtin_amdgcn_sched_barrier(0);
      // One k of every tile after the other: neighbouring instructions do not wait for each other's sums.
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt)
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            acc[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][rt][i], b[q][mt][i], q == 0 && i == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[rt][mt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
    constexpr int kChains = kSegment / kChain;
    const bool ends = t % kChains == kChains - 1 || t + 1 == chains;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        part[rt][mt] = (t % kChains == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : part[rt][mt]) + acc[rt][mt];
        if (ends) total[rt][mt] += part[rt][mt];
      }
  };
  if (whole > 0) copy(0, 0);
  int at = 0;
  for (int t = 0; t < whole; ++t, at ^= STAGE) {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(wait_for_copies(0));
    __builtin_amdgcn_s_barrier();                                      // chain t has arrived, and everybody has read the one before
    __builtin_amdgcn_sched_barrier(0);
    if (t + 1 < whole) copy(t + 1, at ^ STAGE);
    asm volatile("" ::: "memory");                                     // what the copies brought is read behind the barrier
    __builtin_amdgcn_sched_barrier(0);
    multiply(t, at);
  }
  if (whole < chains) {                                                // the last chain in part: zeros behind K, a multiple of 4
    auto put = [&](int to, const char* from, uint32_t off, int row) {
      const int k = kChain * whole + 4 * piece(row);
      *reinterpret_cast<f32x4*>(buffers + at + to + lane * 16) =
          k < K ? *reinterpret_cast<const f32x4*>(from + static_cast<int64_t>(whole) * 256 + off) : f32x4{0.f, 0.f, 0.f, 0.f};
    };
#pragma unroll
    for (int i = 0; i < LW; ++i) put((wave * LW + i) * 1024, wb, w_off[i], (wave * LW + i) * 4 + row0);
#pragma unroll
    for (int i = 0; i < LX; ++i) put(BN * 256 + (wave * LX + i) * 1024, xb, x_off[i], (wave * LX + i) * 4 + row0);
    __syncthreads();                                                   // (this buffer was last read in front of the barrier before)
    multiply(whole, at);
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

template <int BM, int BN, int WM, int WN>
static void launch_tiles(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const int m_tiles = static_cast<int>(ceil_div(M, BM)), tiles = static_cast<int>(ceil_div(N, BN)) * m_tiles;
  const int per_die = static_cast<int>(ceil_div(tiles, 8));
  gemm_f32_kernel<BM, BN, WM, WN><<<dim3(static_cast<unsigned>(8 * per_die)), dim3(64 * WM * WN), 0, s>>>(x, w, out, M, N, K, m_tiles, tiles, per_die);
}

bool linear_f32_takes(const void* x, const void* w, int64_t M, int N, int K) {
  const uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w);
  return K % 4 == 0 && bits % 16 == 0 && M <= (1 << 24) && K <= (1 << 23) &&
         ceil_div(M, 32) * ceil_div(N, 32) < (1LL << 31) - 8;              // a tile's offsets of 32 bits
}

// Which kernel, us at one MI355X (K = 2,048 unless given; every one gives the same bits):
//  * K of one segment, and up to 16 tokens or so few tiles as below: a wave per chain.
//  * up to 8 tokens, or 16 where the columns are fewer than 16,384: 16 rows of w per workgroup. 2,048 columns at 8 tokens 13
//    (tiles of 32 tokens 36), 128,256 at 1 token 187 (234); at 16 tokens 282 (224).
//  * tiles of 32 tokens x 64 columns for a quarter of the compute units at most: the same kernel with 32 tokens. 64 tokens x 2,048 columns 16 (tiles 17),
//    33 x 2,048 x 8,192 50 (79), 24 x 3,072 16 (24).
//  * tiles: what the compute unit with the most of them takes, in columns x tokens over the share of its rate that a shape gets from as many
//    workgroups as it has. 600 x 16,384 in tiles of 64 x 64 / 32 x 64 / 32 x 32 346 / 335 / 366, 2,048 x 16,384 1,093 / 1,117 / 1,281, 600 x 3,072 73 / 78 / 80, 600 x 2,048
//    71 / 56 / 60, x 8,192 271 / 210 / 231, 300 x 2,048 40 / 42 / 34, 150 x 2,048 x 8,192 153 / 100 / 90, 17 x 16,384 45 / 34 / 32, 128 x 3,072 41 / 28 / 25.
int launch_linear_f32(hipStream_t s, const float* x, const float* w, float* out, int M, int N, int K) {
  const int64_t tiles32 = ceil_div(M, 32) * ceil_div(N, 64);
  auto cost = [&](int bm, int bn, double share) {
    const int64_t each = ceil_div(ceil_div(M, bm) * ceil_div(N, bn), 256);
    return static_cast<double>(each) * bm * bn / (share * (bm * bn > 2048 || each > 2 ? 1.0 : (each == 2 ? 0.85 : 0.62)));
  };
  if (K <= kSegment && M <= 16) launch_rows_short<1>(s, x, w, out, M, N, K);
  else if (K <= kSegment && tiles32 <= 128) launch_rows_short<2>(s, x, w, out, M, N, K);
  else if (M <= 8 || (M <= 16 && N < 16384)) launch_rows<1>(s, x, w, out, M, N, K);
  else if (tiles32 <= 64) launch_rows<2>(s, x, w, out, M, N, K);
  else if (cost(64, 64, 1.0) <= std::min(cost(32, 64, 0.94), cost(32, 32, 0.78))) launch_tiles<64, 64, 2, 4>(s, x, w, out, M, N, K);
  else if (cost(32, 64, 0.94) <= cost(32, 32, 0.78)) launch_tiles<32, 64, 1, 4>(s, x, w, out, M, N, K);
  else launch_tiles<32, 32, 2, 2>(s, x, w, out, M, N, K);
  return check_launch("psamd_linear");
}

}  // namespace psamd
