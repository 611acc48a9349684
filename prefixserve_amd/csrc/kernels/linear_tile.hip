// bfloat16 products of more than 128 tokens with what follows them in the same kernel, out[M,N] = x[M,K] * w[N,K]^T: the
// activation of a gated feed-forward, the rotation and the pages of a q/k/v projection, the sum into the float32 residual stream,
// or K-slices that the norm behind it adds up. tile_product.h has the loop.

#include <algorithm>

#include "api.h"
#include "common.h"
#include "linear_stream.h"
#include "tile_product.h"
#include "wide_tile.h"

namespace psamd {
namespace {

// What becomes of the sums: float32 K-slices, added into a float32 output, act(gate) * up in bfloat16, q/k/v. In the last
// two they are rounded to bfloat16 in front of what follows them, as the library leaves them to the kernels behind it: with its order
// of sums the results have its bits, and no router behind them sees another token.
constexpr int kTileSlices = 0, kTileAdd = 1, kTileGated = 2, kTileQkv = 3;

// A workgroup of WM x WN waves makes TM tokens x TN rows of w. GATED and QKV: a wave's rows of w are RN / 2 tiles of 16 columns (gate
// rows; first halves of rotation pairs) and then their partners (up rows; second halves), so that a lane holds both of a pair.
// Tiles are dealt out to the eight dies in stretches, the tiles of the same columns side by side, whose rows of w then stand in
// that die's L2. blockIdx.y is the K-slice.
template <int TM, int TN, int WM, int WN, int STAGES, int OCC, int FORM>
__global__ __launch_bounds__(64 * WM * WN, OCC) void linear_tile_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                        void* __restrict__ out, int M, int N, int K, int slice_steps,
                                                                        int row_tiles, int col_tiles, int act, QkvOut q) {
  constexpr int WV = WM * WN, RM = TM / WM / 16, RN = TN / WN / 16, WROWS = TN / WN, LA = TM / 8 / WV, LB = TN / 8 / WV;
  constexpr bool PAIRED = FORM == kTileGated || FORM == kTileQkv;
  constexpr int WCOLS = PAIRED ? WROWS / 2 : WROWS, COLS = PAIRED ? TN / 2 : TN;
  static_assert(LA * 8 * WV == TM && LB * 8 * WV == TN && (!PAIRED || RN % 2 == 0), "whole copies and pairs per wave");
  extern __shared__ __align__(16) unsigned char linear_tile_smem[];
  const int tiles = row_tiles * col_tiles, per_die = (tiles + 7) / 8;
  const int id = static_cast<int>(blockIdx.x & 7) * per_die + static_cast<int>(blockIdx.x >> 3);
  if (static_cast<int>(blockIdx.x >> 3) >= per_die || id >= tiles) return;       // uniform for the workgroup
  const int m0 = id % row_tiles * TM, n0 = id / row_tiles * COLS;                // QKV: n0 counts pairs
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4, wm = wave / WN * (TM / WM), wn = wave % WN;
  const int first = blockIdx.y * slice_steps, steps = min(slice_steps, K / 64 - first);
  const int half = FORM == kTileQkv ? q.d >> 1 : 1;
  auto pair_col = [&](int p) { return p / half * q.d + p % half; };              // QKV: the column of a pair's first half
  uint32_t a_off[LA], b_off[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i) {
    const int row = (wave * LA + i) * 8 + (lane >> 3);
    a_off[i] = static_cast<uint32_t>(min(m0 + row, M - 1)) * (2u * K) + 16u * tile_copy_piece(row, lane);
  }
#pragma unroll
  for (int i = 0; i < LB; ++i) {
    const int row = (wave * LB + i) * 8 + (lane >> 3);
    int col = n0 + row / WROWS * WCOLS + row % WROWS % WCOLS;
    const bool second = row % WROWS >= WCOLS;
    if (FORM == kTileQkv) col = pair_col(min(col, N / 2 - 1)) + (second ? half : 0);
    else col = min(col, N - 1) + (second ? N : 0);
    b_off[i] = static_cast<uint32_t>(col) * (2u * K) + 16u * tile_copy_piece(row, lane);
  }
  tile_f32x4 acc[RN][RM];
#pragma unroll
  for (int i = 0; i < RN; ++i)
#pragma unroll
    for (int j = 0; j < RM; ++j) acc[i][j] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
  tile_product<STAGES, TM, TN>(acc, linear_tile_smem, reinterpret_cast<const char*>(x) + static_cast<int64_t>(first) * 128,
                               reinterpret_cast<const char*>(w) + static_cast<int64_t>(first) * 128, a_off, b_off, wm, wn * WROWS, wave, lane,
                               steps, m0 + wm < M);
  auto pack = [](tile_f32x4 v) { return ushort4{float_to_bf16(v[0]), float_to_bf16(v[1]), float_to_bf16(v[2]), float_to_bf16(v[3])}; };
  auto rounded = [](tile_f32x4 v) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = bf16_to_float(float_to_bf16(v[e]));
    return v;
  };
#pragma unroll
  for (int j = 0; j < RM; ++j) {
    const int m = m0 + wm + 16 * j + r;
    if (m >= M) continue;
#pragma unroll
    for (int i = 0; i < WCOLS / 16; ++i) {
      const int n = n0 + wn * WCOLS + 16 * i + 4 * g;                            // this lane's four columns (pairs) of token m
      if (n >= (FORM == kTileQkv ? N / 2 : N)) continue;                         // N is a multiple of 16
      if constexpr (FORM == kTileQkv) {
        tile_f32x4 a = rounded(acc[i][j]), b = rounded(acc[(i + RN / 2) % RN][j]);
        const int head = n / half, p = n % half;                                 // half is a multiple of 8: four pairs of one head
        if (q.table != nullptr && head < q.hq + q.hkv) {
          const float4* cs = reinterpret_cast<const float4*>(q.table + static_cast<int64_t>(q.positions[m]) * half + p);
          const float4 c01 = cs[0], c23 = cs[1];
          const float c[4] = {c01.x, c01.z, c23.x, c23.z}, s[4] = {c01.y, c01.w, c23.y, c23.w};
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            const float lo = a[v] * c[v] - b[v] * s[v], hi = b[v] * c[v] + a[v] * s[v];
            a[v] = lo;
            b[v] = hi;
          }
        }
        const ushort4 lo = pack(a), hi = pack(b);
        bf16_t* o = static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + head * q.d + p;
        *reinterpret_cast<ushort4*>(o) = lo;
        *reinterpret_cast<ushort4*>(o + half) = hi;
        if (q.kv == nullptr || head < q.hq) continue;
        const int slot = q.write_slot[m], off = slot % kPage;
        bf16_t* page = q.kv + static_cast<int64_t>(slot / kPage) * (2LL * q.hkv * kPage * q.d);
        if (head < q.hq + q.hkv) {                                               // key row [16][D]
          bf16_t* k = page + (static_cast<int64_t>(head - q.hq) * kPage + off) * q.d + p;
          *reinterpret_cast<ushort4*>(k) = lo;
          *reinterpret_cast<ushort4*>(k + half) = hi;
        } else {                                                                 // value, transposed [D][16], behind the keys
          bf16_t* vp = page + (static_cast<int64_t>(head - q.hq) * q.d + p) * kPage + off;
          vp[0] = lo.x;
          vp[kPage] = lo.y;
          vp[2 * kPage] = lo.z;
          vp[3 * kPage] = lo.w;
          vp += half * kPage;
          vp[0] = hi.x;
          vp[kPage] = hi.y;
          vp[2 * kPage] = hi.z;
          vp[3 * kPage] = hi.w;
        }
      } else if constexpr (FORM == kTileGated) {
        tile_f32x4 v = rounded(acc[i][j]);
        const tile_f32x4 up = rounded(acc[(i + RN / 2) % RN][j]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = gate_act(v[e], act) * up[e];
        *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + n) = pack(v);
      } else {
        tile_f32x4* o = reinterpret_cast<tile_f32x4*>(static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n);
        *o = FORM == kTileAdd ? *o + acc[i][j] : acc[i][j];
      }
    }
  }
}

// The largest tiles (256 x 256; wide_tile.h has the loop): workgroups of four waves that walk their die's stretch of the tiles.
// ACT: the activation of the gated form (asked for number by number, it took 12 us a tile).
template <int FORM, int ACT>
struct DenseTiles {
  void* __restrict__ out;
  int M, N, K, row_tiles, to, at_once;
  const char* w;
  int cur, next_a, next_w, lane, wave;                 // tiles: multiplied, copied next

  static constexpr int kMinSteps = 2;                  // the tiles that are copied are counted apart from the one that is multiplied
  static constexpr int WROWS = kWideTile / 2, WCOLS = FORM == kTileGated ? WROWS / 2 : WROWS, COLS = 2 * WCOLS;
  // (What follows from the lane alone would be computed in front of all tiles and held through them, where no register is free.)
  __device__ __forceinline__ int own_lane() const {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  }
  __device__ __forceinline__ bool a_rows(uint32_t (&off)[8]) {
    if (next_a >= to) return false;
    const int lane = own_lane(), m0 = next_a % row_tiles * kWideTile;
    next_a += at_once;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      off[i] = wide_row(min(m0 + 64 * wave + 8 * i + (lane >> 3), M - 1), K) + wide_piece(8 * i + (lane >> 3), lane);
    return true;
  }
  // GATED: a lane's four columns of two neighbouring tiles of 16 stand side by side, 16 bytes of the output.
  __device__ __forceinline__ bool w_rows(uint32_t (&off)[8]) {
    if (next_w >= to) return false;
    const int lane = own_lane(), n0 = next_w / row_tiles * COLS;
    next_w += at_once;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = (wave * 8 + i) * 8 + (lane >> 3), in = row % WCOLS;
      const int c = FORM == kTileGated ? (in & ~31) + (in >> 2 & 3) * 8 + (in >> 4 & 1) * 4 + (in & 3) : in;
      const int col = min(n0 + row / WROWS * WCOLS + c, N - 1);
      off[i] = wide_row(FORM == kTileGated && row % WROWS >= WCOLS ? N + col : col, K) + wide_piece(8 * i + (lane >> 3), lane);
    }
    return true;
  }
  __device__ __forceinline__ int rows() const { return min(kWideTile, M - cur % row_tiles * kWideTile); }
  __device__ __forceinline__ void ahead() {}
  template <int RM>
  __device__ __forceinline__ bool finish(tile_f32x4 (&acc)[8][RM]) {
    const int lane = own_lane(), r = lane & 15, g = lane >> 4;
    const int c0 = cur / row_tiles * COLS + (wave & 1) * WCOLS, m0 = cur % row_tiles * kWideTile + (wave >> 1) * (16 * RM) + r;
#pragma unroll
    for (int j = 0; j < RM; ++j) {
      const int m = m0 + 16 * j;
      if (m >= M) continue;
#pragma unroll
      for (int i = 0; i < WCOLS / 16; i += FORM == kTileGated ? 2 : 1) {
        const int n = c0 + 16 * i + (FORM == kTileGated ? 8 : 4) * g;
        if (n >= N) continue;                          // N is a multiple of 16
        if constexpr (FORM == kTileGated) {
          union {
            bf16_t h[8];
            uint4 v;
          } res;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float gate = bf16_to_float(float_to_bf16(acc[i + e / 4][j][e % 4])), up = bf16_to_float(float_to_bf16(acc[(i + e / 4 + 4) % 8][j][e % 4]));
            res.h[e] = float_to_bf16(gate_act(gate, ACT) * up);
          }
          *reinterpret_cast<uint4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + n) = res.v;
        } else {
          *reinterpret_cast<tile_f32x4*>(static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n) = acc[i][j];
        }
        __builtin_amdgcn_sched_barrier(0);             // a few sums at a time leave the accumulator registers
      }
    }
    cur += at_once;
    return cur < to;
  }
};

template <int FORM, int ACT>
__global__ __launch_bounds__(kWideThreads, 1) void linear_wide_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                      void* __restrict__ out, int M, int N, int K, int slice_steps,
                                                                      int row_tiles, int col_tiles) {
  extern __shared__ __align__(16) unsigned char linear_wide_smem[];
  const int tiles = row_tiles * col_tiles, per_die = (tiles + 7) / 8, die = static_cast<int>(blockIdx.x & 7);
  const int64_t first = static_cast<int64_t>(blockIdx.y) * slice_steps;
  DenseTiles<FORM, ACT> work;
  work.out = out, work.M = M, work.N = N, work.K = K, work.row_tiles = row_tiles;
  work.to = min((die + 1) * per_die, tiles), work.at_once = static_cast<int>(gridDim.x >> 3);
  work.cur = work.next_a = work.next_w = die * per_die + static_cast<int>(blockIdx.x >> 3);
  work.lane = threadIdx.x & 63, work.wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  work.w = reinterpret_cast<const char*>(w) + first * 128;
  wide_tiles(work, reinterpret_cast<const char*>(x) + first * 128, linear_wide_smem, min(slice_steps, K / 64 - static_cast<int>(first)));
}

// Whether every slice of K has the steps that the largest tiles work with.
bool wide_takes(int K, int ksplit) {
  const int64_t steps = ceil_div(K / 64, ksplit);
  return K / 64 - (ksplit - 1) * steps >= DenseTiles<kTileSlices, 0>::kMinSteps;
}

// How many workgroups of the largest tiles a slice of K has, one a compute unit: each die's eighth of them walks the die's eighth of the
// slice's tiles. (What they take is counted in these rounds: 252 tiles of three slices, 33 of them on a die, are two, 516 tokens x 6,960 x 5,440 97 us where
// tiles of 192 x 128 take 65.)
int64_t wide_workgroups(int ksplit) { return std::max<int64_t>(8, 256 / ksplit / 8 * 8); }

template <int FORM, int ACT>
int launch_wide(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit) {
  if (!wide_takes(K, ksplit)) return fail("linear_tile: too few steps of k for the largest tiles");
  auto kernel = linear_wide_kernel<FORM, ACT>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kWideSmem) != hipSuccess)
    return fail("linear_tile: " + std::to_string(kWideSmem) + " bytes of LDS were refused");
  const int row_tiles = static_cast<int>(ceil_div(M, kWideTile)), col_tiles = static_cast<int>(ceil_div(N, FORM == kTileGated ? kWideTile / 2 : kWideTile));
  const int64_t most = 8 * ceil_div(static_cast<int64_t>(row_tiles) * col_tiles, 8);
  kernel<<<dim3(static_cast<unsigned>(std::min(most, wide_workgroups(ksplit))), static_cast<unsigned>(ksplit)), dim3(kWideThreads), kWideSmem, s>>>(
      static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), out, M, N, K, static_cast<int>(ceil_div(K / 64, ksplit)), row_tiles, col_tiles);
  return check_launch("linear_tile");
}

template <int TM, int TN, int WM, int WN, int STAGES, int OCC, int FORM>
int launch_tile(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act, const QkvOut& q) {
  constexpr size_t smem = static_cast<size_t>(STAGES) * (TM + TN) * 128;
  constexpr bool PAIRED = FORM == kTileGated || FORM == kTileQkv;
  auto kernel = linear_tile_kernel<TM, TN, WM, WN, STAGES, OCC, FORM>;
  if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("linear_tile: " + std::to_string(smem) + " bytes of LDS were refused");
  const int row_tiles = static_cast<int>(ceil_div(M, TM));
  const int col_tiles = static_cast<int>(ceil_div(FORM == kTileQkv ? N / 2 : N, PAIRED ? TN / 2 : TN));
  const int slice_steps = static_cast<int>(ceil_div(K / 64, ksplit));
  kernel<<<dim3(static_cast<unsigned>(8 * ceil_div(static_cast<int64_t>(row_tiles) * col_tiles, 8)), static_cast<unsigned>(ksplit)),
           dim3(64 * WM * WN), smem, s>>>(static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), out, M, N, K, slice_steps,
                                          row_tiles, col_tiles, act, q);
  return check_launch("linear_tile");
}

// The forms that add into a float32 output and that write q/k/v come in the two smallest shapes alone: the others were never the fastest.
constexpr bool tile_shape_built(int form, int shape) { return shape >= 3 || form == kTileSlices || form == kTileGated; }
constexpr int kTileShapeCount = 5;

template <int FORM>
int launch_form(hipStream_t s, int shape, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                const QkvOut& q = {}) {
  if constexpr (tile_shape_built(FORM, 0)) {
    if (shape == 0 && !wide_takes(K, ksplit)) shape = 3;       // the same sums
    if (shape == 0) {
      if constexpr (FORM == kTileGated) {
        if (act == 1) return launch_wide<FORM, 1>(s, x, w, out, M, N, K, ksplit);
        if (act == 2) return launch_wide<FORM, 2>(s, x, w, out, M, N, K, ksplit);
      }
      return launch_wide<FORM, 0>(s, x, w, out, M, N, K, ksplit);
    }
    if (shape == 1) return launch_tile<192, 128, 2, 2, 2, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
    if (shape == 2) return launch_tile<192, 128, 2, 4, 3, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  }
  if (shape == 3) return launch_tile<128, 128, 2, 4, 4, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  if (shape == 4) return launch_tile<64, 128, 2, 2, 3, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  return fail("linear_tile: this form has no such shape");
}

// The shapes above and what they take, in us: `step` for 64 k in a round that fills the chip (`at_once` workgroups a compute unit),
// `half_step` where two share a unit and the round has only one for each, `round` beside the steps; a million bytes of w on their way
// from memory, and each time another row of tiles asks for them; `start` once. Fitted, as the forms below, to the device's time
// of 15,000 kernels, with weights that lay in no cache, as in a step: 130 to 8,192 tokens, 56 products from 64 x 64 to 2 x 28,672 x
// 8,192. One in ten is off by 12% or more, and one in ten of those near the library's time by 9% or more. The largest shape's were fitted again to its loop of
// four waves, with SiLU: over 260 gated products 0.92 to 1.12 of the measured time but for one in ten at either end, over 163 for the stream 0.98 on average.
struct TileShape {
  int rows, cols, at_once;
  double step, half_step, round, weights, reads, start;
};
constexpr TileShape kTileShapes[kTileShapeCount] = {
    {256, 256, 1, 0.956, 0.0, 4.21, 0.0, 0.0355, 3.66},       // asks for the fewest bytes a product; four waves that walk its tiles
    {192, 128, 2, 1.127, 0.841, 0.27, 0.032, 0.023, 5.06},    // two on a unit: one's loop beside the other's beginning and end
    {192, 128, 1, 0.627, 0.0, 2.71, 0.023, 0.027, 2.78},      // three steps under way, for one round
    {128, 128, 1, 0.469, 0.0, 2.24, 0.011, 0.028, 2.91},      // four
    {64, 128, 2, 0.606, 0.373, 0.26, 0.066, 0.011, 4.01},
};
// What a form takes beside that (`start`, and for a million numbers that it leaves), and what the library and the kernel that is then
// needed behind it take: once, for 10^9 operations, a million bytes of w, a million results and 64 k.
struct TileForm {
  double start, numbers, library, library_gflop, library_mb, library_numbers, library_step;
};
constexpr TileForm kStreamForm{2.83, 1.517, 6.99, 0.787, 0.145, 2.709, 0.090};   // both with the norm that adds up
constexpr TileForm kGatedForm{0.0, 0.703, 6.27, 0.398, 0.104, 2.620, 0.194};
constexpr TileForm kQkvForm{0.0, 1.504, 7.37, 0.524, 0.206, 2.026, 0.132};

// What a round of the largest tiles takes longer with GELU than with SiLU, for which the table holds: its activations run with no matrix
// instruction beside them (7.3 to 10.5 us over 48 products; ReLU takes 3 less than SiLU), less what the activation kernel behind the library's
// product takes longer too. Anything from 5.5 to 7.5 decides alike over those products. Without it, gated products with GELU ran in these tiles where
// something else is the faster (us, the largest tiles / what runs now): 2 x 8,192 x 2,048 at 640 tokens 54.9 / 47.0, 2 x 6,144 x 1,024 at 640 37.2 /
// 26.8, 2 x 2,816 x 1,024 at 2,048 35.6 / 31.4, 2 x 8,192 x 2,048 at 4,096 235 / 223; 2 x 8,192 x 3,072 at 900 keeps them, 81 / 97, and 2 x 8,192 x 2,048 at 2,048,
// which takes 118 / 118 one after the other and 136 to 141 / 130 to 137 among a step's other kernels. Over 36 products with GELU 0.98 of the time that it is without this;
// the library's fit, on its fast side, keeps some that these tiles do faster (2 x 11,008 x 1,536 at 2,048 tokens 143 / 165, at 4,096 290 / 300).
constexpr double kWideGelu = 6.5;
// By what part products for the stream must be faster in the largest tiles than in smaller ones by the table, whose figures are good to that: of
// 129 products that it would have do otherwise by any lead, 38 were slower by more than 2% (262 tokens x 6,944 x 7,552 54.0 -> 60.7 us) and 44 faster; with this
// one 3 are slower (at most 9%) and the sum of the times is the same; of 110 others that run in the largest tiles by it, at 0.88 of the time, 6 are slower, by 2 to 7%. Two slices of them, which are only ever chosen close to the library, lost to it by 3 to 8% in
// all of four products (555 x 7,552 x 5,696 71.4 / 77.1) and are not taken.
constexpr double kWideLead = 1.06;

constexpr int kTileMinTokens = 129;         // fewer: linear_stream.hip
constexpr int kStreamMaxTokens = 1023;      // above, the library's product adds into the stream itself: tiles 0.97 to 1.32 of its time
constexpr int64_t kStreamMaxNumbers = 4200000;   // tokens x columns, and columns: above, the library has work for the whole chip without
constexpr int kStreamMaxColumns = 8192;          // slices (237 tokens x 11,008 x 5,760 91.8 / 114 us)
constexpr int64_t kMostGatedWeights = 70000000;  // above, the library was the faster from 200 tokens on and 2 to 10% slower below
constexpr int kThirdsMaxK = 16384;          // three slices of a K of 18,944 took 1.65 times the table's time (3,584 columns: 384 tokens 121 us, four 73)
constexpr int kMostSliceRows = 4608;        // K-slices x tokens that there is room for

struct TilePlan {
  int shape = -1, ksplit = 1;               // shape -1: the library; of a product for the stream ksplit 1 adds into it
};

// The shape (and K-slices) of the least time by the table, if that is less than what the library takes by it. The library's figures are
// fitted with errors towards more counted up to twice and lowered by up to 3%: its times of neighbouring sizes differ by a tenth and more, and no
// product that it does faster should be taken from it. Of 220 products for the stream, 220 gated ones with SiLU and 220 with GELU, drawn at random (129 to 1,023
// and 4,096 tokens), 120, 113 and 92 run in tiles; those of them that take the library 30 us or more (36, 27, 23) at 0.73, 0.67 and 0.77 of its time; three,
// none and two are slower by more than 2%, at most by 16% (387 tokens x 2,640 x 10,880 59.5 / 69.1). Of q/k/v products, whose shapes are older, 0.78 to 0.83. us,
// the library and what follows > the tiles, or (the best tiles) where it stays with the library:
//   tokens                        150          256          384          535          640          900          1,023        1,531         2,048
//   q/k/v 3,072 x 2,048           16.4 (18.9)  17.5 (19.6)  19.3 (20.1)  21.7 > 20.3  22.4 > 21.1  28.4 (24.7)  30.8 (26.9)  33.4 (43.2)   38.6 (51.3)
//   q/k/v 6,144 x 4,096           43.3 (33.3)  46.6 > 35.1  42.7 (38.8)  47.7 (44.6)  49.4 > 45.8  59.9 (81.0)  63.7 (86.2)  91.3 (127)    99.6 (138)
//   gated 2 x 1,024 x 2,048       14.9 (17.3)  15.0 (17.9)  16.0 (17.9)  18.4 (17.5)  18.7 (18.0)  20.1 > 17.9  21.2 > 18.7  26.4 (23.1)   28.6 > 24.4
//   gated 2 x 8,192 x 2,048       29.8 > 22.1  33.2 > 25.6  35.4 > 30.2  45.2 (43.8)  46.7 > 45.0  62.8 > 52.4  65.0 > 54.0  98.0 (96.2)   118 > 104
//   gated 2 x 14,336 x 4,096      59.7 (57.0)  71.5 (83.3)  84.7 (89.7)  133 (144)    139 (159)    190 (174)    197 (179)    280 (274)     364 (371)
//   with the norm 2,048 x 2,048   15.2 > 12.4  15.5 > 14.7  16.9 (17.2)  19.1 (19.6)  20.1 (20.2)  22.7 (22.7)  24.0 (23.7)
//   2,048 x 8,192                 29.5 > 19.3  30.4 > 22.9  36.6 > 27.5  46.7 > 34.0  47.3 > 36.6  50.5 > 45.0  54.8 > 50.3  69.2 (82.9)   83.3 (93.6)
//   4,096 x 4,096                 26.0 > 20.1  27.2 > 23.5  30.7 > 28.5  41.5 (37.9)  41.6 > 38.6  46.6 (44.7)  49.7 > 47.9  65.3 (67.1)   78.1 (102)
//   4,096 x 14,336                62.4 > 38.3  66.8 > 50.9  85.4 > 61.4  114 > 88.2   117 > 88.5   125 > 103    138 > 108    192 (197)     236 (301)
// (From 1,024 tokens on the tiles add into the stream.) With four waves of 128 x 128 in the largest shape instead of eight of 128 x 64 that began each tile
// anew (both sides on one card): gated 2 x 8,192 x 2,048 at 2,048 tokens 122 by the library and the activation -> 110, 2 x 4,096 x 2,048 63 -> 56 (at 1,531
// 52 -> 48), 2 x 2,816 x 1,024 43 -> 29, 2 x 8,192 x 3,072 172 -> 153; with the norm 4,096 x 14,336 at 767 tokens 105 -> 97, 4,096 x 11,008 at 640 81 -> 73. 2 x 14,336 x
// 4,096 would gain 9% at 900 and 1,023 tokens and 2% at 1,531, and lose 2% at 2,048 and 15% at 640: left to the library. In bfloat16 for the other norms the tiles had no lead: 2,048 x 2,048 15.1 / 19.0 at
// 130 tokens, 19.3 / 21.1 at 535, 34.8 / 34.9 at 2,048; such products are the library's.
TilePlan tile_plan(int form, int M, int N, int K, int act = 0) {
  const bool stream = form == kTileSlices || form == kTileAdd;
  const int64_t rows = form == kTileGated ? 2LL * N : N;
  if (stream && (M > kStreamMaxTokens || N > kStreamMaxColumns || static_cast<int64_t>(M) * N > kStreamMaxNumbers)) return TilePlan{};
  if (form == kTileGated && rows * K > kMostGatedWeights) return TilePlan{};
  const TileForm& f = stream ? kStreamForm : (form == kTileGated ? kGatedForm : kQkvForm);
  const double mb = 2e-6 * rows * K, numbers = 1e-6 * M * N;
  double least = f.library + f.library_gflop * 1e-3 * M * mb + f.library_mb * mb + f.library_numbers * numbers + f.library_step * (K / 64);
  TilePlan plan;
  for (int shape : {1, 2, 3, 4, 0}) {
    const TileShape& t = kTileShapes[shape];
    for (int slices : {1, 2, 3, 4, 6, 8}) {
      if (slices % 3 == 0 && K > kThirdsMaxK) continue;
      if (slices > 1 && (!stream || K / 64 < 2 * slices || static_cast<int64_t>(slices) * M > kMostSliceRows)) break;
      const int64_t steps = ceil_div(K / 64, slices);
      if (ceil_div(K / 64, steps) != slices || !tile_shape_built(stream && slices == 1 ? kTileAdd : form, shape)) continue;
      if (shape == 0 && (!wide_takes(K, slices) || (stream && slices == 2))) continue;
      const int64_t row_tiles = ceil_div(M, t.rows), groups = row_tiles * ceil_div(rows, t.cols) * slices, at_once = 256 * t.at_once;
      const int64_t left = groups % at_once;
      const bool half = t.at_once == 2 && left > 0 && left <= 256;
      const int64_t rounds = shape == 0 ? ceil_div(ceil_div(groups / slices, 8), wide_workgroups(slices) / 8)
                                        : groups / at_once + (left > 0 && !half ? 1 : 0);
      const double full = static_cast<double>(rounds);
      const double time = t.start + f.start + full * (steps * t.step + t.round) + (half ? steps * t.half_step : 0.0) +
                          mb * (t.weights + t.reads * row_tiles) + f.numbers * numbers * slices +
                          (form == kTileGated && shape == 0 && act == 2 ? full * kWideGelu : 0.0);
      if ((shape == 0 && stream && plan.shape > 0 ? kWideLead * time : time) < least) {
        least = time;
        plan = TilePlan{shape, slices};
      }
    }
  }
  return plan;
}

bool tile_takes(const void* x, const void* w, const void* out, int M, int N, int rows, int K) {
  return M >= kTileMinTokens && N > 0 && N % 16 == 0 && K >= 64 && K % 64 == 0 && 2LL * M * K < (1LL << 32) && 2LL * rows * K < (1LL << 32) &&
         (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
}

}  // namespace
}  // namespace psamd

using namespace psamd;

extern "C" {

int psamd_linear_tile_slices(const void* x, const void* w, int M, int n_out, int K) {
  if (!tile_takes(x, w, nullptr, M, n_out, n_out, K)) return -1;
  const TilePlan plan = tile_plan(kTileSlices, M, n_out, K);
  return plan.shape < 0 ? -1 : (plan.ksplit == 1 ? 0 : plan.ksplit);
}

int psamd_linear_tile_slice_rows(int n_out, int K) {
  int most = 0;
  if (n_out <= 0 || n_out % 16 != 0 || K < 64 || K % 64 != 0) return 0;
  for (int M = kTileMinTokens; M <= kStreamMaxTokens; ++M)
    if (const TilePlan plan = tile_plan(kTileSlices, M, n_out, K); plan.shape >= 0 && plan.ksplit > 1) most = max(most, plan.ksplit * M);
  return most;
}

int psamd_linear_tile_plan(int form, int M, int n_out, int K, int activation) {
  if (form < kTileSlices || form > kTileQkv || n_out > INT32_MAX / 2 ||
      !tile_takes(nullptr, nullptr, nullptr, M, n_out, form == kTileGated ? 2 * n_out : n_out, K))
    return -1;
  const TilePlan plan = tile_plan(form, M, n_out, K, activation);
  return plan.shape < 0 ? -1 : 16 * plan.shape + plan.ksplit;
}

int psamd_linear_tile_stream(void* stream, const void* x, const void* w, float* out, int M, int n_out, int K) {
  PSAMD_REQUIRE(tile_takes(x, w, out, M, n_out, n_out, K), "operands that psamd_linear_tile_slices does not take");
  const TilePlan plan = tile_plan(kTileSlices, M, n_out, K);
  PSAMD_REQUIRE(plan.shape >= 0, "psamd_linear_tile_slices leaves this product to the library");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (plan.ksplit == 1) return launch_form<kTileAdd>(s, plan.shape, x, w, out, M, n_out, K, 1, 0);
  return launch_form<kTileSlices>(s, plan.shape, x, w, out, M, n_out, K, plan.ksplit, 0);
}

int psamd_linear_tile_gated(void* stream, const void* x, const void* w, void* out, int M, int n_out, int K, int activation) {
  PSAMD_REQUIRE(activation >= 0 && activation <= 2, "activation 0 (silu), 1 (relu) or 2 (gelu)");
  if (!tile_takes(x, w, out, M, n_out, 2 * n_out, K)) return 2;
  const TilePlan plan = tile_plan(kTileGated, M, n_out, K, activation);
  if (plan.shape < 0) return 2;
  return launch_form<kTileGated>(static_cast<hipStream_t>(stream), plan.shape, x, w, out, M, n_out, K, 1, activation);
}

int psamd_linear_tile_qkv(void* stream, const void* x, const void* w, void* qkv_out, int M, int K, int hq, int hkv, int head_dim,
                          const int32_t* positions, const float* table, void* kv, const int32_t* write_slot) {
  PSAMD_REQUIRE(hq > 0 && hkv > 0 && head_dim > 0 && positions != nullptr, "bad sizes");
  PSAMD_REQUIRE(kv == nullptr || write_slot != nullptr, "pages come with their slots");
  const int64_t rows = (static_cast<int64_t>(hq) + 2LL * hkv) * head_dim;
  if (head_dim % 16 != 0 || rows > INT32_MAX || reinterpret_cast<uintptr_t>(table) % 16 != 0 ||
      !tile_takes(x, w, qkv_out, M, static_cast<int>(rows), static_cast<int>(rows), K))
    return 2;
  const TilePlan plan = tile_plan(kTileQkv, M, static_cast<int>(rows), K);
  if (plan.shape < 0) return 2;
  const QkvOut q{hq, hkv, head_dim, positions, reinterpret_cast<const float2*>(table), static_cast<bf16_t*>(kv), write_slot};
  return launch_form<kTileQkv>(static_cast<hipStream_t>(stream), plan.shape, x, w, qkv_out, M, static_cast<int>(rows), K, 1, 0, q);
}

int psamd_linear_tile_shaped(void* stream, int form, int shape, int ksplit, const void* x, const void* w, void* out, int M, int n_out, int K,
                             int activation, int hq, int hkv, int head_dim, const int32_t* positions, const float* table, void* kv,
                             const int32_t* write_slot) {
  PSAMD_REQUIRE(form >= kTileSlices && form <= kTileQkv && shape >= 0 && shape < kTileShapeCount && tile_shape_built(form, shape),
                "this form has no such shape");
  PSAMD_REQUIRE(activation >= 0 && activation <= 2, "activation 0 (silu), 1 (relu) or 2 (gelu)");
  PSAMD_REQUIRE(n_out > 0 && n_out <= INT32_MAX / 2 && tile_takes(x, w, out, M, n_out, form == kTileGated ? 2 * n_out : n_out, K),
                "operands that the tiles do not take");
  PSAMD_REQUIRE(ksplit >= 1 && ksplit <= K / 64 && (ksplit == 1 || form == kTileSlices) &&
                    ceil_div(K / 64, ceil_div(K / 64, ksplit)) == ksplit, "slices with whole steps of 64 k in each");
  QkvOut q{};
  if (form == kTileQkv) {
    PSAMD_REQUIRE(hq > 0 && hkv > 0 && head_dim > 0 && head_dim % 16 == 0 && (static_cast<int64_t>(hq) + 2LL * hkv) * head_dim == n_out &&
                      positions != nullptr && reinterpret_cast<uintptr_t>(table) % 16 == 0 && (kv == nullptr || write_slot != nullptr),
                  "bad sizes");
    q = QkvOut{hq, hkv, head_dim, positions, reinterpret_cast<const float2*>(table), static_cast<bf16_t*>(kv), write_slot};
  }
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (form == kTileSlices) return launch_form<kTileSlices>(s, shape, x, w, out, M, n_out, K, ksplit, 0);
  if (form == kTileAdd) return launch_form<kTileAdd>(s, shape, x, w, out, M, n_out, K, 1, 0);
  if (form == kTileGated) return launch_form<kTileGated>(s, shape, x, w, out, M, n_out, K, 1, activation);
  return launch_form<kTileQkv>(s, shape, x, w, out, M, n_out, K, 1, 0, q);
}

}  // extern "C"
