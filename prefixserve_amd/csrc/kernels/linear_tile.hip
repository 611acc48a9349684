// bfloat16 products of more than 128 tokens with what follows them in the same kernel, out[M,N] = x[M,K] * w[N,K]^T: the
// activation of a gated feed-forward, the rotation and the pages of a q/k/v projection, the sum into the float32 residual stream,
// or K-slices that the norm behind it adds up. tile_product.h has the loop.

#include <algorithm>
#include <iterator>

#include "api.h"
#include "common.h"
#include "linear_stream.h"
#include "tile_product.h"

namespace psamd {
namespace {

// What becomes of the sums: float32 K-slices, added into a float32 output, bfloat16, act(gate) * up in bfloat16, q/k/v. In the last
// two they are rounded to bfloat16 in front of what follows them, as the library leaves them to the kernels behind it: with its order
// of sums the results have its bits, and no router behind them sees another token.
constexpr int kTileSlices = 0, kTileAdd = 1, kTilePlain = 2, kTileGated = 3, kTileQkv = 4;

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
      } else if constexpr (FORM == kTilePlain) {
        *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + n) = pack(acc[i][j]);
      } else {
        tile_f32x4* o = reinterpret_cast<tile_f32x4*>(static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n);
        *o = FORM == kTileAdd ? *o + acc[i][j] : acc[i][j];
      }
    }
  }
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

template <int FORM>
int launch_form(hipStream_t s, int shape, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                const QkvOut& q = {}) {
  switch (shape) {
    case 0: return launch_tile<256, 256, 2, 4, 2, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
    case 1: return launch_tile<192, 128, 2, 2, 2, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
    case 2: return launch_tile<192, 128, 2, 4, 3, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
    case 3: return launch_tile<128, 128, 2, 4, 4, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
    default: return launch_tile<64, 128, 2, 2, 3, 2, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  }
}

// The shapes above and what they take, in us: `full` for a step of 64 k in a round that fills the chip (`at_once` workgroups a compute
// unit), `half` where two share a unit and the round has only one for each; `round` and `half_round` beside the steps, `start` once, and
// a million bytes of sums in 32 bits (to memory and back through the norm) or of bfloat16 (to memory).
struct TileShape {
  int rows, cols, at_once;
  double full, half, round, half_round, start, per_mb_f32, per_mb_bf16;
};
constexpr TileShape kTileShapes[] = {
    {256, 256, 1, 1.332, 0.0, 4.05, 0.0, 5.65, 0.163, 0.90},   // asks for the fewest bytes a product
    {192, 128, 2, 1.208, 0.86, 0.22, 0.0, 3.63, 0.151, 0.81},  // two on a unit: one's loop beside the other's beginning and end
    {192, 128, 1, 0.637, 0.0, 2.46, 0.0, 2.62, 0.159, 1.06},   // three steps under way, for one round
    {128, 128, 1, 0.495, 0.0, 1.21, 0.0, 2.58, 0.235, 1.13},   // four
    {64, 128, 2, 0.639, 0.302, 0.0, 4.82, 1.12, 0.287, 0.82},
};
constexpr int kMostSliceRows = 4608;   // K-slices x tokens that there is room for
constexpr int kAddMinTokens = 1024;    // from here on a product for the stream is added into it and leaves no slices, as the library's is

struct TilePlan {
  int shape = -1, ksplit = 1;
  bool add = false;
};

// The shape (and K-slices) of the least time by the table, if that is under what the library and the kernels that are then needed
// behind it take (within 10% of 80 measured products of 130 to 2,048 tokens; the table within 7%). Over those products, from
// 3,072 x 2,048 to 2 x 14,336 x 4,096, the choice is 17 to 18% under the library on average and 1% over the better of the two. us,
// library and what follows / here:
//   tokens                                    150          256          384          535          1,000        1,531        2,048
//   q/k/v 3,072 x 2,048                       32.0 / 17.7  26.0 / 17.6  27.1 / 18.1  26.7 / 18.8  29.4 / 26.6  33.6         38.1
//   q/k/v 6,144 x 4,096                       50.6 / 31.8  34.9 / 32.4  38.7 / 41.6  47.8 / 42.7  61.9         88.5         94.6
//   gated 2 x 8,192 x 2,048                   31.1 / 22.4  33.9 / 26.0  36.1 / 31.1  46.3         74.7 / 64.0  99.1         120
//   into the stream, norm incl. 2,048 x 2,048 28.6 / 18.2  24.9 / 18.0  25.1 / 18.8  25.5 / 19.6  25.4 / 21.8  29.6 / 30.7  33.5 / 32.9
//   2,048 x 8,192                             30.5 / 22.5  31.2 / 25.1  37.6 / 28.7  47.2 / 36.0  57.1 / 51.0  68.5 / 64.9  79.2
//   4,096 x 14,336                            62.0 / 38.7  78.8 / 53.6  83.9 / 70.6  114 / 93     137 / 116    171 / 193    212 / 212
TilePlan tile_plan(int form, bool may_add, int M, int N, int K) {
  const bool stream = form == kTileSlices || form == kTilePlain, slice = form == kTileSlices;
  const double rows = form == kTileGated ? 2.0 * N : N, gflop = 2e-9 * M * rows * K, mb = 2e-6 * rows * K, numbers = 1e-6 * M * N;
  double least = form == kTileQkv ? 21.3 + 0.562 * gflop + 0.228 * mb
                                  : (stream ? 21.5 + 0.733 * gflop + 0.211 * mb : 20.3 + 0.684 * gflop + 0.056 * mb);
  // In bfloat16 nothing but the product is saved, and beside a step's cold weights the small tiles, which ask for the tokens often, lose
  // some of their lead: 2,048 tokens x 2,048 x 2,048 31 us there where the library took 25.6, and the table says 33 against 36 with the norm.
  least *= form == kTilePlain ? 0.85 : 0.97;
  TilePlan plan;
  for (int shape = 0; shape < static_cast<int>(std::size(kTileShapes)); ++shape) {
    const TileShape& t = kTileShapes[shape];
    for (int slices : {1, 2, 3, 4, 6, 8}) {
      if (slices > 1 && (!slice || M >= kAddMinTokens || K / 64 < 2 * slices || static_cast<int64_t>(slices) * M > kMostSliceRows)) break;
      const int64_t steps = ceil_div(K / 64, slices), used = ceil_div(K / 64, steps);
      const int64_t groups = ceil_div(M, t.rows) * ceil_div(static_cast<int64_t>(rows), t.cols) * used, at_once = 256 * t.at_once;
      const int64_t left = groups % at_once;
      const bool half = t.at_once == 2 && left > 0 && left <= 256;
      const double full = static_cast<double>(groups / at_once + (left > 0 && !half ? 1 : 0));
      const double time = t.start + full * (steps * t.full + t.round) + (half ? steps * t.half + t.half_round : 0.0) +
                          (stream ? 5.0 : 0.0) + (slice ? 8.0 * t.per_mb_f32 * numbers * used : 2.0 * t.per_mb_bf16 * numbers);
      if (time < least) {
        least = time;
        plan = TilePlan{shape, static_cast<int>(used), may_add && used == 1};
      }
    }
  }
  return plan;
}

bool tile_takes(const void* x, const void* w, const void* out, int M, int N, int rows, int K) {
  return M > 128 && N > 0 && N % 16 == 0 && K >= 64 && K % 64 == 0 && 2LL * M * K < (1LL << 32) && 2LL * rows * K < (1LL << 32) &&
         (reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
}

}  // namespace
}  // namespace psamd

using namespace psamd;

extern "C" {

int psamd_linear_tile_slices(const void* x, const void* w, int M, int n_out, int K) {
  if (!tile_takes(x, w, nullptr, M, n_out, n_out, K)) return -1;
  const TilePlan plan = tile_plan(kTileSlices, true, M, n_out, K);
  return plan.shape < 0 ? -1 : (plan.add ? 0 : plan.ksplit);
}

int psamd_linear_tile_stream(void* stream, const void* x, const void* w, float* out, int M, int n_out, int K) {
  PSAMD_REQUIRE(tile_takes(x, w, out, M, n_out, n_out, K), "operands that psamd_linear_tile_slices does not take");
  const TilePlan plan = tile_plan(kTileSlices, true, M, n_out, K);
  PSAMD_REQUIRE(plan.shape >= 0, "psamd_linear_tile_slices leaves this product to the library");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (plan.add) return launch_form<kTileAdd>(s, plan.shape, x, w, out, M, n_out, K, 1, 0);
  return launch_form<kTileSlices>(s, plan.shape, x, w, out, M, n_out, K, plan.ksplit, 0);
}

int psamd_linear_tile_plain(void* stream, const void* x, const void* w, void* out, int M, int n_out, int K) {
  if (!tile_takes(x, w, out, M, n_out, n_out, K)) return 2;
  const TilePlan plan = tile_plan(kTilePlain, false, M, n_out, K);
  if (plan.shape < 0) return 2;
  return launch_form<kTilePlain>(static_cast<hipStream_t>(stream), plan.shape, x, w, out, M, n_out, K, 1, 0);
}

int psamd_linear_tile_gated(void* stream, const void* x, const void* w, void* out, int M, int n_out, int K, int activation) {
  PSAMD_REQUIRE(activation >= 0 && activation <= 2, "activation 0 (silu), 1 (relu) or 2 (gelu)");
  if (!tile_takes(x, w, out, M, n_out, 2 * n_out, K)) return 2;
  const TilePlan plan = tile_plan(kTileGated, false, M, n_out, K);
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
  const TilePlan plan = tile_plan(kTileQkv, false, M, static_cast<int>(rows), K);
  if (plan.shape < 0) return 2;
  const QkvOut q{hq, hkv, head_dim, positions, reinterpret_cast<const float2*>(table), static_cast<bf16_t*>(kv), write_slot};
  return launch_form<kTileQkv>(static_cast<hipStream_t>(stream), plan.shape, x, w, qkv_out, M, static_cast<int>(rows), K, 1, 0, q);
}

}  // extern "C"
