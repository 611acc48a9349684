// bfloat16 products of up to 16 tokens that are rows of the float32 residual stream, normalized on the way in, with the rows of w
// through LDS: out[M,N] = norm(rows) * w^T, act(gate) * up, or q/k/v with rotation and pages.
//
// They are bound by reading w once; the kernels of linear.hip (stream_kernel, qkv_rope_append_kernel) do not get there, because
//  * a workgroup's first rows of w are asked for when its tokens have been normalized: here half of the waves ask for w at once and
//    the others bring the tokens (a wave's loads come back in order, so one that did both would wait for w in front of the tokens);
//  * their loads are a matrix instruction's operand, 16 rows x 64 bytes, which the path from L2 carries at 9.7 TB/s over the chip where it
//    carries whole lines at 28 to 32: here w goes to LDS in whole lines (global_load_lds), and no register holds what is under way;
//  * all workgroups ask the same few memory channels in step: here each begins at another place of K (see linear_stream.hip).
#include <algorithm>

#include "api.h"
#include "common.h"
#include "linear_stream.h"
#include "stream_operands.h"

namespace psamd {
namespace {

constexpr int kEnoughBlocks = 136;                                             // tiles of 64 or 32 rows: as in linear_stream.hip
constexpr int wait_for_lds = 15 | (3 << 14) | (7 << 4);                        // s_waitcnt lgkmcnt(0) alone

// Bytes of LDS for the tokens and their sums of squares.
constexpr size_t normed_tokens_bytes(int rows, int K) { return static_cast<size_t>(K / 64) * rows * 128 + sizeof(float) * rows * 4; }

// Wave `wave` of XW brings its share of the M tokens: xs[K / 64][ROWS][128 bytes] = bfloat16(row x the norm's weight), the 16-byte pieces of a
// unit's row exchanged as those of w, and its part of a row's sum of squares in ss[row][wave of the row]. Either wpr waves share
// a row (TOGETHER = 1) or a wave has up to TOGETHER rows, whose loads are under way together.
template <int ROWS, int XW, int TOGETHER>
__device__ __forceinline__ void stage_tokens(const Tokens& tk, unsigned char* xs, float* ss, int M, int K, int wave, int lane, int wpr) {
  const int pieces = K >> 3, per_part = (pieces + wpr - 1) / wpr, part = TOGETHER == 1 ? wave % wpr : 0, row0 = TOGETHER == 1 ? wave / wpr : wave;
  if (row0 >= M) return;
  const float* src[TOGETHER];
  float sum[TOGETHER];
#pragma unroll
  for (int j = 0; j < TOGETHER; ++j) {
    const int row = min(row0 + j * XW, M - 1);
    src[j] = tk.resid + static_cast<int64_t>(tk.rows != nullptr ? tk.rows[row] : row) * K;
    sum[j] = 0.f;
  }
  const int c_end = min(pieces, (part + 1) * per_part);
#pragma unroll TOGETHER > 2 ? 2 : 4
  for (int c = part * per_part + lane; c < c_end; c += 64) {
    float4 a[TOGETHER], b[TOGETHER];
#pragma unroll
    for (int j = 0; j < TOGETHER; ++j) {
      a[j] = *reinterpret_cast<const float4*>(src[j] + 8 * c);
      b[j] = *reinterpret_cast<const float4*>(src[j] + 8 * c + 4);
    }
    float wn[8];
    if (tk.norm_w_bf16) {
      const bf16x8 wv = *reinterpret_cast<const bf16x8*>(static_cast<const bf16_t*>(tk.norm_w) + 8 * c);
#pragma unroll
      for (int i = 0; i < 8; ++i) wn[i] = static_cast<float>(wv[i]);
    } else {
      const float4 w0 = *reinterpret_cast<const float4*>(static_cast<const float*>(tk.norm_w) + 8 * c);
      const float4 w1 = *reinterpret_cast<const float4*>(static_cast<const float*>(tk.norm_w) + 8 * c + 4);
      wn[0] = w0.x, wn[1] = w0.y, wn[2] = w0.z, wn[3] = w0.w, wn[4] = w1.x, wn[5] = w1.y, wn[6] = w1.z, wn[7] = w1.w;
    }
#pragma unroll
    for (int j = 0; j < TOGETHER; ++j) {
      const int row = row0 + j * XW;
      const float v[8] = {a[j].x, a[j].y, a[j].z, a[j].w, b[j].x, b[j].y, b[j].z, b[j].w};
      bf16x8 o;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        sum[j] = fmaf(v[i], v[i], sum[j]);
        o[i] = static_cast<__bf16>(v[i] * wn[i]);
      }
      if (row < ROWS) *reinterpret_cast<bf16x8*>(xs + (c >> 3) * (ROWS * 128) + row * 128 + (((c & 7) ^ ((row >> 1) & 7)) << 4)) = o;   // behind M: a repeated row
    }
  }
#pragma unroll
  for (int j = 0; j < TOGETHER; ++j) {
    const float all = wave_sum(sum[j]);
    if (lane == 0 && row0 + j * XW < M) ss[(row0 + j * XW) * XW + part] = all;
  }
}

// TN rows of w (gated: TN gate rows and the TN up rows of the same columns) x all M <= ROWS tokens; layouts, steps of KG units of 64 k and q/k/v
// tiles as in stream_tiles_kernel. TN / 16 x KG waves: each multiplies one unit of a step for 16 columns, NW of them ask for w.
template <int ROWS, int TN, int KG, int STAGES, int NW, int FORM>
__global__ __launch_bounds__(64 * (TN / 16) * KG) void normed_tiles_kernel(Tokens tk, const bf16_t* __restrict__ w, void* __restrict__ out,
                                                                          int M, int N, int K, int act, int rotated, QkvOut q) {
  constexpr int CT = TN / 16, RT = FORM == kGated ? 2 : 1, WROWS = TN * RT, W = CT * KG, LW = KG * WROWS / 8 / NW, STEP = KG * WROWS * 128;
  constexpr int XW = W - NW;                                                   // waves that bring the tokens while the others ask for w
  static_assert(LW * 8 * NW == KG * WROWS && XW >= 1, "whole copies per wave");
  static_assert(W * RT * 1024 <= STAGES * STEP, "the sums of the units' waves fit where the steps were");
  extern __shared__ __align__(16) unsigned char normed_smem[];                 // STAGES x [KG][WROWS][128] of w, [K / 64][ROWS][128] of the tokens, ss
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN, half = FORM == kQkv ? q.d >> 1 : 0;
  const int units = K / 64, steps = (units + KG - 1) / KG;
  unsigned char* const xs = normed_smem + STAGES * STEP;
  float* const ss = reinterpret_cast<float*>(xs + units * ROWS * 128);         // [ROWS][XW]
  const int rot = rotated ? static_cast<int>(blockIdx.x >> 3) * units / static_cast<int>((gridDim.x + 7) >> 3) : 0;
  const char* wb = reinterpret_cast<const char*>(w);
  uint32_t off[LW];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int at = wave * LW + i, row = at % (WROWS / 8) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    int col = min(n0 + row % TN, N - 1);
    if (FORM == kQkv) {                                                        // as in stream_tiles_kernel
      const int pair = col / 16 * 8 + col % 8, head = pair / half;
      col = head * q.d + (pair - head * half) + (col % 16 < 8 ? 0 : half);
    }
    off[i] = static_cast<uint32_t>(row >= TN ? N + col : col) * (2u * K) + 16u * piece;
  }
  const int end = units * 128;
  int from = rot * 128, to = 0;
  auto copy = [&]() {                                                          // the next step into the next buffer
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      const int at = wave * LW + i, k = from + at / (WROWS / 8) * 128;
      __builtin_amdgcn_global_load_lds((global_ptr)(wb + min(k >= end ? k - end : k, end - 128) + off[i]), (lds_ptr)(normed_smem + to + at * 1024), 16, 0, 0);
    }
    from = min(from + KG * 128 >= end ? from + KG * 128 - end : from + KG * 128, end - 128);
    to = to + STEP == STAGES * STEP ? 0 : to + STEP;
  };
  const int wpr = M == 1 ? XW : (2 * M <= XW ? XW / 2 : 1);                    // waves that share a token's row
  if (wave < NW) {
#pragma unroll
    for (int t = 0; t < STAGES - 1; ++t)
      if (t < steps) copy();
  } else {
    if (M <= XW) stage_tokens<ROWS, XW, 1>(tk, xs, ss, M, K, wave - NW, lane, wpr);
    else stage_tokens<ROWS, XW, ROWS / XW>(tk, xs, ss, M, K, wave - NW, lane, 1);
    __builtin_amdgcn_s_waitcnt(wait_for_lds);                                  // what this wave stored is there behind the barrier
  }
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  int slot = 0;                                                                // what the finishing waves need, asked for in front of the products
  float2 angle[4];
  if (FORM == kQkv && wave < CT) {
    const int pair = (n0 + 16 * wave) / 2 + 4 * (g & 1), head = pair / half, m = min(r, M - 1);
    if (q.kv != nullptr && head >= q.hq && n0 + 16 * wave < N) slot = q.write_slot[m];
    const bool rotate = q.table != nullptr && head < q.hq + q.hkv;
    const float2* cs = rotate ? q.table + static_cast<int64_t>(q.positions[m]) * half + (pair - head * half) : nullptr;
#pragma unroll
    for (int i = 0; i < 4; ++i) angle[i] = rotate ? cs[i] : float2{1.f, 0.f};
  }
  const int tile = wave % CT, unit = wave / CT;                                // this wave's column tile and unit of a step
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes)normed_smem));
  const int xr = r % ROWS;                                                     // with 8 rows, lanes 8..15 of a group repeat tokens: their columns are not stored
  const uint32_t w_at = base + (unit * WROWS + 16 * tile + r) * 128 + 16u * (g ^ ((r >> 1) & 7));
  const uint32_t x_at = base + STAGES * STEP + xr * 128 + 16u * (g ^ ((xr >> 1) & 7));
  uint32_t at = 0;
  int k = rot + unit;                                                          // the unit of K that this wave multiplies next
  if (k >= units) k -= units;
  for (int t = 0; t < steps; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    if (wave < NW) wait_for_step<LW, STAGES - 2>(steps - 1 - t);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (wave < NW && t + STAGES - 1 < steps) copy();
    __builtin_amdgcn_sched_barrier(0);
    if (t * KG + unit < units) {
      Operands<TN, RT, 1> ops;
      ops.read(w_at + at, x_at + k * (ROWS * 128));
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ops.w[h][rt], ops.x[h][0], acc[rt], 0, 0, 0);
    }
    at = at + STEP == STAGES * STEP ? 0 : at + STEP;
    k = k + KG >= units ? k + KG - units : k + KG;
  }
  f32x4* const parts = reinterpret_cast<f32x4*>(normed_smem);                  // [KG][CT][RT][64 lanes]
  __syncthreads();                                                             // the last step has been read by everybody
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) parts[(wave * RT + rt) * 64 + lane] = acc[rt];
  __syncthreads();
  if (wave >= CT) return;
  const int n = n0 + 16 * tile + 4 * g;
  float sum = 0.f;
  for (int p = 0; p < wpr; ++p) sum += ss[min(r, M - 1) * XW + p];
  const float scale = rsqrtf(sum / static_cast<float>(K) + tk.eps);
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    acc[rt] = parts[(wave * RT + rt) * 64 + lane];
#pragma unroll
    for (int p = 1; p < KG; ++p) acc[rt] += parts[((p * CT + wave) * RT + rt) * 64 + lane];
    acc[rt] *= scale;
  }
  f32x4 v = acc[0];
  if constexpr (FORM == kGated) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = gate_act(v[i], act) * acc[RT - 1][i];
  }
  const bool second = g >= 2;
  if constexpr (FORM == kQkv) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float other = __shfl_xor(v[i], 32, kWave);                         // the pair's other half
      v[i] = second ? v[i] * angle[i].x + other * angle[i].y : v[i] * angle[i].x - other * angle[i].y;
    }
  }
  if (r >= M || n >= N) return;                                                // N is a multiple of 4 (q/k/v: of 16)
  const ushort4 pk = {float_to_bf16(v[0]), float_to_bf16(v[1]), float_to_bf16(v[2]), float_to_bf16(v[3])};
  if constexpr (FORM == kQkv) {
    const int pair = (n0 + 16 * tile) / 2 + 4 * (g & 1), head = pair / half;
    put_qkv(static_cast<bf16_t*>(out), N, r, head, (second ? half : 0) + pair - head * half, pk, slot, q);
  } else {
    *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(r) * N + n) = pk;
  }
}

template <int ROWS, int TN, int STAGES, int FORM>
int launch_normed_tiles(hipStream_t s, const Tokens& tk, const void* w, void* out, int M, int N, int K, int act, const QkvOut& q) {
  constexpr int KG = 128 / TN, NW = 4;
  constexpr size_t step = static_cast<size_t>(KG) * TN * (FORM == kGated ? 2 : 1) * 128;
  const size_t smem = STAGES * step + normed_tokens_bytes(ROWS, K);
  auto kernel = normed_tiles_kernel<ROWS, TN, KG, STAGES, NW, FORM>;
  if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("linear_normed: " + std::to_string(smem) + " bytes of LDS were refused");
  const int64_t blocks = ceil_div(N, TN);
  kernel<<<dim3(static_cast<unsigned>(blocks)), dim3(512), smem, s>>>(tk, static_cast<const bf16_t*>(w), out, M, N, K, act, blocks <= 1024 ? 1 : 0, q);
  return check_launch("linear_normed");
}

// Rows of w per workgroup as in linear_stream.hip; as many buffers as fit beside the tokens.
template <int ROWS, int FORM>
int launch_normed_rows(hipStream_t s, const Tokens& tk, const void* w, void* out, int M, int N, int K, int act, const QkvOut& q) {
  constexpr int deep = FORM == kGated ? 3 : 6, step = FORM == kGated ? 32 * 1024 : 16 * 1024;
  const bool fits = deep * step + normed_tokens_bytes(ROWS, K) <= 160 * 1024;
#define PSAMD_NORMED(TN_)                                                                             \
  return fits ? launch_normed_tiles<ROWS, TN_, deep, FORM>(s, tk, w, out, M, N, K, act, q)            \
              : launch_normed_tiles<ROWS, TN_, deep - deep / 3, FORM>(s, tk, w, out, M, N, K, act, q)
  if (ceil_div(N, 64) >= kEnoughBlocks) PSAMD_NORMED(64);
  if (ceil_div(N, 32) >= kEnoughBlocks) PSAMD_NORMED(32);
  PSAMD_NORMED(16);
#undef PSAMD_NORMED
}

template <int FORM>
int launch_normed(hipStream_t s, const Tokens& tk, const void* w, void* out, int M, int N, int K, int act, const QkvOut& q) {
  return M <= 8 ? launch_normed_rows<8, FORM>(s, tk, w, out, M, N, K, act, q) : launch_normed_rows<16, FORM>(s, tk, w, out, M, N, K, act, q);
}

}  // namespace

// Where every compute unit's one workgroup has rows enough to hide the staging of the tokens, which grows with them, and buffers enough for its rows of w:
// beside the tokens there is room for three buffers of the gated form up to K = 4,032 (9 and more tokens: 1,984), for two behind that. us with
// weights that are in no cache at 1, 4, 5, 8, 9 and 16 tokens, kernels of linear.hip and here (q/k/v: heads of 128):
//   tiles of 16 rows (below 4,321)
//     gated 2 x 1,536 x 2,048   8.8, 8.9, 9.0, 9.0, 10.1, 10.3 -> 7.6, 8.2, 9.0, 9.0, 11.3, 11.4       2 x 2,048 x 4,096  14.4, 15.0, 16.0, 15.9 -> 14.1, 16.1, 17.3, 17.2
//           2 x 4,096 x 1,536   9.1, 9.3, 9.5, 9.3, 10.4, 10.5 -> 8.8, 9.4, 10.1, 10.1, 11.1, 11.2     2 x 2,816 x 5,120  19.1, 19.5, 21.0, 20.9 -> 18.8, 21.1, 22.6, 22.6
//     plain 2,048 x 2,048       6.3, 6.6, 6.8, 6.7 -> 5.9, 6.4, -, -      4,096 x 4,096  10.7, 11.5 -> 9.9, 12.0      q/k/v 3,072 x 2,048  6.7, 7.0, -, 7.4, -, 8.8 -> 6.9, 7.3, -, 8.4, -, 9.3
//   tiles of 32 (below 8,641)
//     gated 2 x 8,192 x 2,048   17.1, 17.4, 17.9, 17.9, 20.5, 21.2 -> 15.1, 16.0, 16.7, 16.8, 19.2, 19.2     x 1,024  10.0, 10.0, 10.3, 10.4, 12.8, 13.2 -> 10.0, 10.2, 10.7, 10.8, 11.5, 11.6
//           2 x 8,192 x 2,880   21.0, 21.8, 23.1, 22.8, 26.3, 26.8 -> 20.4, 21.7, 23.0, 22.9, 27.7, 27.9     x 4,096  34.3, 35.4, 37.2, 37.2 -> 29.1, 30.9, 32.1, 32.2
//     q/k/v 4,608 x 2,048       9.1, 10.0, 9.8, 10.5, 11.3, 12.1 -> 8.2, 8.9, 9.6, 9.6, 10.9, 11.0           4,608 x 1,536  7.9, 8.4, 8.3, 8.8, 9.6, 10.3 -> 7.7, 8.2, 8.8, 8.8, 9.8, 10.0
//           6,144 x 4,096       14.8, 15.4, 15.6, 16.5 -> 13.9, 15.9, 17.0, 17.1                             8,192 x 4,096  16.7, 17.8, 18.4, 19.1 -> 17.2, 19.4, 20.4, 20.4
//           6,144 x 5,120       21.2, 22.9, 25.4, 26.1 -> 16.4, 18.6, 20.1, 20.3                             8,192 x 2,560  12.3, 13.0, 12.9, 13.6, 15.3, 16.2 -> 12.2, 13.1, 14.0, 14.2, 15.7, 15.8
//     plain 6,144 x 2,048       9.3, 9.7, 10.1, 10.0, 11.7, 12.0 -> 8.4, 9.1, 9.8, 9.8, 11.3, 11.5           6,144 x 1,536  7.8, 8.0, 8.1, 8.2, 9.2, 9.4 -> 7.6, 8.0, 8.7, 8.7, 9.7, 9.9
//   tiles of 64
//     gated 2 x 14,336 x 4,096  49.2, 50.3, 51.5, 51.6 -> 43.2, 45.0, 45.9, 46.2       2 x 11,008 x 2,560  30.9, 32.4, 32.6, 32.8, 31.4, 32.2 -> 24.7, 25.5, 26.3, 26.5, 34.9, 35.2
//     q/k/v 9,216 x 2,048       13.3, 14.6, 15.1, 15.6, 20.7, 22.0 -> 11.3, 12.1, 12.8, 12.9, 14.0, 14.2     plain  13.2, 13.6, 13.0, 13.9, 17.4, 18.4 -> 10.9, 11.6, 12.3, 12.3, 13.6, 13.8
// Float32 outputs (the output matrix) stay in linear.hip, whose workgroups stage the
// tokens once for several groups of rows: 32,000 x 2,048 28.7, 29.0, 31.4, 37.2 there, 29.3, 30.4, 32.4, 35.5 here, 128,256 x 2,048 93.9 to 112 there, 101 to 131 here.
static bool normed_pays(int form, int M, int n_out, int K) {
  const int64_t of16 = ceil_div(n_out, 16), of32 = ceil_div(n_out, 32);
  const bool narrow = of32 < kEnoughBlocks, wide = ceil_div(n_out, 64) >= kEnoughBlocks;   // tiles of 16 and of 64 rows
  if (form == kGated) {
    const bool three = 96 * 1024 + normed_tokens_bytes(M <= 8 ? 8 : 16, K) <= 160 * 1024;  // buffers
    if (narrow) return M <= 2 || (three && (M <= 4 || K > 1536 || of16 < 160));            // few steps do not pay for many tokens
    if (wide) return M <= 8 || three || K <= 2048;
    return M <= 8 ? (M <= 4 || K > 1024 || of32 <= 200) : (three || K <= 2560);
  }
  if (narrow) return form == kPlain && (M <= 2 || (M <= 4 && (K <= 2816 || of16 <= 160)));
  if (wide || K >= 4608) return true;
  if (K < 2048) return M <= 4 && (K <= 512 || (K >= 1536 && of32 <= 192));
  if (K <= 2816) return M <= 4 || M > 8 || of32 <= 192;
  if (M > 8) return form == kPlain || of32 <= 192;
  return of32 <= 192 && M <= (of32 <= 176 ? 4 : 2);
}

bool linear_normed_takes(const void* w, const void* out, int form, int M, int n_out, int K) {
  if (form == kSlices || !normed_pays(form, M, n_out, K)) return false;
  return M >= 1 && M <= 16 && n_out > 0 && n_out % 4 == 0 && K >= 64 && K % 64 == 0 && (form == kGated ? 4LL : 2LL) * n_out * K < (1LL << 32) &&
         64 * 1024 + normed_tokens_bytes(M <= 8 ? 8 : 16, K) <= 160 * 1024 &&
         (reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out)) % 16 == 0;
}

int launch_linear_normed(hipStream_t s, const Tokens& tk, const void* w, void* out, int form, int M, int n_out, int K, int gate_act, const QkvOut& q) {
  if (form == kGated) return launch_normed<kGated>(s, tk, w, out, M, n_out, K, gate_act, q);
  if (form == kQkv) return launch_normed<kQkv>(s, tk, w, out, M, n_out, K, 0, q);
  return launch_normed<kPlain>(s, tk, w, out, M, n_out, K, 0, q);
}

}  // namespace psamd
