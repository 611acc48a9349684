// bfloat16 products of 17 to 128 tokens, out[M,N] = x[M,K] * w[N,K]^T, with both operands through LDS.
//
// They are bound by reading w once, but the kernels of linear.hip read the tokens from L2 beside it, in pieces of 64 bytes
// of 16 rows: as many bytes as w at 64 tokens, through the path that carries w. Here a workgroup copies whole lines of both into
// LDS (global_load_lds, 16 bytes a lane, nothing through registers), several steps ahead, for up to 64 rows of w at a time, and the
// matrix instructions read them there. Microseconds of a product whose weights are not in any cache (from 65 tokens on the other
// side is the library, with the rotation or the activation in a kernel behind it):
//   rows x K            17 tokens      32             64             77             128
//   2,048 x 2,048       4.9 -> 4.5     5.3 -> 4.6     7.1 -> 5.4     8.5 -> 5.9     8.8 -> 6.5
//   2,048 x 8,192      11.7 -> 8.9    13.5 -> 9.4    15.6 -> 10.5   21.0 -> 11.8   21.8 -> 14.0
//   4,096 x 14,336     35.1 -> 22.7   40.2 -> 23.2   41.2 -> 26.5   49.5 -> 29.5   75.9 -> 36.6
//   2 x 8,192 x 2,048  20.3 -> 14.6   21.4 -> 14.6   22.0 -> 15.1   23.3 -> 17.1   25.7 -> 19.8   (gated)
//   2 x 14,336 x 4,096 58.4 -> 42     62.0 -> 42     58.3 -> 43     60   -> 45     62.7 -> 51     (gated)
//   6,144 x 4,096      19.6 -> 14.0   22.4 -> 15.8   30.5 -> 20.2   28.9 -> 21.7   31.4 -> 27.4   (q/k/v)
//   128,256 x 2,048     131 -> 101     138 -> 105     159 -> 120    (float32 out; above 64 tokens the library's product is as fast)
// So do the bfloat16 products above 64 tokens (16,384 x 2,048 at 77: 18.4 there, 19.1 here), which stay with the library.

#include <algorithm>

#include "api.h"
#include "common.h"
#include "linear_stream.h"
#include "stream_operands.h"

namespace psamd {

// grid (ceil(rows of w / TN), K-slices): TN rows of w for all of up to TM tokens; the gated form takes TN gate rows and
// the TN up rows of the same columns, the q/k/v form lays 8 rotation pairs of a head into each tile of 16 rows: 8 rows of its
// first half and their partners in the second, whose sums then lie two lane groups apart. A step is KG units of 64 k. A wave
// multiplies one unit of a step, 16 columns for TM / TG tokens: TN / 16 x TG x KG waves, the sums of the KG added through LDS at the end.
// A unit's rows are 128 bytes whose 16-byte pieces are exchanged by row / 2, so that 16 rows' reads meet every bank once.
// Buffer t % STAGES holds step t, which is asked for STAGES - 1 steps ahead, into the buffer that everybody has read when the
// barrier in front of its asking has been passed.
// What bounds it, found by leaving parts out (3,072 x 2,048 q/k/v at 77 tokens, 14.0 us): a fifth is memory; the loop without copies and
// without products took 6 us (its divisions, an epilogue whose positions, angles and slots came from memory one after the other)
// and a wave's products 4.5, reads and matrix instructions in turn. Hence counters in place of divisions, the epilogue's operands
// asked for in front of the loop, and several waves that share a unit's tokens (TG) or a step's units (KG): 9.7 us.
// Rows of w lie a power of two apart as a rule, so that workgroups that walk K in step ask the same few memory channels: each starts
// at another step (`rotated`) and comes round. 2 x 11,008 x 4,096 gated at 32 tokens 45.6 -> 33.6 us, 2 x 14,336 x 4,096 50.2 -> 40.1,
// 2 x 8,192 x 2,048 16.3 -> 13.5, 32,000 x 2,048 30.2 -> 26.2. K-slices start apart as it is (at 96 and more tokens turning them lost 10%),
// and the workgroups of a long grid soon are (128,256 rows: 106.6 us, 108.4 turned).
template <int TM, int TN, int TG, int KG, int STAGES, int FORM>
__global__ __launch_bounds__(64 * (TN / 16) * TG * KG) void stream_tiles_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                                                                                void* __restrict__ out, int M, int N, int K,
                                                                                int slice_units, int act, int rotated, QkvOut q) {
  constexpr int CT = TN / 16, RM = TM / 16 / TG, RT = FORM == kGated ? 2 : 1, ROWS = TN * RT, W = CT * TG * KG;
  constexpr int LW = KG * ROWS / 8 / W, LX = KG * TM / 8 / W, W_STEP = KG * ROWS * 128, STAGE = W_STEP + KG * TM * 128;   // copies of 8 rows per wave and step
  static_assert(RM * 16 * TG == TM && LW * 8 * W == KG * ROWS && LX * 8 * W == KG * TM, "whole copies per wave");
  static_assert(KG == 1 || W * RT * RM * 1024 <= STAGES * STAGE, "the sums of the units' waves fit where the steps were");
  extern __shared__ __align__(16) unsigned char stream_smem[];                 // STAGES x [KG][ROWS rows of w][128], [KG][TM of x][128]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * TN;
  const int first = blockIdx.y * slice_units, units = min(slice_units, K / 64 - first), steps = (units + KG - 1) / KG;
  const char* xb = reinterpret_cast<const char*>(x) + static_cast<int64_t>(first) * 128;
  const char* wb = reinterpret_cast<const char*>(w) + static_cast<int64_t>(first) * 128;
  const int half = FORM == kQkv ? q.d >> 1 : 0;
  uint32_t w_off[LW], x_off[LX];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int at = wave * LW + i, row = at % (ROWS / 8) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    int col = min(n0 + row % TN, N - 1);
    if (FORM == kQkv) {                                                        // N is a multiple of 16: whole tiles of 8 pairs
      const int pair = col / 16 * 8 + col % 8, head = pair / half;
      col = head * q.d + (pair - head * half) + (col % 16 < 8 ? 0 : half);
    }
    w_off[i] = static_cast<uint32_t>(row >= TN ? N + col : col) * (2u * K) + 16u * piece;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {
    const int at = wave * LX + i, row = at % (TM / 8) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    x_off[i] = static_cast<uint32_t>(min(row, M - 1)) * (2u * K) + 16u * piece;
  }
  const int end = units * 128;
  int from = rotated ? static_cast<int>(blockIdx.x >> 3) * units / static_cast<int>((gridDim.x + 7) >> 3) * 128 : 0, to = 0;
  // Of a step's units, the one behind the last is the first again; what the last step has no unit for is copied and not multiplied.
  auto unit_at = [&](int unit) {
    const int k = from + unit * 128;
    return KG == 1 ? k : min(k >= end ? k - end : k, end - 128);
  };
  auto copy = [&]() {                                                          // the next step into the next buffer
#pragma unroll
    for (int i = 0; i < LW; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr)(wb + unit_at((wave * LW + i) / (ROWS / 8)) + w_off[i]),
                                       (lds_ptr)(stream_smem + to + (wave * LW + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < LX; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr)(xb + unit_at((wave * LX + i) / (TM / 8)) + x_off[i]),
                                       (lds_ptr)(stream_smem + to + W_STEP + (wave * LX + i) * 1024), 16, 0, 0);
    from = from + KG * 128 >= end ? from + KG * 128 - end : from + KG * 128;
    if (KG > 1) from = min(from, end - 128);                                   // fewer units than a step has: it is the only one
    to = to + STAGE == STAGES * STAGE ? 0 : to + STAGE;
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
  const int tile = wave % CT, share = wave / CT % TG, unit = wave / (CT * TG);  // this wave's column tile, tokens and unit of a step
  const int tokens = share * (16 * RM);
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes)stream_smem));
  const uint32_t piece0 = 16u * (g ^ ((r >> 1) & 7));
  const uint32_t w_at = base + (unit * ROWS + 16 * tile + r) * 128 + piece0;
  const uint32_t x_at = base + W_STEP + (unit * TM + tokens + r) * 128 + piece0;
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < steps) copy();
  // Of the KG waves with the same columns and tokens, this one finishes token tiles unit, unit + KG, ...
  constexpr int MINE = (RM + KG - 1) / KG;
  int slot_of[MINE];
  float2 angle[MINE][4];
  if constexpr (FORM == kQkv) {
    const int pair = (n0 + 16 * tile) / 2 + 4 * (g & 1), head = pair / half, p = pair - head * half;
    const bool rotate = q.table != nullptr && head < q.hq + q.hkv, stored = q.kv != nullptr && head >= q.hq && n0 + 16 * tile < N;
#pragma unroll
    for (int k = 0; k < MINE; ++k) {
      const int m = min(tokens + 16 * (k * KG + unit) + r, M - 1);
      slot_of[k] = stored ? q.write_slot[m] : 0;
      const float2* cs = rotate ? q.table + static_cast<int64_t>(q.positions[m]) * half + p : nullptr;
#pragma unroll
      for (int i = 0; i < 4; ++i) angle[k][i] = rotate ? cs[i] : float2{1.f, 0.f};
    }
  }
  uint32_t at = 0;
  for (int t = 0; t < steps; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    wait_for_step<LW + LX, STAGES - 2>(steps - 1 - t);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + STAGES - 1 < steps) copy();
    __builtin_amdgcn_sched_barrier(0);
    if (KG == 1 || t * KG + unit < units) {
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
    }
    at = at + STAGE == STAGES * STAGE ? 0 : at + STAGE;
    if (!RUNS) continue;
    if ((t & 1) != 0 || t + 1 == steps || units < 8) {
#pragma unroll
      for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int j = 0; j < RM; ++j) {
          acc[rt][j] += part[rt][j];
          part[rt][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
  }
  f32x4* const parts = reinterpret_cast<f32x4*>(stream_smem);                  // [KG][TG][CT][RT][RM][64 lanes]
  if (KG > 1) {
    __syncthreads();                                                           // the last step has been read by everybody
#pragma unroll
    for (int i = 0; i < RT * RM; ++i) parts[(wave * RT * RM + i) * 64 + lane] = acc[i / RM][i % RM];
    __syncthreads();
  }
  auto sums = [&](int rt, int j) {
    if (KG == 1) return acc[rt][j];
    const f32x4* p = parts + (wave % (CT * TG) * RT * RM + rt * RM + j) * 64 + lane;
    f32x4 v = *p;
#pragma unroll
    for (int k = 1; k < KG; ++k) v += p[k * CT * TG * RT * RM * 64];
    return v;
  };
  const int n = n0 + 16 * tile + 4 * g;                                        // this lane's four columns of token tokens + 16 j + r
  auto pack = [](f32x4 v) { return ushort4{float_to_bf16(v[0]), float_to_bf16(v[1]), float_to_bf16(v[2]), float_to_bf16(v[3])}; };
#pragma unroll
  for (int j = 0; j < RM; ++j) {
    if (KG > 1 && j % KG != unit) continue;
    const int m = tokens + 16 * j + r;
    if constexpr (FORM == kQkv) {
      const bool second = g >= 2;
      const int pair = (n0 + 16 * tile) / 2 + 4 * (g & 1), head = pair / half, p = pair - head * half;
      f32x4 v = sums(0, j);
      const bool here = m < M && n < N;                                        // N is a multiple of 16: both halves of a pair or none
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float other = __shfl_xor(v[i], 32, kWave);                       // the pair's other half
        const float2 c = angle[j / KG][i];
        v[i] = second ? v[i] * c.x + other * c.y : v[i] * c.x - other * c.y;
      }
      if (here) put_qkv(static_cast<bf16_t*>(out), N, m, head, (second ? half : 0) + p, pack(v), slot_of[j / KG], q);
      continue;
    }
    if (m >= M || n >= N) continue;                                            // N is a multiple of 4
    if constexpr (FORM == kSlices) {
      float* o = static_cast<float*>(out) + (static_cast<int64_t>(blockIdx.y) * M + m) * N + n;
      *reinterpret_cast<f32x4*>(o) = sums(0, j);
    } else {
      f32x4 v = sums(0, j);
      if constexpr (FORM == kGated) {
        const f32x4 up = sums(RT - 1, j);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = gate_act(v[i], act) * up[i];
      }
      *reinterpret_cast<ushort4*>(static_cast<bf16_t*>(out) + static_cast<int64_t>(m) * N + n) = pack(v);
    }
  }
}

constexpr int kUnits = 256;                                                    // compute units

// The most rows of w per workgroup, which read the tokens least often, that still give about half of the 256 compute units one and
// leave no second round of workgroups that take a whole unit's LDS: 5,632 gated columns are 352 workgroups of 16 (23.1 us at 77 tokens) or 176
// of 32 (18.0), 11,008 344 of 32 (54.4) or 172 of 64 (43.2), 4,608 rows of q/k/v 288 of 16 (33.5) or 144 of 32 (19.5); the six fastest
// forms tried for 8,192 gated columns x 2,048 were all 256 of 32, not 128 of 64. With K-slices, which linear_stream_ksplit chooses for 64 rows,
// fewer only where even eight slices leave units idle (1,024 x 1,024: 3.5, 3.2, 3.2) and those of fewer rows, one to a unit, are still one round.
// us with the norm behind it, two rounds of 32 / one of 64: 1,408 x 1,536 at 33 tokens 9.9 / 8.4, at 128 13.6 / 11.3, 1,280 x 2,048 at 97 12.4 / 10.4, 5,632 x 256 at
// 33 12.3 / 10.9; of 16 / of 32: 2,816 x 256 at 128 11.6 / 9.7.
static int stream_columns(int N, int ksplit) {
  const int64_t of64 = ceil_div(N, 64) * ksplit, of32 = ceil_div(N, 32) * ksplit, of16 = ceil_div(N, 16) * ksplit;
  if (ksplit > 1) return of64 >= 192 || of32 > kUnits ? 64 : (of32 >= 192 || of16 > kUnits ? 32 : 16);
  return of64 >= 136 ? 64 : (of32 >= 136 ? 32 : 16);
}

// How a tile of TM tokens and TN rows is shared out: TG, KG and the number of buffers. Few rows a workgroup (16, 32) leave a unit of
// K one or two waves: there the units of a step go to waves of their own (KG); with 64 rows the waves share the tokens.
// us (waves as for one unit, then this; 17 / 32 / 64 / 77 / 128 tokens): q/k/v 3,072 x 2,048 7.6, 8.3, 10.3, 13.9, 14.3 -> 6.2, 6.4, 7.8, 10.6, 12.2;
// 4,608 x 3,584 (16 rows then, 32 now) 20.1, 17.2, 23.7, 29.2, 36.5 -> 13.2, 14.3, 17.5, 19.5, 24.6; 6,144 x 4,096 16.1, 16.8, 20.6, 25.2, 28.4 -> 14.0, 15.8,
// 20.2, 21.7, 27.4. Gated (turned): 2 x 8,192 x 2,048 17.0, 17.3, 17.9, 20.7, 21.6 -> 14.6, 14.6, 15.1, 17.1, 19.8; 2 x 11,008 x 4,096 (32 rows then, 64 now)
// 43.9, 45.1, 49.4, 54.4, 61.5 -> 34.3, 35.2, 39.2, 43.2, 50.6; 2 x 14,336 x 4,096 54.2, 55.2, 57.1, 57.3, 59.2 -> 42.2, 42.4, 43.4, 45.1, 51.1. bfloat16 1,024 x 4,096
// 11.7, 11.7, 13.7 -> 7.1, 7.2, 9.2. K-slices of 64 rows gain from the loop (2,048 x 2,048 4.9 -> 4.5 at 17), and around 80 tokens from KG where a
// slice is long enough to pay for its sum (2,048 x 8,192 12.9 -> 11.8, 4,096 x 14,336 34.3 -> 29.5; 2,048 x 2,048, four units, 5.8 -> 6.3).
struct StreamShape { int tg, kg, stages; };
constexpr StreamShape stream_shape(bool gated, int tm, int tn) {
  if (tn == 64) {
    if (gated) return tm == 32 ? StreamShape{1, 1, 4} : (tm == 64 ? StreamShape{2, 1, 6} : StreamShape{4, 1, 4});
    return tm == 32 ? StreamShape{1, 1, 6} : (tm == 64 ? StreamShape{2, 1, 5} : (tm == 96 ? StreamShape{1, 2, 3} : StreamShape{2, 1, 3}));
  }
  if (tn == 32) {
    if (gated) return tm == 64 ? StreamShape{4, 1, 5} : StreamShape{tm == 128 ? 4 : (tm == 96 ? 2 : 1), 2, 3};
    return {2, 2, tm <= 64 ? 5 : 3};
  }
  if (gated && tm == 128) return {4, 2, 3};
  return {2, 4, tm <= 64 ? 3 : 2};
}

template <int TM, int TN, int FORM>
static int launch_stream_tiles(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                               const QkvOut& q) {
  constexpr StreamShape S = stream_shape(FORM == kGated, TM, TN);
  constexpr size_t smem = static_cast<size_t>(S.stages) * S.kg * ((FORM == kGated ? 2 : 1) * TN + TM) * 128;
  static_assert(smem <= 160 * 1024, "a compute unit's LDS");
  auto kernel = stream_tiles_kernel<TM, TN, S.tg, S.kg, S.stages, FORM>;
  if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("linear_stream: " + std::to_string(smem) + " bytes of LDS were refused");
  const int64_t blocks = ceil_div(N, TN);
  kernel<<<dim3(static_cast<unsigned>(blocks), static_cast<unsigned>(ksplit)), dim3(64 * (TN / 16) * S.tg * S.kg), smem, s>>>(
      static_cast<const bf16_t*>(x), static_cast<const bf16_t*>(w), out, M, N, K, static_cast<int>(ceil_div(K / 64, ksplit)), act,
      ksplit == 1 && blocks <= 1024 ? 1 : 0, q);
  return check_launch("linear_stream");
}

template <int FORM, int TN>
static int launch_stream_tokens(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                                const QkvOut& q) {
  if (M <= 32) return launch_stream_tiles<32, TN, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  if (M <= 64) return launch_stream_tiles<64, TN, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  // Tiles of 96 tokens, whose slices have a unit each to themselves, not where that makes a second round: those of 128 share one (2,816 x 4,096, 264
  // workgroups, the norm behind it included, 77 tokens 18.7 / 16.0 us, x 512 at 65 11.9 / 10.5).
  if constexpr (!(FORM == kGated && TN == 64)) {       // (2 x 14,336 x 4,096 gated at 96 tokens: 45.4 us as 96, 46.3 as 128; 2 x 11,008 43.7, 41.9)
    if (M <= 96 && (TN < 64 || (ceil_div(K / 64, ksplit) >= 8 && ceil_div(N, 64) * ksplit <= kUnits))) return launch_stream_tiles<96, TN, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
  }
  return launch_stream_tiles<128, TN, FORM>(s, x, w, out, M, N, K, ksplit, act, q);
}

template <int FORM>
static int launch_stream_form(hipStream_t s, const void* x, const void* w, void* out, int M, int N, int K, int ksplit, int act,
                              const QkvOut& q = {}) {
  const int tn = stream_columns(N, ksplit);
  if (tn == 64) return launch_stream_tokens<FORM, 64>(s, x, w, out, M, N, K, ksplit, act, q);
  if (tn == 32) return launch_stream_tokens<FORM, 32>(s, x, w, out, M, N, K, ksplit, act, q);
  return launch_stream_tokens<FORM, 16>(s, x, w, out, M, N, K, ksplit, act, q);
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
