// Mixture-of-experts feed-forward: the router, and the experts in two forms.
//
// * Pair by pair: one (token, choice) pair per workgroup row, the expert's matrices read once per
//   pair. It is the form of the 32-bit path at every size (templated on the element type, sums in
//   float, in an order that does not depend on the step) and of bfloat16 steps of one or two tokens.
// * Grouped (bfloat16): the step's pairs are sorted by expert, and every expert's pairs go through
//   its matrices in tiles of 16 or 64 pairs on the matrix cores (v_mfma_f32_16x16x32_bf16), so an
//   expert is read once per tile of pairs instead of once per pair: a decode batch reads each
//   expert it uses once, a prompt's portion runs as grouped products.
//
// Router: z = x . w_r[e] (+ bias[e]) in float; the `top` largest are taken, the lower index among
// equals. mode 0: the score is sigmoid(z) and is the weight as it is; mode 1: the weights are the
// softmax over the chosen z alone; mode 2: the score is the softmax over all z, the choice goes by score +
// correction[e] (which may be negative) and the weight is the score as it is. Expert: with h = weight * x, g = min(gate h, limit), u = clamp(up h,
// -limit, limit), act = g * sigmoid(gate_alpha * g) * (u + up_shift), out = down act. There the weight
// multiplies the expert's input, so it cannot be pulled out of the clamps; with weight_on_output the
// expert sees x itself and the weight multiplies out (limit = infinity, gate_alpha = 1, up_shift = 0
// then make the plain SiLU-gated expert). The other kind of expert has no gate: act = max(up h, 0)^2
// (kExpertSquaredRelu), its first matrix is [F, K].
//
// With groups (modes 0 and 2): the experts form `groups` equal runs of neighbours, a run's score is the sum of its
// two largest scores (group_max: its largest), each with its correction, and only experts of the `keep` best runs
// (the lower index among equals) can be chosen. The weights are multiplied by `factor`.
//
// Choices from `experts` on are identity experts: they have no matrices, their output is the token itself times the
// weight. The grouped form lists their pairs behind the experts' and lets the second product's launch copy them.
//
// `out` is float slices [top][tokens][K], or, for a small bfloat16 step, the float residual stream itself
// (`into_stream`): every pair then adds col_scale[k] * weight * value with float atomics, and nobody adds
// slices up afterwards (the order of the additions differs from run to run).

#include <algorithm>
#include <cmath>

#include "api.h"
#include "common.h"
#include "linear_stream.h"
#include "stream_operands.h"
#include "tile_product.h"
#include "wide_tile.h"

namespace psamd {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kExpertGated = 0, kExpertSquaredRelu = 1;
constexpr int kMaxRouterGroups = 4 * kWave;

// How a router turns scores into a choice (see above). groups 0: every expert can be chosen.
struct RouterRule {
  int mode;
  int groups;
  int keep;
  float factor;
  int group_max;
  const float* correction;             // mode 2: [experts] or null
};

// dst += v at the memory side, nothing returned.
__device__ __forceinline__ void add_float(float* dst, float v) { (void)unsafeAtomicAdd(dst, v); }

// Dot product of a row of n elements with a float vector in LDS, dealt out over the 64 lanes;
// every lane returns the whole sum. bfloat16 rows whose length is a multiple of 8 are read in
// 16-byte pieces.
template <typename W>
__device__ __forceinline__ float wave_dot(const W* __restrict__ row, const float* __restrict__ xs, int n, int lane) {
  float acc = 0.f;
  if (sizeof(W) == 2 && (n & 7) == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0) {
    const int chunks = n >> 3;
    for (int c = lane; c < chunks; c += kWave) {
      const uint4 q = *reinterpret_cast<const uint4*>(reinterpret_cast<const bf16_t*>(row) + 8 * c);
      const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
      const float* xp = xs + 8 * c;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        acc = fmaf(__uint_as_float(w4[i] << 16), xp[2 * i], acc);
        acc = fmaf(__uint_as_float(w4[i] & 0xffff0000u), xp[2 * i + 1], acc);
      }
    }
  } else if (sizeof(W) == 4 && (n & 3) == 0 && (reinterpret_cast<uintptr_t>(row) & 15) == 0) {
    const int chunks = n >> 2;
    float acc2 = 0.f;
    for (int c = lane; c < chunks; c += 2 * kWave) {
      const int c2 = c + kWave;
      const float4 q = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(row) + 4 * c);
      const float4 q2 = c2 < chunks ? *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(row) + 4 * c2)
                                    : float4{0.f, 0.f, 0.f, 0.f};
      const float* xp = xs + 4 * c;
      const float* xp2 = xs + 4 * min(c2, chunks - 1);
      acc = fmaf(q.x, xp[0], acc); acc = fmaf(q.y, xp[1], acc); acc = fmaf(q.z, xp[2], acc); acc = fmaf(q.w, xp[3], acc);
      acc2 = fmaf(q2.x, xp2[0], acc2); acc2 = fmaf(q2.y, xp2[1], acc2); acc2 = fmaf(q2.z, xp2[2], acc2); acc2 = fmaf(q2.w, xp2[3], acc2);
    }
    acc += acc2;
  } else {
    for (int i = lane; i < n; i += kWave) acc = fmaf(to_float<W>(row[i]), xs[i], acc);
  }
  return wave_sum(acc);
}

// ------------------------------------------------------------------ router

// The largest of every lane's (value, index), the lower index among equals, in every lane.
__device__ __forceinline__ void wave_best(float& best, int& at) {
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    const float ob = __shfl_xor(best, o, kWave);
    const int oa = __shfl_xor(at, o, kWave);
    if (ob > best || (ob == best && oa < at)) {
      best = ob;
      at = oa;
    }
  }
}

// Takes the experts outside the best groups out of the choice: their entries of score[] (LDS) become kTaken.
// Lane l holds the scores of groups l, l + 64, ... (at most kMaxRouterGroups in all).
__device__ __forceinline__ void keep_best_groups(float* score, int experts, const RouterRule& rule, int lane) {
  const int groups = rule.groups, keep = rule.keep;
  constexpr int kPer = kMaxRouterGroups / kWave;
  const float kTaken = -__builtin_inff();
  const int size = experts / groups;
  float sum[kPer];
  bool kept[kPer];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int grp = lane + i * kWave;
    kept[i] = false;
    sum[i] = kTaken;
    if (grp < groups) {
      float a = kTaken, b = 0.f;                          // the two largest; a group of one expert has one
      for (int e = grp * size; e < (grp + 1) * size; ++e) {
        const float s = rule.correction != nullptr ? score[e] + rule.correction[e] : score[e];
        if (s > a) {
          b = a == kTaken ? 0.f : a;
          a = s;
        } else if (e > grp * size + 1 ? s > b : e > grp * size) {
          b = s;
        }
      }
      sum[i] = rule.group_max ? a : a + b;
    }
  }
  for (int j = 0; j < keep; ++j) {
    float best = kTaken;
    int at = 0x7fffffff;
#pragma unroll
    for (int i = 0; i < kPer; ++i)
      if (!kept[i] && sum[i] > best) {                    // ascending groups: the first of equals stays
        best = sum[i];
        at = lane + i * kWave;
      }
    wave_best(best, at);
#pragma unroll
    for (int i = 0; i < kPer; ++i) kept[i] = kept[i] || at == lane + i * kWave;
  }
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int grp = lane + i * kWave;
    if (grp < groups && !kept[i])
      for (int e = grp * size; e < (grp + 1) * size; ++e) score[e] = kTaken;
  }
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
}

// The same choice for up to 64 experts without LDS: lane e holds expert e's score (lanes past the last hold nothing of
// use) and counts who comes in front of it.
__device__ __forceinline__ void pick_top_in_lanes(float s, int experts, int top, RouterRule rule, int32_t* __restrict__ chosen,
                                                  float* __restrict__ weight, int lane) {
  const float kTaken = -__builtin_inff();
  auto of = [](float v, int from) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), from)); };
  if (lane >= experts) s = kTaken;
  float w = s;
  if (rule.mode == 2) {
    const float m = wave_max(s);                          // by all lanes: the moves between lanes need every one of them
    const float p = lane < experts ? expf(s - m) : 0.f;
    w = p / wave_sum(p);
    s = lane >= experts ? kTaken : rule.correction != nullptr ? w + rule.correction[lane] : w;
  }
  if (rule.groups > 0) {
    const int size = experts / rule.groups, mine = lane / size;
    float a = kTaken, b = kTaken;                         // the two largest of the lane's own group
    for (int grp = 0; grp < rule.groups; ++grp)
      for (int i = 0; i < size; ++i) {
        const float v = of(s, grp * size + i);
        if (grp == mine) {
          b = fmaxf(b, fminf(a, v));
          a = fmaxf(a, v);
        }
      }
    const float sum = rule.group_max ? a : a + (size > 1 ? b : 0.f);
    int ahead = 0;                                        // groups in front of the lane's own
    for (int grp = 0; grp < rule.groups; ++grp) {
      const float v = of(sum, grp * size);
      ahead += (v > sum || (v == sum && grp < mine)) ? 1 : 0;
    }
    if (ahead >= rule.keep) s = kTaken;
  }
  int rank = 0;
  for (int e = 0; e < experts; ++e) {
    const float v = of(s, e);
    rank += (v > s || (v == s && e < lane)) ? 1 : 0;
  }
  const bool taken = lane < experts && rank < top && s > kTaken;
  if (rule.mode == 0) w = s;
  if (rule.mode == 1) {
    const float m = wave_max(taken ? s : kTaken);
    // Summed in the order of the choice, largest first.
    float sum = 0.f;
    for (int j = 0; j < top; ++j) {
      const unsigned long long at = __ballot(taken && rank == j);
      if (at != 0) sum += expf(of(s, __ffsll(static_cast<unsigned long long>(at)) - 1) - m);
    }
    w = expf(s - m) / sum;
  }
  if (taken) {
    chosen[rank] = lane;
    weight[rank] = rule.factor * w;
  }
}

// The router's choice for one token by one wave: score[] (LDS, `experts` entries: sigmoid(z) in mode
// 0, z in modes 1 and 2) -> chosen / weight [top], largest first, the lower index among equals; taken
// entries are overwritten. Mode 1 then turns the chosen z into their softmax; mode 2 turns all z into their softmax first.
__device__ __forceinline__ void pick_top(float* score, int experts, int top, RouterRule rule, int32_t* __restrict__ chosen,
                                         float* __restrict__ weight, int lane) {
  const float kTaken = -__builtin_inff();
  if (experts <= kWave) {
    pick_top_in_lanes(lane < experts ? score[lane] : 0.f, experts, top, rule, chosen, weight, lane);
    return;
  }
  if (rule.mode == 2) {
    float m = kTaken, sum = 0.f;
    for (int e = lane; e < experts; e += kWave) m = fmaxf(m, score[e]);
    m = wave_max(m);
    for (int e = lane; e < experts; e += kWave) {
      score[e] = expf(score[e] - m);
      sum += score[e];
    }
    sum = wave_sum(sum);
    for (int e = lane; e < experts; e += kWave) score[e] /= sum;
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
  }
  if (rule.groups > 0) keep_best_groups(score, experts, rule, lane);
  for (int j = 0; j < top; ++j) {
    float best = kTaken;
    int at = 0x7fffffff;
    for (int e = lane; e < experts; e += kWave) {
      const float s = rule.correction != nullptr ? score[e] + rule.correction[e] : score[e];
      if (s > best) {                                    // ascending e: the first of equals stays
        best = s;
        at = e;
      }
    }
    wave_best(best, at);
    if (lane == 0) {
      chosen[j] = at;
      weight[j] = rule.mode == 0 ? rule.factor * best : rule.mode == 2 ? (at != 0x7fffffff ? rule.factor * score[at] : 0.f) : best;
      if (at != 0x7fffffff) score[at] = kTaken;
    }
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
  }
  if (rule.mode == 1 && lane == 0) {
    const float m = weight[0];                           // the largest comes first
    float sum = 0.f;
    for (int j = 0; j < top; ++j) sum += expf(weight[j] - m);
    for (int j = 0; j < top; ++j) weight[j] = rule.factor * (expf(weight[j] - m) / sum);
  }
}

__device__ __forceinline__ float router_score(float z, const float* __restrict__ bias, int e, int mode) {
  if (bias != nullptr) z += bias[e];
  return mode == 0 ? 1.f / (1.f + expf(-z)) : z;
}

// One block of four waves per token: the waves share the experts' dot products, then wave 0
// picks the `top` largest scores one after the other (each pick: a strided scan and a wave
// reduction that prefers the lower index among equals).
template <typename A>
__global__ __launch_bounds__(256) void moe_route_kernel(const A* __restrict__ x, const float* __restrict__ w_router,
                                                        int32_t* __restrict__ chosen, float* __restrict__ weight,
                                                        int K, int experts, int top, const float* __restrict__ bias,
                                                        RouterRule rule) {
  extern __shared__ __align__(16) float route_smem[];    // xs[K], score[experts]
  float* xs = route_smem;
  float* score = route_smem + K;
  const int64_t t = blockIdx.x;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  for (int i = threadIdx.x; i < K; i += blockDim.x) xs[i] = to_float<A>(x[t * K + i]);
  __syncthreads();
  for (int e = wave; e < experts; e += 4) {
    const float z = wave_dot<float>(w_router + static_cast<int64_t>(e) * K, xs, K, lane);
    if (lane == 0) score[e] = router_score(z, bias, e, rule.mode);
  }
  __syncthreads();
  if (wave != 0) return;
  pick_top(score, experts, top, rule, chosen + t * top, weight + t * top, lane);
}

// The same choice from logits a product has already written (z[t, :] float). One wave per token,
// four tokens per block.
__global__ __launch_bounds__(256) void moe_topk_kernel(const float* __restrict__ z, int32_t* __restrict__ chosen,
                                                       float* __restrict__ weight, int64_t tokens, int experts, int top,
                                                       const float* __restrict__ bias, RouterRule rule) {
  extern __shared__ __align__(16) float topk_smem[];     // score[4][experts]
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 4 + wave;
  if (t >= tokens) return;
  float* score = topk_smem + wave * experts;
  for (int e = lane; e < experts; e += kWave) score[e] = router_score(z[t * experts + e], bias, e, rule.mode);
  __builtin_amdgcn_wave_barrier();
  __threadfence_block();
  pick_top(score, experts, top, rule, chosen + t * top, weight + t * top, lane);
}

// ------------------------------------------------------------------ experts, pair by pair

constexpr int kRowsPerWave = 4;
constexpr int kRowsPerBlock = 4 * kRowsPerWave;

// grid (pairs, ceil(F / 16)): the block stages h = weight * x[t] in LDS and each wave computes
// kRowsPerWave activations of the pair's expert.
template <typename A>
__global__ __launch_bounds__(256) void moe_gate_up_rows_kernel(
    const A* __restrict__ x, const int32_t* __restrict__ chosen, const float* __restrict__ weight,
    const A* __restrict__ w_gate_up, A* __restrict__ act, int K, int F, int experts, int top, float gate_alpha,
    float limit, float up_shift, int weight_on_output, int kind) {
  extern __shared__ __align__(16) float rows_smem[];     // h[K]
  const int64_t pair = blockIdx.x;
  const int64_t t = pair / top;
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  if (chosen[pair] >= experts) return;                   // an identity expert has no activations
  const int e = max(chosen[pair], 0);
  const float wgt = weight_on_output ? 1.f : weight[pair];
  for (int i = threadIdx.x; i < K; i += blockDim.x) rows_smem[i] = wgt * to_float<A>(x[t * K + i]);
  __syncthreads();
  const A* we = w_gate_up + static_cast<int64_t>(e) * (kind == kExpertGated ? 2 : 1) * F * K;
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int f = static_cast<int>(blockIdx.y) * kRowsPerBlock + wave * kRowsPerWave + r;
    if (f >= F) break;
    float g = wave_dot<A>(we + static_cast<int64_t>(f) * K, rows_smem, K, lane);
    if (kind == kExpertSquaredRelu) {
      g = fmaxf(g, 0.f);
      if (lane == 0) act[pair * F + f] = from_float<A>(g * g);
      continue;
    }
    float u = wave_dot<A>(we + static_cast<int64_t>(F + f) * K, rows_smem, K, lane);
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    if (lane == 0) act[pair * F + f] = from_float<A>(g / (1.f + expf(-gate_alpha * g)) * (u + up_shift));
  }
}

// grid (pairs, ceil(K / 16)): out[j][t][k] = down[e][k] . act[pair].
template <typename A>
__global__ __launch_bounds__(256) void moe_down_rows_kernel(
    const A* __restrict__ act, const int32_t* __restrict__ chosen, const A* __restrict__ w_down,
    float* __restrict__ out, int64_t tokens, int K, int F, int experts, int top, const float* __restrict__ out_weight,
    int into_stream, const float* __restrict__ col_scale, const A* __restrict__ x, const float* __restrict__ weight) {
  extern __shared__ __align__(16) float rows_smem[];     // act[F]
  const int64_t pair = blockIdx.x;
  const int64_t t = pair / top;
  const int j = static_cast<int>(pair - t * top);
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
  if (chosen[pair] >= experts) {                         // an identity expert: the token itself
    const int k = static_cast<int>(blockIdx.y) * kRowsPerBlock + threadIdx.x;
    if (threadIdx.x >= kRowsPerBlock || k >= K) return;
    const float y = weight[pair] * to_float<A>(x[t * K + k]);
    if (into_stream) add_float(out + t * K + k, col_scale != nullptr ? col_scale[k] * y : y);
    else out[(static_cast<int64_t>(j) * tokens + t) * K + k] = y;
    return;
  }
  const int e = max(chosen[pair], 0);
  for (int i = threadIdx.x; i < F; i += blockDim.x) rows_smem[i] = to_float<A>(act[pair * F + i]);
  __syncthreads();
  const A* we = w_down + static_cast<int64_t>(e) * K * F;
  float* o = out + (into_stream ? t : static_cast<int64_t>(j) * tokens + t) * K;
#pragma unroll
  for (int r = 0; r < kRowsPerWave; ++r) {
    const int k = static_cast<int>(blockIdx.y) * kRowsPerBlock + wave * kRowsPerWave + r;
    if (k >= K) break;
    const float v = wave_dot<A>(we + static_cast<int64_t>(k) * F, rows_smem, F, lane);
    if (lane != 0) continue;
    const float y = out_weight != nullptr ? out_weight[pair] * v : v;
    if (into_stream) add_float(o + k, col_scale != nullptr ? col_scale[k] * y : y);
    else o[k] = y;
  }
}


// ------------------------------------------------------------------ experts, grouped by expert

// How an expert's pairs are cut into tiles: up to `rows` of them each, the last with what is left, or, with rows 0, into as few as the
// limit of 256, 192 or 128 pairs that is best for this step's counts (tiles_time) allows (TileCut).
struct TileRule {
  int rows;
  int columns[2], length[2];           // rows == 0: columns of tiles and length of a tile's sums in the two products
};

// An expert's pairs in tiles as even as whole 64s allow: the first `larger` hold units + 1 64s, the others `units`, the last what is left.
// (Evenly by the pair, 800 are four tiles of 200, each as long as one of 256; so 256 + 192 + 192 + 160.)
struct TileCut {
  int tiles, units, larger;
  __device__ __forceinline__ TileCut(int pairs, int limit) {
    const int all = (pairs + 63) / 64;
    tiles = (pairs + limit - 1) / limit;                   // limit: a multiple of 64, so no tile holds more
    units = all / max(tiles, 1);
    larger = all - units * tiles;
  }
  __device__ __forceinline__ int first(int tile) const { return 64 * (tile * units + min(tile, larger)); }
};

// The time of a large tile by its 64s of pairs, in 1/64 of a full one's, as measured of the loop of eight waves that stood in wide_tile.h's place. There 128
// experts of 2,048 x 1,024 with 64, 128, 192 and 256 pairs each take 338, 388, 449 and 514 us (42, 48, 56, 64; before 342, 398, 485, 582); over 480
// steps (ten shapes, 64 to 2,000 pairs an expert, even to uneven) the limit that these numbers choose takes 0.3% more than the best of the three, 9% at most, and those of
// the new loop choose no better.
__device__ __forceinline__ int tile_cost(int units) { return units <= 2 ? 42 : units == 3 ? 54 : 64; }

// The time of the step's tiles under a limit of pairs, computed by one wave: every die runs an eighth of the tiles, 32 at once, and a
// round of them takes as long as its tiles do on average.
__device__ __forceinline__ int64_t tiles_time(const int32_t* count, int experts, int limit, const TileRule& rule, int lane) {
  int tiles = 0, cost = 0;
  for (int e = lane; e < experts; e += kWave) {
    const TileCut cut(count[e], limit);
    tiles += cut.tiles;
    cost += cut.larger * tile_cost(cut.units + 1) + (cut.tiles - cut.larger) * tile_cost(cut.units);
  }
#pragma unroll
  for (int o = kWave / 2; o > 0; o >>= 1) {
    tiles += __shfl_xor(tiles, o, kWave);
    cost += __shfl_xor(cost, o, kWave);
  }
  int64_t time = 0;
#pragma unroll
  for (int p = 0; p < 2; ++p)
    time += static_cast<int64_t>(((tiles * rule.columns[p] + 7) / 8 + 31) / 32) * rule.length[p] * (64 * cost / max(tiles, 1));
  return time;
}

constexpr size_t group_smem_ints(int experts) { return 4 * static_cast<size_t>(experts) + 5; }
// Whether the sorted pairs are laid out in LDS before they leave, in whole lines (us of the kernel and two products of next to nothing,
// straight / through LDS: 32 experts 1,024 pairs 10.9 / 11.1, 4,096 17.7 / 17.4, 16,384 23.8 / 22.1; 256 experts 11.6 / 11.7, 14.3 / 13.3,
// 27.0 / 22.2; 4 experts, whose pairs make long rows anyway, 4,096 18.8 / 19.2, 16,384 27.3 / 28.8).
static bool group_staged(int64_t pairs, int experts) { return experts >= 16 && pairs >= 2048 && pairs <= 16384; }

// One workgroup of 16 waves sorts the step's pairs by expert and lists the tiles that the products run over.
// ints: sorted[pairs] (pair indices, expert by expert), then per tile slot
// tile_expert, tile_first (index into sorted), tile_count; slots past the last tile hold -1; then the number of tiles.
// The order of an expert's pairs among themselves is whatever the atomics gave: every pair's
// result is computed from its own row alone, so it does not matter which rows share a tile.
// `identity`: the pairs of the last of the `experts` buckets have no tiles; where they begin in `sorted` stands in tile_first
// behind the last tile. One counter an expert: counters of the waves' own, added up, were slower at every size (measured as above, 32
// experts: 64 pairs 10.6 / 11.4, 1,024 10.9 / 11.6, 16,384 22.1 / 23.3).
__device__ __forceinline__ void group_pairs(const int32_t* __restrict__ chosen, int pairs, int experts, const TileRule& rule, bool identity,
                                            int max_tiles, int32_t* __restrict__ sorted, int32_t* __restrict__ tile_expert,
                                            int32_t* __restrict__ tile_first, int32_t* __restrict__ tile_count,
                                            int32_t* tiles_out, int32_t* smem, int32_t* staged) {
  int32_t *count = smem, *start = smem + experts, *tstart = smem + 2 * experts, *cursor = smem + 3 * experts, *listed = smem + 4 * experts;
  const int tiled = identity ? experts - 1 : experts;                            // buckets that have tiles
  for (int e = threadIdx.x; e < experts; e += blockDim.x) count[e] = 0;
  // Four choices a load, all of a step's first 16 x 1,024 asked for at once and kept for the second look.
  constexpr int kKept = 4;
  const int quads = reinterpret_cast<uintptr_t>(chosen) % 16 == 0 ? pairs / 4 : 0;
  auto bucket = [&](int c) { return min(max(c, 0), experts - 1); };
  int4 kept[kKept];
#pragma unroll
  for (int i = 0; i < kKept; ++i) {
    const int q = threadIdx.x + i * blockDim.x;
    kept[i] = q < quads ? reinterpret_cast<const int4*>(chosen)[q] : int4{0, 0, 0, 0};
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kKept; ++i) {
    if (static_cast<int>(threadIdx.x + i * blockDim.x) >= quads) break;
    atomicAdd(&count[bucket(kept[i].x)], 1);
    atomicAdd(&count[bucket(kept[i].y)], 1);
    atomicAdd(&count[bucket(kept[i].z)], 1);
    atomicAdd(&count[bucket(kept[i].w)], 1);
  }
  const int done = 4 * min(quads, kKept * static_cast<int>(blockDim.x));
#pragma unroll 4
  for (int p = done + threadIdx.x; p < pairs; p += blockDim.x) atomicAdd(&count[bucket(chosen[p])], 1);
  __syncthreads();
  if (rule.rows == 0) {                          // a wave each for limits of 256, 192 and 128 pairs
    if (const int w = threadIdx.x >> 6; w < 3) {
      const int64_t time = tiles_time(count, tiled, 256 - 64 * w, rule, threadIdx.x & 63);
      if ((threadIdx.x & 63) == 0) listed[2 + w] = static_cast<int>(min(time >> 8, static_cast<int64_t>(INT32_MAX)));
    }
    __syncthreads();
  }
  if (threadIdx.x < kWave) {                     // where every expert's pairs and tiles begin: sums over the wave's lanes
    const int lane = threadIdx.x;
    int limit = rule.rows;
    if (limit == 0) {
      int best = 0;
      for (int w = 1; w < 3; ++w)
        if (listed[2 + w] < listed[2 + best]) best = w;
      limit = 256 - 64 * best;
    }
    int at = 0, nt = 0;                          // of the experts in front of this run of 64
    for (int e0 = 0; e0 < experts; e0 += kWave) {
      const int e = e0 + lane;
      const int pairs_e = e < experts ? count[e] : 0, tiles_e = e < tiled ? (pairs_e + limit - 1) / limit : 0;
      int p_sum = pairs_e, t_sum = tiles_e;
#pragma unroll
      for (int o = 1; o < kWave; o <<= 1) {
        const int pp = __shfl_up(p_sum, o, kWave), tt = __shfl_up(t_sum, o, kWave);
        if (lane >= o) {
          p_sum += pp;
          t_sum += tt;
        }
      }
      if (e < experts) {
        start[e] = cursor[e] = at + p_sum - pairs_e;
        tstart[e] = nt + t_sum - tiles_e;
      }
      at += __shfl(p_sum, kWave - 1, kWave);
      nt += __shfl(t_sum, kWave - 1, kWave);
    }
    if (lane == 0) {
      listed[0] = min(nt, max_tiles);
      listed[1] = limit;
    }
  }
  __syncthreads();
  const int n_tiles = listed[0], limit = listed[1];
  for (int e = threadIdx.x; e < tiled; e += blockDim.x) {
    const int c = count[e], n = (c + limit - 1) / limit;
    const TileCut cut(c, limit);
    for (int i = 0, nt = tstart[e]; i < n && nt < max_tiles; ++i, ++nt) {
      const int from = rule.rows == 0 ? cut.first(i) : i * limit, to = rule.rows == 0 ? cut.first(i + 1) : from + limit;
      tile_expert[nt] = e;
      tile_first[nt] = start[e] + from;
      tile_count[nt] = min(to, c) - from;
    }
  }
  if (threadIdx.x == 0) *tiles_out = n_tiles;
  for (int nt = n_tiles + threadIdx.x; nt < max_tiles; nt += blockDim.x) tile_expert[nt] = -1;
  if (tiled < experts && threadIdx.x == 0 && n_tiles < max_tiles) tile_first[n_tiles] = start[tiled];
  int32_t* to = staged != nullptr ? staged : sorted;
#pragma unroll
  for (int i = 0; i < kKept; ++i) {
    const int q = threadIdx.x + i * blockDim.x;
    if (q >= quads) break;
    to[atomicAdd(&cursor[bucket(kept[i].x)], 1)] = 4 * q;
    to[atomicAdd(&cursor[bucket(kept[i].y)], 1)] = 4 * q + 1;
    to[atomicAdd(&cursor[bucket(kept[i].z)], 1)] = 4 * q + 2;
    to[atomicAdd(&cursor[bucket(kept[i].w)], 1)] = 4 * q + 3;
  }
#pragma unroll 4
  for (int p = done + threadIdx.x; p < pairs; p += blockDim.x) to[atomicAdd(&cursor[bucket(chosen[p])], 1)] = p;
  if (staged == nullptr) return;
  __syncthreads();
#pragma unroll 4
  for (int p = threadIdx.x; p < pairs; p += blockDim.x) sorted[p] = staged[p];
}

__global__ __launch_bounds__(1024) void moe_group_kernel(const int32_t* __restrict__ chosen, int pairs, int experts,
                                                         TileRule rule, int identity, int max_tiles, int staged,
                                                         int32_t* __restrict__ sorted, int32_t* __restrict__ tile_expert,
                                                         int32_t* __restrict__ tile_first, int32_t* __restrict__ tile_count) {
  extern __shared__ int32_t group_smem[];
  group_pairs(chosen, pairs, experts, rule, identity != 0, max_tiles, sorted, tile_expert, tile_first, tile_count, tile_count + max_tiles,
              group_smem, staged != 0 ? group_smem + group_smem_ints(experts) : nullptr);
}

// The choice from logits and the sorting in one workgroup of 16 waves, for steps of so few tokens
// that one workgroup does the choice at once (a decode step): a wave per token, then the sorting above.
__global__ __launch_bounds__(1024) void moe_topk_group_kernel(const float* __restrict__ z, int32_t* __restrict__ chosen,
                                                              float* __restrict__ weight, int tokens, int experts, int buckets, int top,
                                                              int tile_rows, int max_tiles, int32_t* __restrict__ sorted,
                                                              int32_t* __restrict__ tile_expert, int32_t* __restrict__ tile_first,
                                                              int32_t* __restrict__ tile_count, const float* __restrict__ bias,
                                                              RouterRule rule) {
  extern __shared__ int32_t group_smem[];      // the sorting's integers, then score[16][experts]
  float* score = reinterpret_cast<float*>(group_smem + group_smem_ints(buckets)) + (threadIdx.x >> 6) * experts;
  const int lane = threadIdx.x & (kWave - 1);
  for (int t = threadIdx.x >> 6; t < tokens; t += 16) {
    for (int e = lane; e < experts; e += kWave) score[e] = router_score(z[static_cast<int64_t>(t) * experts + e], bias, e, rule.mode);
    __builtin_amdgcn_wave_barrier();
    __threadfence_block();
    pick_top(score, experts, top, rule, chosen + t * top, weight + t * top, lane);
  }
  __threadfence_block();
  __syncthreads();                             // the workgroup's own writes of `chosen` are read below
  group_pairs(chosen, tokens * top, buckets, TileRule{tile_rows, {0, 0}, {0, 0}}, false, max_tiles, sorted, tile_expert, tile_first, tile_count,
              tile_count + max_tiles, group_smem, nullptr);
}

// k per staging round: with one tile of pairs a round of 64 leaves a wave two pieces of its matrix in flight, too few to
// hide a trip to memory.
constexpr int group_bk(int mt) { return mt == 1 ? 128 : 64; }

// One workgroup (4 waves) per (64 * RT output columns, tile of MT * 16 pairs of one expert). The
// pairs' input rows pass through LDS 64 k at a time (gathered through `sorted`). GATED: the
// pair's weight on the expert's input is applied to the float32 sums, gate (w x) = w (gate x),
// before the clamps: the same number without a rounding of w x, and no arithmetic while staging
// (scaling and rounding the rows there cost as many vector cycles as the matrix instructions). Every
// wave streams its 16 * RT rows of the expert's matrix from memory (GATED: gate rows and the up
// rows that belong to them) and multiplies them with all MT tiles of pairs. The next round's
// rows of both operands are asked for before the current round is multiplied (registers, then
// the other of two LDS buffers), so one barrier per round is all the waves wait for.
//   kFormGated:       out_act[pair][n] = act(gate, up) in bfloat16, N = F columns, w = [E][2N][K].
//   kFormSquaredRelu: out_act[pair][n] = max(sum, 0)^2 in bfloat16, N = F columns, w = [E][N][K].
//   kFormDown: out_f32[(pair % top) * tokens + pair / top][n] = sum, N = hidden columns, w = [E][N][K],
//              rows of `a` are indexed by pair; into_stream: out_f32[pair / top][n] += col_scale[n] * sum.
constexpr int kFormDown = 0, kFormGated = 1, kFormSquaredRelu = 2;
template <int MT, int RT, int FORM>
__global__ __launch_bounds__(256) void moe_grouped_kernel(
    const bf16_t* __restrict__ a, const float* __restrict__ pair_weight, const bf16_t* __restrict__ w,
    const int32_t* __restrict__ sorted, const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_first,
    const int32_t* __restrict__ tile_count, bf16_t* __restrict__ out_act, float* __restrict__ out_f32, int64_t tokens,
    int K, int N, int top, float gate_alpha, float limit, float up_shift, int into_stream,
    const float* __restrict__ col_scale, int experts, const bf16_t* __restrict__ x, const float* __restrict__ weight) {
  constexpr bool GATED = FORM == kFormGated;
  constexpr int kGroupBK = group_bk(MT);
  constexpr int kGroupLD = kGroupBK + 8;                     // LDS row stride of the staged pairs, in elements
  constexpr int ROWS = MT * 16;
  constexpr int PIECES = ROWS * (kGroupBK / 8);              // 16-byte pieces of a round's pairs
  constexpr int PPT = (PIECES + 255) / 256;                  // pieces per thread
  constexpr int KK = kGroupBK / 32;
  __shared__ __align__(16) bf16_t as[2][ROWS * kGroupLD];
  __shared__ int32_t pair_s[ROWS];
  const int slot = blockIdx.y;
  const int e = tile_expert[slot];
  if (e < 0) return;                            // uniform for the workgroup
  const int first = tile_first[slot], count = tile_count[slot];
  if (e >= experts) {                           // a tile of identity pairs: the tokens themselves times their weights
    if (FORM != kFormDown) return;
    constexpr int COLS = 64 * RT;
    for (int idx = threadIdx.x; idx < count * COLS; idx += 256) {
      const int pair = sorted[first + idx / COLS], n = static_cast<int>(blockIdx.x) * COLS + idx % COLS;
      if (n >= N) continue;
      const int64_t t = pair / top;
      const float y = weight[pair] * bf16_to_float(x[t * N + n]);
      if (into_stream) add_float(out_f32 + t * N + n, col_scale != nullptr ? col_scale[n] * y : y);
      else out_f32[(static_cast<int64_t>(pair % top) * tokens + t) * N + n] = y;
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int n0 = (static_cast<int>(blockIdx.x) * 4 + wave) * 16 * RT;     // this wave's first column
  if (threadIdx.x < ROWS) pair_s[threadIdx.x] = threadIdx.x < count ? sorted[first + threadIdx.x] : -1;
  const bf16_t* wg[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    const int nrow = min(n0 + rt * 16 + r, N - 1);
    wg[rt] = w + (static_cast<int64_t>(e) * (GATED ? 2 : 1) * N + nrow) * K + 8 * g;
  }
  const int64_t up_off = static_cast<int64_t>(N) * K;                      // GATED: from a gate row to its up row
  f32x4 acc_g[RT][MT], acc_u[RT][MT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc_g[rt][mt] = acc_u[rt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  __syncthreads();

  // This thread's pieces of a round: which pair's row, where from, its weight.
  const bf16_t* src[PPT];
#pragma unroll
  for (int p = 0; p < PPT; ++p) {
    const int idx = static_cast<int>(threadIdx.x) + p * 256;
    const int row = min(idx, PIECES - 1) / (kGroupBK / 8), c = min(idx, PIECES - 1) % (kGroupBK / 8);
    const int pair = pair_s[row];
    src[p] = (pair >= 0 && idx < PIECES) ? a + static_cast<int64_t>(FORM != kFormDown ? pair / top : pair) * K + 8 * c : nullptr;
  }
  uint4 areg[PPT];
  bf16x8 wa[KK][RT], wb[KK][RT];
  auto ask = [&](int k0) {                       // the round's rows of both operands, into registers
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int c8 = 8 * ((static_cast<int>(threadIdx.x) + p * 256) % (kGroupBK / 8));
      areg[p] = (src[p] != nullptr && k0 + c8 < K) ? *reinterpret_cast<const uint4*>(src[p] + k0) : make_uint4(0u, 0u, 0u, 0u);
    }
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      const int k = k0 + kk * 32;
      const bool in = k + 8 * g < K;            // K is a multiple of 8: a piece is inside or outside as a whole
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
#pragma unroll
        for (int i = 0; i < 8; ++i) wa[kk][rt][i] = wb[kk][rt][i] = static_cast<__bf16>(0.f);
        if (in) {
          wa[kk][rt] = *reinterpret_cast<const bf16x8*>(wg[rt] + k);
          if (GATED) wb[kk][rt] = *reinterpret_cast<const bf16x8*>(wg[rt] + up_off + k);
        }
      }
    }
  };
  auto stage = [&](int buf) {                    // the pairs' pieces from registers into LDS
#pragma unroll
    for (int p = 0; p < PPT; ++p) {
      const int idx = static_cast<int>(threadIdx.x) + p * 256;
      if (idx >= PIECES) continue;
      *reinterpret_cast<uint4*>(as[buf] + (idx / (kGroupBK / 8)) * kGroupLD + 8 * (idx % (kGroupBK / 8))) = areg[p];
    }
  };
  ask(0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int k0 = 0; k0 < K; k0 += kGroupBK, buf ^= 1) {
    bf16x8 ca[KK][RT], cb[KK][RT];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        ca[kk][rt] = wa[kk][rt];
        cb[kk][rt] = wb[kk][rt];
      }
    const bool more = k0 + kGroupBK < K;
    if (more) ask(k0 + kGroupBK);               // in flight while this round is multiplied
    // The pairs' operand of every step is read from LDS two steps ahead of the matrix instructions
    // that use it (read right in front of them, every group of four waited for its operand first).
    const bf16_t* bsrc = as[buf] + r * kGroupLD + 8 * g;
    auto b_of = [&](int step) {
      return *reinterpret_cast<const bf16x8*>(bsrc + (step % MT) * 16 * kGroupLD + (step / MT) * 32);
    };
    bf16x8 bq[3];
    bq[0] = b_of(0);
    if (KK * MT > 1) bq[1] = b_of(1);
#pragma unroll
    for (int step = 0; step < KK * MT; ++step) {
      const int kk = step / MT, mt = step % MT;
      if (step + 2 < KK * MT) bq[(step + 2) % 3] = b_of(step + 2);
      __builtin_amdgcn_sched_barrier(0);        // the read stays in front of this step's matrix instructions
      const bf16x8 b = bq[step % 3];
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) {
        acc_g[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ca[kk][rt], b, acc_g[rt][mt], 0, 0, 0);
        if (GATED) acc_u[rt][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cb[kk][rt], b, acc_u[rt][mt], 0, 0, 0);
      }
    }
    if (more) stage(buf ^ 1);                   // nobody reads that buffer: all passed the last barrier after reading it
    __syncthreads();
  }
  // Lane (r, g) holds, for the pair in row mt * 16 + r, the four columns n0 + rt * 16 + 4 g .. + 3.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int pair = pair_s[mt * 16 + r];
    if (pair < 0) continue;
    const float pw = pair_weight != nullptr ? pair_weight[pair] : 1.f;   // on the input's sums (GATED) or on the output's
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int nc = n0 + rt * 16 + 4 * g;
      if (FORM != kFormDown) {
        bf16_t* o = out_act + static_cast<int64_t>(pair) * N + nc;
        bf16_t res[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (!GATED) {
            const float p = fmaxf(pw * acc_g[rt][mt][v], 0.f);
            res[v] = float_to_bf16(p * p);
            continue;
          }
          const float gg = fminf(pw * acc_g[rt][mt][v], limit);
          const float uu = fminf(fmaxf(pw * acc_u[rt][mt][v], -limit), limit);
          res[v] = float_to_bf16(gg / (1.f + __expf(-gate_alpha * gg)) * (uu + up_shift));
        }
        if (nc + 3 < N && (N & 3) == 0) {
          *reinterpret_cast<ushort4*>(o) = ushort4{res[0], res[1], res[2], res[3]};
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nc + v < N) o[v] = res[v];
        }
      } else if (into_stream) {
        float* o = out_f32 + static_cast<int64_t>(pair / top) * N + nc;
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (nc + v < N) add_float(o + v, (col_scale != nullptr ? col_scale[nc + v] : 1.f) * (pw * acc_g[rt][mt][v]));
      } else {
        float* o = out_f32 + (static_cast<int64_t>(pair % top) * tokens + pair / top) * N + nc;
        if (nc + 3 < N && (N & 3) == 0) {
          *reinterpret_cast<float4*>(o) = float4{pw * acc_g[rt][mt][0], pw * acc_g[rt][mt][1], pw * acc_g[rt][mt][2], pw * acc_g[rt][mt][3]};
        } else {
#pragma unroll
          for (int v = 0; v < 4; ++v)
            if (nc + v < N) o[v] = pw * acc_g[rt][mt][v];
        }
      }
    }
  }
}

// The same tiles of up to 16 pairs with both operands through LDS in whole lines, for K and F multiples of 64 (the kernel above loads its matrix as a
// matrix instruction's operand, 16 rows x 64 bytes, one round ahead). TN columns a workgroup; steps, units, buffers and waves as in
// stream_tiles_kernel (linear_stream.hip). Bound by reading the used experts' matrices once; each workgroup begins at another place of K, as rows
// of w lie a power of two apart (that alone gave the kernel above 10%). us of routing and experts, above / here (TB/s of the used experts' matrices):
//   32 experts of 2,048 x 1,024, 8 choices, 1, 2, 4, 8, 16 and 64 tokens   45.8, 52.5, 78.0, 96.6, 104.7, 126.6 / 34.7, 42.9, 69.0, 81.1, 88.3 (4.6), 101.7
//    the same without gates                                              32.4, 43.6, 65.7, 75.5,  74.0,  85.2 / 26.7, 38.9, 57.2, 65.2, 65.8, 76.1
//    8 of 4,096 x 3,584, 2 choices, 1, 8, 16, 64                         78.1, 145.9, 158.8, 210.5 / 51.0, 122.3, 134.8 (5.2), 160.5
//   64 of 2,048 x 1,408, 6 choices, 1, 2, 8, 16                          39.5, 57.9, 140.9, 206.0 / 33.0, 62.4, 110.7, 169.9
// (1 and 2 tokens: pair by pair before.)
template <int TN, int KG, int STAGES, int FORM>
__global__ __launch_bounds__(64 * (TN / 16) * KG) void moe_stream_kernel(
    const bf16_t* __restrict__ a, const float* __restrict__ pair_weight, const bf16_t* __restrict__ w,
    const int32_t* __restrict__ sorted, const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_first,
    const int32_t* __restrict__ tile_count, bf16_t* __restrict__ out_act, float* __restrict__ out_f32, int64_t tokens,
    int K, int N, int top, float gate_alpha, float limit, float up_shift, int into_stream,
    const float* __restrict__ col_scale, int experts, const bf16_t* __restrict__ x, const float* __restrict__ weight) {
  constexpr bool GATED = FORM == kFormGated;
  constexpr int CT = TN / 16, RT = GATED ? 2 : 1, ROWS = TN * RT, W = CT * KG, LW = KG * ROWS / 8 / W;
  constexpr int XC = 2 * KG, LX = (XC + W - 1) / W;                              // copies of 8 pairs a step, of a wave
  constexpr int W_STEP = KG * ROWS * 128, STEP = W_STEP + KG * 2048;
  static_assert(LW * 8 * W == KG * ROWS && (XC % W == 0 || W % XC == 0), "whole copies per wave");
  static_assert(W * RT * 1024 <= STAGES * STEP, "the sums of the units' waves fit where the steps were");
  extern __shared__ __align__(16) unsigned char moe_smem[];                      // STAGES x [KG][ROWS rows of w][128], [KG][16 pairs][128]
  const int slot = blockIdx.y;
  const int e = tile_expert[slot];
  if (e < 0) return;                            // uniform for the workgroup
  const int first = tile_first[slot], count = tile_count[slot];
  const int n0 = static_cast<int>(blockIdx.x) * TN;
  if (e >= experts) {                           // a tile of identity pairs: the tokens themselves times their weights
    if (FORM != kFormDown) return;
    for (int idx = threadIdx.x; idx < count * TN; idx += blockDim.x) {
      const int pair = sorted[first + idx / TN], n = n0 + idx % TN;
      if (n >= N) continue;
      const int64_t t = pair / top;
      const float y = weight[pair] * bf16_to_float(x[t * N + n]);
      if (into_stream) add_float(out_f32 + t * N + n, col_scale != nullptr ? col_scale[n] * y : y);
      else out_f32[(static_cast<int64_t>(pair % top) * tokens + t) * N + n] = y;
    }
    return;
  }
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4;
  const char* wb = reinterpret_cast<const char*>(w + static_cast<int64_t>(e) * (GATED ? 2 : 1) * N * K);
  const char* ab = reinterpret_cast<const char*>(a);
  uint32_t w_off[LW], x_off[LX];
#pragma unroll
  for (int i = 0; i < LW; ++i) {
    const int row = (wave * LW + i) % (ROWS / 8) * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    const int col = min(n0 + row % TN, N - 1);
    w_off[i] = static_cast<uint32_t>(row >= TN ? N + col : col) * (2u * K) + 16u * piece;
  }
#pragma unroll
  for (int i = 0; i < LX; ++i) {                // where waves outnumber the copies, some bring the same rows to the same place
    const int row = (wave * LX + i) % 2 * 8 + (lane >> 3), piece = (lane & 7) ^ ((row >> 1) & 7);
    const int pair = sorted[first + min(row, count - 1)];
    x_off[i] = static_cast<uint32_t>(FORM != kFormDown ? pair / top : pair) * (2u * K) + 16u * piece;
  }
  const int units = K / 64, steps = (units + KG - 1) / KG, end = units * 128;
  // By columns and expert, never by the tile: the sorting puts an expert's pairs into its tiles in any order, and a pair's sums keep theirs.
  int from = static_cast<int>((blockIdx.x + 5u * static_cast<unsigned>(e)) % static_cast<unsigned>(units)) * 128, to = 0;
  auto unit_at = [&](int unit) {
    const int k = from + unit * 128;
    return min(k >= end ? k - end : k, end - 128);
  };
  auto copy = [&]() {
#pragma unroll
    for (int i = 0; i < LW; ++i) {
      const int at = wave * LW + i;
      __builtin_amdgcn_global_load_lds((global_ptr)(wb + unit_at(at / (ROWS / 8)) + w_off[i]), (lds_ptr)(moe_smem + to + at * 1024), 16, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < LX; ++i) {
      const int at = (wave * LX + i) % XC;
      __builtin_amdgcn_global_load_lds((global_ptr)(ab + unit_at(at / 2) + x_off[i]), (lds_ptr)(moe_smem + to + W_STEP + at * 1024), 16, 0, 0);
    }
    from = min(from + KG * 128 >= end ? from + KG * 128 - end : from + KG * 128, end - 128);
    to = to + STEP == STAGES * STEP ? 0 : to + STEP;
  };
#pragma unroll
  for (int t = 0; t < STAGES - 1; ++t)
    if (t < steps) copy();
  f32x4 acc[RT];
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) acc[rt] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int tile = wave % CT, unit = wave / CT;
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_bytes)moe_smem)), piece0 = 16u * (g ^ ((r >> 1) & 7));
  const uint32_t w_at = base + (unit * ROWS + 16 * tile + r) * 128 + piece0, x_at = base + W_STEP + (unit * 16 + r) * 128 + piece0;
  uint32_t at = 0;
  for (int t = 0; t < steps; ++t) {
    __builtin_amdgcn_sched_barrier(0);
    wait_for_step<LW + LX, STAGES - 2>(steps - 1 - t);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + STAGES - 1 < steps) copy();
    __builtin_amdgcn_sched_barrier(0);
    if (t * KG + unit < units) {
      Operands<TN, RT, 1> ops;
      ops.read(w_at + at, x_at + at);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int rt = 0; rt < RT; ++rt) acc[rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ops.w[h][rt], ops.x[h][0], acc[rt], 0, 0, 0);
    }
    at = at + STEP == STAGES * STEP ? 0 : at + STEP;
  }
  f32x4* const parts = reinterpret_cast<f32x4*>(moe_smem);                       // [KG][CT][RT][64 lanes]
  __syncthreads();
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) parts[(wave * RT + rt) * 64 + lane] = acc[rt];
  __syncthreads();
  if (wave >= CT) return;
#pragma unroll
  for (int rt = 0; rt < RT; ++rt) {
    acc[rt] = parts[(wave * RT + rt) * 64 + lane];
#pragma unroll
    for (int q = 1; q < KG; ++q) acc[rt] += parts[((q * CT + wave) * RT + rt) * 64 + lane];
  }
  // Lane (r, g) holds, for the pair in row r, columns 4 g .. + 3 of its wave's sixteen.
  const int nc = n0 + 16 * tile + 4 * g;
  if (r >= count || nc >= N) return;                                             // N is a multiple of 8
  const int pair = sorted[first + r];
  const float pw = pair_weight != nullptr ? pair_weight[pair] : 1.f;             // on the input's sums (GATED) or on the output's
  if (FORM != kFormDown) {
    bf16_t res[4];
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      if (!GATED) {
        const float p = fmaxf(pw * acc[0][v], 0.f);
        res[v] = float_to_bf16(p * p);
        continue;
      }
      const float gg = fminf(pw * acc[0][v], limit);
      const float uu = fminf(fmaxf(pw * acc[RT - 1][v], -limit), limit);
      res[v] = float_to_bf16(gg / (1.f + __expf(-gate_alpha * gg)) * (uu + up_shift));
    }
    *reinterpret_cast<ushort4*>(out_act + static_cast<int64_t>(pair) * N + nc) = ushort4{res[0], res[1], res[2], res[3]};
  } else if (into_stream) {
    float* o = out_f32 + static_cast<int64_t>(pair / top) * N + nc;
#pragma unroll
    for (int v = 0; v < 4; ++v) add_float(o + v, (col_scale != nullptr ? col_scale[nc + v] : 1.f) * (pw * acc[0][v]));
  } else {
    *reinterpret_cast<float4*>(out_f32 + (static_cast<int64_t>(pair % top) * tokens + pair / top) * N + nc) =
        float4{pw * acc[0][0], pw * acc[0][1], pw * acc[0][2], pw * acc[0][3]};
  }
}

// ------------------------------------------------------------------ experts, many pairs each

// A tile of up to 256 pairs by 256 rows of the expert's matrix, or 128 by 128, per workgroup, both operands through LDS 64 k at a
// time (wide_tile.h and tile_product.h have the loops). The matrices of all experts are read at the rate the matrix cores use them only if a
// workgroup multiplies each byte often: 256 x 256 asks for half the bytes per product of the kernel above, whose rows of the matrix go
// from memory to registers for one tile of 128 pairs (14 TB/s out of the L2s). What it does about each bound:
//  * an expert's tiles run on one die (its L2 then holds the expert's rows): die d takes the d-th eighth of the work;
//  * a chip of 256 units runs large tiles in a few rounds, whose last one is seldom full, and an expert with a few pairs more than
//    whole tiles costs one more: the sorting cuts every expert's pairs into near-even tiles under the limit (256, 192 or 128)
//    that gives the step's counts the least time, and a tile runs the loop that is made for its size;
//  * us of sorting and products, tiles of 256 and a rest in one loop / cut evenly by the pair / so, 32 experts of 2,048 x 1,024: 66 pairs
//    an expert 119 / 119 / 112, 160 136 / 142 / 134, 256 208 / 189 / 164, 512 328 / 294 / 287, 1,000 552 / 561 / 584, 1,400 681 / 693 / 704; 8 of
//    4,096 x 3,584: 256 356 / 340 / 317, 512 590 / 573 / 562, 1,400 1,165 / 1,197 / 1,182. Over 274 steps (eight shapes, 52 to 2,000 pairs, even and
//    uneven) 0.91 of the time of tiles of 256 and a rest, 0.97 of that of the even cut (all of them with the loop before wide_tile.h's);
//  * as many workgroups as there are units stay and walk the large tiles, the copies of one under the end of the one before: that and waves of 128
//    x 128 against eight of 128 x 64 that began each tile anew, us of sorting and both products, 32 experts of 2,048 x 1,024: 448 pairs an expert
//    225 -> 204, 512 273 -> 249 (all even 242 -> 227), 1,024 525 -> 455; 8 of 4,096 x 3,584 at 512 526 -> 469; 64 of 2,048 x 1,408 at 192 345 -> 314. Over 480 steps
//    0.88 of the time, and 1.02 to 1.05 in twelve of them, mostly of 90 to 128 pairs an expert (32 of 2,048 x 1,024 at 90 116 -> 118, at 128 123 -> 127, 32 of 4,096 x
//    2,048 at 90 349 -> 357): every tile's copies are those of 256 rows, and eight waves asked for a step more of the matrices where a tile had fewer.
//    What is left of 249: gate and up 136 (one tile after the other 1.6 us a step of 64 k where the dense product takes 1.4: 268 MB of matrices come from
//    memory meanwhile; 4 us of activations behind each tile, under which no matrix core works), down 90 (134 MB of float32 leave, 134 MB of matrices come).
// GATED: a wave's rows of the matrix are gate rows and then the up rows of the same columns.

// The identity pairs lie behind the experts' and have no tiles: the tokens themselves times their weights, dealt out over all threads.
__device__ __forceinline__ void copy_identity(const int32_t* __restrict__ sorted, int begin, int end, const bf16_t* __restrict__ x,
                                              const float* __restrict__ weight, float* __restrict__ out_f32, int64_t tokens, int N, int top,
                                              int into_stream, const float* __restrict__ col_scale) {
  const int quads = N / 4;                                                       // N is a multiple of 8
  const int64_t all = static_cast<int64_t>(end - begin) * quads, step = static_cast<int64_t>(gridDim.x) * blockDim.x;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < all; i += step) {
    const int pair = sorted[begin + i / quads], n = static_cast<int>(i % quads) * 4;
    const int64_t t = pair / top;
    const float wt = weight[pair];
    const ushort4 in = *reinterpret_cast<const ushort4*>(x + t * N + n);
    const float4 y{wt * bf16_to_float(in.x), wt * bf16_to_float(in.y), wt * bf16_to_float(in.z), wt * bf16_to_float(in.w)};
    if (into_stream) {
      const float* ys = &y.x;
#pragma unroll
      for (int v = 0; v < 4; ++v) add_float(out_f32 + t * N + n + v, col_scale != nullptr ? col_scale[n + v] * ys[v] : ys[v]);
    } else {
      *reinterpret_cast<float4*>(out_f32 + (static_cast<int64_t>(pair % top) * tokens + t) * N + n) = y;
    }
  }
}

// The small tiles: one a workgroup, two workgroups a unit.
constexpr int kSmallTile = 128, kSmallSmem = 2 * 2 * kSmallTile * 128;

template <int FORM>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(
    const bf16_t* __restrict__ a, const float* __restrict__ pair_weight, const bf16_t* __restrict__ w,
    const int32_t* __restrict__ sorted, const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_first,
    const int32_t* __restrict__ tile_count, const int32_t* __restrict__ n_tiles, bf16_t* __restrict__ out_act,
    float* __restrict__ out_f32, int64_t tokens, int K, int N, int top, float gate_alpha, float limit, float up_shift,
    int into_stream, const float* __restrict__ col_scale, int identity_to, const bf16_t* __restrict__ x,
    const float* __restrict__ weight, int column_tiles) {
  constexpr bool GATED = FORM == kFormGated;
  constexpr int TM = kSmallTile, TN = kSmallTile, BK = 64, RM = 4, RN = 4, WROWS = TN / 2, LA = 4, LB = 4;   // four waves of 64 x 64
  constexpr int COLS = GATED ? TN / 2 : TN, WCOLS = GATED ? WROWS / 2 : WROWS;   // columns of the workgroup, of a wave
  extern __shared__ __align__(16) unsigned char tile_smem[];                     // two steps, then int32_t[TM]
  int32_t* pair_s = reinterpret_cast<int32_t*>(tile_smem + kSmallSmem);
  // The work of this workgroup's die: an eighth of all (tile, columns).
  const int tiles = *n_tiles, die = static_cast<int>(blockIdx.x & 7);
  const int from = static_cast<int>(static_cast<int64_t>(tiles) * column_tiles * die / 8);
  const int to = static_cast<int>(static_cast<int64_t>(tiles) * column_tiles * (die + 1) / 8);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4, wn = wave & 1;
  if (const int at = from + static_cast<int>(blockIdx.x >> 3); at < to) {        // uniform for the workgroup
    const int slot = at / column_tiles, n0 = at % column_tiles * COLS;
    const int e = tile_expert[slot], first = tile_first[slot], count = min(tile_count[slot], TM);
    const char* w_base = reinterpret_cast<const char*>(w + static_cast<int64_t>(e) * (GATED ? 2 : 1) * N * K);
    if (threadIdx.x < TM) pair_s[threadIdx.x] = static_cast<int>(threadIdx.x) < count ? sorted[first + threadIdx.x] : -1;
    __syncthreads();
    uint32_t a_off[LA], b_off[LB];
#pragma unroll
    for (int i = 0; i < LA; ++i) {
      const int row = (wave * LA + i) * 8 + (lane >> 3);
      const int pair = pair_s[min(row, count - 1)];
      a_off[i] = static_cast<uint32_t>(FORM != kFormDown ? pair / top : pair) * (2u * K) + 16u * tile_copy_piece(row, lane);
    }
#pragma unroll
    for (int i = 0; i < LB; ++i) {
      const int row = (wave * LB + i) * 8 + (lane >> 3);
      const int col = min(n0 + (row / WROWS) * WCOLS + row % WCOLS, N - 1);
      b_off[i] = static_cast<uint32_t>(GATED && row % WROWS >= WCOLS ? N + col : col) * (2u * K) + 16u * tile_copy_piece(row, lane);
    }
    const int wm = wave / 2 * (RM * 16);
    const bool works = wm < count;               // the waves for pairs that a tile does not have skip the arithmetic
    tile_f32x4 acc[RN][RM];
#pragma unroll
    for (int i = 0; i < RN; ++i)
#pragma unroll
      for (int j = 0; j < RM; ++j) acc[i][j] = tile_f32x4{0.f, 0.f, 0.f, 0.f};
    tile_product<2, TM, TN>(acc, tile_smem, reinterpret_cast<const char*>(a), w_base, a_off, b_off, wm, wn * WROWS, wave, lane, K / BK, works);
    // Lane (r, g) holds, for the pair in row wm + 16 j + r, columns 4 g .. + 3 of every 16 of the wave's.
#pragma unroll
    for (int j = 0; j < RM; ++j) {
      const int pair = pair_s[wm + j * 16 + r];
      if (pair < 0) continue;
      const float pw = pair_weight != nullptr ? pair_weight[pair] : 1.f;       // on the input's sums (GATED) or on the output's
#pragma unroll
      for (int i = 0; i < WCOLS / 16; ++i) {
        const int nc = n0 + wn * WCOLS + i * 16 + 4 * g;
        if (nc >= N) continue;                                                 // N is a multiple of 8
        if (FORM != kFormDown) {
          bf16_t res[4];
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            if (!GATED) {
              const float p = fmaxf(pw * acc[i][j][v], 0.f);
              res[v] = float_to_bf16(p * p);
              continue;
            }
            const float gg = fminf(pw * acc[i][j][v], limit);
            const float uu = fminf(fmaxf(pw * acc[(i + RN / 2) % RN][j][v], -limit), limit);
            res[v] = float_to_bf16(gg / (1.f + __expf(-gate_alpha * gg)) * (uu + up_shift));
          }
          *reinterpret_cast<ushort4*>(out_act + static_cast<int64_t>(pair) * N + nc) = ushort4{res[0], res[1], res[2], res[3]};
        } else if (into_stream) {
          float* o = out_f32 + static_cast<int64_t>(pair / top) * N + nc;
#pragma unroll
          for (int v = 0; v < 4; ++v) add_float(o + v, (col_scale != nullptr ? col_scale[nc + v] : 1.f) * (pw * acc[i][j][v]));
        } else {
          float* o = out_f32 + (static_cast<int64_t>(pair % top) * tokens + pair / top) * N + nc;
          *reinterpret_cast<float4*>(o) = float4{pw * acc[i][j][0], pw * acc[i][j][1], pw * acc[i][j][2], pw * acc[i][j][3]};
        }
      }
    }
  }
  if (FORM == kFormDown && identity_to != 0)
    copy_identity(sorted, tile_first[tiles], identity_to, x, weight, out_f32, tokens, N, top, into_stream, col_scale);
}

// The large ones of these tiles (256 x 256; wide_tile.h has the loop): workgroups of four waves that stay and walk their die's eighth of the work.
template <int FORM>
struct ExpertTiles {
  const float* __restrict__ pair_weight;
  const bf16_t* __restrict__ matrices;
  const int32_t* __restrict__ sorted;
  const int32_t* __restrict__ tile_expert;
  const int32_t* __restrict__ tile_first;
  const int32_t* __restrict__ tile_count;
  bf16_t* __restrict__ out_act;
  float* __restrict__ out_f32;
  const float* __restrict__ col_scale;
  int64_t tokens;
  int K, N, top, into_stream, column_tiles, from, to, at_once;
  float gate_alpha, limit, up_shift;

  static constexpr bool GATED = FORM == kFormGated;
  static constexpr int kMinSteps = 4;           // a_rows takes the pairs that ahead() asked for
  static constexpr int WROWS = kWideTile / 2, WCOLS = GATED ? WROWS / 2 : WROWS, COLS = 2 * WCOLS;
  struct Item {
    int expert, first, count, n0;
  };
  const char* w;
  int round, lane, wave;
  bool has_next;
  Item cur, nxt;                                // the tile that is multiplied, the one behind it
  int row_pair, out_pair[2];                    // of the copies' row 64 wave + lane of the next tile; of this tile's rows of this wave

  // What follows from the lane alone would be computed in front of all tiles and held through them, where no register is free.
  __device__ __forceinline__ int own_lane() const {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  }
  // Each round its place moves on by a tile's columns: an expert's last tile is often a smaller one, and a workgroup that always took the
  // same place would have it every time, or never.
  __device__ __forceinline__ void look() {
    const int at = from + round * at_once + static_cast<int>((blockIdx.x >> 3) + static_cast<unsigned>(round) * column_tiles) % at_once;
    has_next = at < to;
    if (!has_next) return;
    const int slot = at / column_tiles;
    auto one = [](int v) { return __builtin_amdgcn_readfirstlane(v); };          // uniform, where the compiler can't see it
    nxt = Item{one(tile_expert[slot]), one(tile_first[slot]), one(min(tile_count[slot], kWideTile)), one(at % column_tiles * COLS)};
    ++round;
  }
  __device__ __forceinline__ void start() {
    lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    round = 0;
    look();
    if (has_next) ask_rows();
  }
  __device__ __forceinline__ void ask_rows() { row_pair = sorted[nxt.first + min(64 * wave + lane, nxt.count - 1)]; }
  __device__ __forceinline__ void ahead() {
    if (has_next) ask_rows();
  }
  __device__ __forceinline__ int rows() {
    cur = nxt;
    look();
    const int at = (wave >> 1) * (16 * rows16(cur.count)) + lane;
#pragma unroll
    for (int h = 0; h < 2; ++h) out_pair[h] = sorted[cur.first + min(at + 64 * h, cur.count - 1)];
    return cur.count;
  }
  static __device__ __forceinline__ int rows16(int count) { return count <= 64 ? 2 : (count <= 128 ? 4 : (count <= 192 ? 6 : 8)); }
  __device__ __forceinline__ bool a_rows(uint32_t (&off)[8]) {
    if (!has_next) return false;
    const int lane = own_lane();
    const int at = static_cast<int>(static_cast<uint32_t>(FORM != kFormDown ? row_pair / top : row_pair) * (2u * K));
#pragma unroll
    for (int i = 0; i < 8; ++i) off[i] = static_cast<uint32_t>(__shfl(at, 8 * i + (lane >> 3), kWave)) + wide_piece(8 * i + (lane >> 3), lane);
    return true;
  }
  // Columns of the two bfloat16 forms: a lane's four of two neighbouring tiles of 16 stand side by side, 16 bytes of the output.
  __device__ __forceinline__ bool w_rows(uint32_t (&off)[8]) {
    if (!has_next) return false;
    const int lane = own_lane();
    w = reinterpret_cast<const char*>(matrices + static_cast<int64_t>(nxt.expert) * (GATED ? 2 : 1) * N * K);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = (wave * 8 + i) * 8 + (lane >> 3), in = row % WCOLS;
      const int c = FORM == kFormDown ? in : (in & ~31) + (in >> 2 & 3) * 8 + (in >> 4 & 1) * 4 + (in & 3);
      const int col = min(nxt.n0 + row / WROWS * WCOLS + c, N - 1);
      off[i] = wide_row(GATED && row % WROWS >= WCOLS ? N + col : col, K) + wide_piece(8 * i + (lane >> 3), lane);
    }
    return true;
  }
  template <int RM>
  __device__ __forceinline__ bool finish(tile_f32x4 (&acc)[8][RM]) {
    const int lane = own_lane(), r = lane & 15, g = lane >> 4, wm = (wave >> 1) * (16 * RM);
    int pair[RM];
    float weight[RM];
#pragma unroll
    for (int j = 0; j < RM; ++j) {
      pair[j] = __shfl(out_pair[j / 4], (16 * j + r) % kWave, kWave);
      weight[j] = pair_weight != nullptr ? pair_weight[pair[j]] : 1.f;            // on the input's sums (GATED) or on the output's
    }
#pragma unroll
    for (int j = 0; j < RM; ++j) {
      if (wm + 16 * j + r >= cur.count) continue;
      const float pw = weight[j];
      const int c0 = cur.n0 + (wave & 1) * WCOLS;
      if constexpr (FORM != kFormDown) {
        bf16_t* o = out_act + static_cast<int64_t>(pair[j]) * N;
#pragma unroll
        for (int i = 0; i < WCOLS / 16; i += 2) {
          const int nc = c0 + i * 16 + 8 * g;
          if (nc >= N) continue;                                                 // N is a multiple of 64
          union {
            bf16_t h[8];
            uint4 v;
          } res;
#pragma unroll
          for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              if (!GATED) {
                const float p = fmaxf(pw * acc[i + q][j][v], 0.f);
                res.h[4 * q + v] = float_to_bf16(p * p);
                continue;
              }
              const float gg = fminf(pw * acc[i + q][j][v], limit);
              const float uu = fminf(fmaxf(pw * acc[(i + q + 4) % 8][j][v], -limit), limit);
              res.h[4 * q + v] = float_to_bf16(gg / (1.f + __expf(-gate_alpha * gg)) * (uu + up_shift));
            }
          *reinterpret_cast<uint4*>(o + nc) = res.v;
          __builtin_amdgcn_sched_barrier(0);                                     // a few sums at a time leave the accumulator registers
        }
      } else {
        const int64_t row = into_stream ? pair[j] / top : static_cast<int64_t>(pair[j] % top) * tokens + pair[j] / top;
        float* o = out_f32 + row * N;
#pragma unroll
        for (int i = 0; i < WCOLS / 16; ++i) {
          const int nc = c0 + i * 16 + 4 * g;
          if (nc >= N) continue;
          const tile_f32x4 y = {pw * acc[i][j][0], pw * acc[i][j][1], pw * acc[i][j][2], pw * acc[i][j][3]};
          if (!into_stream) {
            *reinterpret_cast<tile_f32x4*>(o + nc) = y;
          } else {
#pragma unroll
            for (int v = 0; v < 4; ++v) add_float(o + nc + v, (col_scale != nullptr ? col_scale[nc + v] : 1.f) * y[v]);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    return has_next;
  }
};

template <int FORM>
__global__ __launch_bounds__(kWideThreads, 1) void moe_wide_kernel(
    const bf16_t* __restrict__ a, const float* __restrict__ pair_weight, const bf16_t* __restrict__ w,
    const int32_t* __restrict__ sorted, const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ tile_first,
    const int32_t* __restrict__ tile_count, const int32_t* __restrict__ n_tiles, bf16_t* __restrict__ out_act,
    float* __restrict__ out_f32, int64_t tokens, int K, int N, int top, float gate_alpha, float limit, float up_shift,
    int into_stream, const float* __restrict__ col_scale, int identity_to, const bf16_t* __restrict__ x,
    const float* __restrict__ weight, int column_tiles) {
  extern __shared__ __align__(16) unsigned char wide_smem[];
  const int64_t work = static_cast<int64_t>(*n_tiles) * column_tiles;
  const int die = static_cast<int>(blockIdx.x & 7);
  ExpertTiles<FORM> tiles;
  tiles.pair_weight = pair_weight, tiles.matrices = w, tiles.sorted = sorted, tiles.tile_expert = tile_expert, tiles.tile_first = tile_first;
  tiles.tile_count = tile_count, tiles.out_act = out_act, tiles.out_f32 = out_f32, tiles.col_scale = col_scale, tiles.tokens = tokens;
  tiles.K = K, tiles.N = N, tiles.top = top, tiles.into_stream = into_stream, tiles.column_tiles = column_tiles;
  tiles.from = static_cast<int>(work * die / 8), tiles.to = static_cast<int>(work * (die + 1) / 8), tiles.at_once = static_cast<int>(gridDim.x >> 3);
  tiles.gate_alpha = gate_alpha, tiles.limit = limit, tiles.up_shift = up_shift;
  tiles.start();
  wide_tiles(tiles, reinterpret_cast<const char*>(a), wide_smem, K / 64);
  if (FORM == kFormDown && identity_to != 0)
    copy_identity(sorted, tile_first[*n_tiles], identity_to, x, weight, out_f32, tokens, N, top, into_stream, col_scale);
}

// What the experts' two products have in common.
struct ExpertCall {
  const void* x;
  const int32_t* chosen;
  const float* weight;
  const void* w_in;                    // [E, 2F, K] (gated) or [E, F, K]
  const void* w_down;                  // [E, K, F]
  void* act;
  float* out;
  int64_t tokens;
  int K, F, experts, identity, top, kind;        // experts: those with matrices
  float gate_alpha, limit, up_shift;
  int weight_on_output, into_stream;
  const float* col_scale;
};

template <int MT, int RT, int FORM>
static void run_grouped(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  const int32_t* sorted = ints;
  const int32_t* t_e = ints + c.tokens * c.top;
  const int32_t* t_f = t_e + max_tiles;
  const int32_t* t_c = t_f + max_tiles;
  constexpr bool down = FORM == kFormDown;
  const int N = down ? c.K : c.F, K = down ? c.F : c.K;
  const dim3 grid(static_cast<unsigned>(ceil_div(N, 64 * RT)), static_cast<unsigned>(max_tiles));
  moe_grouped_kernel<MT, RT, FORM><<<grid, dim3(256), 0, s>>>(
      static_cast<const bf16_t*>(down ? c.act : c.x), (c.weight_on_output != 0) == down ? c.weight : nullptr,
      static_cast<const bf16_t*>(down ? c.w_down : c.w_in), sorted, t_e, t_f, t_c, down ? nullptr : static_cast<bf16_t*>(c.act),
      down ? c.out : nullptr, c.tokens, K, N, c.top, c.gate_alpha, c.limit, c.up_shift, c.into_stream, c.col_scale, c.experts,
      static_cast<const bf16_t*>(c.x), c.weight);
}

template <int MT, int RT>
static int launch_grouped(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  if (c.kind == kExpertGated) run_grouped<MT, RT, kFormGated>(s, c, ints, max_tiles);
  else run_grouped<MT, RT, kFormSquaredRelu>(s, c, ints, max_tiles);
  if (check_launch("psamd_moe_experts_grouped (in)")) return 1;
  run_grouped<MT, RT, kFormDown>(s, c, ints, max_tiles);
  return check_launch("psamd_moe_experts_grouped (down)");
}

template <int TN, int FORM>
static int run_stream(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  constexpr int KG = 128 / TN, STAGES = FORM == kFormGated ? 2 : 3;              // two workgroups share a compute unit
  constexpr size_t smem = static_cast<size_t>(STAGES) * KG * ((FORM == kFormGated ? 2 : 1) * TN + 16) * 128;
  auto kernel = moe_stream_kernel<TN, KG, STAGES, FORM>;
  if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("psamd_moe_experts_grouped: " + std::to_string(smem) + " bytes of LDS were refused");
  const int32_t* t_e = ints + c.tokens * c.top;
  constexpr bool down = FORM == kFormDown;
  const int N = down ? c.K : c.F, K = down ? c.F : c.K;
  kernel<<<dim3(static_cast<unsigned>(ceil_div(N, TN)), static_cast<unsigned>(max_tiles)), dim3(512), smem, s>>>(
      static_cast<const bf16_t*>(down ? c.act : c.x), (c.weight_on_output != 0) == down ? c.weight : nullptr,
      static_cast<const bf16_t*>(down ? c.w_down : c.w_in), ints, t_e, t_e + max_tiles, t_e + 2 * max_tiles,
      down ? nullptr : static_cast<bf16_t*>(c.act), down ? c.out : nullptr, c.tokens, K, N, c.top, c.gate_alpha, c.limit, c.up_shift,
      c.into_stream, c.col_scale, c.experts, static_cast<const bf16_t*>(c.x), c.weight);
  return check_launch("psamd_moe_experts_grouped (small tiles)");
}

// Columns a workgroup: the most that leave it a few hundred workgroups, were there a tile a slot. us of a whole step's experts (sorting included), columns
// of the first product / the second: 32 experts of 2,048 x 1,024, 8 tokens x 8 choices 32/64 74.8, 32/32 75.0, 64/64 77.1, 16/64 85.8, 16/16 101; 24 of
// 1,024 x 320, 8 x 4 17.4, 18.1, 19.1, 18.6, 23.7; 4 of 1,024 x 512, 5 x 2 14.8, 14.0, 17.1, 13.8, 13.1.
template <int FORM>
static int launch_stream_form(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  const int64_t N = FORM == kFormDown ? c.K : c.F;
  if (FORM == kFormDown && ceil_div(N, 64) * max_tiles >= 384) return run_stream<64, FORM>(s, c, ints, max_tiles);
  if (ceil_div(N, 32) * max_tiles >= 192) return run_stream<32, FORM>(s, c, ints, max_tiles);
  return run_stream<16, FORM>(s, c, ints, max_tiles);
}

static int launch_stream(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  if (c.kind == kExpertGated ? launch_stream_form<kFormGated>(s, c, ints, max_tiles) : launch_stream_form<kFormSquaredRelu>(s, c, ints, max_tiles))
    return 1;
  return launch_stream_form<kFormDown>(s, c, ints, max_tiles);
}

template <int FORM>
static int run_tiles(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  constexpr size_t kSmem = kSmallSmem + kSmallTile * sizeof(int32_t);
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(moe_tile_kernel<FORM>), hipFuncAttributeMaxDynamicSharedMemorySize,
                          static_cast<int>(kSmem)) != hipSuccess)
    return fail("psamd_moe_experts_grouped: " + std::to_string(kSmem) + " bytes of LDS were refused");
  const int32_t* sorted = ints;
  const int32_t* t_e = ints + c.tokens * c.top;
  const int32_t* t_f = t_e + max_tiles;
  const int32_t* t_c = t_f + max_tiles;
  constexpr bool down = FORM == kFormDown;
  const int N = down ? c.K : c.F, K = down ? c.F : c.K;
  const int column_tiles = static_cast<int>(ceil_div(N, FORM == kFormGated ? kSmallTile / 2 : kSmallTile));
  const dim3 grid(static_cast<unsigned>(8 * ceil_div(static_cast<int64_t>(max_tiles) * column_tiles, 8)));
  moe_tile_kernel<FORM><<<grid, dim3(256), kSmem, s>>>(
      static_cast<const bf16_t*>(down ? c.act : c.x), (c.weight_on_output != 0) == down ? c.weight : nullptr,
      static_cast<const bf16_t*>(down ? c.w_down : c.w_in), sorted, t_e, t_f, t_c, t_c + max_tiles,
      down ? nullptr : static_cast<bf16_t*>(c.act), down ? c.out : nullptr, c.tokens, K, N, c.top, c.gate_alpha, c.limit,
      c.up_shift, c.into_stream, c.col_scale, c.identity > 0 ? static_cast<int>(c.tokens * c.top) : 0,
      static_cast<const bf16_t*>(c.x), c.weight, column_tiles);
  return check_launch("psamd_moe_experts_grouped (tiles)");
}

static int launch_tiles(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  if (c.kind == kExpertGated ? run_tiles<kFormGated>(s, c, ints, max_tiles) : run_tiles<kFormSquaredRelu>(s, c, ints, max_tiles)) return 1;
  return run_tiles<kFormDown>(s, c, ints, max_tiles);
}

template <int FORM>
static int run_wide(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  if ((FORM == kFormDown ? c.F : c.K) < 64 * ExpertTiles<FORM>::kMinSteps)
    return fail("psamd_moe_experts_grouped: too few steps of k for tiles of 256 pairs");
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(moe_wide_kernel<FORM>), hipFuncAttributeMaxDynamicSharedMemorySize, kWideSmem) != hipSuccess)
    return fail("psamd_moe_experts_grouped: " + std::to_string(kWideSmem) + " bytes of LDS were refused");
  const int32_t* t_e = ints + c.tokens * c.top;
  constexpr bool down = FORM == kFormDown;
  const int N = down ? c.K : c.F, K = down ? c.F : c.K;
  const int column_tiles = static_cast<int>(ceil_div(N, FORM == kFormGated ? kWideTile / 2 : kWideTile));
  const dim3 grid(static_cast<unsigned>(std::min<int64_t>(8 * ceil_div(static_cast<int64_t>(max_tiles) * column_tiles, 8), 256)));
  moe_wide_kernel<FORM><<<grid, dim3(kWideThreads), kWideSmem, s>>>(
      static_cast<const bf16_t*>(down ? c.act : c.x), (c.weight_on_output != 0) == down ? c.weight : nullptr,
      static_cast<const bf16_t*>(down ? c.w_down : c.w_in), ints, t_e, t_e + max_tiles, t_e + 2 * max_tiles, t_e + 3 * max_tiles,
      down ? nullptr : static_cast<bf16_t*>(c.act), down ? c.out : nullptr, c.tokens, K, N, c.top, c.gate_alpha, c.limit,
      c.up_shift, c.into_stream, c.col_scale, c.identity > 0 ? static_cast<int>(c.tokens * c.top) : 0,
      static_cast<const bf16_t*>(c.x), c.weight, column_tiles);
  return check_launch("psamd_moe_experts_grouped (large tiles)");
}

static int launch_wide(hipStream_t s, const ExpertCall& c, const int32_t* ints, int max_tiles) {
  if (c.kind == kExpertGated ? run_wide<kFormGated>(s, c, ints, max_tiles) : run_wide<kFormSquaredRelu>(s, c, ints, max_tiles)) return 1;
  return run_wide<kFormDown>(s, c, ints, max_tiles);
}

// Whether the tiles of the kernel for many pairs take these experts: whole steps of 64 k in both products, and offsets inside
// an operand that fit 32 bits.
static bool tiles_take(int64_t tokens, int64_t pairs, int K, int F) {
  const int64_t most = (1LL << 32) - 1;
  return K % 64 == 0 && F % 64 == 0 && 2 * tokens * K <= most && 2 * pairs * F <= most && 4LL * K * F <= most;
}

// From how many pairs an expert on a step that sorts its pairs itself takes the large tiles; below, moe_stream_kernel reads an expert once per 16 pairs. The
// large tiles take nearly the same time at any of these counts, which is that of their steps of K one after the other, if there are too few of them: `filled`
// counts those of 128 columns that the smaller of the two products has with one tile an expert. us of routing and experts, small tiles / large, at 24, 32, 40 and 47
// pairs an expert (filled):
//   64 of 2,048 x 1,408 gated (1,024) 230, 273, 313, 339 / 197, 202, 218, 228       32 of 2,048 x 1,024 gated (512) 122, 134, 150, 160 / 118, 120, 122, 123
//    8 of 4,096 x 3,584 gated (256)   182, 209, 235, 244 / 185, 188, 189, 191       16 of 2,048 x 2,816 gated (256) 152, 170, 188, 201 / 168, 171, 174, 176
//   24 of 1,024 x 320 gated (120)      34, 39, 41, 42 / 38, 39, 40, 40                8 of 2,048 x 1,024 gated (128)  38, 44, 44, 47 / 53, 55, 55, 56
//   16 of 4,096 x 1,024 ungated (128)  78, 87, 99, 103 / 98, 102, 109, 114            8 of 1,024 x 8,192 gated (64)  124, 154, 165, 177 / 178, 181, 183, 184
//    4 of 1,024 x 512 gated (32)       18, 19, 21, 22 / 31, 32, 33, 35               32 of 512 x 256 ungated (64)     23, 27, 29, 31 / 30, 32, 35, 36
static int64_t tiles_from_pairs(int experts, int K, int F, int kind) {
  const int64_t filled = experts * std::min(ceil_div(K, 128), ceil_div(F, kind == kExpertGated ? 64 : 128));
  return filled >= 320 ? 24 : (filled >= 200 ? 28 : 48);
}

// ... and their rows: 0 where the kernel for small tiles takes the step, 256 where the device chooses tiles of up to 256 x 256 by the step's
// counts. Those ask for half the bytes per product, but one workgroup of them fills a compute unit, two of 128 x 128 share one, and a
// last round that is not full costs nearly as much as one that is: the time is that of the rounds, K long in the first product and F
// in the second, and 300 more for what a large tile does in front of and behind its loop, which the two small ones on a unit do beside
// each other's. An expert's last tile is half empty on average. us of both products and the sorting, 256 / 128 (E experts of K x F,
// choices at random):
//   32 of 2,048 x 1,024:  50 pairs an expert 111 / 108, 140 129 / 151, 260 161 / 208, 448 204 / 253, 1,000 467 / 586
//    8 of 2,048 x 1,024:  64 63 / 57, 260 67 / 63, 512 77 / 100, 1,000 138 / 155, 2,000 224 / 272
//    8 of 4,096 x 3,584:  64 170 / 165, 260 271 / 395, 448 324 / 540, 1,000 709 / 1,123
//   24 of 1,024 x 320:    64 42 / 35, 512 65 / 70, 2,000 207 / 200
//    4 of 1,024 x 512:    64 35 / 29, 512 41 / 33, 2,000 56 / 65
//   64 of 2,048 x 1,408:  140 284 / 378, 448 530 / 721, 1,000 1,093 / 1,497
// The 1.2 and the 300 were fitted to the loop of eight waves, whose tiles did not begin under the end of the one before: over 724 steps (ten shapes, 64 to 2,000
// pairs an expert, even to uneven) the choice is 1.5% over the faster on average (always 256: 0.7%, always 128: 21%), 30% at worst, all of them left to 128.
static int wide_tile_rows(int64_t pairs, int experts, int K, int F, int kind) {
  if (pairs < tiles_from_pairs(experts, K, F, kind) * experts) return 0;
  auto rounds = [&](int rows, int at_once, int beside) {
    const double tiles = std::max<double>(experts, static_cast<double>(pairs) / rows + 0.5 * experts);
    auto of = [&](int64_t columns) {
      const double full = tiles * columns / at_once;
      return 0.5 * (std::ceil(full) + std::max(full, 1.0));
    };
    return of(ceil_div(F, kind == kExpertGated ? rows / 2 : rows)) * (K + beside) + of(ceil_div(K, rows)) * (F + beside);
  };
  if (std::min(K, F) < 64 * ExpertTiles<kFormGated>::kMinSteps) return 128;
  return 1.2 * rounds(256, 256, 300) < rounds(128, 512, 0) ? 256 : 128;
}

template <typename A>
static int launch_experts_rows(hipStream_t s, const ExpertCall& c) {
  const unsigned pairs = static_cast<unsigned>(c.tokens * c.top);
  moe_gate_up_rows_kernel<A><<<dim3(pairs, static_cast<unsigned>(ceil_div(c.F, kRowsPerBlock))), dim3(256),
                               sizeof(float) * c.K, s>>>(
      static_cast<const A*>(c.x), c.chosen, c.weight, static_cast<const A*>(c.w_in), static_cast<A*>(c.act), c.K, c.F,
      c.experts, c.top, c.gate_alpha, c.limit, c.up_shift, c.weight_on_output, c.kind);
  if (check_launch("psamd_moe_experts_rows (in)")) return 1;
  moe_down_rows_kernel<A><<<dim3(pairs, static_cast<unsigned>(ceil_div(c.K, kRowsPerBlock))), dim3(256),
                            sizeof(float) * c.F, s>>>(
      static_cast<const A*>(c.act), c.chosen, static_cast<const A*>(c.w_down), c.out, c.tokens, c.K, c.F, c.experts, c.top,
      c.weight_on_output ? c.weight : nullptr, c.into_stream, c.col_scale, static_cast<const A*>(c.x), c.weight);
  return check_launch("psamd_moe_experts_rows (down)");
}

// The rule as the entry points take it, checked on the host.
static const char* bad_rule(const RouterRule& r, int experts, int top) {
  if (r.mode < 0 || r.mode > 2) return "router mode 0 (sigmoid scores), 1 (softmax over the chosen) or 2 (softmax over all)";
  if (r.correction != nullptr && r.mode != 2) return "a correction of the choice goes with the softmax over all experts";
  if (r.groups == 0) return nullptr;
  if (r.mode == 1) return "groups of experts go with scores that do not depend on the choice";
  if (r.groups < 1 || r.groups > kMaxRouterGroups || experts % r.groups != 0) return "the experts must form at most 256 equal groups";
  if (r.keep < 1 || r.keep > r.groups || top > r.keep * (experts / r.groups)) return "the kept groups hold fewer experts than are chosen";
  return nullptr;
}

// out[t, :] *= sigmoid(x[t] . w): one number per token on the output of a branch every token takes.
// One workgroup per token, the dot product in float.
template <typename A>
__global__ __launch_bounds__(256) void row_gate_kernel(float* __restrict__ out, const A* __restrict__ x,
                                                       const float* __restrict__ w, int out_hidden, int hidden) {
  __shared__ float parts[4];
  const int64_t t = blockIdx.x;
  float acc = 0.f;
  for (int i = threadIdx.x; i < hidden; i += 256) acc = fmaf(to_float<A>(x[t * hidden + i]), w[i], acc);
  const float g = 1.f / (1.f + expf(-block_sum(acc, parts, 4)));
  float* o = out + t * out_hidden;
  for (int i = threadIdx.x; i < out_hidden; i += 256) o[i] *= g;
}

// What the grouped form refuses, on the host.
static const char* bad_experts(const ExpertCall& c, const int32_t* ints) {
  if (c.kind != kExpertGated && c.kind != kExpertSquaredRelu) return "experts are gated (0) or squared ReLU without a gate (1)";
  if (c.tokens < 0 || c.K <= 0 || c.F <= 0 || c.experts <= 0 || c.identity < 0 || c.top < 1 || c.top > c.experts + c.identity) return "bad sizes";
  if (c.K % 8 != 0 || c.F % 8 != 0) return "K and F must be multiples of 8";
  if (c.experts > 4096 || c.tokens * c.top > (1 << 24)) return "too many experts or pairs";
  return ints == nullptr ? "the grouping needs its integer scratch" : nullptr;
}

// `wide`: the pairs of a large tile, 256 (at most) or 128, or 0 for the kernels of small ones.
static int run_experts(hipStream_t s, const ExpertCall& c, int32_t* ints, int grouped_already, int wide) {
  if (c.tokens == 0) return 0;
  const int64_t pairs = c.tokens * c.top;
  const int buckets = c.experts + (c.identity > 0 ? 1 : 0);  // all identity pairs lie in one, behind the experts'
  const int rows = wide != 0 ? wide : psamd_moe_grouped_tile_rows(pairs, buckets);
  const int least = rows == 256 ? 128 : rows;                // the device may cut into tiles of 128
  const int max_tiles = static_cast<int>(std::min<int64_t>(ceil_div(pairs, least) + buckets, pairs));
  if (wide == 0 && max_tiles > 65535) return fail("psamd_moe_experts_grouped: too many tiles for one launch");   // they are gridDim.y of moe_grouped_kernel alone
  if (grouped_already == 0) {
    const TileRule rule{rows == 256 ? 0 : rows,
                        {static_cast<int>(ceil_div(c.F, c.kind == kExpertGated ? 128 : 256)), static_cast<int>(ceil_div(c.K, 256))}, {c.K, c.F}};
    const bool staged = group_staged(pairs, buckets);
    const size_t smem = sizeof(int32_t) * (group_smem_ints(buckets) + (staged ? pairs : 0));
    if (smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(moe_group_kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                                static_cast<int>(smem)) != hipSuccess)
      return fail("psamd_moe_experts_grouped: " + std::to_string(smem) + " bytes of LDS were refused");
    moe_group_kernel<<<dim3(1), dim3(1024), smem, s>>>(
        c.chosen, static_cast<int>(pairs), buckets, rule, c.identity > 0 && wide != 0, max_tiles, staged, ints, ints + pairs,
        ints + pairs + max_tiles, ints + pairs + 2 * max_tiles);
    if (check_launch("psamd_moe_experts_grouped (grouping)")) return 1;
  }
  if (wide == 256) return launch_wide(s, c, ints, max_tiles);
  if (wide == 128) return launch_tiles(s, c, ints, max_tiles);
  if (rows == 128) return launch_grouped<8, 2>(s, c, ints, max_tiles);
  if (rows == 64) return launch_grouped<4, 2>(s, c, ints, max_tiles);
  if (tiles_take(c.tokens, pairs, c.K, c.F)) return launch_stream(s, c, ints, max_tiles);
  return launch_grouped<1, 1>(s, c, ints, max_tiles);
}

}  // namespace psamd

using namespace psamd;

extern "C" {

int psamd_moe_route(void* stream, const void* x, int x_dtype, const float* w_router, int32_t* chosen, float* weight,
                    int64_t tokens, int K, int experts, int top, const float* bias, int mode,
                    int groups, int keep, float factor, int group_max, const float* correction) {
  PSAMD_REQUIRE(tokens >= 0 && K > 0 && experts > 0 && top >= 1 && top <= experts, "bad sizes");
  const RouterRule rule{mode, groups, keep, factor, group_max, correction};
  if (const char* bad = bad_rule(rule, experts, top)) return fail(bad);
  PSAMD_REQUIRE(sizeof(float) * (static_cast<size_t>(K) + experts) <= 64 * 1024, "row and scores do not fit in LDS");
  PSAMD_REQUIRE(tokens <= 2147483647LL, "too many tokens for one launch");
  if (tokens == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t smem = sizeof(float) * (static_cast<size_t>(K) + experts);
  const dim3 grid(static_cast<unsigned>(tokens));
  if (x_dtype == kBF16) {
    moe_route_kernel<bf16_t><<<grid, dim3(256), smem, s>>>(static_cast<const bf16_t*>(x), w_router, chosen, weight, K,
                                                          experts, top, bias, rule);
  } else if (x_dtype == kF32) {
    moe_route_kernel<float><<<grid, dim3(256), smem, s>>>(static_cast<const float*>(x), w_router, chosen, weight, K,
                                                         experts, top, bias, rule);
  } else {
    return fail("psamd_moe_route: x must be float32 or bfloat16");
  }
  return check_launch("psamd_moe_route");
}

int psamd_moe_topk(void* stream, const float* logits, int32_t* chosen, float* weight, int64_t tokens, int experts,
                   int top, const float* bias, int mode,
                   int groups, int keep, float factor, int group_max, const float* correction) {
  PSAMD_REQUIRE(tokens >= 0 && experts > 0 && top >= 1 && top <= experts, "bad sizes");
  const RouterRule rule{mode, groups, keep, factor, group_max, correction};
  if (const char* bad = bad_rule(rule, experts, top)) return fail(bad);
  PSAMD_REQUIRE(sizeof(float) * 4 * static_cast<size_t>(experts) <= 64 * 1024, "scores do not fit in LDS");
  PSAMD_REQUIRE(ceil_div(tokens, 4) <= 2147483647LL, "too many tokens for one launch");
  if (tokens == 0) return 0;
  moe_topk_kernel<<<dim3(static_cast<unsigned>(ceil_div(tokens, 4))), dim3(256), sizeof(float) * 4 * experts,
                    static_cast<hipStream_t>(stream)>>>(logits, chosen, weight, tokens, experts, top, bias, rule);
  return check_launch("psamd_moe_topk");
}

int psamd_moe_topk_group(void* stream, const float* logits, int32_t* chosen, float* weight, int32_t* ints, int64_t tokens,
                         int experts, int buckets, int top, const float* bias, int mode,
                         int groups, int keep, float factor, int group_max, const float* correction) {
  PSAMD_REQUIRE(tokens >= 1 && tokens <= 64 && experts > 0 && experts <= 1024 && top >= 1 && top <= experts, "bad sizes");
  const RouterRule rule{mode, groups, keep, factor, group_max, correction};
  if (const char* bad = bad_rule(rule, experts, top)) return fail(bad);
  PSAMD_REQUIRE(ints != nullptr && buckets >= 1 && buckets <= experts, "the grouping needs its integer scratch, and buckets for the experts");
  const int64_t pairs = tokens * top;
  const int rows = psamd_moe_grouped_tile_rows(pairs, buckets);
  const int max_tiles = psamd_moe_grouped_max_tiles(pairs, buckets);
  moe_topk_group_kernel<<<dim3(1), dim3(1024), sizeof(int32_t) * group_smem_ints(buckets) + sizeof(float) * 16 * experts,
                          static_cast<hipStream_t>(stream)>>>(logits, chosen, weight, static_cast<int>(tokens), experts, buckets, top, rows,
                                                              max_tiles, ints, ints + pairs, ints + pairs + max_tiles,
                                                              ints + pairs + 2 * max_tiles, bias, rule);
  return check_launch("psamd_moe_topk_group");
}

int psamd_moe_experts_rows(void* stream, const void* x, const int32_t* chosen, const float* weight,
                           const void* w_in, const void* w_down, void* act, float* out, int dtype,
                           int64_t tokens, int K, int F, int experts, int identity, int top, float gate_alpha, float limit,
                           float up_shift, int weight_on_output, int kind, int into_stream, const float* col_scale) {
  PSAMD_REQUIRE(tokens >= 0 && K > 0 && F > 0 && experts > 0 && identity >= 0 && top >= 1 && top <= experts + identity, "bad sizes");
  PSAMD_REQUIRE(kind == kExpertGated || kind == kExpertSquaredRelu, "experts are gated (0) or squared ReLU without a gate (1)");
  PSAMD_REQUIRE(sizeof(float) * static_cast<size_t>(std::max(K, F)) <= 64 * 1024, "a row does not fit in LDS");
  PSAMD_REQUIRE(tokens * top <= 2147483647LL && ceil_div(std::max(K, F), kRowsPerBlock) <= 65535, "too large for one launch");
  if (tokens == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const ExpertCall c{x, chosen, weight, w_in, w_down, act, out, tokens, K, F, experts, identity, top, kind,
                     gate_alpha, limit, up_shift, weight_on_output, into_stream, col_scale};
  if (dtype == kBF16) return launch_experts_rows<bf16_t>(s, c);
  if (dtype == kF32) return launch_experts_rows<float>(s, c);
  return fail("psamd_moe_experts_rows: dtype must be float32 or bfloat16");
}

// Pairs per tile of the grouped form for a step of this many pairs over this many experts: 128 when
// the experts have at least twice that many pairs each on average (an expert's last tile is half
// empty on average: 512 tokens of 8 choices over 32 experts took 204 us in tiles of 128, one full
// and one nearly empty per expert), 64 from 48 pairs per expert on, 16 below. Where K and F are multiples of 64, wide_tile_rows is asked first.
int psamd_moe_grouped_tile_rows(int64_t pairs, int experts) {
  return pairs >= 256LL * experts ? 128 : (pairs >= 48LL * experts ? 64 : 16);
}

// Tile slots the grouped form's grid has for such a step (every expert may end in a tile that is not full).
int psamd_moe_grouped_max_tiles(int64_t pairs, int experts) {
  const int rows = psamd_moe_grouped_tile_rows(pairs, experts);
  return static_cast<int>(std::min<int64_t>(ceil_div(pairs, rows) + experts, pairs));
}

int psamd_moe_expert_tile_rows(int64_t tokens, int K, int F, int experts, int identity, int top, int kind) {
  const int64_t pairs = tokens * top;
  return tiles_take(tokens, pairs, K, F) ? wide_tile_rows(pairs, experts + (identity > 0 ? 1 : 0), K, F, kind) : 0;
}

int psamd_moe_experts_grouped(void* stream, const void* x, const int32_t* chosen, const float* weight,
                              const void* w_in, const void* w_down, void* act, float* out, int32_t* ints,
                              int64_t tokens, int K, int F, int experts, int identity, int top, float gate_alpha, float limit,
                              float up_shift, int grouped_already, int weight_on_output, int kind, int into_stream,
                              const float* col_scale) {
  const ExpertCall c{x, chosen, weight, w_in, w_down, act, out, tokens, K, F, experts, identity, top, kind,
                     gate_alpha, limit, up_shift, weight_on_output, into_stream, col_scale};
  if (const char* bad = bad_experts(c, ints)) return fail(std::string(__func__) + ": " + bad);
  // Pairs that the router's kernel has sorted lie in the tiles of a small step.
  return run_experts(static_cast<hipStream_t>(stream), c, ints, grouped_already,
                     grouped_already == 0 ? psamd_moe_expert_tile_rows(tokens, K, F, experts, identity, top, kind) : 0);
}

int psamd_moe_experts_tiled(void* stream, const void* x, const int32_t* chosen, const float* weight,
                            const void* w_in, const void* w_down, void* act, float* out, int32_t* ints,
                            int64_t tokens, int K, int F, int experts, int identity, int top, float gate_alpha, float limit,
                            float up_shift, int weight_on_output, int kind, int into_stream, const float* col_scale, int tile_rows) {
  const ExpertCall c{x, chosen, weight, w_in, w_down, act, out, tokens, K, F, experts, identity, top, kind,
                     gate_alpha, limit, up_shift, weight_on_output, into_stream, col_scale};
  if (const char* bad = bad_experts(c, ints)) return fail(std::string(__func__) + ": " + bad);
  PSAMD_REQUIRE(tiles_take(tokens, tokens * top, K, F) && (tile_rows == 128 || tile_rows == 256), "operands and tiles that these kernels take");
  PSAMD_REQUIRE(tile_rows == 128 || std::min(K, F) >= 64 * ExpertTiles<kFormGated>::kMinSteps, "too few steps of k for tiles of 256 pairs");
  return run_experts(static_cast<hipStream_t>(stream), c, ints, 0, tile_rows);
}

int psamd_row_gate(void* stream, float* out, const void* x, int act_dtype, const float* w, int64_t tokens, int out_hidden,
                   int hidden) {
  PSAMD_REQUIRE(tokens >= 0 && out_hidden > 0 && hidden > 0 && tokens <= 2147483647LL, "bad sizes");
  if (tokens == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(tokens));
  if (act_dtype == kBF16) {
    row_gate_kernel<bf16_t><<<grid, dim3(256), 0, s>>>(out, static_cast<const bf16_t*>(x), w, out_hidden, hidden);
  } else if (act_dtype == kF32) {
    row_gate_kernel<float><<<grid, dim3(256), 0, s>>>(out, static_cast<const float*>(x), w, out_hidden, hidden);
  } else {
    return fail("psamd_row_gate: activation dtype must be float32 or bfloat16");
  }
  return check_launch("psamd_row_gate");
}

}  // extern "C"
