// Causal grouped-query attention over the paged cache for the 32-bit path, on the float32 matrix instructions
// (v_mfma_f32_16x16x4_f32): scores, softmax and weighted sums in float32. Optional sliding window, sink, bias by distance and
// gate as in attention_generic.hip, whose one-wave-per-(token, head) form stays for the shapes this one does not take.
//
// A tile is 16 columns: 16 / G queries of one request for all G query heads of one kv head, so that a key is read once
// for the group. Keys are taken in runs of kRun positions counted from position 0; a run gives (maximum, sum, weighted
// values) on its own, and the runs are merged in ascending order. A run that lies outside a query's keys leaves its sums as they
// are, so a query's result is the same bit for bit whichever queries share its tile and however its sequence was cut. So does
// a value that is not finite behind a query or in front of its window, which a weight of zero would not hide: in pages that some
// query of the tile does not see whole such values are added on their own.
//
// Bound by the matrix instructions (1,024 cycles of them per 16 columns and page at a head size of 64 against 8 KB read).
// 600 tokens x 32 heads of 64 on 8: 820 us (one wave per token and head, every key read four times over) -> 53, of 128 1,655 -> 99
// (110 with a page's values asked for 16 dimensions at a time). A few tokens in front of nothing are bound by the launch and two
// trips to memory: two of 32 heads of 64 4.7 us there, 5.8 with a whole run's exponentials and the merge, 4.6 with neither.

#include "api.h"
#include "common.h"

namespace psamd {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kRunPages = 8, kRun = kRunPages * kPage;   // keys per run
constexpr int kAttnWaves = 4;

struct AttentionF32 {
  const float* qkv;
  int q_stride;
  float* out;
  const float* kv;
  const int32_t* pf_tiles;     // [n_pf][2]: item, first query of the tile within the item
  int n_pf, subs;              // tiles of the list, and how many tiles of 16 columns each is
  const int32_t* dec_items;
  const int32_t* item_start;
  const int32_t* item_pos0;
  const int32_t* table_off;
  const int32_t* block_ids;
  int hq, hkv;
  float scale;
  int window;
  const float* sink;
  const float* dist_bias;
  int n_dist;
  const float* gate;
  int64_t gate_row;
};

// Lane (r = l % 16, g = l / 16). Scores: rows are the page's keys, columns the tile's; lane (r, g) supplies dimensions 16 s +
// 4 g .. + 3 of key r and of column r, and receives keys 4 g .. 4 g + 3 of column r, which is the operand the product with the
// values wants of it: there rows are dimensions (the page holds values as [D][16]), and a lane receives four dimensions.
// Chains of matrix instructions are at most 64 products long (see linear_f32.hip).
template <int DT>
__global__ __launch_bounds__(64 * kAttnWaves) void attention_f32_kernel(AttentionF32 c) {
  constexpr int D = DT * 16, OWN = (DT + kAttnWaves - 1) / kAttnWaves;
  __shared__ f32x4 acc_s[kAttnWaves][DT][64];
  __shared__ float max_s[kAttnWaves][16], sum_s[kAttnWaves][16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int kvh = blockIdx.y, group = c.hq / c.hkv, per_tile = 16 / group;
  int item, q0 = 0, nq = 1;
  if (static_cast<int>(blockIdx.x) < c.n_pf * c.subs) {
    const int tile = blockIdx.x / c.subs, sub = blockIdx.x - tile * c.subs;
    item = c.pf_tiles[2 * tile];
    q0 = c.pf_tiles[2 * tile + 1] + sub * per_tile;
    nq = min(per_tile, c.item_start[item + 1] - c.item_start[item] - q0);
    if (nq <= 0) return;                               // uniform for the workgroup
  } else {
    item = c.dec_items[blockIdx.x - c.n_pf * c.subs];
  }
  const int qi = min(r / group, nq - 1), h = kvh * group + r % group;
  const int64_t t = c.item_start[item] + q0 + qi;
  const int first_pos = c.item_pos0[item] + q0, last_pos = first_pos + nq - 1, pos = first_pos + qi;
  const int lo = c.window > 0 ? pos - c.window + 1 : 0;                // this column's first key (may be negative)
  const int last_lo = c.window > 0 ? last_pos - c.window + 1 : 0;      // the last column's
  const int32_t* table = c.block_ids + c.table_off[item];
  const int64_t page_elems = 2LL * c.hkv * kPage * D, half_elems = static_cast<int64_t>(c.hkv) * kPage * D;
  const float* kv = c.kv + static_cast<int64_t>(kvh) * kPage * D;

  f32x4 q[DT];
  const float* qp = c.qkv + t * c.q_stride + static_cast<int64_t>(h) * D + 4 * g;
#pragma unroll
  for (int s = 0; s < DT; ++s) q[s] = *reinterpret_cast<const f32x4*>(qp + 16 * s);

  const int p_begin = c.window > 0 ? max(0, first_pos - c.window + 1) / kPage : 0;   // pages some column sees
  const int p_end = last_pos / kPage + 1;
  const int run_end = (p_end + kRunPages - 1) / kRunPages;
  // A tile whose keys are one run has nothing to merge: its first wave writes what it has, the others leave.
  const bool one_run = run_end - p_begin / kRunPages == 1;
  if (one_run && wave != 0) return;
  auto put = [&](int d, f32x4 y) {
    if (c.gate != nullptr) {
      const float* gp = c.gate + t * c.gate_row + static_cast<int64_t>(h) * D + d;
#pragma unroll
      for (int v = 0; v < 4; ++v) y[v] *= 1.f / (1.f + expf(-gp[v]));
    }
    *reinterpret_cast<f32x4*>(c.out + (t * c.hq + h) * D + d) = y;
  };
  f32x4 total[OWN];
#pragma unroll
  for (int o = 0; o < OWN; ++o) total[o] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  for (int run0 = p_begin / kRunPages; run0 < run_end; run0 += kAttnWaves) {
    const int run = run0 + wave;
    if (run < run_end) {
      f32x4 s[kRunPages];
      float top = -INFINITY;
#pragma unroll
      for (int i = 0; i < kRunPages; ++i) {
        const int p = run * kRunPages + i;
        s[i] = f32x4{-INFINITY, -INFINITY, -INFINITY, -INFINITY};
        if (p < p_begin || p >= p_end) continue;
        const float* kr = kv + table[p] * page_elems + r * D + 4 * g;
        f32x4 k[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d) k[d] = *reinterpret_cast<const f32x4*>(kr + 16 * d);
        f32x4 dot = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int d0 = 0; d0 < DT; d0 += 4) {
          f32x4 chain = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int d = d0; d < (d0 + 4 < DT ? d0 + 4 : DT); ++d)
#pragma unroll
            for (int j = 0; j < 4; ++j) chain = __builtin_amdgcn_mfma_f32_16x16x4f32(k[d][j], q[d][j], chain, 0, 0, 0);
          dot += chain;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int key = p * kPage + 4 * g + v;
          if (key > pos || key < lo) continue;
          float x = dot[v] * c.scale;
          if (c.dist_bias != nullptr) x += c.dist_bias[static_cast<int64_t>(h) * c.n_dist + min(pos - key, c.n_dist - 1)];
          s[i][v] = x;
          top = fmaxf(top, x);
        }
      }
      top = fmaxf(top, __shfl_xor(top, 16, kWave));
      top = fmaxf(top, __shfl_xor(top, 32, kWave));
      const float base = top == -INFINITY ? 0.f : top;                 // a run without a key of this column: all weights 0
      float sum = 0.f;
#pragma unroll
      for (int i = 0; i < kRunPages; ++i) {
        const int p = run * kRunPages + i;
        if (p < p_begin || p >= p_end) {                               // nobody's: weights of 0, without 4 exponentials for each
          s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
          continue;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          s[i][v] = expf(s[i][v] - base);
          sum += s[i][v];
        }
      }
      sum += __shfl_xor(sum, 16, kWave);
      sum += __shfl_xor(sum, 32, kWave);
      f32x4 acc[DT];
#pragma unroll
      for (int d = 0; d < DT; ++d) acc[d] = f32x4{0.f, 0.f, 0.f, 0.f};
      unsigned odd = 0;                                                // pages whose values are not all finite (the same in all lanes)
#pragma unroll
      for (int i0 = 0; i0 < kRunPages; i0 += 4) {
        f32x4 chain[DT];
#pragma unroll
        for (int d = 0; d < DT; ++d) chain[d] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = i0; i < i0 + 4; ++i) {
          const int p = run * kRunPages + i;
          if (p < p_begin || p >= p_end) continue;
          const float* vp = kv + table[p] * page_elems + half_elems;
          const float* vr = vp + r * kPage + 4 * g;
          const int key0 = p * kPage + 4 * g;
          f32x4 val[DT];
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            val[d] = *reinterpret_cast<const f32x4*>(vr + d * 16 * kPage);
#pragma unroll
            for (int j = 0; j < 4; ++j) val[d][j] = key0 + j <= last_pos ? val[d][j] : 0.f;   // what lies behind the last position is nobody's
          }
          // Where some column does not see all of the page's keys: a weight of zero does not hide a value that is not finite.
          if (p * kPage + kPage - 1 > first_pos || p * kPage < last_lo) {
            float zeros = 0.f;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
              for (int j = 0; j < 4; ++j) zeros = fmaf(val[d][j], 0.f, zeros);
            if (__any(zeros != 0.f)) {
              odd |= 1u << i;
#pragma unroll
              for (int d = 0; d < DT; ++d)
#pragma unroll
                for (int j = 0; j < 4; ++j) val[d][j] = fabsf(val[d][j]) < INFINITY ? val[d][j] : 0.f;
            }
          }
#pragma unroll
          for (int d = 0; d < DT; ++d)
#pragma unroll
            for (int j = 0; j < 4; ++j) chain[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(val[d][j], s[i][j], chain[d], 0, 0, 0);
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) acc[d] += chain[d];
      }
      // What was left out is added for the columns that see its key; the others keep their bits.
      for (; odd != 0; odd &= odd - 1) {
        const int i = __builtin_ctz(odd), p = run * kRunPages + i;
        f32x4 weights = s[0];
#pragma unroll
        for (int k = 1; k < kRunPages; ++k) weights = i == k ? s[k] : weights;
        const float* vp = kv + table[p] * page_elems + half_elems + 4 * g * kPage;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          for (int src = 0; src < 4; ++src) {                          // the lanes of group src hold key 4 src + j
            const float weight = __shfl(weights[j], 16 * src + r, kWave);
            const int at = 4 * src + j, key = p * kPage + at;
            if (key > pos || key < lo) continue;
#pragma unroll
            for (int d = 0; d < DT; ++d)
#pragma unroll
              for (int v = 0; v < 4; ++v) {
                const float y = vp[(16 * d + v) * kPage + at];
                if (!(fabsf(y) < INFINITY)) acc[d][v] += weight * y;
              }
          }
      }
      if (one_run) {
        if (r / group >= nq) return;
        const float b = top == -INFINITY ? 0.f : 1.f;                  // as the merge below weighs it
        float all = sum * b;
        if (c.sink != nullptr) all += expf(c.sink[h] - top);
        const float inv = 1.f / all;
#pragma unroll
        for (int d = 0; d < DT; ++d) put(16 * d + 4 * g, acc[d] * b * inv);
        return;
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) acc_s[wave][d][lane] = acc[d];
      if (g == 0) {
        max_s[wave][r] = top;
        sum_s[wave][r] = sum;
      }
    }
    __syncthreads();
    const int n = min(kAttnWaves, run_end - run0);
    for (int i = 0; i < n; ++i) {
      const float mi = max_s[i][r], m_new = fmaxf(m, mi);
      const float a = m == -INFINITY ? 0.f : expf(m - m_new), b = mi == -INFINITY ? 0.f : expf(mi - m_new);
      l = fmaf(l, a, sum_s[i][r] * b);
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        const int d = wave + o * kAttnWaves;
        if (d >= DT) break;
        const f32x4 x = acc_s[i][d][lane];
#pragma unroll
        for (int v = 0; v < 4; ++v) total[o][v] = fmaf(total[o][v], a, x[v] * b);
      }
      m = m_new;
    }
    __syncthreads();
  }
  if (r / group >= nq) return;
  if (c.sink != nullptr) l += expf(c.sink[h] - m);                     // the query's own key is always seen: m is finite
  const float inv = 1.f / l;
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int d = (wave + o * kAttnWaves) * 16 + 4 * g;
    if (d >= D) break;
    put(d, total[o] * inv);
  }
}

template <int DT>
static int launch_attention_f32(hipStream_t s, dim3 grid, const AttentionF32& c) {
  attention_f32_kernel<DT><<<grid, dim3(64 * kAttnWaves), 0, s>>>(c);
  return check_launch("psamd_attention_f32");
}

}  // namespace psamd

using namespace psamd;

extern "C" {

// 1 if psamd_attention_f32 takes this shape: whole 16-byte pieces, a head size whose sums of four waves fit in static LDS, and
// a kv head's query heads divide a tile of 16 columns.
int psamd_attention_f32_supports(int hq, int hkv, int head_dim, int q_stride) {
  if (hq < 1 || hkv < 1 || hq % hkv != 0 || 16 % (hq / hkv) != 0 || q_stride % 4 != 0 || hkv > 65535) return 0;
  return head_dim == 16 || head_dim == 32 || head_dim == 64 || head_dim == 128 ? 1 : 0;
}

int psamd_attention_f32(void* stream, const float* qkv, int q_stride, float* out, const float* kv, const int32_t* pf_tiles,
                        int n_pf, int tile_queries, const int32_t* dec_items, int n_dec, const int32_t* item_start, const int32_t* item_pos0,
                        const int32_t* table_off, const int32_t* block_ids, int hq, int hkv, int head_dim, float scale,
                        int window, const float* sink, const float* dist_bias, int n_dist, const float* gate, int64_t gate_row) {
  PSAMD_REQUIRE(psamd_attention_f32_supports(hq, hkv, head_dim, q_stride), "unsupported head counts or head size");
  PSAMD_REQUIRE((reinterpret_cast<uintptr_t>(qkv) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(kv)) % 16 == 0,
                "operands must lie on 16 bytes");
  PSAMD_REQUIRE(n_pf >= 0 && n_dec >= 0, "bad tile counts");
  PSAMD_REQUIRE(dist_bias == nullptr || n_dist >= 1, "a distance bias needs at least one entry per head");
  PSAMD_REQUIRE(gate == nullptr || gate_row >= static_cast<int64_t>(hq) * head_dim, "the gate's rows");
  if (n_pf + n_dec == 0) return 0;
  const int per_tile = 16 / (hq / hkv);
  PSAMD_REQUIRE(tile_queries >= 1 && tile_queries % per_tile == 0, "the list's tiles must be whole tiles of 16 columns");
  const int subs = tile_queries / per_tile;
  PSAMD_REQUIRE(static_cast<int64_t>(n_pf) * subs + n_dec <= 2147483647LL, "too many tiles for one launch");
  const AttentionF32 c{qkv, q_stride, out, kv, pf_tiles, n_pf, subs, dec_items, item_start, item_pos0, table_off, block_ids,
                       hq, hkv, scale, window, sink, dist_bias, n_dist, gate, gate_row};
  const dim3 grid(static_cast<unsigned>(n_pf * subs + n_dec), static_cast<unsigned>(hkv));
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (head_dim) {
    case 16: return launch_attention_f32<1>(s, grid, c);
    case 32: return launch_attention_f32<2>(s, grid, c);
    case 64: return launch_attention_f32<4>(s, grid, c);
    default: return launch_attention_f32<8>(s, grid, c);
  }
}

}  // extern "C"
