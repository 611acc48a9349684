// The recurrences of delta.hip over prompts, run by run on the matrix cores (float32: v_mfma_f32_16x16x4_f32).
//
// Token by token (delta_scan_kernel) a head's 2,048 tokens are 2,048 sums that wait for each other, 0.19 us each, on half
// the compute units: 385 us for 16 heads of 128 x 128, 394 for 32 of 64 x 64. In a run of kRunTokens tokens the state S0 in
// front of the run enters linearly. With D_t the product of the decays up to token t of the run (a number per head, or a
// vector over the key channels), in the gated form (p = ps k, c = k, both with the decayed state)
//     w_t = ps_t k_t^T (D_t S0) + sum_{s<t} L_ts w_s + xs_t x_t,     L_ts = ps_t (D_t / D_s) (k_t . k_s)
//     o_t = (D_t q_t)^T S0 + sum_{s<=t} (D_t / D_s) (q_t . k_s) w_s
//     S   = D_n S0 + sum_s (D_n / D_s) k_s w_s^T
// so with T = (1 - L)^-1 (unit lower triangular) the run is W = Wx + Kt S0 with Wx = T diag(xs) X and Kt = T diag(ps D) K,
// known without S0. The general form (a decay per channel, the removal reads the state before the decay) has the same shape with
//     L_ts = (c_t D_{t-1}) . (p_s / D_s), W = U (what is taken out), Wx = T (M X), M_ts = (c_t D_{t-1}) . (k_s / D_s),
//     Kt = T (c D_{-1}), and what the values alone leave in the output (Y) and the state (Z).
// Three launches: runs_prepare (all runs side by side: everything that does not need S0), runs_chain (an item's runs in turn:
// two small products each), runs_output (all runs side by side). 2,048 tokens as above: 39 + 90 + 27 us (gated), 106 + 60 + 24
// (general). The chain is what bounds a long prompt: 64 matrix instructions and two barriers a run, 2.9 us of 32 runs in turn.
//
// Numerics: everything is float32. T is built by substitution, 16 x 16 on the diagonal and block by block below it (a product
// of powers of L is shorter and loses everything where keys repeat). The gated form's ratios D_t / D_s are products of the
// decays between the two tokens, so a decay may be 0; the general form divides by D_s and is only taken where the decays'
// floor keeps D_s far from underflow. A product over tokens multiplies those behind a token by zeros, which does not hide what is
// not finite: it then stands in that token's W, and the chain walks such a run token by token for the 16 value channels it
// concerns, as delta_scan_kernel would have. The state is as near 64 bits as the walk's (2.0e-8 to 2.3e-8 either way), the outputs are
// 1.18e-7 off with heads of 128 and the gated form (the walk 1.05e-7), 1.07e-7 (1.03e-7) plain, 1.20e-7 (0.95e-7) general: the
// operands that carry a decay are rounded once more.
//
// Operand layout of a 16 x 16 x 4 instruction: lane (r = l % 16, g = l / 16) gives k = 4 g + i, i = 0..3, of row r and of column
// r, and receives rows 4 g .. 4 g + 3 of column r: what it receives is the column operand of a product over those rows.

#include <algorithm>

#include "api.h"
#include "common.h"

namespace psamd {

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int kRunTokens = 64, kRunTiles = kRunTokens / 16;
constexpr int kLd = kRunTokens + 4;                      // LDS row stride of [.][run] arrays, in floats

struct DeltaRuns {
  const float* kvec;
  const float* cvec;
  const float* pvec;
  const float* rvec;
  int64_t key_row;
  int heads_per_group;
  const float* dvec;
  int64_t dvec_row;
  const float* dscal;
  const float* pscal;
  const float* xscal;
  int64_t scal_row;
  const float* x;
  int64_t x_row;
  float* out;
  int64_t out_row;
  float* state;
  int64_t state_row;
  const int32_t* slots;
  int heads, vdim;
  float* scratch;              // [kMaxRuns at most][heads][run_layout().total]
};

// The runs that one round of launches makes, in the order of their tokens, and the items that they are of. The host lists them (it
// has the items' lengths) and hands the list over as a kernel argument.
constexpr int kMaxRuns = 64;
constexpr int64_t kRunScratch = 384LL << 20;             // bytes
struct RunList {
  int32_t t0[kMaxRuns];        // a run's first token of the step
  int32_t tokens[kMaxRuns];    // how many it has
  int32_t item[kMaxRuns];      // parts: an item, its first run of the list, how many follow each other there
  int32_t first[kMaxRuns];
  int32_t runs[kMaxRuns];
};

// Where a run's arrays lie in its scratch.
struct RunLayout {
  int kt, kd, qd, w, p, s0, z, dc, walked, total;
};
__host__ __device__ constexpr RunLayout run_layout(int dim, int vdim, bool general) {
  RunLayout l{};
  int at = 0;
  l.kt = at, at += kRunTokens * dim;                     // [t][dim]
  l.kd = at, at += kRunTokens * dim;                     // [dim][t]
  l.qd = at, at += kRunTokens * dim;                     // [t][dim]
  l.w = at, at += kRunTokens * vdim;                     // [vdim][t]: Wx, then W
  l.p = at, at += kRunTokens * kRunTokens;               // [t][s]
  l.s0 = at, at += dim * vdim;                           // [vdim][dim]
  l.z = at, at += general ? dim * vdim : 0;              // [vdim][dim]
  l.dc = at, at += dim;
  l.walked = at, at += 16;                               // [vdim / 16]: not 0 where these channels' outputs are finished
  l.total = at;
  return l;
}

// acc + 16 products. The products are summed on their own first: chains of 64 left the outputs 1.7 times as far from 64 bits
// as the token-by-token walk, whose sums over the key channels are sums of 8 added in a tree.
__device__ __forceinline__ f32x4 mma(f32x4 a, f32x4 b, f32x4 acc) {
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 4; ++i) sum = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], sum, 0, 0, 0);
  return acc + sum;
}

// A barrier for what passes through LDS alone: loads from memory stay under way across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kGatedForm = 0, kPlainForm = 1, kGeneralForm = 2;   // plain: the gated form with nothing taken out

// grid (runs, heads), four waves: wave w makes the rows of tokens 16 w .. 16 w + 15 of what is between tokens, then the columns
// 16 w, 64 + 16 w, .. of Wx, Kt, Kd and Z. With one to three waves a SIMD, what bounds it is each wave's chain of loads and
// products: 16 heads of 128, 2,048 tokens, 61 -> 39 us with the columns divided (wave 3 was at it 74 us while wave 0 took 42) and
// the operands asked for ahead; the general form's 32 heads of 64 118 -> 106. There the divisions by D_s, the rows that
// wave 3 has four times as many of as wave 0 and two workgroups of 70 KB of LDS a compute unit are left. Same sums, same bits.
template <int DT, int FORM>
__global__ __launch_bounds__(256) void runs_prepare_kernel(DeltaRuns c, RunList list) {
  constexpr int D = DT * 16, LD = D + 4;
  constexpr bool GENERAL = FORM == kGeneralForm, SOLVES = FORM != kPlainForm;
  extern __shared__ __align__(16) float run_smem[];
  float* tm = run_smem;                                  // [t][s]: the ratios D_t / D_s, later T
  float* lm = tm + kRunTokens * kLd;                     // [t][s]: L
  float* ds = lm + kRunTokens * kLd;                     // general: D [t][dim]
  float* mx = ds + (GENERAL ? kRunTokens * LD : 0);      // general: M X, [vdim][t]
  __shared__ float num[5][kRunTokens];                   // per token: decay, D_t, D_n / D_t, ps, xs
  const int64_t t0 = list.t0[blockIdx.x];
  const int n = list.tokens[blockIdx.x];
  const int h = blockIdx.y, grp = h / c.heads_per_group;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const RunLayout lay = run_layout(D, c.vdim, GENERAL);
  float* sc = c.scratch + (static_cast<int64_t>(blockIdx.x) * c.heads + h) * lay.total;
  const int64_t key0 = t0 * c.key_row + static_cast<int64_t>(grp) * D;
  const int64_t x0 = t0 * c.x_row + static_cast<int64_t>(h) * c.vdim;

  // The run's products over the key channels, a lane's rows and columns read 16 bytes at a time. What is read is asked for ahead
  // of where it is used and without a branch, behind the run the last token again; zeros are used for it.
  const int t = 16 * wave + r;
  const bool has = t < n;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  auto row4 = [&](const float* v, int tok, int d) {      // dimensions 16 d + 4 g .. of a token's vector
    return *reinterpret_cast<const f32x4*>(v + key0 + min(tok, n - 1) * c.key_row + 16 * d + 4 * g);
  };
  f32x4 ct[DT], qt[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    ct[d] = row4(GENERAL ? c.cvec : c.kvec, t, d);
    qt[d] = row4(c.rvec, t, d);
  }
  if (threadIdx.x < kRunTokens) {
    const int t = threadIdx.x;
    const int64_t at = (t0 + t) * c.scal_row + h;
    num[0][t] = !GENERAL && t < n && c.dscal != nullptr ? c.dscal[at] : 1.f;
    num[3][t] = t >= n ? 0.f : c.pscal != nullptr ? c.pscal[at] : 1.f;
    num[4][t] = t >= n ? 0.f : c.xscal != nullptr ? c.xscal[at] : 1.f;
  }
  if constexpr (GENERAL) {
    for (int idx = threadIdx.x; idx < kRunTokens * D; idx += 256) {
      const int t = idx / D, i = idx % D;
      const float w = c.dvec[(t0 + min(t, n - 1)) * c.dvec_row + static_cast<int64_t>(h) * D + i];
      ds[t * LD + i] = t < n ? w : 1.f;
    }
    __syncthreads();
    if (threadIdx.x < D) {
      float d = 1.f;
#pragma unroll 8
      for (int t = 0; t < kRunTokens; ++t) {
        d *= ds[t * LD + threadIdx.x];
        ds[t * LD + threadIdx.x] = d;
      }
    }
  }
  __syncthreads();
  if constexpr (!GENERAL) {
    if (threadIdx.x < kRunTokens) {
      const int s = threadIdx.x;
      float ratio = 1.f;
#pragma unroll 16
      for (int t = 0; t < kRunTokens; ++t) {             // all lanes at one t: the decays are read ahead
        ratio *= t > s ? num[0][t] : 1.f;
        if (t >= s) tm[t * kLd + s] = ratio;
      }
      num[2][s] = ratio;
    }
    __syncthreads();
    if (threadIdx.x < kRunTokens) num[1][threadIdx.x] = tm[threadIdx.x * kLd] * num[0][0];
    __syncthreads();
  }

  f32x4 first[DT], second[DT];                           // a block of tokens s, asked for a block ahead
  auto ask_rows = [&](int st) {
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      first[d] = row4(GENERAL ? c.pvec : c.kvec, 16 * st + r, d);
      if constexpr (GENERAL) second[d] = row4(c.kvec, 16 * st + r, d);
    }
  };
  ask_rows(0);
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    ct[d] = has ? ct[d] : zero;
    qt[d] = has ? qt[d] : zero;
    if constexpr (GENERAL) {
      if (t > 0) ct[d] *= *reinterpret_cast<const f32x4*>(ds + (t - 1) * LD + 16 * d + 4 * g);
      qt[d] *= *reinterpret_cast<const f32x4*>(ds + t * LD + 16 * d + 4 * g);
    }
    *reinterpret_cast<f32x4*>(sc + lay.qd + t * D + 16 * d + 4 * g) = GENERAL ? qt[d] : qt[d] * num[1][t];
  }
  f32x4 m_reg[kRunTiles], pk_reg[kRunTiles];             // general: M and (D_t r_t) . (k_s / D_s), rows s, column t
#pragma unroll
  for (int st = 0; st < kRunTiles; ++st) {
    m_reg[st] = pk_reg[st] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (st > wave) continue;
    const int sr = 16 * st + r;                          // the row this lane supplies
    f32x4 cc = {0.f, 0.f, 0.f, 0.f}, qc = cc, ck = cc, qk = cc;
    f32x4 one[DT], two[DT];
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      one[d] = sr < n ? first[d] : zero;
      if constexpr (GENERAL) two[d] = sr < n ? second[d] : zero;
    }
    if (st < wave) ask_rows(st + 1);
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if constexpr (GENERAL) {
        const f32x4 dd = *reinterpret_cast<const f32x4*>(ds + sr * LD + 16 * d + 4 * g);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          one[d][i] /= dd[i];
          two[d][i] /= dd[i];
        }
        ck = mma(two[d], ct[d], ck);
        qk = mma(two[d], qt[d], qk);
      }
      if constexpr (SOLVES) cc = mma(one[d], ct[d], cc);
      qc = mma(one[d], qt[d], qc);
    }
    f32x4 l, p;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int s = 16 * st + 4 * g + v;
      const float ratio = GENERAL ? 1.f : (s <= t ? tm[t * kLd + s] : 0.f);
      l[v] = s < t ? (GENERAL ? cc[v] : num[3][t] * (ratio * cc[v])) : 0.f;
      p[v] = s <= t ? (GENERAL ? qc[v] : ratio * qc[v]) : 0.f;
      if constexpr (GENERAL) {
        m_reg[st][v] = s < t ? ck[v] : 0.f;
        pk_reg[st][v] = s <= t ? qk[v] : 0.f;
      }
    }
    if constexpr (SOLVES) *reinterpret_cast<f32x4*>(lm + t * kLd + 16 * st + 4 * g) = l;
    *reinterpret_cast<f32x4*>(sc + lay.p + t * kRunTokens + 16 * st + 4 * g) = p;
  }
  // A lane's four tokens s of column j of the values (k = 4 g + i of the operand of either kind), a column at a time.
  f32x4 xs[kRunTiles];
  auto ask_x = [&](int j, int blocks) {
#pragma unroll
    for (int st = 0; st < kRunTiles; ++st) {
      if (st >= blocks) continue;
#pragma unroll
      for (int i = 0; i < 4; ++i) xs[st][i] = c.x[x0 + min(16 * st + 4 * g + i, n - 1) * c.x_row + j];
    }
  };
  auto x4 = [&](int st) {
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = 16 * st + 4 * g + i < n ? xs[st][i] : 0.f;
    return v;
  };
  if constexpr (GENERAL) {
    ask_x(r, wave + 1);
    for (int j0 = 0; j0 < c.vdim; j0 += 16) {
      f32x4 y = zero, m = zero, x[kRunTiles];
#pragma unroll
      for (int st = 0; st < kRunTiles; ++st) x[st] = x4(st);
      ask_x(min(j0 + 16, c.vdim - 16) + r, wave + 1);
#pragma unroll
      for (int st = 0; st < kRunTiles; ++st) {
        if (st > wave) continue;
        y = mma(x[st], pk_reg[st], y);
        m = mma(x[st], m_reg[st], m);
      }
      if (has) *reinterpret_cast<f32x4*>(c.out + (t0 + t) * c.out_row + static_cast<int64_t>(h) * c.vdim + j0 + 4 * g) = y;
#pragma unroll
      for (int v = 0; v < 4; ++v) mx[(j0 + 4 * g + v) * kLd + t] = m[v];
    }
  }
  if constexpr (!GENERAL) ask_x(min(16 * wave, c.vdim - 16) + r, kRunTiles);
  __syncthreads();                                       // L is whole, the ratios have been read
  if constexpr (SOLVES) {
    // T = (1 - L)^-1: the blocks on the diagonal by substitution, a column per lane, ...
    float col[16];
    const float* lb = lm + 16 * wave * kLd + 16 * wave;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      float v = i == r ? 1.f : 0.f;
#pragma unroll
      for (int s = 0; s < i; ++s) v = fmaf(lb[i * kLd + s], col[s], v);
      col[i] = v;
    }
    if (g == 0) {
#pragma unroll
      for (int i = 0; i < 16; ++i) tm[(16 * wave + i) * kLd + 16 * wave + r] = col[i];
    }
    __syncthreads();
    // ... and T_ij = T_ii sum_k L_ik T_kj below it, by distance from the diagonal.
#pragma unroll
    for (int off = 1; off < kRunTiles; ++off) {
      if (wave >= off) {
        const int bj = wave - off;
        f32x4 sum = {0.f, 0.f, 0.f, 0.f};
        for (int bk = bj; bk < wave; ++bk) {
          f32x4 b;
#pragma unroll
          for (int i = 0; i < 4; ++i) b[i] = tm[(16 * bk + 4 * g + i) * kLd + 16 * bj + r];
          sum = mma(*reinterpret_cast<const f32x4*>(lm + (16 * wave + r) * kLd + 16 * bk + 4 * g), b, sum);
        }
        const f32x4 res = mma(*reinterpret_cast<const f32x4*>(tm + (16 * wave + r) * kLd + 16 * wave + 4 * g), sum, f32x4{0.f, 0.f, 0.f, 0.f});
#pragma unroll
        for (int v = 0; v < 4; ++v) tm[(16 * wave + 4 * g + v) * kLd + 16 * bj + r] = res[v];
      }
      __syncthreads();
    }
  }
  // Behind here a wave has columns of its own for all four blocks of tokens: with blocks of tokens of its own wave 3 made four
  // times the products of wave 0, and each wave fetched the operands again.
  f32x4 tr[kRunTiles][kRunTiles];                        // rows 16 tt + r of T
  if constexpr (SOLVES) {
#pragma unroll
    for (int tt = 0; tt < kRunTiles; ++tt)
#pragma unroll
      for (int st = 0; st <= tt; ++st) tr[tt][st] = *reinterpret_cast<const f32x4*>(tm + (16 * tt + r) * kLd + 16 * st + 4 * g);
  }
  for (int j0 = 16 * wave; j0 < c.vdim; j0 += 64) {      // Wx, rows t, column j
    f32x4 b[kRunTiles];
#pragma unroll
    for (int st = 0; st < kRunTiles; ++st) {
      if constexpr (GENERAL) {
        b[st] = *reinterpret_cast<const f32x4*>(mx + (j0 + r) * kLd + 16 * st + 4 * g);
      } else {
        b[st] = x4(st);
#pragma unroll
        for (int i = 0; i < 4; ++i) b[st][i] *= num[4][16 * st + 4 * g + i];
      }
    }
    if constexpr (!GENERAL) ask_x(min(j0 + 64, c.vdim - 16) + r, kRunTiles);
#pragma unroll
    for (int tt = 0; tt < kRunTiles; ++tt) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
      if constexpr (SOLVES) {
#pragma unroll
        for (int st = 0; st <= tt; ++st) acc = mma(tr[tt][st], b[st], acc);
      } else {
        acc = b[tt];
      }
      *reinterpret_cast<f32x4*>(sc + lay.w + (j0 + r) * kRunTokens + 16 * tt + 4 * g) = acc;
    }
  }
  for (int i0 = 16 * wave; i0 < D; i0 += 64) {           // Kt, rows i, column t; Kd
    const int i = i0 + r;
    f32x4 a[kRunTiles];
#pragma unroll
    for (int st = 0; st < kRunTiles; ++st) {
      f32x4 kd;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int s = 16 * st + 4 * g + v;
        const float key = (GENERAL ? c.cvec : c.kvec)[key0 + min(s, n - 1) * c.key_row + i], k = s < n ? key : 0.f;
        a[st][v] = GENERAL ? (s > 0 ? k * ds[(s - 1) * LD + i] : k) : num[3][s] * num[1][s] * k;
        if constexpr (GENERAL) {
          const float taken = c.pvec[key0 + min(s, n - 1) * c.key_row + i];
          kd[v] = s < n ? taken * (ds[(kRunTokens - 1) * LD + i] / ds[s * LD + i]) : 0.f;
        } else {
          kd[v] = num[2][s] * k;
        }
      }
      *reinterpret_cast<f32x4*>(sc + lay.kd + i * kRunTokens + 16 * st + 4 * g) = kd;
    }
    if constexpr (SOLVES) {
#pragma unroll
      for (int tt = 0; tt < kRunTiles; ++tt) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int st = 0; st <= tt; ++st) acc = mma(a[st], tr[tt][st], acc);
        *reinterpret_cast<f32x4*>(sc + lay.kt + (16 * tt + r) * D + i0 + 4 * g) = acc;
      }
    }
  }
  if constexpr (GENERAL) {
    for (int it = wave; it < DT; it += 4) {              // Z, rows i, column j
      f32x4 kk[kRunTiles];
      ask_x(r, kRunTiles);
      const int i = 16 * it + r;
#pragma unroll
      for (int st = 0; st < kRunTiles; ++st)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int s = 16 * st + 4 * g + v;
          const float key = c.kvec[key0 + min(s, n - 1) * c.key_row + i];
          kk[st][v] = s < n ? key * (ds[(kRunTokens - 1) * LD + i] / ds[s * LD + i]) : 0.f;
        }
      for (int j0 = 0; j0 < c.vdim; j0 += 16) {
        f32x4 acc = {0.f, 0.f, 0.f, 0.f}, x[kRunTiles];
#pragma unroll
        for (int st = 0; st < kRunTiles; ++st) x[st] = x4(st);
        ask_x(min(j0 + 16, c.vdim - 16) + r, kRunTiles);
#pragma unroll
        for (int st = 0; st < kRunTiles; ++st) acc = mma(kk[st], x[st], acc);
        *reinterpret_cast<f32x4*>(sc + lay.z + (j0 + r) * D + 16 * it + 4 * g) = acc;
      }
    }
  }
  for (int i = threadIdx.x; i < D; i += 256) sc[lay.dc + i] = GENERAL ? ds[(kRunTokens - 1) * LD + i] : num[1][kRunTokens - 1];
}

// grid (parts, heads, vdim / 16), four waves: an item's runs in turn for 16 value channels, from the state in its slot, which is
// left as it is behind them (the item's next runs, in another round of launches, begin there). Wave w makes the rows of tokens
// 16 w .. of W and keeps the state's key channels 16 (w + 4 o) .. in registers.
template <int DT, int FORM>
__global__ __launch_bounds__(256, 1) void runs_chain_kernel(DeltaRuns c, RunList list) {
  constexpr int D = DT * 16, LD = D + 4, OWN = (DT + 3) / 4;
  constexpr bool GENERAL = FORM == kGeneralForm, SOLVES = FORM != kPlainForm;
  __shared__ __align__(16) float st_s[16 * LD];          // the state, [value channel][key channel]
  __shared__ f32x4 w_s[kRunTiles][64];
  __shared__ int odd_s[kRunTiles];                       // per wave: W is not finite
  __shared__ float sum_s[2][2][kRunTiles][16];
  const int item = list.item[blockIdx.x], first = list.first[blockIdx.x], runs = list.runs[blockIdx.x];
  const int h = blockIdx.y, j0 = blockIdx.z * 16;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const RunLayout lay = run_layout(D, c.vdim, GENERAL);
  const int64_t run_stride = static_cast<int64_t>(c.heads) * lay.total;
  float* sc = c.scratch + (static_cast<int64_t>(first) * c.heads + h) * lay.total;
  float* st = c.state + static_cast<int64_t>(c.slots[item]) * c.state_row + (static_cast<int64_t>(h) * c.vdim + j0 + r) * D + 4 * g;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  f32x4 s[OWN];
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int it = wave + 4 * o;
    s[o] = it < DT ? *reinterpret_cast<const f32x4*>(st + 16 * it) : zero;
  }
  // What a run needs from memory. Two runs' operands are held: a run's are asked for as soon as those of the run two in
  // front of it have been used, more than a run's time ahead.
  struct Operands {
    f32x4 kt[DT], wx, kd[OWN][kRunTiles], dc[OWN], z[OWN];
  };
  Operands even, odd;
  auto ask_front = [&](Operands& a, int run) {           // what the first product takes
    const float* q = sc + min(run, runs - 1) * run_stride;             // no branch: what is asked for behind the last is not used
    if constexpr (SOLVES) {
#pragma unroll
      for (int d = 0; d < DT; ++d) a.kt[d] = *reinterpret_cast<const f32x4*>(q + lay.kt + (16 * wave + r) * D + 16 * d + 4 * g);
    }
    a.wx = *reinterpret_cast<const f32x4*>(q + lay.w + (j0 + r) * kRunTokens + 16 * wave + 4 * g);
  };
  auto ask_back = [&](Operands& a, int run) {            // what the second takes
    const float* q = sc + min(run, runs - 1) * run_stride;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int it = min(wave + 4 * o, DT - 1);
#pragma unroll
      for (int t = 0; t < kRunTiles; ++t) a.kd[o][t] = *reinterpret_cast<const f32x4*>(q + lay.kd + (16 * it + r) * kRunTokens + 16 * t + 4 * g);
      a.dc[o] = *reinterpret_cast<const f32x4*>(q + lay.dc + 16 * it + 4 * g);
      if constexpr (GENERAL) a.z[o] = *reinterpret_cast<const f32x4*>(q + lay.z + (j0 + r) * D + 16 * it + 4 * g);
    }
  };
  // Sum over all key channels of a value channel, in every thread of its column.
  auto column_sum = [&](float v, float (*parts)[16]) {
    v += __shfl_xor(v, 16, kWave);
    v += __shfl_xor(v, 32, kWave);
    if (g == 0) parts[wave][r] = v;
    lds_barrier();
    return parts[0][r] + parts[1][r] + parts[2][r] + parts[3][r];
  };
  // A run token by token, outputs included.
  auto walk_tokens = [&](int run) {
    const int64_t t0 = list.t0[first + run];
    const int n = list.tokens[first + run];
    for (int t = 0; t < n; ++t) {
      const int64_t scal = (t0 + t) * c.scal_row + h, head = (t0 + t) * c.out_row + static_cast<int64_t>(h) * c.vdim + j0 + r;
      const int64_t key = (t0 + t) * c.key_row + static_cast<int64_t>(h / c.heads_per_group) * D + 4 * g;
      const float xs = c.xscal != nullptr ? c.xscal[scal] : 1.f, ps = c.pscal != nullptr ? c.pscal[scal] : 1.f;
      const float x = xs * c.x[(t0 + t) * c.x_row + static_cast<int64_t>(h) * c.vdim + j0 + r];
      const float ds = !GENERAL && c.dscal != nullptr ? c.dscal[scal] : 1.f;
      auto row = [&](const float* v, int it) { return *reinterpret_cast<const f32x4*>(v + key + 16 * it); };
      auto dot = [](f32x4 a, f32x4 b) { return a[0] * b[0] + a[1] * b[1] + a[2] * b[2] + a[3] * b[3]; };
      float taken = 0.f, read = 0.f;
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        const int it = wave + 4 * o;
        if (it >= DT) break;
        if constexpr (GENERAL) {
          taken += dot(s[o], row(c.cvec, it));
#pragma unroll
          for (int i = 0; i < 4; ++i) s[o][i] *= c.dvec[(t0 + t) * c.dvec_row + static_cast<int64_t>(h) * D + 16 * it + 4 * g + i];
        } else {
          s[o] = s[o] * ds;
          if constexpr (SOLVES) taken += dot(s[o], row(c.kvec, it));
        }
      }
      if constexpr (SOLVES) taken = ps * column_sum(taken, sum_s[0][t & 1]);
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        const int it = wave + 4 * o;
        if (it >= DT) break;
        if constexpr (SOLVES) s[o] += taken * row(c.pvec, it);
        s[o] += x * row(c.kvec, it);
        read += dot(s[o], row(c.rvec, it));
      }
      read = column_sum(read, sum_s[1][t & 1]);
      if (wave == 0 && g == 0) c.out[head] = read;
    }
  };
  auto walk = [&](Operands& a, int run) {
    float* q = sc + run * run_stride;
#pragma unroll
    for (int o = 0; o < OWN; ++o) {
      const int it = wave + 4 * o;
      if (it >= DT) break;
      *reinterpret_cast<f32x4*>(q + lay.s0 + (j0 + r) * D + 16 * it + 4 * g) = s[o];
      if constexpr (SOLVES) *reinterpret_cast<f32x4*>(st_s + r * LD + 16 * it + 4 * g) = s[o];
    }
    lds_barrier();                                       // the state is whole; the run before's W has been read
    f32x4 w = a.wx;
    if constexpr (SOLVES) {
      f32x4 from_state[4] = {zero, zero, zero, zero};
#pragma unroll
      for (int d = 0; d < DT; ++d) from_state[d % 4] = mma(a.kt[d], *reinterpret_cast<const f32x4*>(st_s + r * LD + 16 * d + 4 * g), from_state[d % 4]);
      w += (from_state[0] + from_state[1]) + (from_state[2] + from_state[3]);
      *reinterpret_cast<f32x4*>(q + lay.w + (j0 + r) * kRunTokens + 16 * wave + 4 * g) = w;
    }
    w_s[wave][lane] = w;
    const float zeros = fmaf(w[0], 0.f, w[1] * 0.f) + fmaf(w[2], 0.f, w[3] * 0.f);
    const bool odd = __any(zeros != 0.f);
    if (lane == 0) odd_s[wave] = odd;
    ask_front(a, run + 2);
    lds_barrier();
    const bool by_token = (odd_s[0] | odd_s[1] | odd_s[2] | odd_s[3]) != 0;
    if (threadIdx.x == 0) q[lay.walked + blockIdx.z] = by_token ? 1.f : 0.f;
    if (by_token) {
      walk_tokens(run);
    } else {
#pragma unroll
      for (int o = 0; o < OWN; ++o) {
        f32x4 sum = zero;
#pragma unroll
        for (int t = 0; t < kRunTiles; ++t) sum = mma(a.kd[o][t], w_s[t][lane], sum);
        if constexpr (GENERAL) sum += a.z[o];
        s[o] = s[o] * a.dc[o] + sum;
      }
    }
    ask_back(a, run + 2);
  };
  ask_front(even, 0);
  ask_back(even, 0);
  ask_front(odd, 1);
  ask_back(odd, 1);
  for (int run = 0; run < runs; run += 2) {
    walk(even, run);
    if (run + 1 < runs) walk(odd, run + 1);
  }
#pragma unroll
  for (int o = 0; o < OWN; ++o) {
    const int it = wave + 4 * o;
    if (it < DT) *reinterpret_cast<f32x4*>(st + 16 * it) = s[o];
  }
}

// grid (runs, heads), four waves: out = Qd S0 + P W (+ Y), rows of values, column t.
template <int DT, int FORM>
__global__ __launch_bounds__(256) void runs_output_kernel(DeltaRuns c, RunList list) {
  constexpr int D = DT * 16;
  constexpr bool GENERAL = FORM == kGeneralForm;
  const int64_t t0 = list.t0[blockIdx.x];
  const int n = list.tokens[blockIdx.x];
  const int h = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4, t = 16 * wave + r;
  if (16 * wave >= n) return;                            // no barrier below
  const RunLayout lay = run_layout(D, c.vdim, GENERAL);
  const float* sc = c.scratch + (static_cast<int64_t>(blockIdx.x) * c.heads + h) * lay.total;
  f32x4 q[DT], p[kRunTiles];
#pragma unroll
  for (int d = 0; d < DT; ++d) q[d] = *reinterpret_cast<const f32x4*>(sc + lay.qd + t * D + 16 * d + 4 * g);
#pragma unroll
  for (int st = 0; st < kRunTiles; ++st)
    p[st] = st <= wave ? *reinterpret_cast<const f32x4*>(sc + lay.p + t * kRunTokens + 16 * st + 4 * g) : f32x4{0.f, 0.f, 0.f, 0.f};
  const uint64_t walked = __ballot(lane < c.vdim / 16 && sc[lay.walked + lane % 16] != 0.f);
  float* o = c.out + (t0 + t) * c.out_row + static_cast<int64_t>(h) * c.vdim + 4 * g;
  for (int j0 = 0; j0 < c.vdim; j0 += 16) {
    if ((walked >> (j0 / 16) & 1) != 0) continue;
    f32x4 a[DT], w[kRunTiles];
#pragma unroll
    for (int d = 0; d < DT; ++d) a[d] = *reinterpret_cast<const f32x4*>(sc + lay.s0 + (j0 + r) * D + 16 * d + 4 * g);
#pragma unroll
    for (int st = 0; st < kRunTiles; ++st)
      if (st <= wave) w[st] = *reinterpret_cast<const f32x4*>(sc + lay.w + (j0 + r) * kRunTokens + 16 * st + 4 * g);
    // Added in pairs: one after the other the general form's outputs were 1.28e-7 and 1.35e-7 off 64 bits, so 1.18e-7 and 1.20e-7.
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    f32x4 left[DT], right[kRunTiles];
#pragma unroll
    for (int d = 0; d < DT; ++d) left[d] = mma(a[d], q[d], zero);
#pragma unroll
    for (int st = 0; st < kRunTiles; ++st) right[st] = st <= wave ? mma(w[st], p[st], zero) : zero;
#pragma unroll
    for (int half = DT / 2; half > 0; half /= 2)
#pragma unroll
      for (int d = 0; d < half; ++d) left[d] += left[d + half];
    f32x4 sum = left[0] + ((right[0] + right[1]) + (right[2] + right[3]));
    if (GENERAL && t < n) sum += *reinterpret_cast<const f32x4*>(o + j0);
    if (t < n) *reinterpret_cast<f32x4*>(o + j0) = sum;
  }
}

template <int DT, int FORM>
static int launch_runs(hipStream_t s, const DeltaRuns& c, const RunList& list, int n_runs, int n_parts) {
  constexpr int D = DT * 16;
  constexpr bool GENERAL = FORM == kGeneralForm;
  const dim3 all(static_cast<unsigned>(n_runs), static_cast<unsigned>(c.heads));
  const size_t smem = sizeof(float) * (2 * kRunTokens * kLd + (GENERAL ? kRunTokens * (D + 4) + c.vdim * kLd : 0));
  auto prepare = runs_prepare_kernel<DT, FORM>;
  if (smem > 60 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(prepare), hipFuncAttributeMaxDynamicSharedMemorySize,
                                              static_cast<int>(smem)) != hipSuccess)
    return fail("psamd_delta_runs: " + std::to_string(smem) + " bytes of LDS were refused");
  prepare<<<all, dim3(256), smem, s>>>(c, list);
  if (check_launch("psamd_delta_runs (prepare)")) return 1;
  runs_chain_kernel<DT, FORM><<<dim3(static_cast<unsigned>(n_parts), static_cast<unsigned>(c.heads), static_cast<unsigned>(c.vdim / 16)),
                                dim3(256), 0, s>>>(c, list);
  if (check_launch("psamd_delta_runs (chain)")) return 1;
  runs_output_kernel<DT, FORM><<<all, dim3(256), 0, s>>>(c, list);
  return check_launch("psamd_delta_runs (output)");
}

static int launch_runs_form(hipStream_t s, const DeltaRuns& c, const RunList& list, int n_runs, int n_parts, int dim, int form) {
  if (form == kGatedForm) return dim == 64 ? launch_runs<4, kGatedForm>(s, c, list, n_runs, n_parts) : launch_runs<8, kGatedForm>(s, c, list, n_runs, n_parts);
  if (form == kPlainForm) return dim == 64 ? launch_runs<4, kPlainForm>(s, c, list, n_runs, n_parts) : launch_runs<8, kPlainForm>(s, c, list, n_runs, n_parts);
  return dim == 64 ? launch_runs<4, kGeneralForm>(s, c, list, n_runs, n_parts) : launch_runs<8, kGeneralForm>(s, c, list, n_runs, n_parts);
}

}  // namespace psamd

using namespace psamd;

extern "C" {

// Whether psamd_delta_runs takes a recurrence of this shape: 1, or 0. general: a decay per key channel, of which decay_least
// is the least a token can have (the run's decays are divided by).
int psamd_delta_runs_supports(int dim, int vdim, int64_t key_row, int64_t x_row, int64_t out_row, int64_t dvec_row, int64_t state_row,
                              int general, float decay_least) {
  if ((dim != 64 && dim != 128) || vdim % 16 != 0 || vdim < 16 || vdim > 256) return 0;
  if (key_row % 4 != 0 || out_row % 4 != 0 || x_row < 1 || dvec_row < 0 || state_row % 4 != 0) return 0;
  // e^-40: D_s and its reciprocal, times operands of any ordinary size, stay far inside float32.
  if (general && !(decay_least > 0.f && kRunTokens * -logf(decay_least) <= 40.f)) return 0;
  return 1;
}

// How many runs of a recurrence of this shape the scratch holds at a time, and its floats. Both follow from the shape alone: the
// scratch is at most 384 MiB whatever a step holds (a step with more runs makes them in several rounds of launches), so that it
// never grows once a first prompt has been run. 64 runs of 16 heads of 128 x 128 (219 MB), 58 of 32 heads, 29 of 64. With 128 MiB
// 2,048 tokens of 32 heads took a second round (300 us instead of 273; 32 heads of 128 x 64 without removal 201 instead of 146).
int psamd_delta_runs_at_once(int heads, int dim, int vdim, int general) {
  const int64_t run = sizeof(float) * static_cast<int64_t>(heads) * run_layout(dim, vdim, general != 0).total;
  return static_cast<int>(std::min<int64_t>(kMaxRuns, kRunScratch / run));
}
int64_t psamd_delta_runs_floats(int heads, int dim, int vdim, int general) {
  return static_cast<int64_t>(psamd_delta_runs_at_once(heads, dim, vdim, general)) * heads * run_layout(dim, vdim, general != 0).total;
}

// starts: item_start on the host. Items of `most` tokens or fewer are left out.
int psamd_delta_runs(void* stream, const float* kvec, const float* cvec, const float* pvec, const float* rvec, int64_t key_row,
                     int key_groups, const float* dvec, int64_t dvec_row, const float* dscal, const float* pscal, const float* xscal,
                     int64_t scal_row, const float* x, int64_t x_row, float* out, int64_t out_row, float* state, int64_t state_row,
                     const int32_t* starts, const int32_t* slots, int items, int most, int heads, int dim, int vdim, int form,
                     float decay_least, float* scratch) {
  PSAMD_REQUIRE(form == kGatedForm || form == kPlainForm || form == kGeneralForm, "form: gated, plain or general");
  PSAMD_REQUIRE(items >= 0 && most >= 0 && heads > 0 && key_groups > 0 && heads % key_groups == 0, "bad sizes");
  const bool general = form == kGeneralForm;
  PSAMD_REQUIRE(psamd_delta_runs_supports(dim, vdim, key_row, x_row, out_row, dvec_row, state_row, general ? 1 : 0, decay_least), "unsupported shape");
  PSAMD_REQUIRE(general ? (dvec != nullptr && dscal == nullptr && pscal == nullptr && xscal == nullptr && key_groups == heads)
                        : (cvec == kvec && pvec == kvec && dvec == nullptr), "operands of another form");
  PSAMD_REQUIRE(kvec && cvec && pvec && rvec && x && out && state && starts && slots && scratch, "missing operands");
  const uintptr_t bits = reinterpret_cast<uintptr_t>(kvec) | reinterpret_cast<uintptr_t>(cvec) | reinterpret_cast<uintptr_t>(pvec) |
                         reinterpret_cast<uintptr_t>(rvec) | reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(state) |
                         reinterpret_cast<uintptr_t>(scratch);
  PSAMD_REQUIRE(bits % 16 == 0, "operands must lie on 16 bytes");
  PSAMD_REQUIRE(state_row >= static_cast<int64_t>(heads) * dim * vdim && heads <= 65535, "state rows too short, or too many heads");
  const int at_once = psamd_delta_runs_at_once(heads, dim, vdim, general ? 1 : 0);
  PSAMD_REQUIRE(at_once >= 1, "more heads than the scratch holds a run of");
  const DeltaRuns c{kvec, cvec, pvec, rvec, key_row, heads / key_groups, dvec, dvec_row, dscal, pscal, xscal, scal_row, x, x_row, out,
                    out_row, state, state_row, slots, heads, vdim, scratch};
  hipStream_t s = static_cast<hipStream_t>(stream);
  RunList list{};
  int n_runs = 0, n_parts = 0;
  for (int i = 0; i < items; ++i) {
    PSAMD_REQUIRE(starts[i] >= 0 && starts[i + 1] >= starts[i], "the items' first tokens must ascend");
    const int n = starts[i + 1] - starts[i];
    if (n <= most) continue;
    for (int q = 0; q < n; q += kRunTokens) {
      if (n_runs == at_once) {
        if (launch_runs_form(s, c, list, n_runs, n_parts, dim, form)) return 1;
        n_runs = n_parts = 0;
      }
      if (q == 0 || n_parts == 0) {
        list.item[n_parts] = i;
        list.first[n_parts] = n_runs;
        list.runs[n_parts++] = 0;
      }
      ++list.runs[n_parts - 1];
      list.t0[n_runs] = starts[i] + q;
      list.tokens[n_runs++] = std::min(kRunTokens, n - q);
    }
  }
  return n_runs == 0 ? 0 : launch_runs_form(s, c, list, n_runs, n_parts, dim, form);
}

}  // extern "C"
