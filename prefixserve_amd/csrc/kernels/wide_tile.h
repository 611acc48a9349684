// bfloat16 products in tiles of 256 x 256 by four waves of 128 x 128 that walk their workgroup's tiles without a break: the experts
// with many pairs (moe.hip) and the dense gated products (linear_tile.hip).
#pragma once

#include <type_traits>

#include "tile_product.h"

namespace psamd {

constexpr int kWideTile = 256;                         // rows of A and of W a tile
constexpr int kWideUnit = kWideTile * 128;             // one operand's 64 k of a tile in LDS
constexpr int kWideSmem = 5 * kWideUnit;               // all of a compute unit's
constexpr int kWideThreads = 256;

// A workgroup's tiles of `steps` times 64 k, one after the other; `Work` says what they are:
//   int kMinSteps                        the fewest steps that it works with, 2 or more; whoever launches it refuses fewer
//   bool a_rows(uint32_t (&off)[8])      the next tile's rows of A for the copies of this wave (copy i: rows 64 wave + 8 i + lane / 8), as
//                                        byte offsets from `a` of 16 bytes each (wide_piece); false: there is no next tile
//   bool w_rows(uint32_t (&off)[8])      likewise of W, behind work.w
//   int rows()                           the rows of A of the tile that is multiplied next (1 to 256)
//   void ahead()                         called behind that tile's first step: what may be loaded for the tiles to come
//   void finish<RM>(acc)                 acc[i][j]: lane (r, g) holds, of row 128 / 8 RM (wave / 2) + 16 j + r of A, rows 128 (wave % 2) + 16 i
//                                        + 4 g .. + 3 of W
// a_rows and w_rows are called once more than there are tiles. Copies run two steps ahead, so both are asked for the tile behind this one three steps in front
// of this one's end: from four steps on behind ahead(), with three in front of it, with two in front of this tile's rows() and two tiles ahead of finish.
//
// What bounds it: the matrix instructions' power at long K (256 x 256 tiles of 2,048 x 16,384 x 8,192: matrix cores busy 73% of the time at 1.93
// GHz; the library's kernel 84% at 1.75), beginnings and ends of tiles at short K. Why so:
//  * 128 x 128 a wave read LDS a third less than 128 x 64 (1,024 + 512 cycles of reads and copies a step beside 2,048 of matrix instructions,
//    where eight waves had 1,536 + 512). The sums then fill the accumulator registers, in place: the instructions are written out
//    because the compiler moves sums between registers where all 256 are in use.
//  * the copies run on from one tile into the next: no beginning waits for memory but the first. Five units of LDS are a ring; W, which
//    comes from memory, is asked for one step earlier than A.
//  * one barrier a step, between its halves: each half's operands are read while the half before is multiplied.
template <class Work>
__device__ __forceinline__ void wide_tiles(Work& work, const char* a, unsigned char* smem, int steps) {
  static_assert(Work::kMinSteps >= 2, "two steps are under way in front of the first");
  constexpr int RN = 8, RING = 5 * kWideUnit, COPIES = 8;
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int r = lane & 15, g = lane >> 4, swap = (r >> 1) & 7;
  const uint32_t share = static_cast<uint32_t>(wave) * (COPIES * 1024);
  uint32_t a_off[COPIES], w_off[COPIES];
  int k_a = 0, k_w = 0;                                // the step that is copied next
  uint32_t to_a = base + kWideUnit, to_w = base;       // and its unit
  auto turn = [&](uint32_t at) __attribute__((always_inline)) { return at + 2 * kWideUnit >= base + RING ? at + 2 * kWideUnit - RING : at + 2 * kWideUnit; };
  auto copy_a = [&](int i) __attribute__((always_inline)) { copy_to_lds(to_a + share + i * 1024, a_off[i], a + static_cast<int64_t>(k_a) * 128); };
  auto copy_w = [&](int i) __attribute__((always_inline)) { copy_to_lds(to_w + share + i * 1024, w_off[i], work.w + static_cast<int64_t>(k_w) * 128); };
  // Behind the last tile the copies go on, all lanes from the first bytes of an operand: every wait counts the same.
  auto next_a = [&]() __attribute__((always_inline)) {
    to_a = turn(to_a);
    if (++k_a == steps) {
      k_a = 0;
      if (!work.a_rows(a_off)) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) a_off[i] = 0;
      }
    }
  };
  auto next_w = [&]() __attribute__((always_inline)) {
    to_w = turn(to_w);
    if (++k_w == steps) {
      k_w = 0;
      if (!work.w_rows(w_off)) {
#pragma unroll
        for (int i = 0; i < COPIES; ++i) w_off[i] = 0;
      }
    }
  };
  if (!work.w_rows(w_off)) return;
  work.a_rows(a_off);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
#pragma unroll
    for (int i = 0; i < COPIES; ++i) copy_w(i);
    next_w();
#pragma unroll
    for (int i = 0; i < COPIES; ++i) copy_a(i);
    next_a();
  }
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(wait_for_copies(2 * COPIES));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  typedef __attribute__((address_space(3))) const tile_bf16x8 lds_piece;
  tile_bf16x8 fa[2][8], fb[2][RN];
  uint32_t at_a = base + kWideUnit, at_w = base;       // the units of the step whose operands are read
  // This lane's first piece of the first half of a unit; the second half's is 64 bytes away, in the sense of an exclusive or.
  const uint32_t lane_at = r * 128 + (g ^ swap) * 16, w_at = lane_at + (wave & 1) * (kWideTile / 2) * 128;
  bool more = true;
  while (more) {
    const int rows = work.rows();
    auto tile = [&](auto rm) __attribute__((always_inline)) {
      constexpr int RM = decltype(rm)::value, READ_EVERY = RM == 8 ? 3 : (RM >= 4 ? 2 : 1);
      // (A tile of fewer rows: the waves' first rows lie closer together. They are read again here, the half before did not know that.)
      uint32_t a_at = lane_at + (wave >> 1) * (RM * 16 * 128);
      asm volatile("" : "+v"(a_at));                   // not held for every size
#pragma unroll
      for (int i = 0; i < RN; ++i) fb[0][i] = *reinterpret_cast<lds_piece*>(at_w + w_at + i * 2048);
#pragma unroll
      for (int j = 0; j < RM; ++j) fa[0][j] = *reinterpret_cast<lds_piece*>(at_a + a_at + j * 2048);
      tile_f32x4 acc[RN][RM];
      auto half = [&](auto which_, auto first, auto last) __attribute__((always_inline)) {
        constexpr int which = decltype(which_)::value;
        if (which == 1) at_a = turn(at_a), at_w = turn(at_w);
        const uint32_t from_a = (at_a + a_at) ^ (which == 0 ? 64u : 0u), from_w = (at_w + w_at) ^ (which == 0 ? 64u : 0u);
#pragma unroll
        for (int i = 0; i < RN; ++i)
#pragma unroll
          for (int j = 0; j < RM; ++j) {
            if constexpr (decltype(first)::value)
              asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc[i][j]) : "v"(fb[which][i]), "v"(fa[which][j]));
            else
              asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[i][j]) : "v"(fb[which][i]), "v"(fa[which][j]));
            __builtin_amdgcn_sched_barrier(0);
            const int n = i * RM + j, q = n / READ_EVERY;
            if (!decltype(last)::value && n % READ_EVERY == 0 && q < RM + RN) {                       // the other half's operands
              if (q == 0) fb[which ^ 1][0] = *reinterpret_cast<lds_piece*>(from_w);
              else if (q <= RM) fa[which ^ 1][q - 1] = *reinterpret_cast<lds_piece*>(from_a + (q - 1) * 2048);
              else fb[which ^ 1][q - RM] = *reinterpret_cast<lds_piece*>(from_w + (q - RM) * 2048);
            }
            if (n % RM == 1) which == 0 ? copy_w(n / RM) : copy_a(n / RM);
            __builtin_amdgcn_sched_barrier(0);
          }
        which == 0 ? next_w() : next_a();
      };
      // The next step has arrived but for the W behind it, and everybody has read this one: its units are free.
      auto middle = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(wait_for_copies(COPIES));
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
      };
      using Zero = std::integral_constant<int, 0>;
      using One = std::integral_constant<int, 1>;
      half(Zero{}, std::true_type{}, std::false_type{});
      middle();
      half(One{}, std::false_type{}, std::false_type{});
      work.ahead();
      for (int t = 2; t < steps; ++t) {
        half(Zero{}, std::false_type{}, std::false_type{});
        middle();
        half(One{}, std::false_type{}, std::false_type{});
      }
      half(Zero{}, std::false_type{}, std::false_type{});
      middle();
      half(One{}, std::false_type{}, std::true_type{});
      asm volatile("s_nop 15\n\ts_nop 15" ::: "memory");                       // the last sums are in their registers
      __builtin_amdgcn_sched_barrier(0);
      more = work.template finish<RM>(acc);
      // An end of its own for each size: where the compiler let finish's branches end in a common one, it took what is uniform behind it for
      // different from lane to lane.
      asm volatile("; rows in %0" ::"n"(RM));
    };
    if (rows <= kWideTile / 4) tile(std::integral_constant<int, 2>{});
    else if (rows <= kWideTile / 2) tile(std::integral_constant<int, 4>{});
    else if (rows <= kWideTile / 4 * 3) tile(std::integral_constant<int, 6>{});
    else tile(std::integral_constant<int, 8>{});
  }
  __builtin_amdgcn_s_waitcnt(wait_for_copies(0));                                // LDS is not given back under a copy
}

// Which 16 bytes of a row's 128 a lane copies: the row's number exchanges them, as in tile_product.
__device__ __forceinline__ uint32_t wide_piece(int copy_row, int lane) { return 16u * tile_copy_piece(copy_row, lane); }

// Byte offset of a row of K numbers. Opaque: product and sum in one would be the 64-bit instruction, and every offset two registers.
__device__ __forceinline__ uint32_t wide_row(int row, int K) {
  uint32_t at = static_cast<uint32_t>(row) * (2u * K);
  asm volatile("" : "+v"(at));
  return at;
}

}  // namespace psamd
