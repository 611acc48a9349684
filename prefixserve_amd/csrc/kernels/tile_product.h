// The loop of the bfloat16 products whose operands both pass through LDS in large tiles: a workgroup's tile of A [rows, K] times
// its tile of W [rows, K]^T, 64 k at a time, for the experts with many pairs (moe.hip) and the dense products (linear_tile.hip). (Tiles of
// 256 x 256: wide_tile.h.)
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace psamd {

typedef __attribute__((ext_vector_type(8))) __bf16 tile_bf16x8;
typedef __attribute__((ext_vector_type(4))) float tile_f32x4;

// 64 lanes x 16 bytes from base + offset (a lane's own) to LDS at `to`, side by side: no register receives them. Written out because
// the compiler waits for every copy under way in front of any read of LDS that it sees; whoever reads them waits for them itself.
__device__ __forceinline__ void copy_to_lds(uint32_t to, uint32_t offset, const char* base) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(to), "v"(offset), "s"(base)
               : "memory", "m0");
}

constexpr int wait_for_copies(int left) { return (left & 15) | ((left >> 4) << 14) | (7 << 4); }   // s_waitcnt vmcnt(left) lgkmcnt(0)

// Rows lie in LDS as 128 bytes, their eight 16-byte pieces exchanged by row / 2, so that the 16 rows that a read touches lie on all
// banks; the exchange is done by which piece a lane fetches. Copy i of a wave brings rows 8 i .. 8 i + 7 of its share.
__device__ __forceinline__ int tile_copy_piece(int row, int lane) { return (lane & 7) ^ ((row >> 1) & 7); }

// acc[i][j] += the 16 x 16 products of W rows b_row + 16 i .. and A rows a_row + 16 j .. of the workgroup's tile: lane (r, g) gets, of
// A's row 16 j + r, columns 16 i + 4 g .. + 3. `smem` holds STAGES x [A_ROWS rows of A, B_ROWS of W]; copy i of this wave is
// a_off[i] bytes behind `a` in k step 0 and goes to row 8 (wave LA + i) (w likewise). Every wave of the workgroup comes here with
// the same `steps` (>= 1); where `works` is false (uniform for the wave) it only copies. What bounds it and what it does about it:
//  * the latency of memory: STAGES - 1 steps are under way behind the one that is multiplied;
//  * LDS, whose reads and writes take as long as the matrix instructions at 192 x 128 a workgroup: the operands
//    of half a step are read between the matrix instructions of the half before, and the one barrier of a step stands
//    between its halves, where the matrix cores still have work; waves in their matrix instructions go first.
// On return nothing is under way and LDS may still be read by other waves.
template <int STAGES, int A_ROWS, int B_ROWS, int RM, int RN, int LA, int LB>
__device__ __forceinline__ void tile_product(tile_f32x4 (&acc)[RN][RM], unsigned char* smem, const char* a, const char* w,
                                             const uint32_t (&a_off)[LA], const uint32_t (&b_off)[LB], int a_row, int b_row, int wave,
                                             int lane, int steps, bool works) {
  constexpr int STAGE = (A_ROWS + B_ROWS) * 128, COPIES = LA + LB;
  const uint32_t base = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)smem));
  auto copy = [&](int t, int buf) {
    const uint32_t to = base + buf * STAGE;
#pragma unroll
    for (int i = 0; i < LA; ++i) copy_to_lds(to + (wave * LA + i) * 1024, a_off[i], a + static_cast<int64_t>(t) * 128);
#pragma unroll
    for (int i = 0; i < LB; ++i) copy_to_lds(to + A_ROWS * 128 + (wave * LB + i) * 1024, b_off[i], w + static_cast<int64_t>(t) * 128);
  };
  const int r = lane & 15, g = lane >> 4, swap = (r >> 1) & 7;
  tile_bf16x8 fa[2][RM], fb[2][RN];
  auto operands = [&](int buf, int half) {
    const unsigned char* at = smem + buf * STAGE + ((half * 4 + g) ^ swap) * 16 + r * 128;
#pragma unroll
    for (int i = 0; i < RN; ++i) fb[half][i] = *reinterpret_cast<const tile_bf16x8*>(at + (A_ROWS + b_row + i * 16) * 128);
#pragma unroll
    for (int j = 0; j < RM; ++j) fa[half][j] = *reinterpret_cast<const tile_bf16x8*>(at + (a_row + j * 16) * 128);
  };
  auto multiply = [&](int half) {
#pragma unroll
    for (int i = 0; i < RN; ++i)
#pragma unroll
      for (int j = 0; j < RM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[half][i], fa[half][j], acc[i][j], 0, 0, 0);
    constexpr int BESIDE = RM * RN / (RM + RN) > 0 ? RM * RN / (RM + RN) : 1;
#pragma unroll
    for (int q = 0; q < RM + RN; ++q) {                                          // one read of the other half's operands, then
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                         // the matrix instructions it hides behind
      __builtin_amdgcn_sched_group_barrier(0x008, BESIDE, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, RM * RN, 0);
  };
#pragma unroll
  for (int t = 0; t < STAGES; ++t)
    if (t < steps) copy(t, t);
  __builtin_amdgcn_sched_barrier(0);
  if (steps >= STAGES) __builtin_amdgcn_s_waitcnt(wait_for_copies((STAGES - 1) * COPIES));
  else __builtin_amdgcn_s_waitcnt(wait_for_copies(0));
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  if (works) operands(0, 0);
  int buf = 0;
  for (int t = 0; t < steps; ++t) {
    const int next = buf + 1 == STAGES ? 0 : buf + 1;
    if (works) {
      __builtin_amdgcn_s_setprio(1);
      operands(buf, 1);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
    }
    // Step t + 1 has arrived (of what was asked for, only the steps behind it may be under way), and everybody has read step t.
    __builtin_amdgcn_sched_barrier(0);
    if (t + STAGES - 1 < steps) __builtin_amdgcn_s_waitcnt(wait_for_copies((STAGES - 2) * COPIES));
    else __builtin_amdgcn_s_waitcnt(wait_for_copies(0));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    if (t + STAGES < steps) copy(t + STAGES, buf);
    __builtin_amdgcn_sched_barrier(0);
    if (works) {
      __builtin_amdgcn_s_setprio(1);
      operands(next, 0);                        // behind the last step: what lies there, not used
      multiply(1);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(0);
    }
    buf = next;
  }
}

}  // namespace psamd
