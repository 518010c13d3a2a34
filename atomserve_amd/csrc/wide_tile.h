// The inner part of products in large tiles: both operands come into LDS by copies that pass no register.
//
// A workgroup of WM x WN waves owns a tile; a wave owns 16 FM rows of a x 16 FN rows of w.  K comes in units of 64 columns, each row of a
// unit one whole 128-byte line.  Units lie in rings: RA of a, RW of w (w comes from memory, a mostly from a cache, so w is asked for
// earlier where LDS has room for one ring more only).  A unit is two halves of 32 columns:
//   first half:   products of the first half, whose operands are in registers; the operands of the second are read; once all
//                 waves have them (a barrier) the unit's slots are free, and the copies of a's unit t + RA begin.
//   second half:  unit t + 1 has arrived (a barrier); products of the second half; the operands of unit t + 1's first are
//                 read; the copies of w's unit t + RW begin.
// Copies are spread between the products: in a burst they queue and hold up the wave that issues them (2,048 x 24,576 x 4,096, tiles of
// 256 x 256: 322 us in a burst, 302 spread; with rings of two for both 306, and with one barrier a unit, copies from its middle on, 332).
//
// PAIRED: which columns the halves are.  false: the first 32 and the second.  true: of every 16 columns the first eight and the second,
// as kernels have them whose lanes load 32 neighbouring bytes of a row: the same sums bit for bit.
// LDS piece (16 bytes) c of row r lies at c ^ swizzle(r): the 16 pieces that the hardware reads at once lie in different banks.
#pragma once
#include <type_traits>

#include "common.h"

namespace wide {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) char lds_char;

constexpr int UNIT = 64, ROW_BYTES = 2 * UNIT;  // columns of K in a unit

// 64 lanes copy 16 bytes each from buf + lane_at + at to lds + 16 lane.  It has no result in registers; the caller waits for it.  (The
// builtin of this instruction makes every later read of LDS wait for every copy in flight.)  m0 is named for the compiler's own users of it: a
// copy by the builtin beside this one is else given the m0 that this one left (the warning says that nobody keeps m0: that is what is wanted).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void copy_to_lds(__amdgpu_buffer_rsrc_t buf, unsigned lane_at, unsigned at, unsigned lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(lane_at), "s"(buf), "s"(at), "s"(lds)
               : "memory", "m0");
}
#pragma clang diagnostic pop

template <int WM, int WN, int FM, int FN, int RA, int RW, bool PAIRED = false>
struct Tile {
  static constexpr int WAVES = WM * WN;
  static constexpr int TM = 16 * WM * FM, TN = 16 * WN * FN;  // rows of a and of w in a tile
  static constexpr int A_UNIT = TM * ROW_BYTES, W_UNIT = TN * ROW_BYTES, LDS = RA * A_UNIT + RW * W_UNIT;
  static constexpr int A_COPIES = A_UNIT / 1024 / WAVES, W_COPIES = W_UNIT / 1024 / WAVES;  // a wave's copies of a unit, eight rows each
  static_assert(A_COPIES * WAVES * 1024 == A_UNIT && W_COPIES * WAVES * 1024 == W_UNIT && RA >= 2 && RW >= RA, "whole copies, rings of two and more");

  static __device__ __forceinline__ int swizzle(int r) { return PAIRED ? 0x32765410 >> ((r & 14) * 2) & 7 : r & 7; }
  // The row of the stage that this lane copies with copy i of its wave, and the byte of a unit's row that it takes.
  static __device__ __forceinline__ int row_of(int i, int wave, int lane) { return (i * WAVES + wave) * 8 + (lane >> 3); }
  static __device__ __forceinline__ unsigned piece_of(int row, int lane) { return ((lane & 7) ^ swizzle(row)) * 16u; }

  // acc += the products of `units` units (at least one).  a_at, w_at: this lane's bytes in the buffers for its copies (row and piece, column
  // 0); column(t): the byte of unit t in a row, for t >= units of one that may be asked for again.  idle: this wave's sums are wanted by
  // nobody; it copies and keeps step.  Ends with no copy in flight.
  template <typename Column>
  static __device__ __forceinline__ void run(char* lds, const __amdgpu_buffer_rsrc_t& a_buf, const __amdgpu_buffer_rsrc_t& w_buf,
                                             const unsigned (&a_at)[A_COPIES], const unsigned (&w_at)[W_COPIES], int wave, int wm, int wn, int lane,
                                             int units, Column column, floatx4 (&acc)[FM][FN], bool idle = false) {
    const int lr = lane & 15, lg = lane >> 4;
    lds_char* const stage_a = (lds_char*)lds;
    lds_char* const stage_w = stage_a + RA * A_UNIT;
    const unsigned to_a = (unsigned)(uintptr_t)stage_a + wave * 1024, to_w = (unsigned)(uintptr_t)stage_w + wave * 1024;
    auto copy_a = [&](int i, int slot, unsigned at) { copy_to_lds(a_buf, a_at[i], at, to_a + slot * A_UNIT + i * WAVES * 1024); };
    auto copy_w = [&](int i, int slot, unsigned at) { copy_to_lds(w_buf, w_at[i], at, to_w + slot * W_UNIT + i * WAVES * 1024); };

    // operands: row lr of every 16, a piece for each lane group; the second half's pieces lie at ^ FLIP
    constexpr unsigned FLIP = PAIRED ? 16 : 64;
    const unsigned swizzled = ((PAIRED ? 2 * lg : lg) ^ swizzle(lr)) * 16;
    const unsigned a_from = (wm * 16 * FM + lr) * ROW_BYTES + swizzled, w_from = (wn * 16 * FN + lr) * ROW_BYTES + swizzled;
    auto read = [](lds_char* at) { return *(const __attribute__((address_space(3))) bf16x8*)at; };

    // The products of a half and what goes between them, in the order in which it is written (a scheduler that moves the reads
    // towards their use leaves the matrix cores waiting).
    auto half = [&](const bf16x8 (&av)[FM], const bf16x8 (&wv)[FN], bf16x8 (&next_a)[FM], bf16x8 (&next_w)[FN], unsigned flip, int a_slot,
                    int w_slot, auto first, int w_free, int t) {
      constexpr int ALL = FM * FN, READS = FM + FN;
      constexpr int READ_OVER = ALL * (first ? 30 : 60) / 100, FREE_AT = ALL * 40 / 100;  // the products that the reads are spread over
      lds_char* const aa = stage_a + a_slot * A_UNIT + (a_from ^ flip);
      lds_char* const ww = stage_w + w_slot * W_UNIT + (w_from ^ flip);
      const unsigned a_column = column(t + RA), w_column = column(t + RW);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < ALL; ++i) {
        acc[i / FN][i % FN] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[i % FN], av[i / FN], acc[i / FN][i % FN], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = min(i, READ_OVER) * READS / READ_OVER; r < min(i + 1, READ_OVER) * READS / READ_OVER; ++r) {
          if (r < FN) next_w[r] = read(ww + r * 16 * ROW_BYTES);
          else next_a[r - FN] = read(aa + (r - FN) * 16 * ROW_BYTES);
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (first) {
          if (i == FREE_AT) {  // every wave has read all of unit t
            asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
          }
          if (i >= FREE_AT) {
#pragma unroll
            for (int d = (i - FREE_AT) * A_COPIES / (ALL - FREE_AT); d < (i + 1 - FREE_AT) * A_COPIES / (ALL - FREE_AT); ++d) {
              copy_a(d, a_slot, a_column);
              __builtin_amdgcn_sched_barrier(0);
            }
          }
        } else {
#pragma unroll
          for (int d = i * W_COPIES / ALL; d < (i + 1) * W_COPIES / ALL; ++d) {
            copy_w(d, w_free, w_column);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };

    // Copies are counted: those of a's unit u + RA and w's unit u + RW follow one another, and where RW is the larger, w's of the
    // units between go first.
    constexpr int LATER = RW > RA ? W_COPIES : 0;
#pragma unroll
    for (int u = 0; u < RW - RA; ++u)
#pragma unroll
      for (int i = 0; i < W_COPIES; ++i) copy_w(i, u, column(u));
#pragma unroll
    for (int u = 0; u < RA; ++u) {
#pragma unroll
      for (int i = 0; i < A_COPIES; ++i) copy_a(i, u, column(u));
#pragma unroll
      for (int i = 0; i < W_COPIES; ++i) copy_w(i, u + RW - RA, column(u + RW - RA));
    }
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((RA - 1) * (A_COPIES + W_COPIES) + LATER) : "memory");
    // of unit t + 1 all has arrived while its followers' copies, those of units t + 2 .. t + RA of a and t + 2 .. t + RW - 1 of w, are in flight
    constexpr int FLIGHT = (RA - 2) * (A_COPIES + W_COPIES) + A_COPIES + LATER;
    int a_slot = 0, w_slot = 0;
    if (idle) {
      for (int t = 0; t < units; ++t) {
        asm volatile("s_barrier" ::: "memory");
#pragma unroll
        for (int d = 0; d < A_COPIES; ++d) copy_a(d, a_slot, column(t + RA));
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(FLIGHT) : "memory");
#pragma unroll
        for (int d = 0; d < W_COPIES; ++d) copy_w(d, w_slot, column(t + RW));
        a_slot = a_slot + 1 == RA ? 0 : a_slot + 1;
        w_slot = w_slot + 1 == RW ? 0 : w_slot + 1;
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      return;
    }
    bf16x8 a0[FM], w0[FN], a1[FM], w1[FN];
#pragma unroll
    for (int f = 0; f < FN; ++f) w0[f] = read(stage_w + w_from + f * 16 * ROW_BYTES);
#pragma unroll
    for (int f = 0; f < FM; ++f) a0[f] = read(stage_a + a_from + f * 16 * ROW_BYTES);
    for (int t = 0; t < units; ++t) {
      half(a0, w0, a1, w1, FLIP, a_slot, w_slot, std::true_type{}, 0, t);
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(FLIGHT) : "memory");
      const int w_free = w_slot;
      a_slot = a_slot + 1 == RA ? 0 : a_slot + 1;
      w_slot = w_slot + 1 == RW ? 0 : w_slot + 1;
      half(a1, w1, a0, w0, 0u, a_slot, w_slot, std::false_type{}, w_free, t);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the LDS is another workgroup's after the end
  }
};

}  // namespace wide
