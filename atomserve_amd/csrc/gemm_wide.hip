// bf16 products of many rows, out[M, N] = a[M, K] @ w[N, K]^T: tiles of up to 256 x 256 outputs whose operands both come into LDS by
// copies that pass no register.
//
// A workgroup of WM x WN waves owns a tile; a wave owns 16 FM rows x 16 FN columns of it.  K comes in units of 64 columns, each row of a
// unit one whole 128-byte line.  Units lie in rings: RA of a, RW of w (w comes from memory, a mostly from a cache, so w is asked for
// earlier where LDS has room for one ring more only).  A unit is two halves of 32 columns:
//   first half:   products of the first 32 columns, whose operands are in registers; the operands of the second 32 are read; once all
//                 waves have them (a barrier) the unit's slots are free, and the copies of a's unit t + RA begin.
//   second half:  unit t + 1 has arrived (a barrier); products of the second 32 columns; the operands of unit t + 1's first 32 are
//                 read; the copies of w's unit t + RW begin.
// Copies are spread between the products: in a burst they queue and hold up the wave that issues them (2,048 x 24,576 x 4,096, tiles of
// 256 x 256: 322 us in a burst, 302 spread; with rings of two for both 306, and with one barrier a unit, copies from its middle on, 332).
// LDS piece (16 bytes) c of row r lies at c ^ (r % 8): the eight rows that neighbouring lanes read lie in different banks (no
// conflicts counted).
//
// What bounds it: with all compute units busy the clock falls to 1.7 to 1.8 GHz (power); at 2,048 x 8,192 outputs a unit of K takes 1.50 us
// (the library's 1.38), on half of the units 1.05 of which the matrix cores' own time is 0.87.  Beyond the units a tile takes 5 to 8 us:
// the first copies' way, and the results, which a lane stores 16 bytes at a time (rows of w are dealt to the stage so that a lane's sums
// are neighbours; 8 bytes at a time cost 6 to 13 us more).  Four waves of 128 x 128 instead of eight of 128 x 64: the same within 4 per cent.
//
//   PLAIN    out bf16
//   GATED    w is [2 N, K], gate rows, then up rows: out = silu(gate) * up, both rounded to bf16 first (the bits of a product and
//            silu_mul).  A stage deals two gate and two up rows to each lane, so nothing has to meet.
//   PARTIAL  blockIdx.y names a range of K, whose fp32 sums go to out[range][M][N] for whoever adds them up
#include <type_traits>

#include "common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) char lds_char;

constexpr int UNIT = 64, ROW_BYTES = 2 * UNIT;  // columns of K in a unit

enum { PLAIN = 0, GATED = 1, PARTIAL = 2 };

// 64 lanes copy 16 bytes each from buf + lane_at + at to lds + 16 lane.  It has no result in registers; the caller waits for it.  (The
// builtin of this instruction makes every later read of LDS wait for every copy in flight.)
__device__ __forceinline__ void copy_to_lds(__amdgpu_buffer_rsrc_t buf, unsigned lane_at, unsigned at, unsigned lds) {
  asm volatile("s_mov_b32 m0, %3\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(lane_at), "s"(buf), "s"(at), "s"(lds) : "memory");
}

// COUNT neighbouring results of which the first `room` exist; o lies on 2 COUNT bytes, on 4 where COUNT is 6
template <int COUNT>
__device__ __forceinline__ void put(bf16* o, const bf16* v, int room) {
  if (room >= COUNT) {
    if constexpr (COUNT == 8) {
      *(u32x4*)o = *(const u32x4*)v;
    } else if constexpr (COUNT == 4) {
      *(u32x2*)o = *(const u32x2*)v;
    } else {
#pragma unroll
      for (int i = 0; i < COUNT; i += 2) *(unsigned*)(o + i) = *(const unsigned*)(v + i);
    }
  } else {
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
      if (i < room) o[i] = v[i];
  }
}

template <int WM, int WN, int FM, int FN, int RA, int RW, int KIND>
__global__ __launch_bounds__(WM * WN * 64, WM * WN / 4) void gemm_wide_kernel(const bf16* __restrict__ a, const bf16* __restrict__ w,
                                                                            void* __restrict__ out, int M, int N, int K, int tiles_m,
                                                                            int tiles_n, int units_per_split) {
  constexpr int WAVES = WM * WN;
  constexpr int TM = 16 * WM * FM, TN = 16 * WN * FN;  // rows of a and of w in a tile
  constexpr int A_UNIT = TM * ROW_BYTES, W_UNIT = TN * ROW_BYTES;
  constexpr int A_COPIES = A_UNIT / 1024 / WAVES, W_COPIES = W_UNIT / 1024 / WAVES;  // a wave's copies of a unit
  static_assert(A_COPIES * WAVES * 1024 == A_UNIT && W_COPIES * WAVES * 1024 == W_UNIT && RA >= 2 && RW >= RA, "whole copies, rings of two and more");
  extern __shared__ __attribute__((aligned(128))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;

  // workgroups are dealt to the eight XCDs in turn: each takes a run of tiles, down the rows of a first, so that what runs on it
  // at one time shares rows of w and of a in its L2
  const int total = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7;
  const int tile = xcd * (total >> 3) + min(xcd, total & 7) + (int)(blockIdx.x >> 3);
  const int tm = tile % tiles_m, tn = tile / tiles_m;
  const int m0 = tm * TM, n0 = tn * (KIND == GATED ? TN / 2 : TN);
  const int u0 = blockIdx.y * units_per_split;
  const int units = min(K / UNIT - u0, units_per_split);
  auto column = [&](int t) { return (unsigned)(u0 + min(t, units - 1)) * ROW_BYTES; };  // units past the last are the last again

  const unsigned pitch = (unsigned)K * 2u;
  const __amdgpu_buffer_rsrc_t a_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, (int)((unsigned)M * pitch), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_buf = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16*>(w), 0, (int)((unsigned)(KIND == GATED ? 2 * N : N) * pitch), 0x00020000);

  // A copy takes eight rows; this lane's piece of them.  Rows beyond the last repeat it: nothing outside the matrices is asked for,
  // and such rows' sums are not stored.
  const int e = lane >> 3;
  const unsigned piece = ((lane & 7) ^ e) * 16u;
  unsigned a_at[A_COPIES], w_at[W_COPIES];
#pragma unroll
  for (int i = 0; i < A_COPIES; ++i) a_at[i] = (unsigned)min(m0 + (i * WAVES + wave) * 8 + e, M - 1) * pitch + piece;
#pragma unroll
  for (int i = 0; i < W_COPIES; ++i) {
    const int row = (i * WAVES + wave) * 8 + e;  // of the stage: of wave column `strip` operand f, row 4 g + r, whose sums lane group g holds
    const int strip = row / (16 * FN), q = row % (16 * FN), f = q >> 4, g = (q >> 2) & 3, r = q & 3;
    int n;
    if constexpr (KIND == GATED) n = min(n0 + strip * 8 * FN + g * 2 * FN + 2 * f + (r & 1), N - 1) + (r >> 1) * N;
    else if constexpr (KIND == PARTIAL) n = min(n0 + row, N - 1);
    else n = min(n0 + strip * 16 * FN + ((f | 1) < FN ? (f & ~1) * 16 + 8 * g + 4 * (f & 1) : f * 16 + 4 * g) + r, N - 1);
    w_at[i] = (unsigned)n * pitch + piece;
  }
  lds_char* const stage_a = (lds_char*)lds;
  lds_char* const stage_w = stage_a + RA * A_UNIT;
  const unsigned to_a = (unsigned)(uintptr_t)stage_a + wave * 1024, to_w = (unsigned)(uintptr_t)stage_w + wave * 1024;
  auto copy_a = [&](int i, int slot, unsigned at) { copy_to_lds(a_buf, a_at[i], at, to_a + slot * A_UNIT + i * WAVES * 1024); };
  auto copy_w = [&](int i, int slot, unsigned at) { copy_to_lds(w_buf, w_at[i], at, to_w + slot * W_UNIT + i * WAVES * 1024); };

  // operands: row lr of every 16, the lg-th eight columns of 32; the second 32 columns lie at ^ 64
  const unsigned swizzled = (lg ^ (lr & 7)) * 16;
  const unsigned a_from = (wm * 16 * FM + lr) * ROW_BYTES + swizzled, w_from = (wn * 16 * FN + lr) * ROW_BYTES + swizzled;
  auto read = [](lds_char* at) { return *(const __attribute__((address_space(3))) bf16x8*)at; };

  floatx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // The products of 32 columns and what goes between them, in the order in which it is written (a scheduler that moves the reads
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
  bf16x8 a0[FM], w0[FN], a1[FM], w1[FN];
#pragma unroll
  for (int f = 0; f < FN; ++f) w0[f] = read(stage_w + w_from + f * 16 * ROW_BYTES);
#pragma unroll
  for (int f = 0; f < FM; ++f) a0[f] = read(stage_a + a_from + f * 16 * ROW_BYTES);
  int a_slot = 0, w_slot = 0;
  for (int t = 0; t < units; ++t) {
    half(a0, w0, a1, w1, 64u, a_slot, w_slot, std::true_type{}, 0, t);
    // unit t + 1 has arrived: beyond its copies those of units t + 2 .. t + RA of a and t + 2 .. t + RW - 1 of w may be in flight
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((RA - 2) * (A_COPIES + W_COPIES) + A_COPIES + LATER) : "memory");
    const int w_free = w_slot;
    a_slot = a_slot + 1 == RA ? 0 : a_slot + 1;
    w_slot = w_slot + 1 == RW ? 0 : w_slot + 1;
    half(a1, w1, a0, w0, 0u, a_slot, w_slot, std::false_type{}, w_free, t);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the LDS is another workgroup's after the end

  // lane (lr, lg) holds sums 4 lg .. 4 lg + 3 of every 16 rows of a stage's w (j) with row lr of every 16 rows of a (i)
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m0 + wm * 16 * FM + i * 16 + lr;
    if (m >= M) continue;
    if constexpr (KIND == GATED) {
      const int n = n0 + wn * 8 * FN + lg * 2 * FN;
      alignas(16) bf16 v[2 * FN];
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          const float g = (float)(bf16)acc[i][j][r];
          v[2 * j + r] = (bf16)(g / (1.0f + expf(-g)) * (float)(bf16)acc[i][j][2 + r]);
        }
#pragma unroll
      for (int j = 0; j < 2 * FN; j += 8) put<(2 * FN < 8 ? 2 * FN : 8)>((bf16*)out + (size_t)m * N + n + j, v + j, N - n - j);
    } else if constexpr (KIND == PARTIAL) {
      const int n = n0 + wn * 16 * FN + lg * 4;
      float* o = (float*)out + ((size_t)blockIdx.y * M + m) * N + n;
#pragma unroll
      for (int j = 0; j < FN; ++j)
        if (n + 16 * j < N) *(floatx4*)(o + 16 * j) = acc[i][j];
    } else {
#pragma unroll
      for (int j = 0; j < FN; j += 2) {
        const bool pair = j + 1 < FN;
        const int n = n0 + wn * 16 * FN + j * 16 + lg * (pair ? 8 : 4);
        bf16* o = (bf16*)out + (size_t)m * N + n;
        alignas(16) bf16 v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = (bf16)acc[i][r < 4 || !pair ? j : j + 1][r & 3];
        if (pair) put<8>(o, v, N - n);
        else put<4>(o, v, N - n);
      }
    }
  }
}

template <int WM, int WN, int FM, int FN, int RA, int RW, int KIND>
int launch(const void* a, const void* w, void* out, int M, int N, int K, int splits, hipStream_t stream) {
  constexpr int TM = 16 * WM * FM, TN = 16 * WN * FN / (KIND == GATED ? 2 : 1);
  constexpr int shmem = 16 * (RA * WM * FM + RW * WN * FN) * ROW_BYTES;
  auto kernel = gemm_wide_kernel<WM, WN, FM, FN, RA, RW, KIND>;
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, shmem) != hipSuccess) return AS_LAUNCH_FAILED;
    raised = true;
  }
  const int tiles_m = (M + TM - 1) / TM, tiles_n = (N + TN - 1) / TN;
  kernel<<<dim3(tiles_m * tiles_n, splits), WM * WN * 64, shmem, stream>>>((const bf16*)a, (const bf16*)w, out, M, N, K, tiles_m, tiles_n,
                                                                          (K / UNIT + splits - 1) / splits);
  return launch_status();
}

}  // namespace

// out[M, N] = a[M, K] @ w[N, K]^T; a, w and out start on 16 bytes, K % 64 == 0, N % 16 == 0, neither matrix beyond 0xf0000000 bytes.
//   kind:    0: out bf16; 1: w [2 N, K], out[M, N] = silu(gate) * up in bf16; 2: out fp32 [splits, M, N], the sums of `splits` ranges
//            of ceil(K / 64 / splits) units of 64 columns (the last may be shorter, none may be empty; other kinds: splits = 1).
//   form:    the tile, rows of a x rows of w (gate and up rows counted): 0: 256 x 256, 1: 256 x 192, 2: 256 x 128, 3: 192 x 256,
//            4: 128 x 128, 5: 128 x 128 in half the LDS, two to a compute unit.
extern "C" int as_gemm_bf16_wide(const void* a, const void* w, void* out, int M, int N, int K, int kind, int splits, int form, hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (N <= 0 || K <= 0 || K % UNIT || N % 16 || splits < 1 || kind < PLAIN || kind > PARTIAL || (kind != PARTIAL && splits != 1)) return AS_BAD_SHAPE;
  const int units = K / UNIT, per = (units + splits - 1) / splits;
  if ((long long)(splits - 1) * per >= units || splits > 65535) return AS_BAD_SHAPE;
  if (!a || !w || !out || (((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) & 15)) return AS_BAD_SHAPE;
  if ((kind == GATED ? 2ull : 1ull) * N * K * 2 > 0xf0000000ull || (unsigned long long)M * K * 2 > 0xf0000000ull) return AS_BAD_SHAPE;
#define FORM(NUMBER, ...)                                                                                          \
  if (form == NUMBER) {                                                                                            \
    if (kind == GATED) return launch<__VA_ARGS__, GATED>(a, w, out, M, N, K, splits, stream);                      \
    if (kind == PARTIAL) return launch<__VA_ARGS__, PARTIAL>(a, w, out, M, N, K, splits, stream);                  \
    return launch<__VA_ARGS__, PLAIN>(a, w, out, M, N, K, splits, stream);                                         \
  }
  FORM(0, 2, 4, 8, 4, 2, 3)
  FORM(1, 2, 4, 8, 3, 2, 3)
  FORM(2, 2, 4, 8, 2, 3, 3)
  FORM(3, 2, 2, 6, 8, 2, 3)
  FORM(4, 2, 4, 4, 2, 4, 4)
  FORM(5, 2, 2, 4, 4, 2, 2)
#undef FORM
  return AS_BAD_SHAPE;
}
