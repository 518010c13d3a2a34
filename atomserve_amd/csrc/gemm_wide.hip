// bf16 products of many rows, out[M, N] = a[M, K] @ w[N, K]^T: tiles of up to 256 x 256 outputs whose operands both come into LDS by
// copies that pass no register (`wide_tile.h`, where the order of copies, reads and products stands).
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
#include "wide_tile.h"

namespace {

using namespace wide;

enum { PLAIN = 0, GATED = 1, PARTIAL = 2 };

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
  using T = Tile<WM, WN, FM, FN, RA, RW>;
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
  const int m0 = tm * T::TM, n0 = tn * (KIND == GATED ? T::TN / 2 : T::TN);
  const int u0 = blockIdx.y * units_per_split;
  const int units = min(K / UNIT - u0, units_per_split);
  auto column = [&](int t) { return (unsigned)(u0 + min(t, units - 1)) * ROW_BYTES; };  // units past the last are the last again

  const unsigned pitch = (unsigned)K * 2u;
  const __amdgpu_buffer_rsrc_t a_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, (int)((unsigned)M * pitch), 0x00020000);
  const __amdgpu_buffer_rsrc_t w_buf = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<bf16*>(w), 0, (int)((unsigned)(KIND == GATED ? 2 * N : N) * pitch), 0x00020000);

  // A copy takes eight rows; this lane's piece of them.  Rows beyond the last repeat it: nothing outside the matrices is asked for,
  // and such rows' sums are not stored.
  unsigned a_at[T::A_COPIES], w_at[T::W_COPIES];
#pragma unroll
  for (int i = 0; i < T::A_COPIES; ++i) {
    const int row = T::row_of(i, wave, lane);
    a_at[i] = (unsigned)min(m0 + row, M - 1) * pitch + T::piece_of(row, lane);
  }
#pragma unroll
  for (int i = 0; i < T::W_COPIES; ++i) {
    const int row = T::row_of(i, wave, lane);  // of the stage: of wave column `strip` operand f, row 4 g + r, whose sums lane group g holds
    const int strip = row / (16 * FN), q = row % (16 * FN), f = q >> 4, g = (q >> 2) & 3, r = q & 3;
    int n;
    if constexpr (KIND == GATED) n = min(n0 + strip * 8 * FN + g * 2 * FN + 2 * f + (r & 1), N - 1) + (r >> 1) * N;
    else if constexpr (KIND == PARTIAL) n = min(n0 + row, N - 1);
    else n = min(n0 + strip * 16 * FN + ((f | 1) < FN ? (f & ~1) * 16 + 8 * g + 4 * (f & 1) : f * 16 + 4 * g) + r, N - 1);
    w_at[i] = (unsigned)n * pitch + T::piece_of(row, lane);
  }
  floatx4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  T::run(lds, a_buf, w_buf, a_at, w_at, wave, wm, wn, lane, units, column, acc);

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
  using T = Tile<WM, WN, FM, FN, RA, RW>;
  constexpr int TM = T::TM, TN = T::TN / (KIND == GATED ? 2 : 1), shmem = T::LDS;
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
