// Matrix products of 32-bit matrices: out[M, N] = a[M, K] @ w[N, K]^T (weights keep the checkpoint's [out, in] layout).
//
// A float is the sum of three bf16 values: its nearest one, the nearest one of what is left, and the rest, which fits
// (8 + 8 + 8 bits).  A product of two floats is then nine products of bf16 values, of which the matrix cores, sixteen times
// faster on bf16 than on fp32, compute the six largest; the three left out are below 2^-24 of the product and of either sign.
// Sums are fp32.  The largest of the six has a chain of sums of its own: small products that are added to a large sum are cut
// off downwards, and that error has one sign.  Against 64 bits (K = 1,024 / 2,048 / 3,072, normal values) the error is 0.76e-7 /
// 0.87e-7 / 0.98e-7 of the result (in one chain 1.15e-7 / 1.7e-7 / 2.1e-7), with the cores' fp32 instruction in the same order
// 1.55e-7 / 2.1e-7 / 2.6e-7; heavy tails, outliers and one sign alike: at most 0.9 of that instruction's error.
// Beside those distributions: numbers below 2^-110 keep an absolute error of 2^-134 instead, and a sum of one product that is not zero
// is not rounded correctly, as the fp32 instruction would (the error is below 2^-23 of it).  Values that are not finite (or that round to
// infinity in bf16) would become NaN in the parts: a result that is not finite is computed again with the fp32 instruction.
//
// The order of every output's sum depends on K alone, so a row's result does not depend on which other rows share the launch,
// nor on the kernel or the tile that the launch chose: K is cut into 16 slices of whole steps of 32 columns, each slice is one
// pair of chains (the largest products; the other five of a step in one order), four neighbouring slices are added up in order, then the four sums of four.
// Up to F32_NARROW columns the sum is one chain of fp32 multiply-adds over k = 0..K-1 in order.
// Plain reference: reference atomserve/quant.py:89-91 (F.linear).
#include "common.h"
#include "float_parts.h"

#define F32_SLICES 16
#define F32_GROUPS 4  // of neighbouring slices
#define F32_NARROW 256

__device__ __forceinline__ void store4(float* p, floatx4 v, int valid) {
  if (valid == 4 && (((uintptr_t)p) & 15) == 0) { *reinterpret_cast<floatx4*>(p) = v; return; }
  for (int i = 0; i < valid; ++i) p[i] = v[i];
}

// Columns k .. k+3 of a row, those from K on as zeros.  VEC: rows start on 16 bytes and K % 4 == 0; else the load needs no
// more than a float's alignment.  It ends where the row ends, and `ragged` puts zeros and moves what belongs elsewhere when the
// columns are used, where K ends: a test here would make every load wait for the one before, or choose eight times a step of 32 bytes.
typedef float floatx4_anywhere __attribute__((ext_vector_type(4), aligned(4)));

template <bool VEC> __device__ __forceinline__ floatx4 fetch(const float* row, int k, int K) {
  if constexpr (VEC) {
    return *reinterpret_cast<const floatx4*>(row + min(k, K - 4));
  } else {
    return *reinterpret_cast<const floatx4_anywhere*>(row + min(k, K - 4));  // K > F32_NARROW
  }
}

template <bool VEC> __device__ __forceinline__ floatx4 ragged(floatx4 v, int k, int K) {  // v: what `fetch` gave for k
  if constexpr (VEC) return k < K ? v : floatx4{0.f, 0.f, 0.f, 0.f};
  const int by = k - min(k, K - 4);
  if (by & 1) v = floatx4{v[1], v[2], v[3], 0.f};
  if (by & 2) v = floatx4{v[2], v[3], 0.f, 0.f};
  return by >= 4 ? floatx4{0.f, 0.f, 0.f, 0.f} : v;
}

// `v`, where it is not finite, again by the fp32 instruction over the steps st0 .. st1 - 1: 16 rows of w (this lane's `wrow`)
// by 16 of a.  All lanes of a wave call it together; seldom taken, so it waits for every step's loads.
template <bool VEC> __device__ __forceinline__ floatx4 again_f32(floatx4 v, const float* wrow, const float* arow, int K, int st0, int st1) {
  const int lg = (threadIdx.x & 63) >> 4;
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  for (int st = st0; st < st1; ++st)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int k = st * 32 + lg * 8 + half * 4;
      const floatx4 wv = ragged<VEC>(fetch<VEC>(wrow, k, K), k, K), av = ragged<VEC>(fetch<VEC>(arow, k, K), k, K);
#pragma unroll
      for (int x = 0; x < 4; ++x) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[x], av[x], acc, 0, 0, 0);
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = (__float_as_uint(v[r]) & 0x7f800000u) == 0x7f800000u ? acc[r] : v[r];
  return v;
}

// What a product carries along when the residual sum and the RMSNorm around it are folded into the products of a decode step
// (a pre-norm layer: x += part(norm(x))), as the few-rows products of bf16 do:
//   producer (LINK): the sum goes on top of the stream x = out[M, N]; scaled[M, N] = x * gain, the input of the next product
//     without its 1/rms factor; ssq_out[M, N / 4] = the sums of x^2 per 4 columns (whatever kernel makes them).
//   consumer (ssq_in): 1/rms of each row comes from the row's sums of squares and multiplies the product's sums.
struct LinkF32 {
  const float* ssq_in;
  int strips_in;
  float eps;
  const float* gain;
  float* scaled;
  float* ssq_out;
};

enum { PLAIN, GATED, LINK };

__device__ __forceinline__ floatx4 silu_times(floatx4 g, floatx4 u) {
#pragma unroll
  for (int r = 0; r < 4; ++r) u[r] *= g[r] / (1.0f + expf(-g[r]));
  return u;
}

template <int LANES> __device__ __forceinline__ bf16x8 rotated(bf16x8 v) {  // within 16 lanes: lane i takes lane (i + LANES) % 16
  if constexpr (LANES == 0) return v;
  uintx4 u = __builtin_bit_cast(uintx4, v);
#pragma unroll
  for (int i = 0; i < 4; ++i) u[i] = __builtin_amdgcn_update_dpp(0, (int)u[i], 0x120 + 16 - LANES, 0xf, 0xf, false);
  return __builtin_bit_cast(bf16x8, u);
}

// Operands straight from memory: a workgroup makes a tile of 16 MT rows of `a` by 16 NT rows of `w`; its waves share the tile
// and take the slices of K (16 waves one each, 8 two, 4 four neighbouring ones), so that no wave needs what another has loaded: 32
// bytes a lane and step, DEPTH steps ahead.  The waves' sums meet in LDS.  `w` is the left operand: a lane's 4 results are
// 4 consecutive outputs of one row of `a`.
// SHARE: with at most 16 / SHARE rows the 16 lanes of a row group hold SHARE steps' rows side by side, which are taken apart
// once for all of them and turned into place by a rotation of the lanes: the vector unit, which takes the floats apart (44
// instructions for 8 columns of 16 rows), is what a product of few rows is made of beside reading w.
// GATED: NT = 2, gate rows and the up rows of the same outputs (w has 2 N rows), or NT = MT = 1, eight rows of each in one strip; LINK: MT = NT = 1; ssq_in: MT = 1.
// VEC: rows start on 16 bytes (K % 4 == 0 and both matrices do).
template <int MT, int NT, int WAVES, int DEPTH, int SHARE, bool VEC, int MODE>
__global__ __launch_bounds__(WAVES * 64, MT * NT >= 8 ? 2 : 1) void gemm_f32_rows_kernel(const float* __restrict__ a,
                                                                                       const float* __restrict__ w, float* __restrict__ out,
                                                                                       int M, int N, int K, int tiles_m, int tiles,
                                                                                       int per_xcd, LinkF32 link) {
  static_assert(DEPTH % SHARE == 0 && (SHARE == 1 || MT == 1), "whole groups of steps, one row tile");
  static_assert(MODE != GATED || NT == 2 || (NT == 1 && MT == 1), "a gate strip and its up strip, or eight rows of both in one");
  constexpr bool HALVES = MODE == GATED && NT == 1;
  static_assert(MODE != LINK || (NT == 1 && MT == 1), "one strip of the stream");
  constexpr int T = MT * NT, SLICES = F32_SLICES / WAVES;  // slices of a wave
  constexpr int ENTRIES = SLICES == 4 ? 4 : F32_SLICES;    // sums that meet in LDS: of groups or of slices
  constexpr int ROWS = 16 / SHARE;
  extern __shared__ floatx4 red[];  // [ENTRIES][T][64]
  __shared__ float inv_rms[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  // Workgroups are dealt to the 8 XCDs in turn; each XCD takes a run of tiles with the tiles of the same rows of `w`
  // side by side, so that its L2 reads its share of the weights once.
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles) return;
  constexpr int ACROSS = HALVES ? 8 : MODE == GATED ? 16 : 16 * NT;
  const int n0 = tile / tiles_m * ACROSS, m0 = tile % tiles_m * (16 * MT);
  const int steps = (K + 31) / 32, per = (steps + F32_SLICES - 1) / F32_SLICES;
  const int st0 = min(steps, wave * SLICES * per), st1 = min(steps, st0 + SLICES * per);

  auto weight = [&](int i) {  // this lane's row of strip i
    if constexpr (HALVES) return w + ((size_t)min(n0 + (lr & 7), N - 1) + (size_t)(lr >> 3) * N) * K;
    return w + (MODE == GATED ? (size_t)min(n0 + lr, N - 1) + (size_t)i * N : (size_t)min(n0 + i * 16 + lr, N - 1)) * K;
  };
  const float* wrow[NT];
  const float* arow[MT];
#pragma unroll
  for (int i = 0; i < NT; ++i) wrow[i] = weight(i);
#pragma unroll
  for (int i = 0; i < MT; ++i) arow[i] = a + (size_t)min(m0 + i * 16 + lr % ROWS, M - 1) * K;

  floatx4 wv[DEPTH][NT][2], av[DEPTH / SHARE][MT][2], acc[NT][MT], low[NT][MT], sum[SLICES == 4 ? NT : 1][MT];
#pragma unroll
  for (int i = 0; i < NT; ++i)
#pragma unroll
    for (int j = 0; j < MT; ++j) { acc[i][j] = low[i][j] = floatx4{0.f, 0.f, 0.f, 0.f}; if (SLICES == 4) sum[i][j] = acc[i][j]; }
  auto load = [&](int u, int st) {  // a step's columns of w, and, for the first of SHARE steps, of a
    const int k = min(st, steps - 1) * 32 + lg * 8;
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int half = 0; half < 2; ++half) wv[u][i][half] = fetch<VEC>(wrow[i], k + 4 * half, K);
    if (u % SHARE == 0) {
      const int ka = SHARE == 1 ? k : min(st + lr / ROWS, steps - 1) * 32 + lg * 8;
#pragma unroll
      for (int j = 0; j < MT; ++j)
#pragma unroll
        for (int half = 0; half < 2; ++half) av[u / SHARE][j][half] = fetch<VEC>(arow[j], ka + 4 * half, K);
    }
  };
  auto slice_done = [&](int slice) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) {
        if constexpr (SLICES == 4) sum[i][j] += acc[i][j] + low[i][j];
        else red[(slice * T + i * MT + j) * 64 + lane] = acc[i][j] + low[i][j];
        acc[i][j] = low[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) load(u, st0 + u);
  if (link.ssq_in != nullptr && wave < M && wave < 16) {  // 1 / rms of the rows, a wave a row; published by the barrier below
    for (int row = wave; row < M && row < 16; row += WAVES) {
      float ss = 0.f;
      for (int j = lane; j < link.strips_in; j += 64) ss += link.ssq_in[(size_t)row * link.strips_in + j];
      ss = wave_sum(ss);
      if (lane == 0) inv_rms[row] = 1.0f / sqrtf(ss / (float)K + link.eps);
    }
  }
  int left = per, slice = wave * SLICES;  // steps until the slice ends
  Parts shared[MT];
  for (int st = st0; st < st1; st += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      if (st + u < st1) {
        Parts as[MT], ws[NT];
        if ((K & 31) && st + u + SHARE >= steps) {  // K may end among these steps' columns
          const int k = (st + u) * 32 + lg * 8, ka = SHARE == 1 ? k : min(st + u + lr / ROWS, steps - 1) * 32 + lg * 8;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
#pragma unroll
            for (int i = 0; i < NT; ++i) wv[u][i][half] = ragged<VEC>(wv[u][i][half], k + 4 * half, K);
            if (u % SHARE == 0) {
#pragma unroll
              for (int j = 0; j < MT; ++j) av[u / SHARE][j][half] = ragged<VEC>(av[u / SHARE][j][half], ka + 4 * half, K);
            }
          }
        }
        if (u % SHARE == 0) {
#pragma unroll
          for (int j = 0; j < MT; ++j) shared[j] = parts(av[u / SHARE][j][0], av[u / SHARE][j][1]);
        }
#pragma unroll
        for (int j = 0; j < MT; ++j) {
          switch (u % SHARE * ROWS) {  // known when compiled
            case 0: as[j] = shared[j]; break;
            case 4: as[j] = Parts{rotated<4>(shared[j].h), rotated<4>(shared[j].m), rotated<4>(shared[j].l)}; break;
            case 8: as[j] = Parts{rotated<8>(shared[j].h), rotated<8>(shared[j].m), rotated<8>(shared[j].l)}; break;
            default: as[j] = Parts{rotated<12>(shared[j].h), rotated<12>(shared[j].m), rotated<12>(shared[j].l)}; break;
          }
        }
#pragma unroll
        for (int i = 0; i < NT; ++i) ws[i] = parts(wv[u][i][0], wv[u][i][1]);
        load(u, st + u + DEPTH);
#pragma unroll
        for (int x = 0; x < 6; ++x)
#pragma unroll
          for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < MT; ++j) {
              floatx4& to = x == 5 ? acc[i][j] : low[i][j];
              to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part(ws[i], PART_W[x]), part(as[j], PART_A[x]), to, 0, 0, 0);
            }
        if (--left == 0) {
          left = per;
          slice_done(slice++);
        }
      }
    }
  }
  if constexpr (SLICES == 4) {
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
      for (int j = 0; j < MT; ++j) red[(wave * T + i * MT + j) * 64 + lane] = sum[i][j] + (acc[i][j] + low[i][j]);  // a slice that K's end cut short
  } else {
    for (; slice < (wave + 1) * SLICES; ++slice) slice_done(slice);  // one that K's end cut short, and empty ones
  }
  __syncthreads();
  auto total = [&](int t) {
    floatx4 v;
#pragma unroll
    for (int g = 0; g < F32_GROUPS; ++g) {
      floatx4 s;
      if constexpr (ENTRIES == F32_GROUPS) {
        s = red[(g * T + t) * 64 + lane];
      } else {
        s = red[(4 * g * T + t) * 64 + lane];
#pragma unroll
        for (int x = 1; x < 4; ++x) s += red[((4 * g + x) * T + t) * 64 + lane];
      }
      v = g == 0 ? s : v + s;
    }
    const int m = m0 + t % MT * 16 + lr;
    const bool mine = m < M && n0 + (MODE == GATED ? 0 : t / MT * 16) + (HALVES ? lg & 1 : lg) * 4 < N;
    if (__any(mine && !finite(v))) v = again_f32<VEC>(v, weight(t / MT), a + (size_t)min(m, M - 1) * K, K, 0, steps);
    return v;
  };
  for (int t = wave; t < (MODE == GATED ? MT : T); t += WAVES) {
    const int n = n0 + t / MT * 16 + lg * 4, m = m0 + t % MT * 16 + lr;
    floatx4 v = total(t);
    if (link.ssq_in != nullptr) v *= inv_rms[lr];  // MT = 1: rows 0 .. 15 are the launch's
    if constexpr (HALVES) {  // lanes 32 .. 63 hold the up rows of lanes 0 .. 31
      floatx4 up;
#pragma unroll
      for (int r = 0; r < 4; ++r) up[r] = __shfl_xor(v[r], 32);
      v = silu_times(v, up);
      if (lg >= 2) continue;
    } else if constexpr (MODE == GATED) {
      floatx4 up = total(MT + t);
      if (link.ssq_in != nullptr) up *= inv_rms[lr];
      v = silu_times(v, up);
    }
    if constexpr (MODE == LINK) {
      if (m < M && n < N) {  // N % 4 == 0
        float* xp = out + (size_t)m * N + n;
        v += *reinterpret_cast<floatx4*>(xp);
        *reinterpret_cast<floatx4*>(xp) = v;
        floatx4 g;
#pragma unroll
        for (int r = 0; r < 4; ++r) g[r] = link.gain[n + r];
        *reinterpret_cast<floatx4*>(link.scaled + (size_t)m * N + n) = v * g;
        link.ssq_out[((size_t)m * N + n) / 4] = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
      }
    } else if (m < M && n < N) {
      store4(out + (size_t)m * N + n, v, min(4, N - n));
    }
  }
}

// Up to 8 rows where strips of 16 rows of w are too few to occupy the compute units: a workgroup makes 16 / SIDE outputs, and the
// 16 rows of a wave's matrix operands are 16 / SIDE rows of w (of a) in SIDE neighbouring slices of K side by side, so that a slice's
// sums stand on the diagonal of the product's SIDE x SIDE blocks (the other blocks mean nothing and are dropped).  Each slice
// is one pair of chains in the order of the others: the same bits.  16 / SIDE waves, DEPTH steps of both operands in flight:
// 4 rows, K = 3,072, N = 1,024 (12.6 MB) 13.0 -> 7.4 us, which 64 strips of 16 rows of w had bound, a quarter of the compute
// units with 64 KB each in flight.
template <int SIDE, int DEPTH, bool VEC, int MODE>
__global__ __launch_bounds__(16 / SIDE * 64) void gemm_f32_side_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                    float* __restrict__ out, int M, int N, int K, LinkF32 link) {
  static_assert(MODE != GATED && (SIDE == 2 || SIDE == 4), "");
  constexpr int R = 16 / SIDE, WAVES = F32_SLICES / SIDE;  // rows of either operand; waves
  __shared__ floatx4 red[F32_SLICES][R / 4][R];             // [slice][outputs / 4][row of a]
  __shared__ float inv_rms[16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int n0 = blockIdx.x * R;
  const int steps = (K + 31) / 32, per = (steps + F32_SLICES - 1) / F32_SLICES;
  const int first = (wave * SIDE + lr / R) * per;  // this lane's slice
  const bool cut = (wave * SIDE + SIDE) * per * 32 > K;  // K ends in the wave's slices
  const float* wrow = w + (size_t)min(n0 + lr % R, N - 1) * K;
  const float* arow = a + (size_t)min(lr % R, M - 1) * K;
  floatx4 wv[DEPTH][2], av[DEPTH][2], acc = {0.f, 0.f, 0.f, 0.f}, low = acc;
  auto load = [&](int u, int st) {  // columns from K on count as zeros; steps past the slice are loaded and not used
    const int k = (first + st) * 32 + lg * 8;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      wv[u][half] = fetch<VEC>(wrow, k + 4 * half, K);
      av[u][half] = fetch<VEC>(arow, k + 4 * half, K);
    }
  };
#pragma unroll
  for (int u = 0; u < DEPTH; ++u) load(u, min(u, per - 1));
  if (link.ssq_in != nullptr) {  // 1 / rms of the rows, a wave a row; published by the barrier below
    for (int row = wave; row < M; row += WAVES) {
      float ss = 0.f;
      for (int j = lane; j < link.strips_in; j += 64) ss += link.ssq_in[(size_t)row * link.strips_in + j];
      ss = wave_sum(ss);
      if (lane == 0) inv_rms[row] = 1.0f / sqrtf(ss / (float)K + link.eps);
    }
  }
  for (int st = 0; st < per; st += DEPTH) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      if (st + u < per) {
        if (cut) {
          const int k = (first + st + u) * 32 + lg * 8;
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            wv[u][half] = ragged<VEC>(wv[u][half], k + 4 * half, K);
            av[u][half] = ragged<VEC>(av[u][half], k + 4 * half, K);
          }
        }
        const Parts ws = parts(wv[u][0], wv[u][1]), as = parts(av[u][0], av[u][1]);
        if (st + u + DEPTH < per) load(u, st + u + DEPTH);
#pragma unroll
        for (int x = 0; x < 6; ++x) {
          floatx4& to = x == 5 ? acc : low;
          to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part(ws, PART_W[x]), part(as, PART_A[x]), to, 0, 0, 0);
        }
      }
    }
  }
  // a lane holds rows 4 lg .. 4 lg + 3 of w's side by side in column lr of a's: outputs 4 lg % R of slice 4 lg / R by row lr % R of slice lr / R
  if (4 * lg / R == lr / R) red[wave * SIDE + lr / R][lg % (R / 4)][lr % R] = acc + low;
  __syncthreads();
  if (wave) return;
  const int n = n0 + 4 * lg, m = lr;  // this lane's outputs n .. n+3 of row m
  const bool mine = m < M && 4 * lg < R && n < N;
  floatx4 v = {0.f, 0.f, 0.f, 0.f};
  if (m < R && 4 * lg < R) {
#pragma unroll
    for (int g = 0; g < F32_GROUPS; ++g) {
      floatx4 s = red[4 * g][lg][m];
#pragma unroll
      for (int x = 1; x < 4; ++x) s += red[4 * g + x][lg][m];
      v = g == 0 ? s : v + s;
    }
  }
  if (__any(mine && !finite(v))) {
    const floatx4 f = again_f32<VEC>(v, w + (size_t)min(n0 + lr, N - 1) * K, a + (size_t)min(m, M - 1) * K, K, 0, steps);
    if (mine) v = f;
  }
  if (!mine) return;
  if (link.ssq_in != nullptr) v *= inv_rms[m];
  float* to = out + (size_t)m * N + n;
  if constexpr (MODE == LINK) {  // N % 4 == 0
    v += *reinterpret_cast<floatx4*>(to);
    *reinterpret_cast<floatx4*>(to) = v;
    floatx4 g;
#pragma unroll
    for (int r = 0; r < 4; ++r) g[r] = link.gain[n + r];
    *reinterpret_cast<floatx4*>(link.scaled + (size_t)m * N + n) = v * g;
    link.ssq_out[((size_t)m * N + n) / 4] = v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
  } else {
    store4(to, v, min(4, N - n));
  }
}

// Operands through LDS, for many rows: 8 waves (WM x WN) make a tile of BM = 16 WM MTW rows of `a` by BN = 16 WN NTW rows of
// `w` in steps of 32 columns.  Every float is taken apart once a workgroup, on its way from registers (asked for a step or two ahead) into
// LDS, where the parts of the next step are written while those of this one are multiplied: one barrier a step.
// What bounds it: a step of 128 x 128 takes 1.0 us, its matrix instructions alone 0.77, taking apart 0.16, the writes into LDS 0.08, and the
// waves of a workgroup do these at the same time; so the vector unit's work is dealt out between the matrix instructions, and every wait for
// LDS stands behind some of them.  128 x 128 outputs in which every operand was read before the first product, K = 1,024 / 2,048 at
// up to 256 tiles: 54 / 93 us, now 43 / 75; 64 x 64, one tile a compute unit: 24 / 43, now 19 / 34.
// A place holds 16 bytes, 8 columns of a row; place (row, column block c) of a part is row * 4 + (c ^ f(row / 4 % 4)), f =
// 0, 2, 3, 1: the hardware reads 16-byte operands in the lane groups {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the
// same above 32, which so touch every bank once.
// GATED: half of a tile's rows of w are gate rows, half the up rows of the same outputs.
// SPLIT: blockIdx.y names a group of four slices, whose sums go to out[group][m][n] for whoever adds the groups up in order.
template <int WM, int WN, int MTW, int NTW, bool IS_GATED, bool SPLIT, bool VEC>
__global__ __launch_bounds__(512, 2) void gemm_f32_tile_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                             float* __restrict__ out, int M, int N, int K, int tiles_m, int tiles,
                                                             int per_xcd) {
  constexpr int THREADS = 512;
  constexpr int BM = 16 * WM * MTW, BN = 16 * WN * NTW, ROWS = BM + BN;
  constexpr int PIECES = (ROWS * 8 + THREADS - 1) / THREADS;  // of 4 columns a thread and step; where they do not divide, some are brought twice
  constexpr int AHEAD = MTW > 1 ? 1 : 2;  // steps whose floats wait in registers
  constexpr int PLANE = ROWS * 4;
  constexpr int SPREAD = MTW == 1 ? (22 * PIECES + 6 * NTW - 1) / (6 * NTW) : 4;  // vector instructions a matrix instruction
  static_assert(WM * WN == 8 && ROWS % 16 == 0 && (!IS_GATED || NTW == 2) && !(IS_GATED && SPLIT), "");
  extern __shared__ bf16x8 lds[];  // [2][3][PLANE]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  const int tile = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (tile >= tiles) return;
  const int n0 = tile / tiles_m * (IS_GATED ? BN / 2 : BN), m0 = tile % tiles_m * BM;
  const int wm = wave % WM, wn = wave / WM;
  const int all = (K + 31) / 32, per = (all + F32_SLICES - 1) / F32_SLICES;
  const int st0 = SPLIT ? min(all, (int)blockIdx.y * 4 * per) : 0, st1 = SPLIT ? min(all, st0 + 4 * per) : all;
  if (SPLIT) out += (size_t)blockIdx.y * M * N;
  // row r of the tile's rows of w
  auto weight = [&](int r) -> const float* {
    const int n = IS_GATED ? n0 + (r >> 5) * 16 + (r & 15) : n0 + r;
    return w + (size_t)(min(n, N - 1) + (IS_GATED && (r & 16) ? N : 0)) * K;
  };
  // A thread's pieces: row r of the tile's, columns 4 c .. 4 c + 3 (eight lanes side by side ask for a line).  8 rows are a wave's, of one
  // matrix: their first one's address is uniform.
  const float* from[PIECES];
  unsigned at[PIECES];  // floats from there
  int dst[PIECES];      // halves of a place
#pragma unroll
  for (int p = 0; p < PIECES; ++p) {
    const int r0 = (wave * 64 + p * THREADS) % (ROWS * 8) >> 3, r = r0 + (lane >> 3), c = lane & 7;
    const bool of_a = r0 < BM;
    const int n = n0 + (IS_GATED ? ((r0 - BM) >> 5) * 16 + (r0 & 8) : r0 - BM);
    from[p] = of_a ? a + (size_t)min(m0 + r0, M - 1) * K : w + (size_t)(min(n, N - 1) + (IS_GATED && ((r0 - BM) & 16) ? N : 0)) * K;
    at[p] = (unsigned)(of_a ? min(m0 + r, M - 1) - min(m0 + r0, M - 1) : min(n + (lane >> 3), N - 1) - min(n, N - 1)) * K + c * 4;
    dst[p] = (r * 4 + ((c >> 1) ^ (0x78 >> (r >> 1 & 6) & 3))) * 2 + (c & 1);
  }
  const int last = max(0, K / 32 - 1);
  floatx4 ahead[AHEAD][PIECES];
  auto load = [&](int u, int st) {  // whole steps; those past the last one repeat it and are not used
    const int k = min(st, last) * 32;
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      if constexpr (VEC) ahead[u][p] = *reinterpret_cast<const floatx4*>(from[p] + k + at[p]);
      else ahead[u][p] = *reinterpret_cast<const floatx4_anywhere*>(from[p] + k + at[p]);
    }
  };
  auto place = [&](int u, int buf, int p) {
    bf16x4* base = reinterpret_cast<bf16x4*>(lds + buf * 3 * PLANE) + dst[p];
    const Parts4 s = parts(ahead[u][p]);
    base[0] = s.h;
    base[2 * PLANE] = s.m;
    base[4 * PLANE] = s.l;
  };
  floatx4 acc[NTW][MTW], low[NTW][MTW], group[NTW][MTW], total[NTW][MTW];
#pragma unroll
  for (int i = 0; i < NTW; ++i)
#pragma unroll
    for (int j = 0; j < MTW; ++j) acc[i][j] = low[i][j] = group[i][j] = total[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int u = 0; u < AHEAD; ++u) load(u, st0 + u);
#pragma unroll
  for (int p = 0; p < PIECES; ++p) place(0, 0, p);
  load(0, st0 + AHEAD);
  int slice = 0;  // those that are done
  const int ra = (wm * MTW * 16 + lr) * 4 + (lg ^ (0x78 >> (lr >> 1 & 6) & 3));
  const int rw = (BM + wn * NTW * 16 + lr) * 4 + (lg ^ (0x78 >> (lr >> 1 & 6) & 3));
  bf16x8 av[3], wv[NTW][3];  // the operands of a step's first row tile
  auto read_a = [&](int j, int buf, bf16x8 (&to)[3]) {
#pragma unroll
    for (int x = 0; x < 3; ++x) to[x] = lds[(buf * 3 + x) * PLANE + ra + j * 64];
  };
  auto read_first = [&](int buf, bf16x8 (&ws)[NTW][3], bf16x8 (&as)[3]) {  // the largest parts first: their product needs no others
#pragma unroll
    for (int x = 0; x < 3; ++x) {
#pragma unroll
      for (int i = 0; i < NTW; ++i) ws[i][x] = lds[(buf * 3 + x) * PLANE + rw + i * 64];
      as[x] = lds[(buf * 3 + x) * PLANE + ra];
    }
  };
  auto add_slice = [&](int j) {
#pragma unroll
    for (int i = 0; i < NTW; ++i) group[i][j] += acc[i][j] + low[i][j];
  };
  auto products = [&](int j, const bf16x8 (&ws)[NTW][3], const bf16x8 (&as)[3], auto first) {  // first: of a slice
#pragma unroll
    for (int x = 0; x < 6; ++x)
#pragma unroll
      for (int i = 0; i < NTW; ++i) {
        floatx4& to = x == 0 ? acc[i][j] : low[i][j];  // the largest first, then the five in their order
        const floatx4 before = first.value && x <= 1 ? floatx4{0.f, 0.f, 0.f, 0.f} : to;
        to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ws[i][PART_W[(x + 5) % 6]], as[PART_A[(x + 5) % 6]], before, 0, 0, 0);
      }
  };
  auto spread = [&]() {  // the vector unit's work between a row tile's matrix instructions, whose issue it does not hold up
#pragma unroll
    for (int x = 0; x < 6 * NTW; ++x) {
      __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x2, SPREAD, 0);
    }
  };
  auto group_done = [&]() {
    if (SPLIT || (slice & 3)) return;
#pragma unroll
    for (int i = 0; i < NTW; ++i)
#pragma unroll
      for (int j = 0; j < MTW; ++j) {
        total[i][j] += group[i][j];
        group[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
      }
  };
  auto slice_done = [&]() {  // added up where it ends
#pragma unroll
    for (int j = 0; j < MTW; ++j) {
      add_slice(j);
#pragma unroll
      for (int i = 0; i < NTW; ++i) acc[i][j] = low[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    group_done();
  };
  constexpr std::true_type begins{};
  constexpr std::false_type goes_on{};
  const int whole = min(st1, K / 32);  // steps before one that K ends in
  int st = st0, buf = 0, left = per;   // buf: where step st lies in LDS; left: steps until the slice ends
  if constexpr (MTW == 1) {
    // One row tile a wave: two workgroups on a compute unit fill each other's waits.
    auto step = [&](int u) {  // u: where st + 1 waits in registers
      __syncthreads();
      read_first(buf, wv, av);
#pragma unroll
      for (int p = 0; p < PIECES; ++p) place(u, buf ^ 1, p);
      products(0, wv, av, goes_on);
      load(u, st + 1 + AHEAD);
      __builtin_amdgcn_sched_group_barrier(0x100, 3 * NTW + 3, 0);
      spread();
      if (--left == 0) {
        left = per;
        ++slice;
        slice_done();
      }
      ++st;
      buf ^= 1;
    };
    while (st + 2 <= whole) {
      buf = 0;
      step(AHEAD - 1);
      buf = 1;
      step(0);
    }
    buf = 0;
    if (st < whole) step(AHEAD - 1);
  } else {
    // One workgroup on a compute unit has to fill its own waits: the barrier of a step stands before its last row tile's products, when
    // every read of this step's operands and every write of the next one's is done, so the next step's first operands are on their way
    // under those products; a slice's sums are added up under the next slice's first products.
    auto step = [&](auto first) {
      bf16x8 as[MTW + 1][3], wn[NTW][3];
#pragma unroll
      for (int x = 0; x < 3; ++x) as[0][x] = av[x];
#pragma unroll
      for (int j = 0; j < MTW; ++j) {
        if (j + 1 < MTW) read_a(j + 1, buf, as[j + 1]);
        else {
          __syncthreads();
          read_first(buf ^ 1, wn, av);
        }
#pragma unroll
        for (int p = 0; p < PIECES; ++p)
          if (p * (MTW - 1) / PIECES == j) place(0, buf ^ 1, p);
        if ((PIECES - 1) * (MTW - 1) / PIECES == j) load(0, st + 2);
        if (first.value) add_slice(j);
        products(j, wv, as[j], first);
        if (j + 1 < MTW) __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
        else __builtin_amdgcn_sched_group_barrier(0x100, 3 * NTW + 3, 0);
        spread();
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < NTW; ++i)
#pragma unroll
        for (int x = 0; x < 3; ++x) wv[i][x] = wn[i][x];
      ++st;
      buf ^= 1;
    };
    __syncthreads();
    read_first(0, wv, av);
    if constexpr (SPLIT) {  // a quarter of the slices: added up where they end, which takes fewer registers
#pragma unroll 1
      while (st < whole) {
        step(goes_on);
        if (--left) continue;
        left = per;
        slice_done();
      }
    } else {
#pragma unroll 1
      while (st < whole) {
        step(begins);
        group_done();
        left = per;
#pragma unroll 1
        while (--left && st < whole) step(goes_on);
        if (left == 0) ++slice;
      }
    }
  }
  if (st < st1) {  // columns that are no whole step
    const int k = st * 32 + (lane & 7) * 4;
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PIECES; ++p) {
      ahead[0][p] = ragged<VEC>(fetch<VEC>(from[p] + at[p] - (lane & 7) * 4, k, K), k, K);
      place(0, buf, p);
    }
    __syncthreads();
    if (left == 0) slice_done();
    read_first(buf, wv, av);
#pragma unroll
    for (int j = 0; j < MTW; ++j) {
      if (j) read_a(j, buf, av);
      products(j, wv, av, goes_on);
    }
  }
#pragma unroll
  for (int j = 0; j < MTW; ++j) {
    const int m = m0 + (wm * MTW + j) * 16 + lr;
    floatx4 v[NTW];
#pragma unroll
    for (int i = 0; i < NTW; ++i) {
      v[i] = total[i][j] + (group[i][j] + (acc[i][j] + low[i][j]));
      const int r = (wn * NTW + i) * 16;
      const bool mine = m < M && (IS_GATED ? n0 + wn * 16 : n0 + r) + lg * 4 < N;
      if (__any(mine && !finite(v[i]))) v[i] = again_f32<VEC>(v[i], weight(r + lr), a + (size_t)min(m, M - 1) * K, K, st0, st1);
    }
    if constexpr (IS_GATED) {
      const int n = n0 + wn * 16 + lg * 4;
      if (m < M && n < N) store4(out + (size_t)m * N + n, silu_times(v[0], v[1]), min(4, N - n));
    } else {
#pragma unroll
      for (int i = 0; i < NTW; ++i) {
        const int n = n0 + (wn * NTW + i) * 16 + lg * 4;
        if (m < M && n < N) store4(out + (size_t)m * N + n, v[i], min(4, N - n));
      }
    }
  }
}

// K <= F32_NARROW (toy widths, ranks of two-step projections): there is little to stream and nothing to cut, and the sum
// stays one chain: a workgroup makes 64 x 64 outputs through LDS, a thread 4 x 4 of them, by fp32 multiply-adds.  333 rows of 192
// against 4,096 outputs: 16.4 us; the same chain on the matrix cores, a wave to 16 x 32 outputs straight from memory,
// gives the same bits in 50 us (2,048 rows of 64 against 2,048: 14.3 and 45.8).
#define BM 64
#define BN 64
#define BK 16
__global__ __launch_bounds__(256) void gemm_f32_narrow_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                       float* __restrict__ out, int M, int N, int K) {
  __shared__ float as[BK][BM + 4];
  __shared__ float ws[BK][BN + 4];
  const int tid = threadIdx.x;
  const int tx = tid & 15, ty = tid >> 4;  // 16 x 16 threads, 4 x 4 outputs each
  const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
  const int lr = tid >> 2, lk = (tid & 3) * 4;  // this thread loads 4 consecutive k of row lr
  float acc[4][4] = {};
  const bool vec = (K & 3) == 0;
  for (int kb = 0; kb < K; kb += BK) {
    float av[4] = {0.f, 0.f, 0.f, 0.f}, wv[4] = {0.f, 0.f, 0.f, 0.f};
    const int k = kb + lk;
    if (m0 + lr < M) {
      const float* p = a + (size_t)(m0 + lr) * K + k;
      if (vec && k + 3 < K) { const float4 r = *reinterpret_cast<const float4*>(p); av[0] = r.x; av[1] = r.y; av[2] = r.z; av[3] = r.w; }
      else { for (int i = 0; i < 4; ++i) if (k + i < K) av[i] = p[i]; }
    }
    if (n0 + lr < N) {
      const float* p = w + (size_t)(n0 + lr) * K + k;
      if (vec && k + 3 < K) { const float4 r = *reinterpret_cast<const float4*>(p); wv[0] = r.x; wv[1] = r.y; wv[2] = r.z; wv[3] = r.w; }
      else { for (int i = 0; i < 4; ++i) if (k + i < K) wv[i] = p[i]; }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) { as[lk + i][lr] = av[i]; ws[lk + i][lr] = wv[i]; }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < BK; ++kk) {
      float ar[4], wr[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) { ar[i] = as[kk][ty * 4 + i]; wr[i] = ws[kk][tx * 4 + i]; }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int jn = 0; jn < 4; ++jn) acc[i][jn] = fmaf(ar[i], wr[jn], acc[i][jn]);
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= M) continue;
#pragma unroll
    for (int jn = 0; jn < 4; ++jn) {
      const int n = n0 + tx * 4 + jn;
      if (n < N) out[(size_t)m * N + n] = acc[i][jn];
    }
  }
}

static long f32_tiles(int M, int N, int rows, int columns) {
  return (((long)M + rows - 1) / rows) * (((long)N + columns - 1) / columns);
}
static bool aligned16(const void* a, const void* b) { return ((((uintptr_t)a) | ((uintptr_t)b)) & 15) == 0; }

template <int MT, int NT, int WAVES, int DEPTH, int SHARE, int MODE>
static int launch_rows(const float* a, const float* w, float* out, int M, int N, int K, const LinkF32& link, hipStream_t stream) {
  constexpr size_t lds = (size_t)(WAVES == 4 ? F32_GROUPS : F32_SLICES) * MT * NT * 64 * sizeof(floatx4);
  static_assert(lds + 64 <= 65536, "what a launch may ask for without an attribute");
  const long tiles = f32_tiles(M, N, 16 * MT, MODE == GATED ? 8 * NT : 16 * NT);
  if (tiles > 0x3fffffff) return AS_BAD_SHAPE;
  const int per_xcd = (int)((tiles + 7) / 8), tiles_m = (M + 16 * MT - 1) / (16 * MT);
  if ((K & 3) == 0 && aligned16(a, w))
    gemm_f32_rows_kernel<MT, NT, WAVES, DEPTH, SHARE, true, MODE><<<per_xcd * 8, WAVES * 64, lds, stream>>>(a, w, out, M, N, K, tiles_m,
                                                                                                         (int)tiles, per_xcd, link);
  else
    gemm_f32_rows_kernel<MT, NT, WAVES, DEPTH, SHARE, false, MODE><<<per_xcd * 8, WAVES * 64, lds, stream>>>(a, w, out, M, N, K, tiles_m,
                                                                                                         (int)tiles, per_xcd, link);
  return launch_status();
}

// One row tile: as many steps side by side as its rows leave lanes for.
template <int NT, int WAVES, int DEPTH, int MODE>
static int launch_few(const float* a, const float* w, float* out, int M, int N, int K, const LinkF32& link, hipStream_t stream) {
  if (M <= 4) return launch_rows<1, NT, WAVES, 4, 4, MODE>(a, w, out, M, N, K, link, stream);
  if (M <= 8) return launch_rows<1, NT, WAVES, DEPTH, 2, MODE>(a, w, out, M, N, K, link, stream);
  return launch_rows<1, NT, WAVES, DEPTH, 1, MODE>(a, w, out, M, N, K, link, stream);
}

// Strips of 16 rows of w, one to a workgroup.  A long K goes to sixteen waves while a wave's steps are mostly its loads (N, K at 1, 4, 8
// and 16 rows, eight waves and sixteen, us: 3,072, 8,192 33 27, 33 30, 35 34, 39 43; 4,096, 12,288 50 46, 48 47, 52 52, 57 64; 4,096, 4,096 18 19).
template <int MODE> static int launch_strips(const float* a, const float* w, float* out, int M, int N, int K, const LinkF32& link, hipStream_t stream) {
  if (M <= 8 && K >= 8192 && f32_tiles(M, N, 16, 16) <= compute_units()) return launch_few<1, 16, 4, MODE>(a, w, out, M, N, K, link, stream);
  return launch_few<1, 8, 4, MODE>(a, w, out, M, N, K, link, stream);
}

// Two strips a workgroup: on eight waves while that is one round (8,192, 4,096 at 1 / 16 rows 30 / 31 us, on four 39 / 36; 6,144, 1,024 9.7 / 11.5
// and 10.7 / 11.6), two steps of up to eight rows side by side (gate and up, 3,072 outputs of 1,024 at 4 / 8 rows 9.8 / 10.3 -> 9.35 / 10.0), else on
// four, of which more fit a compute unit (12,288, 2,048 25 / 29, on eight 28 / 33).  Gate and up of few outputs, or of so many that
// several workgroups share a compute unit and up to 4 rows, as one strip of eight rows of either: twice the workgroups (2,048 outputs of 1,024
// at 4 / 16 rows 9.5 / 10.9 -> 7.4 / 8.6, 6,144 of 2,048 at 4 rows 24.5 -> 22.8, at 16 28.2 and 31.0; 9,728 of 2,560 at 4 rows 46 -> 42.8, 12,288 of
// 1,024 24.6 and 26.9: five strips to a compute unit at most).
template <int MODE> static int launch_pairs(const float* a, const float* w, float* out, int M, int N, int K, const LinkF32& link, hipStream_t stream) {
  if constexpr (MODE == GATED) {
    if (f32_tiles(M, N, 16, 8) <= compute_units()) {
      if (M <= 8) return launch_rows<1, 1, 8, 2, 2, MODE>(a, w, out, M, N, K, link, stream);
      return launch_rows<1, 1, 8, 2, 1, MODE>(a, w, out, M, N, K, link, stream);
    }
  }
  if (f32_tiles(M, N, 16, MODE == GATED ? 16 : 32) <= compute_units()) {
    if (M <= 8) return launch_rows<1, 2, 8, 2, 2, MODE>(a, w, out, M, N, K, link, stream);
    return launch_rows<1, 2, 8, 2, 1, MODE>(a, w, out, M, N, K, link, stream);
  }
  if constexpr (MODE == GATED) {
    if (M <= 4 && f32_tiles(M, N, 16, 8) <= 5 * compute_units()) return launch_rows<1, 1, 4, 4, 4, MODE>(a, w, out, M, N, K, link, stream);
  }
  return launch_rows<1, 2, 4, 2, 1, MODE>(a, w, out, M, N, K, link, stream);
}

template <int MODE> static int launch_side(const float* a, const float* w, float* out, int M, int N, int K, const LinkF32& link, hipStream_t stream) {
  const bool vec = (K & 3) == 0 && aligned16(a, w);
#define SIDE_GO(SIDE)                                                                                                            \
  do {                                                                                                                           \
    const int blocks = (N + 16 / SIDE - 1) / (16 / SIDE);                                                                        \
    if (vec) gemm_f32_side_kernel<SIDE, 6, true, MODE><<<blocks, 16 / SIDE * 64, 0, stream>>>(a, w, out, M, N, K, link);         \
    else gemm_f32_side_kernel<SIDE, 6, false, MODE><<<blocks, 16 / SIDE * 64, 0, stream>>>(a, w, out, M, N, K, link);            \
  } while (0)
  if (M <= 4) SIDE_GO(4);
  else SIDE_GO(2);
#undef SIDE_GO
  return launch_status();
}

// Whether a product of few rows goes side by side: while strips of 16 outputs are at most half of the compute units, and, with two
// slices side by side, K is long enough for the second operand's loads to pay.  us, the best of the others and side by side:
// N, K            1 row        4 rows       8 rows           N, K            1 row        4 rows       8 rows
// 1,024, 1,024    6.4  5.3     7.1  6.3     8.0  8.9         2,048, 2,048    9.6  7.9    10.2  9.6    11.3  9.8
// 1,024, 2,048    9.3  6.0    10.0  6.9    11.1  9.5         2,048, 6,144   23.1 18.8    23.7 20.8    26.3 20.5
// 1,024, 3,072   12.0  6.6    13.0  7.4    14.4 10.0         3,072, 1,024    6.9  8.8     7.4 11.6     8.3 16.0
static bool side_by_side(int M, int N, int K) { return N <= 8 * compute_units() && (M <= 4 || (M <= 8 && K >= 2048)); }

template <int WM, int WN, int MTW, int NTW, bool IS_GATED, bool SPLIT, bool VEC>
static int launch_tile_of(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
  constexpr int TM = 16 * WM * MTW, TN = 16 * WN * NTW;
  constexpr int lds = 2 * 3 * (TM + TN) * 64;
  const long tiles = f32_tiles(M, N, TM, IS_GATED ? TN / 2 : TN);
  if (tiles > 0x3fffffff) return AS_BAD_SHAPE;
  const auto kernel = gemm_f32_tile_kernel<WM, WN, MTW, NTW, IS_GATED, SPLIT, VEC>;
  if (lds > 65536 && hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds) != hipSuccess)
    return AS_LAUNCH_FAILED;
  const int per_xcd = (int)((tiles + 7) / 8), tiles_m = (M + TM - 1) / TM;
  kernel<<<dim3(per_xcd * 8, SPLIT ? F32_GROUPS : 1), 512, lds, stream>>>(a, w, out, M, N, K, tiles_m, (int)tiles, per_xcd);
  return launch_status();
}

template <int WM, int WN, int MTW, int NTW, bool IS_GATED, bool SPLIT>
static int launch_tile(const float* a, const float* w, float* out, int M, int N, int K, hipStream_t stream) {
  if ((K & 3) == 0 && aligned16(a, w)) return launch_tile_of<WM, WN, MTW, NTW, IS_GATED, SPLIT, true>(a, w, out, M, N, K, stream);
  return launch_tile_of<WM, WN, MTW, NTW, IS_GATED, SPLIT, false>(a, w, out, M, N, K, stream);
}

// Which kernel: the tile of rows of a by rows of w, and what a workgroup on every compute unit takes per 1,024 of K
// beside the 4.5 us of a launch: the first round, every round.  Measured for N = 1,024 to 12,288 and K = 1,024 to 6,144 at 1 to 512 rows:
// small tiles where the larger ones would leave compute units idle, large ones where operands would be read over and over
// (N = 4,096, K = 1,024: 4 rows 8.3 us with the first and 43 with tiles of 128; N = 12,288, K = 2,048 at 512 rows 624 and 165,
// with the fp32 instruction from memory 272), and 96 rows where those leave fewer compute units idle (6,144 gated, 1,024 at 333
// rows: tiles of 64 45.8, of 128 44.0, of 96 41.2; 12,288, 2,048 149.5, 162.8, 146.9).  The results are the same bit for bit.
struct F32Tile { int rows, columns; float alone_us, round_us; };
static const F32Tile f32_forms[] = {{16, 16, 3.4f, 4.5f},   {16, 16, 4.5f, 3.6f},   {16, 32, 6.2f, 5.6f},    {32, 16, 5.5f, 7.4f},
                                    {32, 32, 7.8f, 9.f},    {64, 32, 12.f, 13.f},   {64, 64, 15.5f, 14.f},   {128, 128, 38.f, 41.f},
                                    {96, 128, 35.f, 35.f}};
#define F32_FORMS 9
#define F32_SIDE 9            // between them
static int f32_form(int i) { return i < F32_SIDE - 1 ? i + 1 : i + 2; }  // of f32_forms[i]
#define F32_ONE_ROW_TILE 3  // so many of one row tile

// split ranges of K are whole slices: up to three of 768 columns' 24 steps walk eight steps, not six, and the fourth has none, whose workgroups end at once
// (700 rows, 768, 768: 64 x 64 12.6 us, 96 x 128 15.6, which counted six steps looked shorter).  A tile of 96 or more rows starts a range
// a microsecond later.  249 products in ranges: 0.2 per cent over the best form on average and 8 at worst (0.6 and 23).
static float f32_cost(const F32Tile& t, int M, int N, int K, int split) {
  const float crowd = t.rows == 16 && t.columns == 16 && M > 8 ? 1.2f : 1.f;  // nothing of a's parts is shared
  float columns = (float)K, start = 4.5f;
  long ranges = 1;
  if (split > 1) {
    const int steps = (K + 31) / 32, walked = (steps + F32_SLICES - 1) / F32_SLICES * (F32_SLICES / split);
    columns = 32.f * (float)walked;
    ranges = (steps + walked - 1) / walked;
    if (t.rows > 64) start += 1.f;
  }
  const long rounds = (f32_tiles(M, N, t.rows, t.columns) * ranges + compute_units() - 1) / compute_units();
  return start + columns / 1024.f * crowd * (t.alone_us + t.round_us * (float)(rounds - 1));
}

// form: 0: chosen here; else the kernel `f32_form` numbers, or the one of slices side by side (tests).
template <int MODE> static int gemm_f32(const float* a, const float* w, float* out, int M, int N, int K, int form, const LinkF32& link,
                                        hipStream_t stream) {
  if constexpr (MODE == PLAIN) {
    if (form == F32_SIDE ? M <= 8 : form == 0 && side_by_side(M, N, K)) return launch_side<PLAIN>(a, w, out, M, N, K, link, stream);
  }
  if (form == 0) {
    float best = 0.f;
    for (int i = MODE == GATED ? 2 : 0; i < (link.ssq_in ? F32_ONE_ROW_TILE : F32_FORMS); ++i) {
      if (MODE == GATED && i == 3) continue;
      const float cost = f32_cost(f32_forms[i], M, MODE == GATED ? 2 * N : N, K, 1);
      if (form == 0 || cost < best) { best = cost; form = f32_form(i); }
    }
  }
  if constexpr (MODE == GATED) {
    switch (form) {
      case 3: return launch_pairs<GATED>(a, w, out, M, N, K, link, stream);
      case 5: return launch_rows<2, 2, 4, 2, 1, GATED>(a, w, out, M, N, K, link, stream);
      case 6: return launch_rows<4, 2, 4, 2, 1, GATED>(a, w, out, M, N, K, link, stream);
      case 7: return launch_tile<4, 2, 1, 2, true, false>(a, w, out, M, N, K, stream);
      case 8: return launch_tile<2, 4, 4, 2, true, false>(a, w, out, M, N, K, stream);
      case 10: return launch_tile<2, 4, 3, 2, true, false>(a, w, out, M, N, K, stream);
    }
  } else {
    switch (form) {
      case 1:
        if (M <= 16) return launch_strips<PLAIN>(a, w, out, M, N, K, link, stream);
        return launch_rows<1, 1, 8, 4, 1, PLAIN>(a, w, out, M, N, K, link, stream);
      case 2:
        if (M <= 16) return launch_few<1, 4, 4, PLAIN>(a, w, out, M, N, K, link, stream);
        return launch_rows<1, 1, 4, 4, 1, PLAIN>(a, w, out, M, N, K, link, stream);
      case 3: return launch_pairs<PLAIN>(a, w, out, M, N, K, link, stream);
      case 4: return launch_rows<2, 1, 8, 2, 1, PLAIN>(a, w, out, M, N, K, link, stream);
      case 5: return launch_rows<2, 2, 4, 2, 1, PLAIN>(a, w, out, M, N, K, link, stream);
      case 6: return launch_rows<4, 2, 4, 2, 1, PLAIN>(a, w, out, M, N, K, link, stream);
      case 7: return launch_tile<4, 2, 1, 2, false, false>(a, w, out, M, N, K, stream);
      case 8: return launch_tile<2, 4, 4, 2, false, false>(a, w, out, M, N, K, stream);
      case 10: return launch_tile<2, 4, 3, 2, false, false>(a, w, out, M, N, K, stream);
    }
  }
  return AS_BAD_SHAPE;
}

extern "C" int as_gemm_f32(const float* a, const float* w, float* out, int M, int N, int K, int form, hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (N <= 0 || K <= 0 || form < 0 || form > F32_FORMS + 1) return AS_BAD_SHAPE;
  if (K <= F32_NARROW) {
    const dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
    if (grid.y > 65535) return AS_BAD_SHAPE;
    gemm_f32_narrow_kernel<<<grid, 256, 0, stream>>>(a, w, out, M, N, K);
    return launch_status();
  }
  return gemm_f32<PLAIN>(a, w, out, M, N, K, form, LinkF32{}, stream);
}

// out[M, N] = silu(a @ w[:N]^T) * (a @ w[N:]^T) for w[2 N, K].  K > F32_NARROW; the activation on the sums that the plain product
// stores: the same bits as the two kernels.
extern "C" int as_gemm_f32_gated(const float* a, const float* w, float* out, int M, int N, int K, int form, hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (N <= 0 || N > 0x3fffffff || K <= F32_NARROW || form < 0 || form > F32_FORMS + 1) return AS_BAD_SHAPE;
  return gemm_f32<GATED>(a, w, out, M, N, K, form, LinkF32{}, stream);
}

// The producer of a LinkF32: x[M, N] += a @ w^T; scaled[M, N] = x * gain; ssq[M, N / 4] = sums of x^2 per 4 columns.
// M <= 16, K > F32_NARROW, N % 4 == 0, x and scaled on 16 bytes.
extern "C" int as_gemm_f32_link(const float* a, const float* w, float* x, const float* gain, float* scaled, float* ssq, int M, int N, int K,
                                hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (M > 16 || N <= 0 || (N & 3) || K <= F32_NARROW || !gain || !scaled || !ssq || !aligned16(x, scaled)) return AS_BAD_SHAPE;
  const LinkF32 link{nullptr, 0, 0.f, gain, scaled, ssq};
  if (side_by_side(M, N, K)) return launch_side<LINK>(a, w, x, M, N, K, link, stream);
  return launch_strips<LINK>(a, w, x, M, N, K, link, stream);
}

// The consumer of a LinkF32: out[M, N] = (scaled @ w^T) / rms(x) with rms from ssq[M, strips_in] (strips_in = K / 4) and eps;
// gated: silu of the first half of w's 2 N rows times the second half, both scaled first.  M <= 16, K > F32_NARROW.
extern "C" int as_gemm_f32_scaled(const float* scaled, const float* ssq, int strips_in, float eps, const float* w, float* out, int M, int N,
                                  int K, int gated, hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (M > 16 || N <= 0 || N > 0x3fffffff || K <= F32_NARROW || (K & 3) || !ssq || strips_in != K / 4) return AS_BAD_SHAPE;
  const LinkF32 link{ssq, strips_in, eps, nullptr, nullptr, nullptr};
  return gated ? gemm_f32<GATED>(scaled, w, out, M, N, K, 0, link, stream) : gemm_f32<PLAIN>(scaled, w, out, M, N, K, 0, link, stream);
}

// sums[4][M, N]: the product's sums over the four quarters of K's slices; added up in order they are the product, bit for bit where
// every sum is finite.  (Of an output with a sum that is not, the product made whole computes all of K again with the fp32 instruction and
// this one that quarter: an operand between bf16's largest number, 3.39e38, and fp32's makes them differ by rounding.)  For
// products of too few outputs to fill the GPU: N = 1,024, K = 2,048 at 333 rows 17.7 us, whole 28.5.  K > F32_NARROW, K % 4 == 0,
// N % 4 == 0.
extern "C" int as_gemm_f32_split(const float* a, const float* w, float* sums, int M, int N, int K, int form, hipStream_t stream) {
  if (M <= 0) return AS_OK;
  if (N <= 0 || (N & 3) || K <= F32_NARROW || (K & 3) || form < 0 || form > 3) return AS_BAD_SHAPE;
  if (form == 0) {
    float best = 0.f;
    for (int i = 6; i < F32_FORMS; ++i) {
      const float cost = f32_cost(f32_forms[i], M, N, K, F32_GROUPS);
      if (form == 0 || cost < best) { best = cost; form = i - 5; }
    }
  }
  if (form == 1) return launch_tile<4, 2, 1, 2, false, true>(a, w, sums, M, N, K, stream);
  if (form == 3) return launch_tile<2, 4, 3, 2, false, true>(a, w, sums, M, N, K, stream);
  return launch_tile<2, 4, 4, 2, false, true>(a, w, sums, M, N, K, stream);
}
