// Shared device helpers for the gfx950 kernels: element types, conversions and
// wave/block reductions.  A wavefront is 64 lanes wide everywhere in this code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16;

#define WAVE 64

// Every entry point returns 0 on success and a negative code when it refuses its
// arguments (the Python wrapper turns the code into an exception).
#define AS_OK 0
#define AS_BAD_DTYPE -1
#define AS_BAD_SHAPE -2
#define AS_LAUNCH_FAILED -3

#define DT_F32 0
#define DT_BF16 1

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16 v) { return (float)v; }

template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f32<bf16>(float v) { return (bf16)v; }  // round to nearest even

// What the cache pools may hold: a value that is not finite (a model that overflowed) is stored
// as zero.  Kernels multiply keys and values of masked places by a weight of zero, which is only
// harmless while every stored value is finite; pages are used again by other requests.
__device__ __forceinline__ float finite_or_zero(float v) {
  return (__float_as_uint(v) & 0x7f800000u) == 0x7f800000u ? 0.f : v;
}
__device__ __forceinline__ bf16 finite_or_zero(bf16 v) {
  return (__builtin_bit_cast(unsigned short, v) & 0x7f80u) == 0x7f80u ? (bf16)0.f : v;
}

// What another lane of the wave holds, without a trip through LDS (a shuffle takes some 100 cycles, these under ten; a sum over
// a wave is six of them in a row, and the short kernels of a decode step wait for nothing else).  All lanes of the wave take part.
template <int CONTROL> __device__ __forceinline__ float dpp(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CONTROL, 0xf, 0xf, true));
}
#define DPP_XOR_1 0xb1        // quad_perm [1, 0, 3, 2]
#define DPP_XOR_2 0x4e        // quad_perm [2, 3, 0, 1]
#define DPP_HALF_MIRROR 0x141  // lane 7 - i of eight: i ^ 4 where the lanes of a quad hold the same
#define DPP_MIRROR 0x140       // lane 15 - i of sixteen: i ^ 8 where those of eight hold the same
#define DPP_ROTATE(N) (0x120 + (N))  // within sixteen; by 8: i ^ 8; by 4: i ^ 4 where lanes eight apart hold the same
struct TwoHalves { float a, b; };
__device__ __forceinline__ TwoHalves halves_32(float v) {  // in every lane: its half of the wave and the other one, in one order
  auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ TwoHalves halves_16(float v) {  // the same for the two sixteens of either half
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return {__uint_as_float(r[0]), __uint_as_float(r[1])};
}
__device__ __forceinline__ float plus_32(float v) { const TwoHalves h = halves_32(v); return h.a + h.b; }
__device__ __forceinline__ float plus_16(float v) { const TwoHalves h = halves_16(v); return h.a + h.b; }

// Lane pairs 32 apart first, then 16, 8, 4, 2, 1.
__device__ __forceinline__ float wave_sum(float v) {
  v = plus_16(plus_32(v));
  v += dpp<DPP_ROTATE(8)>(v);
  v += dpp<DPP_ROTATE(4)>(v);
  v += dpp<DPP_XOR_2>(v);
  return v + dpp<DPP_XOR_1>(v);
}

__device__ __forceinline__ float wave_max(float v) {
  TwoHalves h = halves_32(v);
  h = halves_16(fmaxf(h.a, h.b));
  v = fmaxf(h.a, h.b);
  v = fmaxf(v, dpp<DPP_ROTATE(8)>(v));
  v = fmaxf(v, dpp<DPP_ROTATE(4)>(v));
  v = fmaxf(v, dpp<DPP_XOR_2>(v));
  return fmaxf(v, dpp<DPP_XOR_1>(v));
}

// Sum over a block of up to 1024 threads; every thread gets the result.  `red` is a
// __shared__ float[17].  The order of additions is fixed, so the result is reproducible.  Every thread adds the waves' sums
// up itself: one thread doing it for all costs another barrier.
__device__ __forceinline__ float block_sum(float v, float* red) {
  const int lane = threadIdx.x & (WAVE - 1), wid = threadIdx.x / WAVE;
  const int nw = (blockDim.x + WAVE - 1) / WAVE;
  v = wave_sum(v);
  __syncthreads();  // protects `red` against a previous use
  if (lane == 0) red[wid] = v;
  __syncthreads();
  float s = 0.f;
  for (int i = 0; i < nw; ++i) s += red[i];
  return s;
}

static inline int launch_status() {
  return hipGetLastError() == hipSuccess ? AS_OK : AS_LAUNCH_FAILED;
}

// Compute units of the current device (asked once per device).
static inline int compute_units() {
  static int cached[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cached[dev] = n;
  }
  return cached[dev];
}
