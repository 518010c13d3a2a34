// A float as the sum of three bf16 values (its nearest one, the nearest one of what is left, and the rest, which fits: 8 + 8 + 8
// bits), for products of 32-bit numbers on the matrix cores' bf16 instruction: of the nine products of parts the six largest
// are computed, the three left out are below 2^-24 of the product and of either sign.  Sums are fp32, the largest product's in a
// chain of its own (small products that are added to a large sum are cut off downwards, an error of one sign).
#pragma once
#include "common.h"

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef unsigned uintx2 __attribute__((ext_vector_type(2)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

struct Parts { bf16x8 h, m, l; };   // eight floats as h + m + l
struct Parts4 { bf16x4 h, m, l; };  // four

__device__ __forceinline__ floatx8 widen(bf16x8 v) {
  const uintx4 u = __builtin_bit_cast(uintx4, v);
  floatx8 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    r[2 * i] = __uint_as_float(u[i] << 16);
    r[2 * i + 1] = __uint_as_float(u[i] & 0xffff0000u);
  }
  return r;
}

__device__ __forceinline__ Parts parts(floatx4 p, floatx4 q) {
  floatx8 x = __builtin_shufflevector(p, q, 0, 1, 2, 3, 4, 5, 6, 7);
  Parts s;
  s.h = __builtin_convertvector(x, bf16x8);  // to nearest
  x -= widen(s.h);
  s.m = __builtin_convertvector(x, bf16x8);
  x -= widen(s.m);
  s.l = __builtin_convertvector(x, bf16x8);
  return s;
}

__device__ __forceinline__ floatx4 widen(bf16x4 v) {
  const uintx2 u = __builtin_bit_cast(uintx2, v);
  return floatx4{__uint_as_float(u[0] << 16), __uint_as_float(u[0] & 0xffff0000u), __uint_as_float(u[1] << 16), __uint_as_float(u[1] & 0xffff0000u)};
}

__device__ __forceinline__ Parts4 parts(floatx4 x) {
  Parts4 s;
  s.h = __builtin_convertvector(x, bf16x4);  // to nearest
  x -= widen(s.h);
  s.m = __builtin_convertvector(x, bf16x4);
  x -= widen(s.m);
  s.l = __builtin_convertvector(x, bf16x4);
  return s;
}

// Which parts of w and of a the six products of a step take, the smallest first; the largest (x = 5) has a chain of its own
__device__ __forceinline__ bf16x8 part(const Parts& s, int i) { return i == 0 ? s.h : i == 1 ? s.m : s.l; }
constexpr int PART_W[6] = {2, 0, 1, 1, 0, 0}, PART_A[6] = {0, 2, 1, 0, 1, 0};

__device__ __forceinline__ bool finite(floatx4 v) {
  bool ok = true;
#pragma unroll
  for (int r = 0; r < 4; ++r) ok = ok && (__float_as_uint(v[r]) & 0x7f800000u) != 0x7f800000u;
  return ok;
}
