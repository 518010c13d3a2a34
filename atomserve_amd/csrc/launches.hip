// Calls of entry points that were written down, made again with other addresses: host code only.
//
// Between two launches of a list stood 2 to 3 us of Python beside the 4 us inside HIP, and a small model's prompt waits for both: one
// call of this function makes all launches of a stretch of layers: 3.1 us each, with the layer's addresses looked up 4.3 (a prompt of
// 37 tokens at Qwen3-0.6B sizes, 229 launches: the host 1,840 us before, 1,430 to 1,600 now, with the caches' views made once).
#include <stdint.h>
#include <string.h>

#include "common.h"

#if !defined(__x86_64__)
#error "arguments are passed as the x86-64 System V convention has them"
#endif

// In that convention integers and addresses take their places (six registers, then the stack) in the order in which they come,
// whatever floats stand between them, and floats the vector registers in theirs; the caller clears the stack.  So a function of up to MOST
// integers and FLOATS floats in any order can be called through this one type, with more arguments than it has: those it never reads.
constexpr int MOST = 32, FLOATS = 4;
#define WORD int64_t
typedef int (*Entry)(WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD,
                     WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, WORD, float, float, float, float);
#undef WORD

// program: `words` words, for every call in turn: the function, its numbers of integers, of floats and of patches; its integers;
// its floats (the low 32 bits of a word each); its patches, two words each: the place among the integers and that among `targets`,
// which holds `num_targets` values, of what stands there this time.  Returns 0, or the first failing call's status and in `failed` its
// number (the later ones are not made); AS_BAD_SHAPE and -1 for a program that does not add up, before any call.
extern "C" int as_launch_list(const int64_t* program, int64_t words, const int64_t* targets, int num_targets, int* failed) {
  *failed = -1;
  if (!program || words < 0) return AS_BAD_SHAPE;
  for (int64_t at = 0; at < words;) {
    if (words - at < 4) return AS_BAD_SHAPE;
    const int64_t ints = program[at + 1], floats = program[at + 2], patches = program[at + 3];
    if (!program[at] || ints < 0 || ints > MOST || floats < 0 || floats > FLOATS || patches < 0 || patches > MOST) return AS_BAD_SHAPE;
    const int64_t patch = at + 4 + ints + floats;
    if (words - patch < 2 * patches) return AS_BAD_SHAPE;
    for (int64_t p = patch; p < patch + 2 * patches; p += 2)
      if (program[p] < 0 || program[p] >= ints || program[p + 1] < 0 || program[p + 1] >= num_targets) return AS_BAD_SHAPE;
    at = patch + 2 * patches;
  }
  int call = 0;
  for (int64_t at = 0; at < words; ++call) {
    const int64_t ints = program[at + 1], floats = program[at + 2], patches = program[at + 3];
    int64_t a[MOST] = {};
    float f[FLOATS] = {};
    for (int64_t i = 0; i < ints; ++i) a[i] = program[at + 4 + i];
    for (int64_t i = 0; i < floats; ++i) {
      const uint32_t bits = (uint32_t)program[at + 4 + ints + i];
      memcpy(&f[i], &bits, sizeof(float));
    }
    const int64_t* patch = program + at + 4 + ints + floats;
    for (int64_t p = 0; p < patches; ++p) a[patch[2 * p]] = targets[patch[2 * p + 1]];
    const int status = ((Entry)(uintptr_t)program[at])(
        a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15], a[16], a[17], a[18], a[19], a[20],
        a[21], a[22], a[23], a[24], a[25], a[26], a[27], a[28], a[29], a[30], a[31], f[0], f[1], f[2], f[3]);
    if (status != AS_OK) {
      *failed = call;
      return status;
    }
    at += 4 + ints + floats + 2 * patches;
  }
  return AS_OK;
}
