// Attention over the paged cache.
//
// Cache pages of one layer: k_pages [num_pages, KV, block_size, D] and v_pages
// [num_pages, KV, D, block_size] (values transposed within a page); a token at position p
// of a request lives in page table[p / block_size] at offset p % block_size.  A query at position p sees the keys at positions lo..p, with
// lo = max(0, p - window + 1) if window > 0, the start of p's chunk if the sequence is cut into chunks, else 0, and beside a
// window the first `keep` of the sequence (`Sight`).
// Query head h reads kv head h / (H / KV).  Scores, softmax and the weighted sum are fp32.
//
// attn_single_query: one work item per query token.  A workgroup (4 waves) takes one
// token, one kv head, up to GT query heads of its group, and one partition of
// `part_size` keys.  Inside a wave, LPK lanes share a key (each holds 16 bytes of
// the head) and 64 / LPK keys are in flight at once, each such lane group keeping an
// online-softmax stream (m, l, acc) of its own; streams are merged by shuffles, waves
// through LDS, partitions by attn_reduce.  Serves fp32 (every row) and bf16 (decode).
// Plain reference: reference atomserve/kernels.py:167-334, atomserve/model.py:269-289.
#include "common.h"
#include "no_alloc.h"
#include <type_traits>

#define NEG_INF (-__builtin_inff())

// exp of the fp32 path is the precise one; bf16 serving uses the hardware approximation.
template <typename T> __device__ __forceinline__ float fexp(float x);
template <> __device__ __forceinline__ float fexp<float>(float x) { return expf(x); }
template <> __device__ __forceinline__ float fexp<bf16>(float x) { return __expf(x); }

// What a query at position p sees, and how scores become weights.
struct Sight {
  int window;  // > 0: keys p - window + 1 .. p; 0: every key up to p
  int keep;    // with a window: the sequence's first `keep` keys stay visible behind it
  int chunk;   // > 0: keys of the query's own chunk only, chunks of this many positions counted from 0 (without a window)
  float cap;   // > 0: a score s counts as cap tanh(s / cap)
  int sink;    // 1: the denominator has one more score, which has no value
  const float* sinks;  // [H]: that score per query head (not scaled); null: 0 for all
  int wide;    // 1: the kernels of bfloat16 heads write their results in fp32 (for a consumer that takes differences of them)
};
// The result of a head's coordinate i, in the type of the heads or in fp32 (`Sight::wide`).
template <typename T>
__device__ __forceinline__ void put(T* out, size_t i, float v, int wide) {
  if (wide) reinterpret_cast<float*>(out)[i] = v;
  else out[i] = from_f32<T>(v);
}
__device__ __forceinline__ int first_in_window(const Sight& sight, int ctx) {
  if (sight.chunk > 0) return (ctx - 1) / sight.chunk * sight.chunk;
  return sight.window > 0 ? max(0, ctx - sight.window) : 0;
}
__device__ __forceinline__ float sink_score(int sink, const float* sinks, int head) { return sink && sinks ? sinks[head] : 0.f; }
static inline bool sight_ok(const Sight& s) {
  return s.window >= 0 && s.keep >= 0 && (s.keep == 0 || s.window > 0) && s.cap >= 0.f && (s.sink == 0 || s.sink == 1) &&
         (s.wide == 0 || s.wide == 1) && s.chunk >= 0 && (s.chunk == 0 || s.window == 0);
}
// Which instance of the matrix-core kernels computes it (`SEE` below).
static inline int needed_sight(const Sight& s) { return s.cap > 0.f ? 2 : (s.keep > 0 || s.sink || s.wide || s.chunk > 0) ? 1 : 0; }

// tanh through the hardware's exponential and reciprocal: an absolute error of 1e-7, which is what a capped score
// (times the cap) of the bf16 kernels may carry.
__device__ __forceinline__ float quick_tanh(float x) {
  return 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(2.8853900817779268f * x));
}

template <typename T> struct Chunk;  // 16 bytes of a head
template <> struct Chunk<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load(const float* p, float* v) {
    const float4 r = *reinterpret_cast<const float4*>(p);
    v[0] = r.x; v[1] = r.y; v[2] = r.z; v[3] = r.w;
  }
};
template <> struct Chunk<bf16> {
  static constexpr int N = 8;
  static __device__ __forceinline__ void load(const bf16* p, float* v) {
    const uint4 r = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};

template <typename T, int GT>
__global__ __launch_bounds__(256) void attn_single_query_kernel(
    const T* __restrict__ q, const T* __restrict__ k_pages, const T* __restrict__ v_pages,
    const int* __restrict__ items, const int* __restrict__ positions, const int* __restrict__ tok_row,
    const int* __restrict__ block_tables, int table_width, T* __restrict__ out,
    float* __restrict__ part_m, float* __restrict__ part_l, float* __restrict__ part_acc, int H, int KV,
    int D, int bs, float scale, Sight sight, int part_size, int P, int lpk) {
  constexpr int CH = Chunk<T>::N;
  extern __shared__ float smem[];  // [4][GT] m, [4][GT] l, [4][GT][D] acc
  const int G = H / KV;
  const int HC = (G + GT - 1) / GT;
  const int item = blockIdx.x, kvh = blockIdx.y / HC, hc = blockIdx.y % HC, part = blockIdx.z;
  const int t = items ? items[item] : item;  // null: every token, in order
  const int pos = positions[t];
  const int ctx = pos + 1;
  // the visible keys in order, the kept first ones and then the window's: partitions cut this list
  const int lo = first_in_window(sight, ctx), kept = min(sight.keep, lo);
  const int k0 = part * part_size, k1 = min(kept + ctx - lo, (part + 1) * part_size);
  const int h0 = kvh * G + hc * GT;       // first query head of this workgroup
  const int ng = min(GT, G - hc * GT);    // valid heads among the GT
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

  if (k0 >= k1) {  // an empty partition (P > 1 only): mark it so for the reduce
    if (tid < ng) {
      const size_t o = ((size_t)item * H + h0 + tid) * P + part;
      part_m[o] = NEG_INF;
      part_l[o] = 0.f;
    }
    for (int idx = tid; idx < ng * D; idx += 256)
      part_acc[(((size_t)item * H + h0 + idx / D) * P + part) * D + idx % D] = 0.f;
    return;
  }

  const int nsub = 64 / lpk;  // keys in flight per wave
  const int sub = lane / lpk, j = lane % lpk;
  const bool active = j * CH < D;
  const int* table = block_tables + (size_t)(tok_row ? tok_row[t] : t) * table_width;  // null: token t is row t

  float qr[GT][CH];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    if (active && g < ng) {
      Chunk<T>::load(q + ((size_t)t * H + h0 + g) * D + j * CH, qr[g]);
#pragma unroll
      for (int c = 0; c < CH; ++c) qr[g][c] *= scale;
    } else {
#pragma unroll
      for (int c = 0; c < CH; ++c) qr[g][c] = 0.f;
    }
  }

  float m[GT], l[GT], acc[GT][CH];
#pragma unroll
  for (int g = 0; g < GT; ++g) {
    m[g] = NEG_INF;
    l[g] = 0.f;
#pragma unroll
    for (int c = 0; c < CH; ++c) acc[g][c] = 0.f;
  }

  const int stride = 4 * nsub;
  const int iters = (k1 - k0 + stride - 1) / stride;  // uniform over the workgroup
  for (int it = 0; it < iters; ++it) {
    const int place = k0 + it * stride + wave * nsub + sub;
    const bool valid = place < k1;
    const int key = place < kept ? place : place - kept + lo;
    float kv[CH], vv[CH];
    if (valid && active) {
      const int page = table[key / bs];
      const size_t head = ((size_t)page * KV + kvh) * bs * D;
      Chunk<T>::load(k_pages + head + (size_t)(key % bs) * D + j * CH, kv);
      const T* vt = v_pages + head + (size_t)(j * CH) * bs + key % bs;
#pragma unroll
      for (int c = 0; c < CH; ++c) vv[c] = to_f32(vt[(size_t)c * bs]);
    } else {
#pragma unroll
      for (int c = 0; c < CH; ++c) { kv[c] = 0.f; vv[c] = 0.f; }
    }
    float s[GT];
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      float d = 0.f;
#pragma unroll
      for (int c = 0; c < CH; ++c) d += qr[g][c] * kv[c];
      for (int off = 1; off < lpk; off <<= 1) d += __shfl_xor(d, off, WAVE);
      s[g] = sight.cap > 0.f ? sight.cap * tanhf(d / sight.cap) : d;
    }
    if (valid) {
#pragma unroll
      for (int g = 0; g < GT; ++g) {
        const float mn = fmaxf(m[g], s[g]);
        const float a = fexp<T>(m[g] - mn);  // m = -inf gives 0
        const float p = fexp<T>(s[g] - mn);
        l[g] = l[g] * a + p;
#pragma unroll
        for (int c = 0; c < CH; ++c) acc[g][c] = acc[g][c] * a + p * vv[c];
        m[g] = mn;
      }
    }
  }

  // merge the streams of a wave
  for (int off = lpk; off < 64; off <<= 1) {
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      const float mo = __shfl_xor(m[g], off, WAVE), lo_ = __shfl_xor(l[g], off, WAVE);
      const float mn = fmaxf(m[g], mo);
      const float a = (m[g] == NEG_INF) ? 0.f : fexp<T>(m[g] - mn);
      const float b = (mo == NEG_INF) ? 0.f : fexp<T>(mo - mn);
      l[g] = l[g] * a + lo_ * b;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        const float ao = __shfl_xor(acc[g][c], off, WAVE);
        acc[g][c] = acc[g][c] * a + ao * b;
      }
      m[g] = mn;
    }
  }

  float* sm = smem;
  float* sl = smem + 4 * GT;
  float* sacc = smem + 8 * GT;
  if (lane < lpk) {
#pragma unroll
    for (int g = 0; g < GT; ++g) {
      if (j == 0) { sm[wave * GT + g] = m[g]; sl[wave * GT + g] = l[g]; }
      if (active) {
#pragma unroll
        for (int c = 0; c < CH; ++c) sacc[((size_t)wave * GT + g) * D + j * CH + c] = acc[g][c];
      }
    }
  }
  __syncthreads();

  for (int idx = tid; idx < ng * D; idx += 256) {
    const int g = idx / D, d = idx % D;
    float mx = NEG_INF;
#pragma unroll
    for (int w = 0; w < 4; ++w) mx = fmaxf(mx, sm[w * GT + g]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = sm[w * GT + g];
      const float e = (mw == NEG_INF) ? 0.f : fexp<T>(mw - mx);
      num += sacc[((size_t)w * GT + g) * D + d] * e;
      den += sl[w * GT + g] * e;
    }
    const int h = h0 + g;
    if (P == 1) {
      if (sight.sink) {
        const float sk = sink_score(1, sight.sinks, h), top = fmaxf(mx, sk), e = fexp<T>(mx - top);
        num *= e;
        den = den * e + fexp<T>(sk - top);
      }
      put(out, ((size_t)t * H + h) * D + d, num / den, sight.wide);
    } else {
      const size_t o = ((size_t)item * H + h) * P + part;
      part_acc[o * D + d] = num;
      if (d == 0) { part_m[o] = mx; part_l[o] = den; }
    }
  }
}

// Merge the partitions of each (item, head): out = sum_p acc_p e^(m_p - M) / sum_p l_p e^(m_p - M).
// One workgroup per (item, head), one thread per output coordinate; every thread derives the
// weights itself, a lane a partition, and hands them round by lane reads: one round of loads for the weights and one, which
// waits for no other, for the sums (a loop over the partitions waited for its loads in each: one request of 800 tokens in 25 partitions,
// 16 heads of 128, attention and merge 13.2 -> 9.1 us, in 7 partitions 10.1 -> 8.6).  Empty partitions carry m = -inf, l = 0 and acc = 0.
template <typename T>
__global__ __launch_bounds__(256) void attn_reduce_kernel(const int* __restrict__ items,
                                                          const float* __restrict__ part_m,
                                                          const float* __restrict__ part_l,
                                                          const float* __restrict__ part_acc, T* __restrict__ out,
                                                          int H, int D, int P, int sink, const float* __restrict__ sinks, int wide) {
  const int item = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & (WAVE - 1);
  const size_t base = ((size_t)item * H + h) * P;
  float mx = NEG_INF;
  for (int p = lane; p < P; p += WAVE) mx = fmaxf(mx, part_m[base + p]);
  mx = wave_max(mx);
  const float sk = sink_score(sink, sinks, h);
  if (sink) mx = fmaxf(mx, sk);
  const int t = items ? items[item] : item;  // null: every token, in order
  for (int d = threadIdx.x; d < (D + WAVE - 1) / WAVE * WAVE; d += blockDim.x) {  // whole waves: lanes hold the partitions' weights
    float num = 0.f, den = sink ? fexp<T>(sk - mx) : 0.f;
    const float* acc = part_acc + base * D + min(d, D - 1);
    for (int p0 = 0; p0 < P; p0 += WAVE) {
      const int here = min(WAVE, P - p0);
      const float mp = lane < here ? part_m[base + p0 + lane] : NEG_INF;
      const float weight = mp == NEG_INF ? 0.f : fexp<T>(mp - mx), l = weight == 0.f ? 0.f : part_l[base + p0 + lane] * weight;
      for (int p = 0; p < here; p += 8) {  // eight at a time; those past the end repeat the last with a weight of 0
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = acc[(size_t)(p0 + min(p + j, here - 1)) * D];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          den += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(l), p + j));
          num = fmaf(v[j], __int_as_float(__builtin_amdgcn_readlane(__float_as_int(weight), p + j)), num);
        }
      }
    }
    if (d < D) put(out, ((size_t)t * H + h) * D + d, num * (1.0f / den), wide);
  }
}

// ---- bf16 decode through the matrix cores ---------------------------------------------
//
// One workgroup (4 waves) per (query token, kv head, partition).  All G <= 16 query heads
// of the group ride in the 16 columns of one MFMA tile, so every key and value is read
// once for the whole group.  Per step a wave takes 32 keys (two tiles of 16):
//
//   S^T[key][head] = K[key][:] . Q[head][:]     A = keys, straight from the page (16 bytes
//                                               per lane), B = queries, kept in registers
//   online softmax per head on the accumulator layout (lane = head column)
//   O^T[d][head]  += V^T[d][key] P^T[key][head] A = the transposed value page, straight from
//                                               memory, B = P, which the lane already holds
//
// The softmax weights are rounded to bf16 for the second product; maxima, sums and the
// output accumulate in fp32.  Needs D % 32 == 0, D <= 256, block_size % 16 == 0.
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// Which of a step's 32 keys row `row` of its score tile `tile` (0, 1) stands for.  Rows 4g..4g+3
// of both tiles are what lane group g holds after the score product, and they are keys
// 8g .. 8g+7: eight neighbours, whose values are one 16-byte piece of a transposed page.
#define KEY_OF_ROW(tile, row) (8 * ((row) >> 2) + ((row) & 3) + 4 * (tile))

// Sums and maxima over the four lanes that share `lane % 16` (lane ^ 16, lane ^ 32) without a
// trip through LDS: v_permlane16_swap / v_permlane32_swap exchange rows of 16 lanes between
// two registers.  With both operands equal to x, the results hold (rows 0 0 2 2, rows 1 1 3 3)
// and (rows 0 1 0 1, rows 2 3 2 3) of x.
__device__ __forceinline__ float quad_rows_max(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float quad_rows_sum(float v) {
  auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// The keys and values of one step (32 keys, two 16-key pieces of pages) of one kv head, as the
// MFMA operands of this lane: keys as rows of A (16 bytes of the head of key KEY_OF_ROW(tile,
// lane % 16)), values as the transposed page gives them (the lane group's 8 keys of one
// coordinate: 16 bytes).  A second piece that starts at or beyond `end` repeats the first one: finite numbers, whose weights are zero.
// Loading the next step before computing the current one keeps memory busy while the matrix
// cores work.  PAGE: tokens of a page where the compiler knows them (divisions by another number are 30 instructions each), or 0;
// `kb` and `table` are uniform over the wave, so that pages are found by its scalar unit.
template <int DC>
struct KVStep {
  bf16x8_t k[2][DC];
  bf16x8_t v[2 * DC];
};

template <int DC, int PAGE>
__device__ __forceinline__ void load_kv_step(KVStep<DC>& st, const bf16* __restrict__ k_pages,
                                             const bf16* __restrict__ v_pages, const int* __restrict__ table,
                                             int kb, int end, int KV, int kvh, int page_size, int col, int grp) {
  constexpr int D = DC * 32, DT = DC * 2;
  const int bs = PAGE ? PAGE : page_size;
  size_t head[2];
  int off0[2];
#pragma unroll
  for (int pc = 0; pc < 2; ++pc) {  // uniform over the wave
    const int key0 = pc == 0 || kb + 16 < end ? kb + 16 * pc : kb;
    head[pc] = ((size_t)table[key0 / bs] * KV + kvh) * bs * D;
    off0[pc] = key0 % bs;
  }
  {  // keys: rows 0-7 of both tiles lie in the first piece, rows 8-15 in the second
    const int pc = col >> 3;
    const bf16* krow = k_pages + (pc ? head[1] + (size_t)off0[1] * D : head[0] + (size_t)off0[0] * D) + ((KEY_OF_ROW(0, col) & 15) * D + grp * 8);
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int c = 0; c < DC; ++c) st.k[tt][c] = *reinterpret_cast<const bf16x8_t*>(krow + tt * 4 * D + c * 32);
  }
  {  // values: keys 8 grp .. 8 grp + 7 of coordinates col, col + 16, ...  One instruction of the wave reads two runs of
     // 512 bytes, every 128-byte line whole, and a decode step reads a value once: marked as not to be kept (batch 64
     // of Qwen3-8B sizes 8,542 -> 8,872 tokens/s).  With pages of more than 32 tokens a step's 32 keys are part of a line,
     // which the next step needs again: no mark there.  The keys' loads share their lines in pairs and stay as they are.
    const bf16* vcol = v_pages + (grp >> 1 ? head[1] + off0[1] : head[0] + off0[0]) + (8 * (grp & 1) + col * bs);
    if (bs <= 32) {  // uniform over the grid: two loops, so that neither holds a choice per load
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
        st.v[dt] = __builtin_nontemporal_load(reinterpret_cast<const bf16x8_t*>(vcol + (size_t)dt * 16 * bs));
    } else {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) st.v[dt] = *reinterpret_cast<const bf16x8_t*>(vcol + (size_t)dt * 16 * bs);
    }
  }
}

// FRESH: the kernel takes the projection's output qkv [T, H + 2 KV, D] instead of finished queries
// and does what the norm-rotate-store kernel does before a decode step, for a step whose tokens
// are their own rows: each workgroup norms and rotates the queries of its group, and the workgroup whose
// partition holds the token's own position makes the token's key and value, writes them to the
// pages and attends them from LDS, so nothing waits for those writes.  A head is one wave's work (a lane
// has coordinates i and i + D/2), the waves take the group's heads, the key and the value in turn, and LDS hands the
// queries to all of them as matrix operands.  Same arithmetic as
// qk_norm_rope_store_bf16x8_kernel; the squares are summed in another order.
// What bounds a short context is the instructions of one wave, of which one that is alone on its SIMD issues one in 4 to
// 8 cycles: with every wave norming all queries as operands (16 columns, most of them empty groups' padding), pages found by divisions in
// the vector unit and partial outputs merged float by float, one token of Qwen3-0.6B sizes behind 100 took 7.6 us, now 5.4.
struct FreshQKV {
  const bf16* qkv;
  const void* qw;      // gains of the per-head norms, D values each, bf16 or fp32
  const void* kw;
  const float2* cs;    // [T, D/2] cos, sin of the whole head's rotation
  const int* slots;    // [T] page * block_size + offset of the new token, -1: keep it out of the pages
  bf16* k_store;       // the pages again, to write through
  bf16* v_store;
  float eps;
  int store;           // 0: queries only, the pages already hold the token's key and value
};

// What one workgroup does: partition `part` of item `item` for kv head `kvh`.
template <int DC, int FRESH, int SEE, int PAGE>
__device__ __forceinline__ void decode_item(
    const bf16* __restrict__ q, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ items, const int* __restrict__ positions, const int* __restrict__ tok_row,
    const int* __restrict__ block_tables, int table_width, bf16* __restrict__ out, float* __restrict__ part_m,
    float* __restrict__ part_l, float* __restrict__ part_acc, int H, int KV, int page_size, float scale, const Sight& sight,
    int part_size, int P, int share, const FreshQKV& fresh, float* smem, int item, int kvh, int part) {
  // smem: [4][16] m, [4][16] l, [4][G][LD] acc; FRESH: [G][D + 8] bf16 queries
  // share > 1: every `share` consecutive kv heads named here are one head of the pages (a group of more query heads
  // than a workgroup takes, cut into several); the pages then hold KV / share heads.
  constexpr int D = DC * 32, DT = DC * 2;  // DT: tiles of 16 output coordinates
  constexpr int LD = D + 4;                // a partial output's row in LDS
  __shared__ __align__(16) bf16 fresh_kv[2][256];  // FRESH: the new token's key and value
  const int G = H / KV, bs = PAGE ? PAGE : page_size;
  const int t = items ? items[item] : item;  // null: every token, in order
  const int pos = positions[t];
  const int ctx = pos + 1;
  // The keys are walked in steps of 32: first those that hold kept tokens (`kept_steps` from the sequence's start), then
  // those of the window (from step `base` on); where the two meet it is one run from the start.  Partitions cut this list.
  // Without kept tokens a place in the list is counted in keys, from the step that the window starts in (`k0` ..).
  const int lo = first_in_window(sight, ctx), kept = SEE >= 1 ? min(sight.keep, lo) : 0;
  int kept_steps = (kept + 31) / 32, base = lo / 32;
  if (kept_steps > 0 && kept_steps >= base) kept_steps = base = 0;
  const int steps = kept_steps + (ctx - 1) / 32 - base + 1;
  const int k0 = 32 * base + part * part_size, k1 = min(ctx, k0 + part_size);
  const int from = SEE >= 1 ? part * (part_size / 32) : k0;
  const int to = SEE >= 1 ? min(steps, from + part_size / 32) : k1;
  constexpr int NEXT = SEE >= 1 ? 1 : 32;  // from a step to the next one
  const int bound = SEE >= 1 ? ctx : k1;
  auto first_key = [&](int at) { return SEE >= 1 ? 32 * (at < kept_steps ? at : at - kept_steps + base) : at; };
  const int h0 = kvh * G;
  const int page_heads = KV / share, page_head = kvh / share;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;  // col: head within the group (and key row of A)

  if (from >= to) {  // an empty partition (P > 1 only): mark it so for the reduce
    if (tid < G) {
      const size_t o = ((size_t)item * H + h0 + tid) * P + part;
      part_m[o] = NEG_INF;
      part_l[o] = 0.f;
    }
    for (int idx = tid; idx < G * D; idx += 256)
      part_acc[(((size_t)item * H + h0 + idx / D) * P + part) * D + idx % D] = 0.f;
    return;
  }
  const int* table = block_tables + (size_t)(tok_row ? tok_row[t] : t) * table_width;  // null: token t is row t

  // Everything is asked for before anything is waited for: the queries (FRESH: this wave's heads as the projection
  // left them, with their gains and angles), then the first keys and values.
  constexpr int HALF = D / 2, PAIRS = (HALF + WAVE - 1) / WAVE, TURNS = FRESH ? 5 : 1;  // 16 heads, a key and a value over four waves
  using W = typename std::conditional<FRESH == 2, float, bf16>::type;  // the gains' type
  bf16x8_t qop[DC];
  const bf16x8_t zero = {0, 0, 0, 0, 0, 0, 0, 0};
  const size_t row = (size_t)t * (H + 2 * KV);  // FRESH: the token's heads in qkv
  [[maybe_unused]] const bool fresh_here = FRESH && fresh.store && pos >= k0 && pos < k1;  // these keys include the token's own
  [[maybe_unused]] const int jobs = G + (fresh_here ? 2 : 0);  // the group's heads, then the key and the value
  [[maybe_unused]] bf16 ha[TURNS][PAIRS], hb[TURNS][PAIRS];
  [[maybe_unused]] float ga[2][PAIRS], gb[2][PAIRS];  // gains of a query and of the key
  [[maybe_unused]] float2 angle[PAIRS];
  [[maybe_unused]] int slot = -1;
  if constexpr (FRESH != 0) {
#pragma unroll
    for (int n = 0; n < TURNS; ++n) {
      const int job = wave + 4 * n;
      if (job < jobs) {  // uniform over the wave
        const bf16* src = fresh.qkv + (row + (job < G ? h0 + job : H + kvh + (job - G) * KV)) * D;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          const int i = min(lane + p * WAVE, HALF - 1);
          ha[n][p] = src[i];
          hb[n][p] = src[i + HALF];
        }
      }
    }
#pragma unroll
    for (int p = 0; p < PAIRS; ++p) {
      const int i = min(lane + p * WAVE, HALF - 1);
      ga[0][p] = (float)((const W*)fresh.qw)[i];
      gb[0][p] = (float)((const W*)fresh.qw)[i + HALF];
      ga[1][p] = (float)((const W*)fresh.kw)[i];
      gb[1][p] = (float)((const W*)fresh.kw)[i + HALF];
      angle[p] = fresh.cs[(size_t)t * HALF + i];
    }
    if (fresh_here) slot = fresh.slots[t];
  } else {
    const bf16* qrow = q + ((size_t)t * H + h0 + min(col, G - 1)) * D + grp * 8;
#pragma unroll
    for (int c = 0; c < DC; ++c) qop[c] = col < G ? *reinterpret_cast<const bf16x8_t*>(qrow + c * 32) : zero;
  }
  KVStep<DC> cur, nxt;
  int at = from + NEXT * wave;
  if (at < to) load_kv_step<DC, PAGE>(cur, k_pages, v_pages, table, first_key(at), bound, page_heads, page_head, bs, col, grp);

  if constexpr (FRESH != 0) {
    bf16* const queries = reinterpret_cast<bf16*>(smem + 128 + 4 * LD * G);
    const size_t head = slot >= 0 ? ((size_t)(slot / bs) * KV + kvh) * bs * D : 0;
#pragma unroll
    for (int n = 0; n < TURNS; ++n) {
      const int job = wave + 4 * n;
      if (job > G && job < jobs) {  // the value, as it is; its page is stored transposed
        bf16* vt = fresh.v_store + head + slot % bs;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          const int i = lane + p * WAVE;
          if (i < HALF) {
            const bf16 ra = finite_or_zero(ha[n][p]), rb = finite_or_zero(hb[n][p]);
            fresh_kv[1][i] = ra;
            fresh_kv[1][i + HALF] = rb;
            if (slot >= 0) { vt[(size_t)i * bs] = ra; vt[(size_t)(i + HALF) * bs] = rb; }
          }
        }
      } else if (job < jobs) {  // a query or the key: norm and rotation, one wave over the pairs
        const int is_key = job == G;
        float ss = 0.f;
#pragma unroll
        for (int p = 0; p < PAIRS; ++p)
          if (lane + p * WAVE < HALF) ss += (float)ha[n][p] * (float)ha[n][p] + (float)hb[n][p] * (float)hb[n][p];
        ss = wave_sum(ss);
        const float inv = 1.0f / sqrtf(ss / (float)D + fresh.eps);
#pragma unroll
        for (int p = 0; p < PAIRS; ++p) {
          const int i = lane + p * WAVE;
          if (i < HALF) {
            const float a = (float)ha[n][p] * inv * (is_key ? ga[1][p] : ga[0][p]), b = (float)hb[n][p] * inv * (is_key ? gb[1][p] : gb[0][p]);
            bf16 ra = (bf16)(a * angle[p].x - b * angle[p].y), rb = (bf16)(b * angle[p].x + a * angle[p].y);
            if (is_key) {
              ra = finite_or_zero(ra);
              rb = finite_or_zero(rb);
              fresh_kv[0][i] = ra;
              fresh_kv[0][i + HALF] = rb;
              bf16* dst = fresh.k_store + head + (size_t)(slot % bs) * D;
              if (slot >= 0) { dst[i] = ra; dst[i + HALF] = rb; }
            } else {
              queries[job * (D + 8) + i] = ra;
              queries[job * (D + 8) + i + HALF] = rb;
            }
          }
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < DC; ++c)
      qop[c] = col < G ? *reinterpret_cast<const bf16x8_t*>(queries + min(col, G - 1) * (D + 8) + c * 32 + grp * 8) : zero;
  }
  f32x4_t o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt) o[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m = NEG_INF, l = 0.f;

  for (; at < to; at += 4 * NEXT) {
    const int kb = first_key(at);
    const bool more = at + 4 * NEXT < to;
    if (more) load_kv_step<DC, PAGE>(nxt, k_pages, v_pages, table, first_key(at + 4 * NEXT), bound, page_heads, page_head, bs, col, grp);
    if constexpr (FRESH != 0) {
      if (fresh_here && pos >= kb && pos < kb + 32) {  // this wave's step holds the token itself: take it from LDS
        const int nth = pos - kb;  // = KEY_OF_ROW(tile, row) for
        const int tile = (nth >> 2) & 1, row = 4 * (nth >> 3) + (nth & 3);
        if (col == row) {
#pragma unroll
          for (int tt = 0; tt < 2; ++tt)
            if (tt == tile) {
#pragma unroll
              for (int c = 0; c < DC; ++c) cur.k[tt][c] = *reinterpret_cast<const bf16x8_t*>(&fresh_kv[0][c * 32 + grp * 8]);
            }
        }
        // the token's half word in the eight keys of its lane group: a mask of bits to take per word, none in other lanes
        const unsigned half = grp == (nth >> 3) ? (nth & 1 ? 0xffff0000u : 0xffffu) : 0u;
        u32x4_t take;
#pragma unroll
        for (int w = 0; w < 4; ++w) take[w] = (nth & 7) >> 1 == w ? half : 0u;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const unsigned value = __builtin_bit_cast(unsigned short, fresh_kv[1][dt * 16 + col]) * 0x10001u;
          const u32x4_t was = __builtin_bit_cast(u32x4_t, cur.v[dt]);
          cur.v[dt] = __builtin_bit_cast(bf16x8_t, (was & ~take) | (value & take));
        }
      }
    }
    // ---- scores of 32 keys
    f32x4_t s[2];
#pragma unroll
    for (int tt = 0; tt < 2; ++tt) {
      s[tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < DC; ++c) s[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.k[tt][c], qop[c], s[tt], 0, 0, 0);
    }
    // ---- online softmax for this lane's head column
    float mx = NEG_INF;
#pragma unroll
    for (int tt = 0; tt < 2; ++tt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int key = kb + KEY_OF_ROW(tt, 4 * grp + r);
        const bool seen = key < bound && (key >= lo || key < kept);
        float sc = s[tt][r] * scale;
        if (SEE == 2) sc = sight.cap * quick_tanh(sc / sight.cap);
        s[tt][r] = seen ? sc : NEG_INF;
        mx = fmaxf(mx, s[tt][r]);
      }
    mx = quad_rows_max(mx);
    const float mn = fmaxf(m, mx);
    float alpha = 1.f, rs = 0.f;
    bf16x8_t pop;
    if (mn == NEG_INF) {  // nothing seen yet (a window may hide whole steps)
#pragma unroll
      for (int j = 0; j < 8; ++j) pop[j] = (bf16)0.f;
    } else {
      alpha = (m == NEG_INF) ? 0.f : __expf(m - mn);
#pragma unroll
      for (int tt = 0; tt < 2; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float pv = __expf(s[tt][r] - mn);  // exp(-inf) = 0 for hidden keys
          rs += pv;
          pop[tt * 4 + r] = (bf16)pv;
        }
      m = mn;
    }
    l = l * alpha + quad_rows_sum(rs);
    // ---- weighted values
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      o[dt] *= alpha;
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cur.v[dt], pop, o[dt], 0, 0, 0);
    }
    if (more) cur = nxt;
  }

  // ---- merge the four waves
  float* sm = smem;
  float* sl = smem + 64;
  float* so = smem + 128;  // [4][G][LD]
  if (grp == 0 && col < G) { sm[wave * 16 + col] = m; sl[wave * 16 + col] = l; }
  if (col < G) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4_t*>(so + (wave * G + col) * LD + dt * 16 + 4 * grp) = o[dt];
  }
  __syncthreads();
  for (int idx = tid; idx < G * D; idx += 256) {
    const int g = idx / D, d = idx % D;
    float mxw = NEG_INF;
#pragma unroll
    for (int w = 0; w < 4; ++w) mxw = fmaxf(mxw, sm[w * 16 + g]);
    float num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = sm[w * 16 + g];
      const float e = (mw == NEG_INF) ? 0.f : __expf(mw - mxw);
      num += so[(w * G + g) * LD + d] * e;
      den += sl[w * 16 + g] * e;
    }
    const int h = h0 + g;
    if (P == 1) {
      if (SEE >= 1 && sight.sink) {
        const float sk = sink_score(1, sight.sinks, h), top = fmaxf(mxw, sk), e = __expf(mxw - top);
        num *= e;
        den = den * e + __expf(sk - top);
      }
      put(out, ((size_t)t * H + h) * D + d, num / den, SEE >= 1 ? sight.wide : 0);
    } else {
      const size_t ob = ((size_t)item * H + h) * P + part;
      part_acc[ob * D + d] = num;
      if (d == 0) { part_m[ob] = mxw; part_l[ob] = den; }
    }
  }
}

// D / 32; FRESH 0: finished queries, 1: qkv with bf16 gains, 2: with fp32 gains; SEE 0: a window at most (nothing of the rest of
// `sight` is read), 1: kept first tokens, chunks, a sink and fp32 outputs too, 2: also capped scores; PAGE: tokens of a page, or 0 for any
template <int DC, int FRESH, int SEE, bool TURNED, int PAGE>
__global__ __launch_bounds__(256) void attn_decode_mfma_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ items, const int* __restrict__ positions, const int* __restrict__ tok_row,
    const int* __restrict__ block_tables, int table_width, bf16* __restrict__ out, float* __restrict__ part_m,
    float* __restrict__ part_l, float* __restrict__ part_acc, int H, int KV, int page_size, float scale, Sight sight,
    int part_size, int P, int cus, int share, FreshQKV fresh) {
  extern __shared__ __align__(16) float smem[];
  int item = blockIdx.x, kvh = blockIdx.y;
  const int part = blockIdx.z;
  if (!TURNED && P == 1) {
    // Whole contexts, one workgroup each, of unequal length: two workgroups share a compute unit, and
    // the first two rounds of `cus` workgroups are placed at once, the second on top of the first.
    // Work is taken eight items at a time, their kv heads one after the other (so neighbours in this
    // order read different pages at the same time), with the second round backwards: with `items`
    // sorted longest first a compute unit's first two are a long and a short one, and what follows
    // goes to whichever compute unit is free, longest first.
    int s = blockIdx.x + gridDim.x * blockIdx.y;
    const int total = gridDim.x * gridDim.y;
    if (s >= cus && s < 2 * cus) s = cus + (min(2 * cus, total) - 1 - s);
    const int N = gridDim.x, first = s / (8 * KV) * 8, r = s % (8 * KV), here = min(8, N - first);
    item = first + r % here;
    kvh = r / here;
  }
  if constexpr (TURNED) {
    // Partitions of many tokens come as a turned grid: workgroups are dealt to the XCDs in turn, and with the tokens changing
    // fastest an XCD had every eighth context, so that the one with the longest worked alone at the end.  With the kv heads
    // changing fastest each has its share of every context: 13 requests of 300 to 7,000 keys in a step of 16 rows 67 -> 46 us, 20
    // of 200 to 3,000 in one of 32 60 -> 41 (equal contexts: within 2 per cent).  Up to eight tokens an XCD has one, and its keys'
    // pages to itself: left so.  (An instance of its own: the same branch at run time costs whole contexts 3 to 5 per cent.)
    item = blockIdx.y;
    kvh = blockIdx.x;
  }
  decode_item<DC, FRESH, SEE, PAGE>(q, k_pages, v_pages, items, positions, tok_row, block_tables, table_width, out, part_m, part_l,
                                    part_acc, H, KV, page_size, scale, sight, part_size, P, share, fresh, smem, item, kvh, part);
}

// ---- bf16 prefill through the matrix cores ----------------------------------------------
//
// Work item: up to 64 consecutive query tokens of one request (`tiles` rows: first flat
// token, count, block-table row, position of the first) for one kv head.  A wave owns 32
// of those queries for one query head, as two MFMA column tiles of 16; the four waves of a
// workgroup take heads of the same group (or the other half of the queries), so they all
// need the same keys and values.  Those come into LDS once per workgroup by loads that write
// LDS directly (global_load_lds_dwordx4: no staging registers), into a ring of four stages
// of 32 keys.  A round of the main loop computes 64 keys (two stages) while the copies of the
// next 64 are in flight into the other two, and costs one barrier; 64 keys give a wave 64
// independent MFMAs between its softmax reductions, which is what hides their latency.
// Two waves copy a stage's keys, two its values (a 16-key piece of a page is contiguous in
// memory both for keys and, thanks to the transposed value pages, for values).
//
// LDS layout of a stage, in 16-byte slots:
//   keys:   slot (chunk * 32 + t) holds coordinates 8 chunk .. + 7 of the key behind row t % 16
//           of score tile t / 16, so the 64 lanes of an MFMA operand (row = lane % 16,
//           chunk = 4 step + lane / 16) read four runs of 16 consecutive slots: no bank
//           conflicts, no padding, any head width;
//   values: per 16-key piece, slot (h * D + d) holds keys 8h .. 8h+7 of coordinate d: the eight
//           keys whose weights a lane holds are one slot, and 16 lanes read 256 consecutive bytes.
// A load instruction fills 64 consecutive slots (slot = first + lane); which 16 bytes of
// memory a lane fetches is free, which is how the key layout comes about.
// A query at position p sees keys lo..p by absolute position, wherever the row starts.
// max(a, b, c) as the one instruction it is; NaN operands lose, as with fmaxf.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float r;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}

#define PF_STAGES 4
// s_waitcnt that only constrains the vector-memory counter (vmcnt: bits 3:0 and 15:14)
#define PF_WAIT_VM(N) __builtin_amdgcn_s_waitcnt(((N) & 15) | (((N) >> 4) << 14) | (7 << 4) | (15 << 8))

// A step of few work items takes as long as its longest one (a portion of a prompt behind thousands of cached
// tokens: a hundred workgroups of hundreds of rounds each, on a GPU with room for five hundred).  With `pieces` > 1
// every work item comes as that many workgroups: an item of more than `piece_rounds` rounds of 64 keys is cut
// along its keys into pieces of that many rounds (the last one, with the causal diagonal, may be shorter), each
// piece leaves the maxima, sums and unnormalised outputs of its queries, and `attn_prefill_merge_kernel` puts them
// together; a shorter item is its first workgroup's alone, as without the cut, and the others leave at once.
struct PrefillSplit {
  int pieces;        // workgroups per item; 1: no item is cut
  int piece_rounds;  // rounds of a piece
  int* cut;          // [items]: the pieces the item was cut into (1: not cut), for the merge
  float* ml;         // [T, H, pieces, 2]: maximum (base 2, scaled) and sum
  float* acc;        // [T, H, pieces, D]: unnormalised output
};
constexpr int PREFILL_MIN_PIECE_ROUNDS = 2;  // an item's last two rounds hold its own tokens: one piece

// A step that has both, portions of prompts and single queries, in one launch (PAGE != 0): the single queries' workgroups come first, a kv
// head of every context after the other, and share the compute units with the portions'.  The ones wait for memory most of
// the time and the others for the matrix cores and the softmax, and the tail of neither leaves compute units idle.
// One kernel's body, not a function that two kernels call: inlined, the compiler schedules portions alone otherwise (1,500 tokens of 16 heads
// on 4 kv heads 33.1 and 34.1 us).
struct Singles {
  const int* items;
  const int* positions;
  const int* tok_row;
  float* part_m;
  float* part_l;
  float* part_acc;
  int count, part_size, P;
};

// With kept first tokens behind a window the rounds of 64 keys are first those from the sequence's start that hold kept
// tokens, then those of the window (`first_key`); pieces cut this list.
// With single queries the kv head changes fastest and a pass is walked backwards by eights.  Workgroups are dealt to the eight XCDs in
// turn, each with an L2 of its own, so that with eight kv heads an XCD brings one head's keys and values from memory (with four, two share
// one).  Beside single queries that is what memory is short of (Qwen3-8B sizes, 8 of 500 to 8,192 keys beside 504 tokens 48.3 -> 44.6 us a
// layer, 2 of 7,000 beside 500 32.9 -> 28.7, 32 of 100 to 2,048 beside 480 behind 7,001 with 64 heads 210 -> 195); portions alone
// wait for the matrix cores, and several of one request lose (480 tokens behind 7,001 95 -> 97): not there.
template <int DC, int QT, int SEE, int PAGE>  // D / 32; column tiles of 16 queries that a wave owns: 2, or 1 (see the launcher); SEE: see above;
                                              // PAGE: 0, or the tokens of a page of the single queries before the portions
__global__ __launch_bounds__(256, 2) void attn_prefill_mfma_kernel(
    const bf16* __restrict__ q, const bf16* __restrict__ k_pages, const bf16* __restrict__ v_pages,
    const int* __restrict__ tiles, const int* __restrict__ block_tables, int table_width,
    bf16* __restrict__ out, int H, int KV, int bs, float scale, Sight sight, int units_z, int pass, PrefillSplit split, Singles single) {
  constexpr int D = DC * 32, DT = DC * 2;
  constexpr int PIECE = 64 * DC;  // 16-byte slots of a 16-key piece: 16 * D / 8
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  typedef const __attribute__((address_space(1))) void* global_ptr_t;
  __shared__ __attribute__((aligned(16))) u32x4_t lds[PF_STAGES][4][PIECE];  // [stage][K0 K1 V0 V1][slot]
  int item = blockIdx.x, blocks = gridDim.x;
  if constexpr (PAGE != 0) {  // a single query of up to 16 heads needs 256 D + 1,536 of the 512 D bytes
    const int singles = single.count * KV * single.P;
    if (item < singles) {
      decode_item<DC, 0, 0, PAGE>(q, k_pages, v_pages, single.items, single.positions, single.tok_row, block_tables, table_width, out,
                                  single.part_m, single.part_l, single.part_acc, H, KV, bs, scale, sight, single.part_size, single.P, 1,
                                  FreshQKV{}, reinterpret_cast<float*>(&lds[0][0][0]), item / KV % single.count, item % KV,
                                  item / (KV * single.count));
      return;
    }
    item -= singles;
    blocks -= singles;
  }

  const int G = H / KV;
  // Work items (tile, kv head, group of four waves) in the order of `tiles`, which the caller
  // sorts by the number of keys seen, most first; blocks of `pass` items alternate direction.
  // With one pass per round of workgroups that the GPU places (its compute units), a compute
  // unit that received one of the longest items in one round receives one of the shortest of
  // the next, so that causal prompts, whose items range from one step to hundreds, finish
  // together.
  const int per_tile = KV * units_z;
  const int block = item / pass, first = block * pass, size = min(pass, blocks - first);
  int piece = 0;  // which of an item's workgroups this is
  if constexpr (PAGE != 0) {
    const int off = item - first, eights = size & ~7, all = per_tile * split.pieces;
    if ((block & 1) && off < eights) item = first + eights - 8 - (off & ~7) + (off & 7);
    piece = item % all / per_tile;
    item = (item / all * KV + item % KV) * units_z + item / KV % units_z;
  } else {
    if (block & 1) item = first + size - 1 - (item - first);
    if (split.pieces > 1) {
      piece = item % split.pieces;
      item /= split.pieces;
    }
  }
  const int tile = item / per_tile, kvh = (item % per_tile) / units_z, bz = item % units_z;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int tok0 = tiles[4 * tile], count = tiles[4 * tile + 1], row = tiles[4 * tile + 2];
  const int pos0 = tiles[4 * tile + 3];
  const int* table = block_tables + (size_t)row * table_width;
  const int window = sight.window;
  auto first_seen = [&](int pos) {  // the oldest key that a query at `pos` sees, kept first ones apart
    return SEE >= 1 ? first_in_window(sight, pos + 1) : window > 0 ? max(0, pos - window + 1) : 0;
  };

  // the keys this workgroup walks: from the first key any of its waves sees to the last
  int wg_lo = 0x7fffffff, wg_last = -1;
  constexpr int WQ = 16 * QT, PARTS = 64 / WQ;  // queries of a wave; waves that share a head's 64 queries
  for (int u = bz * 4; u < bz * 4 + 4 && u < PARTS * G; ++u) {
    const int uq0 = (u / G) * WQ;
    if (uq0 >= count) continue;
    wg_last = max(wg_last, pos0 + min(count, uq0 + WQ) - 1);
    wg_lo = min(wg_lo, first_seen(pos0 + uq0));
  }
  if (wg_last < 0) {  // uniform over the workgroup
    if (split.pieces > 1 && piece == 0 && threadIdx.x == 0) split.cut[item] = 1;
    return;
  }
  const int keep = SEE >= 1 ? sight.keep : 0, kept = min(keep, wg_lo);  // kept tokens that lie before every query's window
  int kept_rounds = (kept + 63) / 64, kb0 = (wg_lo / 32) * 32;
  if (kept_rounds > 0 && 64 * kept_rounds >= kb0) kept_rounds = kb0 = 0;  // one run from the start
  int rd_first = 0, rd_end = kept_rounds + ((wg_last - kb0) / 32 + 2) / 2;
  auto first_key = [&](int rd) { return rd < kept_rounds ? 64 * rd : kb0 + 64 * (rd - kept_rounds); };
  bool partial = false;  // this workgroup leaves its share of a cut item for the merge
  if (split.pieces > 1) {
    const int all_rounds = rd_end;
    const int mine = min(split.pieces, (all_rounds + split.piece_rounds - 1) / split.piece_rounds);  // pieces of this item
    if (piece == 0 && threadIdx.x == 0) split.cut[item] = mine;
    if (piece >= mine) return;
    if (mine > 1) {
      partial = true;
      rd_first = split.piece_rounds * piece;
      if (piece + 1 < mine) rd_end = rd_first + split.piece_rounds;
    }
  }

  // this wave's queries
  const int unit = bz * 4 + wave;
  const int head = kvh * G + unit % G;
  const int q0 = (unit / G) * WQ;
  const bool working = unit < PARTS * G && q0 < count;
  const int nq = working ? min(WQ, count - q0) : 1;
  const int my_last = working ? pos0 + q0 + nq - 1 : -1;
  const int my_first_q = pos0 + q0;                  // position of this wave's first query
  const float scale2 = SEE == 2 ? 1.f : scale * 1.4426950408889634f;  // scores are kept in base 2
  const int my_lo = working ? first_seen(pos0 + q0) : 0x7fffffff;
  [[maybe_unused]] const int last_lo = first_seen(my_last);  // of this wave's last query

  bf16x8_t qop[QT][DC];
  int qpos[QT];
  [[maybe_unused]] int qlo[QT];
  bool qok[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int qi = qt * 16 + col;
    qok[qt] = working && qi < nq;
    const int qc = min(qi, nq - 1);  // columns past the end repeat the last query and are not stored
    qpos[qt] = pos0 + q0 + qc;
    if (SEE >= 1) qlo[qt] = first_seen(qpos[qt]);
    if (working) {
      const bf16* qrow = q + ((size_t)(tok0 + q0 + qc) * H + head) * D + grp * 8;
#pragma unroll
      for (int c = 0; c < DC; ++c) qop[qt][c] = *reinterpret_cast<const bf16x8_t*>(qrow + c * 32);
    } else {
#pragma unroll
      for (int c = 0; c < DC; ++c) qop[qt][c] = bf16x8_t{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }
  f32x4_t o[QT][DT];
  float m[QT], l[QT];
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    m[qt] = NEG_INF;
    l[qt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[qt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // ---- this wave's share of the copies: of every 32-key step, waves 0 and 1 bring the keys
  // (half of the 16-byte chunks of all 32 rows each), waves 2 and 3 the values of keys 0-15 and
  // 16-31.
  const int last_piece = (wg_last / 16) * 16;
  // Where the 16-key pieces lie in memory is worked out 64 pieces at a time, one piece per lane
  // (its page from the block table, asked for one batch of 64 ahead), and a step reads the two
  // it copies out of those lanes.  Done by the scalar unit for every step instead, the divisions
  // by the page size and the 64-bit products took a fifth of the kernel's time: that unit is
  // shared by all waves of the compute unit.  A piece that would start beyond the last key
  // repeats the last one (finite numbers; its scores are masked).
  unsigned long long k_at = 0, v_at = 0;  // byte offsets of this lane's piece in k_pages and v_pages
  auto key_of = [&](int piece) {
    return min(SEE >= 1 ? first_key(rd_first + (piece >> 2)) + 16 * (piece & 3) : first_key(rd_first) + 16 * piece, last_piece);
  };
  auto entry_of = [&](int piece) { return key_of(piece) / bs; };
  int page_ahead = table[entry_of(lane)];
  auto locate = [&](int batch) {  // pieces 64 batch .. 64 batch + 63
    const int piece = 64 * batch + lane, key = key_of(piece);
    const unsigned long long row = (unsigned long long)((unsigned)page_ahead * KV + kvh) * bs;
    k_at = (row + key % bs) * (D * 2);
    v_at = (row * D + key % bs) * 2;
    page_ahead = table[entry_of(piece + 64)];
  };
  auto at = [&](unsigned long long offsets, int piece) {
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)offsets, piece & 63);
    const unsigned hi = __builtin_amdgcn_readlane((unsigned)(offsets >> 32), piece & 63);
    return ((unsigned long long)hi << 32) | lo;
  };
  // what of a copy's address belongs to the lane, in bytes
  int lane_at[DC];
  if (wave >= 2) {
#pragma unroll
    for (int i = 0; i < DC; ++i) {  // values: slot = h * D + d holds keys 8h .. 8h+7 of coordinate d
      const int slot = i * 64 + lane, h = slot / D, d = slot % D;
      lane_at[i] = (d * bs + h * 8) * 2;
    }
  } else {
    // keys: slot = chunk * 32 + t holds coordinates 8 chunk .. + 7 of the key that row t of the
    // step's two score tiles stands for (see KEY_OF_ROW)
    const int t = lane & 31, key = KEY_OF_ROW(t >> 4, t & 15);
    lane_at[0] = ((key & 15) * D + (wave * (2 * DC) + (lane >> 5)) * 8) * 2;  // the further chunks: + 32 bytes each
  }
  const bool second_piece = KEY_OF_ROW((lane & 31) >> 4, lane & 15) >> 4;
  auto issue = [&](int step) {
    if ((step & 31) == 0) locate(step >> 5);
    if (wave >= 2) {
      const char* src = reinterpret_cast<const char*>(v_pages) + at(v_at, 2 * step + wave - 2);
      u32x4_t* dst = &lds[step % PF_STAGES][wave][0];
#pragma unroll
      for (int i = 0; i < DC; ++i)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(src + lane_at[i]), (lds_ptr_t)(dst + i * 64), 16, 0, 0);
    } else {
      const unsigned long long first = at(k_at, 2 * step), second = at(k_at, 2 * step + 1);
      const char* src = reinterpret_cast<const char*>(k_pages) + (second_piece ? second : first) + lane_at[0];
      u32x4_t* dst = &lds[step % PF_STAGES][0][0] + wave * (DC * 64);
#pragma unroll
      for (int i = 0; i < DC; ++i)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(src + i * 32), (lds_ptr_t)(dst + i * 64), 16, 0, 0);
    }
  };
  // The same copies one instruction at a time, for a round's two steps: `aim` works out where they read
  // and write, `copy(k)` issues the k-th of their 2 DC instructions (between the round's matrix products,
  // whose issue otherwise leaves the wave idle, instead of in one block that the wave waits through).
  const char* from[2];
  u32x4_t* to[2];
  auto aim = [&](int step0) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int step = step0 + j;
      if ((step & 31) == 0) locate(step >> 5);
      if (wave >= 2) {
        from[j] = reinterpret_cast<const char*>(v_pages) + at(v_at, 2 * step + wave - 2);
        to[j] = &lds[step % PF_STAGES][wave][0];
      } else {
        const unsigned long long first = at(k_at, 2 * step), second = at(k_at, 2 * step + 1);
        from[j] = reinterpret_cast<const char*>(k_pages) + (second_piece ? second : first) + lane_at[0];
        to[j] = &lds[step % PF_STAGES][0][0] + wave * (DC * 64);
      }
    }
  };
  auto copy = [&](int k) {
    const int j = k / DC, i = k % DC;
    if (wave >= 2) __builtin_amdgcn_global_load_lds((global_ptr_t)(from[j] + lane_at[i]), (lds_ptr_t)(to[j] + i * 64), 16, 0, 0);
    else __builtin_amdgcn_global_load_lds((global_ptr_t)(from[j] + i * 32), (lds_ptr_t)(to[j] + i * 64), 16, 0, 0);
  };
  const int nrounds = rd_end - rd_first;
  issue(0);
  issue(1);  // beyond the last key it repeats the last piece
  for (int rd = 0; rd < nrounds; ++rd) {
    PF_WAIT_VM(0);    // this wave's copies for the round have landed
    __syncthreads();  // ... and everyone's; and everyone is done with the round before
    const bool more = rd + 1 < nrounds;  // copies into the two stages the round before used
    const int kb = first_key(rd_first + rd);
    const bool active = working && kb <= my_last && (kb + 63 >= my_lo || kb < keep);
    if (more) {
      aim(2 * rd + 2);
      if (!active) {
#pragma unroll
        for (int k = 0; k < 2 * DC; ++k) copy(k);
      }
    }
    if (active) {
      // raw scores of 64 keys x 16 QT queries; a key operand is read from LDS once for all of a wave's query tiles
      f32x4_t sc[QT][4];
#pragma unroll
      for (int qt = 0; qt < QT; ++qt)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) sc[qt][tt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      // The operands of a whole tile are asked from LDS before its products start, and the next
      // tile's while they run: a product must not wait for a read issued just before it.
      u32x4_t kraw[2][DC];
      auto read_keys = [&](int tt, u32x4_t (&into)[DC]) {
        // score tile tt: rows KEY_OF_ROW(tt & 1, .) of step tt >> 1
        const u32x4_t* keys = &lds[(2 * rd + (tt >> 1)) % PF_STAGES][0][0] + (tt & 1) * 16 + col;
#pragma unroll
        for (int c = 0; c < DC; ++c) into[c] = keys[(c * 4 + grp) * 32];
      };
      read_keys(0, kraw[0]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        if (tt + 1 < 4) read_keys(tt + 1, kraw[(tt + 1) & 1]);
        __builtin_amdgcn_sched_barrier(0);  // or the compiler moves every read down to its product
#pragma unroll
        for (int c = 0; c < DC; ++c) {
          const bf16x8_t kop = __builtin_bit_cast(bf16x8_t, kraw[tt & 1][c]);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt)
            sc[qt][tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kop, qop[qt][c], sc[qt][tt], 0, 0, 0);
        }
        if (more) {  // a quarter of the round's copies behind each tile's products
#pragma unroll
          for (int k = tt * (2 * DC) / 4; k < (tt + 1) * (2 * DC) / 4; ++k) copy(k);
        }
      }
      // The values are asked for before the softmax, under which they arrive, as far as registers hold them
      // (512 tokens behind 15,872, 32 heads, 16 queries a wave in two pieces: 222 us with all values asked for behind it, 198 now; 32
      // queries a wave, 480 behind 7,001 in four pieces: 97, 92).
      u32x4_t vraw[2][DT];
      auto read_values = [&](int j, u32x4_t (&into)[DT]) {
        // this lane's eight weights of step j belong to keys 8 grp .. 8 grp + 7: one 16-byte slot
        const u32x4_t* values = &lds[(2 * rd + j) % PF_STAGES][2 + (grp >> 1)][(grp & 1) * D + col];
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) into[dt] = values[dt * 16];
      };
      constexpr int EARLY = DC <= 5 ? 3 - QT : 2 - QT;  // of a round's two halves
      if constexpr (EARLY >= 1) read_values(0, vraw[0]);
      if constexpr (EARLY >= 2) read_values(1, vraw[1]);
      __builtin_amdgcn_sched_barrier(0);
      // Only rounds that touch the causal diagonal, the window's edge or the end of the context
      // need a mask; the others see all 64 keys (uniform over the wave).
      const bool masked = kb + 63 > my_first_q || (SEE >= 1 ? kb < last_lo : window > 0 && kb < my_last - window + 1);
      bf16x8_t pop[QT][2];
      float alpha[QT];
      bool rescale = false;
      if (SEE == 2) {  // the capped scores, in base 2 already
        const float inner = scale / sight.cap, outer = sight.cap * 1.4426950408889634f;
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) sc[qt][tt][r] = outer * quick_tanh(sc[qt][tt][r] * inner);
      }
#pragma unroll
      for (int qt = 0; qt < QT; ++qt) {
        if (masked) {
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int key = kb + 32 * (tt >> 1) + KEY_OF_ROW(tt & 1, 4 * grp + r);
              const bool seen = key <= qpos[qt] && (SEE >= 1 ? key >= qlo[qt] || key < keep : window <= 0 || key > qpos[qt] - window);
              sc[qt][tt][r] = seen ? sc[qt][tt][r] : NEG_INF;
            }
        }
        // sixteen scores to one in eight three-way maxima (fmaxf would first quiet every operand)
        const float m0 = max3(sc[qt][0][0], sc[qt][0][1], sc[qt][0][2]), m1 = max3(sc[qt][0][3], sc[qt][1][0], sc[qt][1][1]);
        const float m2 = max3(sc[qt][1][2], sc[qt][1][3], sc[qt][2][0]), m3 = max3(sc[qt][2][1], sc[qt][2][2], sc[qt][2][3]);
        const float m4 = max3(sc[qt][3][0], sc[qt][3][1], sc[qt][3][2]);
        const float mx = quad_rows_max(max3(max3(m0, m1, m2), max3(m3, m4, sc[qt][3][3]), NEG_INF));
        // base-2 softmax: scale and log2(e) are folded into one factor (positive, so maxima agree)
        const float mn = fmaxf(m[qt], mx * scale2);
        // Without a branch, so that the two query tiles' arithmetic can be interleaved: while a row
        // has seen no key, every score and mn are -inf, and 2^(-inf - 0) = 0 is what each weight and
        // the factor of the (empty) past should be.
        const float base = mn == NEG_INF ? 0.f : mn;
        alpha[qt] = __builtin_amdgcn_exp2f(m[qt] - base);
        float part[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int tt = 0; tt < 4; ++tt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float pv = __builtin_amdgcn_exp2f(fmaf(sc[qt][tt][r], scale2, -base));
            part[r] += pv;
            pop[qt][tt >> 1][(tt & 1) * 4 + r] = (bf16)pv;
          }
        const float rs = (part[0] + part[1]) + (part[2] + part[3]);
        m[qt] = mn;
        l[qt] = l[qt] * alpha[qt] + rs;  // of this lane's keys; the four lanes of a query meet at the end
        rescale = rescale || alpha[qt] != 1.f;
      }
      // the accumulated output is rescaled only when some query's maximum moved (rare once the
      // first keys have been seen)
      if (__any(rescale)) {
#pragma unroll
        for (int qt = 0; qt < QT; ++qt)
#pragma unroll
          for (int dt = 0; dt < DT; ++dt) o[qt][dt] *= alpha[qt];
      }
      if constexpr (EARLY < 1) read_values(0, vraw[0]);
      if constexpr (EARLY < 2) read_values(1, vraw[1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) {
          const bf16x8_t vop = __builtin_bit_cast(bf16x8_t, vraw[j][dt]);
#pragma unroll
          for (int qt = 0; qt < QT; ++qt) o[qt][dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vop, pop[qt][j], o[qt][dt], 0, 0, 0);
        }
      }
    }
  }

#pragma unroll
  for (int qt = 0; qt < QT; ++qt) l[qt] = quad_rows_sum(l[qt]);
  if (partial) {
#pragma unroll
    for (int qt = 0; qt < QT; ++qt) {
      if (!qok[qt]) continue;
      const size_t at = ((size_t)(tok0 + q0 + qt * 16 + col) * H + head) * split.pieces + piece;
      if (grp == 0) *reinterpret_cast<float2*>(split.ml + at * 2) = make_float2(m[qt], l[qt]);
      float* arow = split.acc + at * D + 4 * grp;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4_t*>(arow + dt * 16) = o[qt][dt];
    }
    return;
  }
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    if (!qok[qt]) continue;
    float inv = 1.0f / l[qt];
    if (SEE >= 1 && sight.sink) {
      const float sk = sink_score(1, sight.sinks, head) * 1.4426950408889634f, top = fmaxf(m[qt], sk);
      const float e = __builtin_amdgcn_exp2f(m[qt] - top);
      inv = e / (l[qt] * e + __builtin_amdgcn_exp2f(sk - top));
    }
    const size_t at = ((size_t)(tok0 + q0 + qt * 16 + col) * H + head) * D + 4 * grp;
    if (SEE >= 1 && sight.wide) {
      float* orow = reinterpret_cast<float*>(out) + at;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4_t*>(orow + dt * 16) = o[qt][dt] * inv;
      continue;
    }
    bf16* orow = out + at;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const bf16x4_t r4 = {(bf16)(o[qt][dt][0] * inv), (bf16)(o[qt][dt][1] * inv), (bf16)(o[qt][dt][2] * inv),
                           (bf16)(o[qt][dt][3] * inv)};
      *reinterpret_cast<bf16x4_t*>(orow + dt * 16) = r4;
    }
  }
}

// The pieces of every cut item, put together: one workgroup per item, its waves and lanes holding the queries and
// coordinates they hold in the kernel above.  out = sum_j acc_j 2^(m_j - m) / sum_j l_j 2^(m_j - m) with m the
// largest maximum; a piece that saw no key has m = -inf and l = 0.
template <int DC, int QT>
__global__ __launch_bounds__(256) void attn_prefill_merge_kernel(const int* __restrict__ tiles, bf16* __restrict__ out,
                                                                  int H, int KV, int units_z, PrefillSplit split, int sink,
                                                                  const float* __restrict__ sinks, int wide) {
  constexpr int D = DC * 32, DT = DC * 2, WQ = 16 * QT, PARTS = 64 / WQ;
  const int item = blockIdx.x;
  const int n = split.cut[item];
  if (n <= 1) return;
  const int G = H / KV, per_tile = KV * units_z;
  const int tile = item / per_tile, kvh = (item % per_tile) / units_z, bz = item % units_z;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, col = lane & 15, grp = lane >> 4;
  const int tok0 = tiles[4 * tile], count = tiles[4 * tile + 1];
  const int unit = bz * 4 + wave, head = kvh * G + unit % G, q0 = (unit / G) * WQ;
  if (unit >= PARTS * G || q0 >= count) return;
#pragma unroll
  for (int qt = 0; qt < QT; ++qt) {
    const int qi = q0 + qt * 16 + col;
    if (qi >= count) continue;
    const size_t at = ((size_t)(tok0 + qi) * H + head) * split.pieces;
    const float2* ml = reinterpret_cast<const float2*>(split.ml) + at;  // (m, l) of the pieces
    float m = NEG_INF;
    for (int j = 0; j < n; ++j) m = fmaxf(m, ml[j].x);
    const float sk = sink_score(sink, sinks, head) * 1.4426950408889634f;
    if (sink) m = fmaxf(m, sk);
    f32x4_t sum[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) sum[dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float den = sink ? __builtin_amdgcn_exp2f(sk - m) : 0.f;
    for (int j = 0; j < n; ++j) {
      const float2 p = ml[j];
      const float w = p.x == NEG_INF ? 0.f : __builtin_amdgcn_exp2f(p.x - m);
      den += p.y * w;
      const float* a = split.acc + (at + j) * D + 4 * grp;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) sum[dt] += *reinterpret_cast<const f32x4_t*>(a + dt * 16) * w;
    }
    const float inv = 1.0f / den;
    if (wide) {
      float* orow = reinterpret_cast<float*>(out) + ((size_t)(tok0 + qi) * H + head) * D + 4 * grp;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) *reinterpret_cast<f32x4_t*>(orow + dt * 16) = sum[dt] * inv;
      continue;
    }
    bf16* orow = out + ((size_t)(tok0 + qi) * H + head) * D + 4 * grp;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
      const bf16x4_t r4 = {(bf16)(sum[dt][0] * inv), (bf16)(sum[dt][1] * inv), (bf16)(sum[dt][2] * inv), (bf16)(sum[dt][3] * inv)};
      *reinterpret_cast<bf16x4_t*>(orow + dt * 16) = r4;
    }
  }
}

// tiles: [num_tiles, 4] int32 (first flat token, count <= 64, block-table row, first position);
// fastest when sorted by first position + count, largest first.
// query_tiles: 2, a wave owns 32 queries of a head and a workgroup two heads' 64; or 1, a wave owns 16 and a
// workgroup one head's 64: twice the workgroups, each with half the arithmetic for the same keys and values
// brought into LDS, so that a round of 64 keys is shorter.  That pays where few work items decide the time
// (a lone prompt of a few thousand tokens: its last tile's rounds are a chain that nothing shortens).
// pieces > 1: every work item comes as that many workgroups, and items of more than piece_rounds rounds of 64 keys are
// cut along their keys into pieces of that many rounds and merged by a second kernel (see PrefillSplit); the caller
// then brings cut [num_tiles * KV * units] int32 with units = ceil(64 / (16 query_tiles) * (H / KV) / 4), part_ml
// [T, H, pieces, 2] and part_acc [T, H, pieces, D] fp32, T being one more than the largest flat token of a tile, and
// piece_rounds * pieces covers the longest item.  pieces <= 1: none is cut, the three may be null.
extern "C" int as_attn_prefill_mfma(const void* q, const void* k_pages, const void* v_pages, const int* tiles,
                                    int num_tiles, const int* block_tables, int table_width, void* out, int H,
                                    int KV, int D, int bs, float scale, int window, int keep, int chunk, float cap, int sink, const float* sinks,
                                    int wide, int query_tiles, int pieces, int piece_rounds, int* cut, float* part_ml,
                                    float* part_acc, hipStream_t stream) {
  if (num_tiles <= 0) return AS_OK;
  const Sight sight{window, keep, chunk, cap, sink, sinks, wide};
  if (!sight_ok(sight)) return AS_BAD_SHAPE;
  if (H <= 0 || KV <= 0 || H % KV || bs <= 0 || table_width <= 0) return AS_BAD_SHAPE;
  const int G = H / KV;
  if (D % 32 || D <= 0 || D > 256 || bs % 16) return AS_BAD_SHAPE;
  if (query_tiles != 1 && query_tiles != 2) return AS_BAD_SHAPE;
  if (pieces < 1) pieces = 1;
  if (pieces > 1 && (piece_rounds < PREFILL_MIN_PIECE_ROUNDS || !cut || !part_ml || !part_acc)) return AS_BAD_SHAPE;
  const int units_z = (64 / (16 * query_tiles) * G + 3) / 4;
  const long items = (long)num_tiles * KV * units_z;
  const long blocks = items * pieces;
  if (blocks > 0x7fffffffL) return AS_BAD_SHAPE;
  const int pass = compute_units();
  const PrefillSplit split{pieces, piece_rounds, cut, part_ml, part_acc};
  const int see = needed_sight(sight);
#define LAUNCH2(DCV, QTV, SEEV)                                                                       \
  attn_prefill_mfma_kernel<DCV, QTV, SEEV, 0><<<(int)blocks, 256, 0, stream>>>(                       \
      (const bf16*)q, (const bf16*)k_pages, (const bf16*)v_pages, tiles, block_tables, table_width,   \
      (bf16*)out, H, KV, bs, scale, sight, units_z, pass, split, Singles{})
#define LAUNCH1(DCV, QTV)                                                                             \
  if (see == 2) LAUNCH2(DCV, QTV, 2);                                                                 \
  else if (see == 1) LAUNCH2(DCV, QTV, 1);                                                            \
  else LAUNCH2(DCV, QTV, 0);                                                                          \
  if (pieces > 1)                                                                                     \
    attn_prefill_merge_kernel<DCV, QTV><<<(int)items, 256, 0, stream>>>(tiles, (bf16*)out, H, KV, units_z, split, sink, sinks, wide);
#define LAUNCH(DCV)              \
  if (query_tiles == 1) {        \
    LAUNCH1(DCV, 1)              \
  } else {                       \
    LAUNCH1(DCV, 2)              \
  }
  switch (D / 32) {
    case 1: LAUNCH(1); break;
    case 2: LAUNCH(2); break;
    case 3: LAUNCH(3); break;
    case 4: LAUNCH(4); break;
    case 5: LAUNCH(5); break;
    case 6: LAUNCH(6); break;
    case 7: LAUNCH(7); break;
    default: LAUNCH(8); break;
  }
#undef LAUNCH
#undef LAUNCH1
#undef LAUNCH2
  return launch_status();
}

static int launch_decode_mfma(const void* q, const void* k_pages, const void* v_pages, const int* items,
                              int num_items, const int* positions, const int* tok_row, const int* block_tables,
                              int table_width, void* out, float* part_m, float* part_l, float* part_acc, int H,
                              int KV, int D, int bs, float scale, const Sight& sight, int part_size, int P,
                              const FreshQKV* fresh, int gains_dtype, hipStream_t stream, int share = 1) {
  if (!sight_ok(sight) || (fresh && needed_sight(sight) > 0)) return AS_BAD_SHAPE;
  const int G = H / KV;
  if (D % 32 || D > 256 || G > 16 || bs % 16 || part_size % 32) return AS_BAD_SHAPE;
  if (fresh && D % 64) return AS_BAD_SHAPE;
  if (share < 1 || KV % share || (fresh && share != 1)) return AS_BAD_SHAPE;
  const bool turned = P > 1 && num_items > 8 && num_items <= 65535 && needed_sight(sight) == 0;
  const dim3 grid = turned ? dim3(KV, num_items, P) : dim3(num_items, KV, P);
  if (sizeof(float) * (size_t)(128 + 4 * D * G) + 1024 > (64u << 10)) return AS_BAD_SHAPE;  // wide heads in large groups: the general kernel's
  const size_t shmem = sizeof(float) * (size_t)(128 + 4 * (D + 4) * G) + (fresh ? sizeof(bf16) * (size_t)(D + 8) * G : 0);
  const FreshQKV none = {};
  const int see = needed_sight(sight);
  // Pages of 16 tokens, the engine's own, have instances of their own (see `load_kv_step`).
#define LAUNCH5(DCV, FRESHV, SEEV, TURNEDV, PAGEV)                                                        \
  do {                                                                                                    \
    const auto kernel = attn_decode_mfma_kernel<DCV, FRESHV, SEEV, TURNEDV, PAGEV>;                       \
    if (shmem + 1024 > 65536 &&                                                                           \
        hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem) != hipSuccess) \
      return AS_LAUNCH_FAILED;                                                                            \
    kernel<<<grid, 256, shmem, stream>>>(                                                                 \
      (const bf16*)q, (const bf16*)k_pages, (const bf16*)v_pages, items, positions, tok_row, block_tables, \
      table_width, (bf16*)out, part_m, part_l, part_acc, H, KV, bs, scale, sight, part_size, P,           \
      compute_units(), share, FRESHV ? *fresh : none);                                                    \
  } while (0)
#define LAUNCH4(DCV, FRESHV, SEEV, TURNEDV) LAUNCH5(DCV, FRESHV, SEEV, TURNEDV, 0)
#define LAUNCH(DCV, FRESHV)                                        \
  if (turned && bs == 16) LAUNCH5(DCV, FRESHV, 0, true, 16);       \
  else if (turned) LAUNCH5(DCV, FRESHV, 0, true, 0);               \
  else if (bs == 16) LAUNCH5(DCV, FRESHV, 0, false, 16);           \
  else LAUNCH5(DCV, FRESHV, 0, false, 0)
#define LAUNCH_PLAIN(DCV)                          \
  if (see == 2) LAUNCH4(DCV, 0, 2, false);         \
  else if (see == 1) LAUNCH4(DCV, 0, 1, false);    \
  else LAUNCH(DCV, 0)
#define LAUNCH_FRESH(FRESHV)            \
  switch (D / 64) {                     \
    case 1: LAUNCH(2, FRESHV); break;   \
    case 2: LAUNCH(4, FRESHV); break;   \
    case 3: LAUNCH(6, FRESHV); break;   \
    default: LAUNCH(8, FRESHV); break;  \
  }
  if (fresh && gains_dtype == DT_F32) {
    LAUNCH_FRESH(2)
  } else if (fresh) {
    LAUNCH_FRESH(1)
  } else {
    switch (D / 32) {
      case 1: LAUNCH_PLAIN(1); break;
      case 2: LAUNCH_PLAIN(2); break;
      case 3: LAUNCH_PLAIN(3); break;
      case 4: LAUNCH_PLAIN(4); break;
      case 5: LAUNCH_PLAIN(5); break;
      case 6: LAUNCH_PLAIN(6); break;
      case 7: LAUNCH_PLAIN(7); break;
      default: LAUNCH_PLAIN(8); break;
    }
  }
#undef LAUNCH_FRESH
#undef LAUNCH_PLAIN
#undef LAUNCH
#undef LAUNCH4
#undef LAUNCH5
  if (hipGetLastError() != hipSuccess) return AS_LAUNCH_FAILED;
  if (P > 1) {
    attn_reduce_kernel<bf16><<<dim3(num_items, H), D <= 64 ? 64 : (D <= 128 ? 128 : 256), 0, stream>>>(
        items, part_m, part_l, part_acc, (bf16*)out, H, D, P, sight.sink, sight.sinks, sight.wide);
  }
  return launch_status();
}

// Same contract as as_attn_single_query, bf16 only, through the matrix cores.
extern "C" int as_attn_decode_mfma(const void* q, const void* k_pages, const void* v_pages, const int* items,
                                   int num_items, const int* positions, const int* tok_row,
                                   const int* block_tables, int table_width, void* out, float* part_m,
                                   float* part_l, float* part_acc, int H, int KV, int D, int bs, float scale,
                                   int window, int keep, int chunk, float cap, int sink, const float* sinks, int wide, int part_size, int P,
                                   hipStream_t stream) {
  if (num_items <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || H % KV || D <= 0 || bs <= 0 || part_size <= 0 || P <= 0 || table_width <= 0)
    return AS_BAD_SHAPE;
  if (P > 1 && (!part_m || !part_l || !part_acc)) return AS_BAD_SHAPE;
  return launch_decode_mfma(q, k_pages, v_pages, items, num_items, positions, tok_row, block_tables, table_width,
                            out, part_m, part_l, part_acc, H, KV, D, bs, scale, Sight{window, keep, chunk, cap, sink, sinks, wide},
                            part_size, P, nullptr, DT_BF16, stream);
}

// The same where the pages hold KV / share heads and every `share` consecutive groups of H / KV query heads read
// one of them: a group of more than 16 query heads, cut into several of equal size.
extern "C" int as_attn_decode_mfma_shared(const void* q, const void* k_pages, const void* v_pages, const int* items,
                                          int num_items, const int* positions, const int* tok_row,
                                          const int* block_tables, int table_width, void* out, float* part_m,
                                          float* part_l, float* part_acc, int H, int KV, int D, int bs, float scale,
                                          int window, int keep, int chunk, float cap, int sink, const float* sinks, int wide, int part_size, int P,
                                          int share, hipStream_t stream) {
  if (num_items <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || H % KV || D <= 0 || bs <= 0 || part_size <= 0 || P <= 0 || table_width <= 0)
    return AS_BAD_SHAPE;
  if (P > 1 && (!part_m || !part_l || !part_acc)) return AS_BAD_SHAPE;
  return launch_decode_mfma(q, k_pages, v_pages, items, num_items, positions, tok_row, block_tables, table_width,
                            out, part_m, part_l, part_acc, H, KV, D, bs, scale, Sight{window, keep, chunk, cap, sink, sinks, wide},
                            part_size, P, nullptr, DT_BF16, stream, share);
}

// A decode step (token t is row t of the block tables) from the projection's output: per-head norm,
// rotation of the whole head, the new token's key and value written to its slot (store 0: queries
// only, the pages already hold them), and attention, in one kernel.  qkv [T, H + 2 KV, D] bf16;
// qw, kw [D] bf16 or fp32; cs [T, D/2] float2; slots [T]; items [T]: the order in which the tokens are
// taken (null: as they come), best the longest contexts first.  Needs D % 64 == 0.
extern "C" int as_attn_decode_fresh(const void* qkv, const void* qw, const void* kw, int gains_dtype,
                                    const float* cs, const int* slots, float eps, int store, void* k_pages,
                                    void* v_pages, const int* items, int num_tokens, const int* positions,
                                    const int* block_tables, int table_width, void* out, float* part_m,
                                    float* part_l, float* part_acc, int H, int KV, int D, int bs, float scale,
                                    int window, int part_size, int P, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || H % KV || D <= 0 || bs <= 0 || part_size <= 0 || P <= 0 || table_width <= 0)
    return AS_BAD_SHAPE;
  if (P > 1 && (!part_m || !part_l || !part_acc)) return AS_BAD_SHAPE;
  if (!qkv || !qw || !kw || !cs || (store && !slots)) return AS_BAD_SHAPE;
  if (gains_dtype != DT_BF16 && gains_dtype != DT_F32) return AS_BAD_DTYPE;
  const FreshQKV fresh = {(const bf16*)qkv, qw, kw, (const float2*)cs, slots, (bf16*)k_pages, (bf16*)v_pages,
                          eps, store};
  return launch_decode_mfma(nullptr, k_pages, v_pages, items, num_tokens, positions, nullptr, block_tables,
                            table_width, out, part_m, part_l, part_acc, H, KV, D, bs, scale, Sight{window, 0, 0, 0.f, 0, nullptr, 0},
                            part_size, P, &fresh, gains_dtype, stream);
}

// as_attn_prefill_mfma and as_attn_decode_mfma of one step in one launch (with merges behind it where items are cut), for
// heads of 64 and 128, pages of 16 tokens and no more sight than a window: arguments as there.  The two sets of tokens
// are apart, and so are the partial results.
extern "C" int as_attn_mixed_mfma(const void* q, const void* k_pages, const void* v_pages, const int* tiles, int num_tiles,
                                  const int* items, int num_items, const int* positions, const int* tok_row,
                                  const int* block_tables, int table_width, void* out, int H, int KV, int D, int bs, float scale,
                                  int window, int query_tiles, int pieces, int piece_rounds, int* cut, float* piece_ml,
                                  float* piece_acc, float* part_m, float* part_l, float* part_acc, int part_size, int P,
                                  hipStream_t stream) {
  if (num_tiles <= 0 || num_items <= 0) return AS_BAD_SHAPE;
  const Sight sight{window, 0, 0, 0.f, 0, nullptr, 0};
  if (!sight_ok(sight)) return AS_BAD_SHAPE;
  if (H <= 0 || KV <= 0 || H % KV || H / KV > 16 || table_width <= 0 || (D != 64 && D != 128) || bs != 16) return AS_BAD_SHAPE;
  if (query_tiles != 1 && query_tiles != 2) return AS_BAD_SHAPE;
  if (pieces < 1) pieces = 1;
  if (pieces > 1 && (piece_rounds < PREFILL_MIN_PIECE_ROUNDS || !cut || !piece_ml || !piece_acc)) return AS_BAD_SHAPE;
  if (part_size <= 0 || part_size % 32 || P <= 0 || (P > 1 && (!part_m || !part_l || !part_acc))) return AS_BAD_SHAPE;
  const int units_z = (64 / (16 * query_tiles) * (H / KV) + 3) / 4;
  const long tile_items = (long)num_tiles * KV * units_z, blocks = tile_items * pieces + (long)num_items * KV * P;
  if (blocks > 0x7fffffffL) return AS_BAD_SHAPE;
  const PrefillSplit split{pieces, piece_rounds, cut, piece_ml, piece_acc};
  const Singles single{items, positions, tok_row, part_m, part_l, part_acc, num_items, part_size, P};
#define LAUNCH(DCV, QTV)                                                                                                 \
  do {                                                                                                                   \
    attn_prefill_mfma_kernel<DCV, QTV, 0, 16><<<(int)blocks, 256, 0, stream>>>(                                          \
        (const bf16*)q, (const bf16*)k_pages, (const bf16*)v_pages, tiles, block_tables, table_width, (bf16*)out, H, KV, \
        bs, scale, sight, units_z, compute_units(), split, single);                                                      \
    if (hipGetLastError() != hipSuccess) return AS_LAUNCH_FAILED;                                                        \
    if (pieces > 1)                                                                                                      \
      attn_prefill_merge_kernel<DCV, QTV><<<(int)tile_items, 256, 0, stream>>>(tiles, (bf16*)out, H, KV, units_z, split, \
                                                                               0, nullptr, 0);                           \
  } while (0)
  if (D == 64) {
    if (query_tiles == 1) LAUNCH(2, 1);
    else LAUNCH(2, 2);
  } else {
    if (query_tiles == 1) LAUNCH(4, 1);
    else LAUNCH(4, 2);
  }
#undef LAUNCH
  if (hipGetLastError() != hipSuccess) return AS_LAUNCH_FAILED;
  if (P > 1)
    attn_reduce_kernel<bf16><<<dim3(num_items, H), D, 0, stream>>>(items, part_m, part_l, part_acc, (bf16*)out, H, D, P, 0, nullptr, 0);
  return launch_status();
}

static int pow2ceil(int v) { int p = 1; while (p < v) p <<= 1; return p; }

template <typename T>
static int launch_single_query(const void* q, const void* k_pages, const void* v_pages, const int* items,
                               int num_items, const int* positions, const int* tok_row,
                               const int* block_tables, int table_width, void* out, float* part_m,
                               float* part_l, float* part_acc, int H, int KV, int D, int bs, float scale,
                               const Sight& sight, int part_size, int P, hipStream_t stream) {
  if (!sight_ok(sight)) return AS_BAD_SHAPE;
  constexpr int CH = Chunk<T>::N;
  if (D % CH != 0 || D > 64 * CH || D > 256) return AS_BAD_SHAPE;
  const int G = H / KV;
  const int lpk = pow2ceil(D / CH);
  const int GT = G >= 8 ? 8 : (G > 2 ? 4 : (G == 2 ? 2 : 1));
  const int HC = (G + GT - 1) / GT;
  dim3 grid(num_items, KV * HC, P);
  const size_t shmem = sizeof(float) * (size_t)(8 * GT + 4 * GT * D);
#define LAUNCH(GTV)                                                                                      \
  attn_single_query_kernel<T, GTV><<<grid, 256, shmem, stream>>>(                                        \
      (const T*)q, (const T*)k_pages, (const T*)v_pages, items, positions, tok_row, block_tables,       \
      table_width, (T*)out, part_m, part_l, part_acc, H, KV, D, bs, scale, sight, part_size, P, lpk)
  switch (GT) {
    case 1: LAUNCH(1); break;
    case 2: LAUNCH(2); break;
    case 4: LAUNCH(4); break;
    default: LAUNCH(8); break;
  }
#undef LAUNCH
  if (hipGetLastError() != hipSuccess) return AS_LAUNCH_FAILED;
  if (P > 1) {
    attn_reduce_kernel<T><<<dim3(num_items, H), D <= 64 ? 64 : (D <= 128 ? 128 : 256), 0, stream>>>(
        items, part_m, part_l, part_acc, (T*)out, H, D, P, sight.sink, sight.sinks, sight.wide);
  }
  return launch_status();
}

// part_m, part_l: [num_items, H, P] fp32; part_acc: [num_items, H, P, D] fp32 (unused when P == 1).
// P must be >= ceil(n / part_size), n the most keys that an item sees (its context; with a window at most window + keep).
extern "C" int as_attn_single_query(const void* q, const void* k_pages, const void* v_pages, int dtype,
                                    const int* items, int num_items, const int* positions,
                                    const int* tok_row, const int* block_tables, int table_width, void* out,
                                    float* part_m, float* part_l, float* part_acc, int H, int KV, int D,
                                    int bs, float scale, int window, int keep, int chunk, float cap, int sink, const float* sinks, int wide,
                                    int part_size, int P, hipStream_t stream) {
  if (num_items <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || H % KV || D <= 0 || bs <= 0 || part_size <= 0 || P <= 0 || table_width <= 0)
    return AS_BAD_SHAPE;
  if (P > 1 && (!part_m || !part_l || !part_acc)) return AS_BAD_SHAPE;
  if (dtype == DT_F32)
    return launch_single_query<float>(q, k_pages, v_pages, items, num_items, positions, tok_row, block_tables,
                                      table_width, out, part_m, part_l, part_acc, H, KV, D, bs, scale,
                                      Sight{window, keep, chunk, cap, sink, sinks, wide}, part_size, P, stream);
  if (dtype == DT_BF16)
    return launch_single_query<bf16>(q, k_pages, v_pages, items, num_items, positions, tok_row, block_tables,
                                     table_width, out, part_m, part_l, part_acc, H, KV, D, bs, scale,
                                     Sight{window, keep, chunk, cap, sink, sinks, wide}, part_size, P, stream);
  return AS_BAD_DTYPE;
}

// ---- fp32 through the matrix cores -------------------------------------------------------
//
// attn_f32: the attention of 32-bit heads, 16 queries of one kv head to a workgroup as the columns of 16 x 16 tiles:
// the G heads of one token (decode: items), or of 16 / G neighbouring tokens of a prompt (tiles), so that every key and value
// is read once for all of them.  The four waves take the steps of 16 keys in turn, each with maxima, sums and
// outputs of its own, which meet in LDS at the end.  Per step, all products by v_mfma_f32_16x16x4_f32 (32-bit products and sums):
//   S[key][query] = K[key][:] . Q[query][:]     keys straight from the page, 16 bytes a lane
//   O^T[d][query] += V^T[d][key] P[key][query]  values straight from the transposed page; P is what the lane holds
// The next step's keys are asked for when this step's have met the queries, its values when these have been added up.
// Values of places that none of the workgroup's queries sees count as 0 whatever lies there (0.1 us); of keys that only some of
// a tile's queries see they are finite, as every kernel that stores values makes them.
// Bound by the 64 matrix instructions of a step (heads of 128): 0.9 us a wave, and by launch and merge for short
// contexts.  16 heads of 128 on 8 kv heads, in a captured step: 4 requests of 600 tokens 12.2 us, of 2,000 tokens 18.4 (45.2 and 54.4
// on the general kernel, which reads each value of a transposed page alone); a prompt of 333 tokens 24 (147: a workgroup to
// every token read all keys before it).
//
// FRESH (decode steps whose tokens are their own rows): the kernel takes the projection's output qkv [T, H + 2 KV, D] and does what
// qk_norm_rope_store does: every workgroup norms and rotates its group's queries, and the one whose partition holds the token's own position
// makes the key and value, stores them and takes them from LDS where its pages' loads would have found them.  A head is one wave's work
// (a lane has coordinates i and i + D/2), the waves take the group's heads, the key and the value in turn.  Same
// arithmetic; the squares are summed in another order.  All that they are made of is asked for before the first keys and values (behind them
// it waited for those).  In a captured step of 4 requests of 500 to 700 tokens, 16 heads of 128 on 8 kv heads: 4.9 us for the kernel before
// this one and 9.6 for this, as one 11.8 with every wave norming all queries as operands (284 registers), now 10.7 (222).
struct FreshF32 {
  const float* qkv;
  const float* qw;   // gains of the per-head norms, D values each
  const float* kw;
  const float2* cs;  // [T, D/2] cos, sin of the whole head's rotation
  const int* slots;  // [T] page * block_size + offset of the new token, -1: keep it out of the pages
  float* k_store;    // the pages again, to write through
  float* v_store;
  float eps;
  int store;         // 0: queries only, the pages already hold the token's key and value
};

// PAGE: tokens of a page where the compiler knows them (three divisions a step by another number are some 600 cycles), or 0.
template <int DT, bool FRESH, int PAGE>
__global__ __launch_bounds__(256) void attn_f32_kernel(
    const float* __restrict__ q, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int* __restrict__ tiles, const int* __restrict__ items, const int* __restrict__ positions,
    const int* __restrict__ tok_row, const int* __restrict__ block_tables, int table_width, float* __restrict__ out,
    float* __restrict__ part_m, float* __restrict__ part_l, float* __restrict__ part_acc, int H, int KV, int page_size,
    float scale, Sight sight, int subs, int part_size, int P, int N, FreshF32 fresh) {
  constexpr int D = 16 * DT, LD = D + 4;
  const int bs = PAGE ? PAGE : page_size;
  extern __shared__ float smem[];  // [4][16] m, [4][16] l, [4][16][LD] outputs
  const int G = H / KV;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  int t0, count, row, pos0;
  // the kv heads change fastest: workgroups are dealt to the XCDs in turn, and every XCD has its share of every context
  const int place = blockIdx.x + N * (blockIdx.y + KV * blockIdx.z), rest = place / KV;
  const int part = rest / N, item = rest - part * N, kvh = (place - rest * KV + item) % KV;
  if (tiles) {
    const int per = 16 / G;  // tokens of a workgroup
    const int* tile = tiles + (size_t)(item / subs) * 4;
    const int at = item % subs * per;
    count = min(per, tile[1] - at);
    if (count <= 0) return;
    t0 = tile[0] + at;
    row = tile[2];
    pos0 = tile[3] + at;
  } else {
    t0 = items ? items[item] : item;
    count = 1;
    row = tok_row ? tok_row[t0] : t0;
    pos0 = positions[t0];
  }
  const int tok = lr / G, head = kvh * G + lr % G;
  const bool valid = tok < count;
  const int pos = valid ? pos0 + tok : -1;
  const int first = valid ? first_in_window(sight, pos + 1) : 0;       // this column's first visible key
  const int seen = first_in_window(sight, pos0 + 1), start = seen & ~15;  // the workgroup's first, and that in whole steps
  const int k0 = start + part * part_size, k1 = P == 1 ? pos0 + count : min(pos0 + count, k0 + part_size);
  if (k0 >= k1) {  // an empty partition (items only): mark it so for the reduce
    if (tid < G) {
      const size_t o = ((size_t)item * H + kvh * G + tid) * P + part;
      part_m[o] = NEG_INF;
      part_l[o] = 0.f;
    }
    for (int x = tid; x < G * D; x += 256) part_acc[(((size_t)item * H + kvh * G + x / D) * P + part) * D + x % D] = 0.f;
    return;
  }
  const int steps = (k1 - k0 + 15) >> 4;
  const int* table = block_tables + (size_t)row * table_width;

  constexpr int HALF = D / 2, TURNS = FRESH ? 5 : 1;  // 16 heads, a key and a value over four waves
  __shared__ __align__(16) float fresh_kv[2][FRESH ? D : 1];  // the new token's key and value
  [[maybe_unused]] float* const queries = smem + 128 + 4 * 16 * LD;  // FRESH: [G][LD]
  f32x4_t qf[DT], kf[DT], vf[DT], o[DT];
  auto piece_of = [&](int i) { return (i >> 1) * 32 + lg * 8 + (i & 1) * 4; };
  const float* qrow = FRESH ? queries + (valid ? lr : 0) * LD : q + ((size_t)(t0 + (valid ? tok : 0)) * H + (valid ? head : kvh * G)) * D;
#pragma unroll
  for (int i = 0; i < DT; ++i) {
    if constexpr (!FRESH) qf[i] = *reinterpret_cast<const f32x4_t*>(qrow + piece_of(i));
    o[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  auto page_of = [&](int step) {  // the 16 keys' place: page and offset, as an offset into one head's pages
    const int key = k0 + min(step, steps - 1) * 16;
    return ((size_t)table[key / bs] * KV + kvh) * bs * D;
  };
  auto load_keys = [&](size_t base, int step) {
    const float* p = k_pages + base + (size_t)((k0 + min(step, steps - 1) * 16) % bs + lr) * D + lg * 8;
#pragma unroll
    for (int i = 0; i < DT; ++i) kf[i] = *reinterpret_cast<const f32x4_t*>(p + (i >> 1) * 32 + (i & 1) * 4);
  };
  auto load_values = [&](size_t base, int step) {
    const float* p = v_pages + base + (size_t)lr * bs + (k0 + min(step, steps - 1) * 16) % bs + lg * 4;
#pragma unroll
    for (int i = 0; i < DT; ++i) vf[i] = *reinterpret_cast<const f32x4_t*>(p + (size_t)i * 16 * bs);
  };
  float m = NEG_INF, l = 0.f;
  size_t base = page_of(wave), next = page_of(wave + 4);
  // FRESH: the new token's key and value, in this partition at key `mine` of step `own_step`, or nowhere.
  [[maybe_unused]] int own_step = -1, slot = -1, jobs = G;  // jobs: the group's heads, then the key and the value
  [[maybe_unused]] const int mine = (pos0 - k0) & 15;
  [[maybe_unused]] float ha[TURNS], hb[TURNS], ga[2], gb[2];
  [[maybe_unused]] float2 angle;
  if constexpr (FRESH) {
    if (fresh.store && pos0 < k1) {  // k0 <= pos0 where the partition is not empty
      own_step = (pos0 - k0) >> 4;
      jobs = G + 2;
      slot = fresh.slots[t0];
    }
    const int i = min(lane, HALF - 1);
#pragma unroll
    for (int n = 0; n < TURNS; ++n) {
      const int job = wave + 4 * n;
      if (job < jobs) {  // uniform over the wave
        const float* src = fresh.qkv + ((size_t)t0 * (H + 2 * KV) + (job < G ? kvh * G + job : H + kvh + (job - G) * KV)) * D;
        ha[n] = src[i];
        hb[n] = src[i + HALF];
      }
    }
    ga[0] = fresh.qw[i];
    gb[0] = fresh.qw[i + HALF];
    ga[1] = fresh.kw[i];
    gb[1] = fresh.kw[i + HALF];
    angle = fresh.cs[(size_t)t0 * HALF + i];
    __builtin_amdgcn_sched_barrier(0);
  }
  if (wave < steps) {
    load_keys(base, wave);
    load_values(base, wave);
  }
  if constexpr (FRESH) {
    __builtin_amdgcn_sched_barrier(0);
    const size_t head_at = slot >= 0 ? ((size_t)(slot / bs) * KV + kvh) * bs * D : 0;
#pragma unroll
    for (int n = 0; n < TURNS; ++n) {
      const int job = wave + 4 * n;
      if (job > G && job < jobs) {  // the value, as it is; its page is stored transposed
        const float ra = finite_or_zero(ha[n]), rb = finite_or_zero(hb[n]);
        if (lane < HALF) {
          fresh_kv[1][lane] = ra;
          fresh_kv[1][lane + HALF] = rb;
          float* vt = fresh.v_store + head_at + slot % bs;
          if (slot >= 0) { vt[(size_t)lane * bs] = ra; vt[(size_t)(lane + HALF) * bs] = rb; }
        }
      } else if (job < jobs) {  // a query or the key
        const bool is_key = job == G;
        const float ss = wave_sum(lane < HALF ? ha[n] * ha[n] + hb[n] * hb[n] : 0.f), inv = 1.0f / sqrtf(ss / (float)D + fresh.eps);
        const float a = ha[n] * inv * (is_key ? ga[1] : ga[0]), b = hb[n] * inv * (is_key ? gb[1] : gb[0]);
        float ra = a * angle.x - b * angle.y, rb = b * angle.x + a * angle.y;
        if (is_key) {
          ra = finite_or_zero(ra);
          rb = finite_or_zero(rb);
        }
        float* to = is_key ? fresh_kv[0] : queries + job * LD;
        if (lane < HALF) {
          to[lane] = ra;
          to[lane + HALF] = rb;
          float* dst = fresh.k_store + head_at + (size_t)(slot % bs) * D;
          if (is_key && slot >= 0) { dst[lane] = ra; dst[lane + HALF] = rb; }
        }
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DT; ++i) qf[i] = *reinterpret_cast<const f32x4_t*>(qrow + piece_of(i));
  }
#pragma unroll
  for (int i = 0; i < DT; ++i) qf[i] = qf[i] * scale;
  for (int step = wave; step < steps; step += 4) {
    if constexpr (FRESH) {
      if (step == own_step) {
#pragma unroll
        for (int i = 0; i < DT; ++i) {
          if (lr == mine) kf[i] = *reinterpret_cast<const f32x4_t*>(&fresh_kv[0][piece_of(i)]);
          const float value = fresh_kv[1][i * 16 + lr];
#pragma unroll
          for (int x = 0; x < 4; ++x) vf[i][x] = lg * 4 + x == mine ? value : vf[i][x];
        }
      }
    }
    f32x4_t s0 = f32x4_t{0.f, 0.f, 0.f, 0.f}, s1 = s0;
#pragma unroll
    for (int i = 0; i < DT; i += 2)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][x], qf[i][x], s0, 0, 0, 0);
        s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i + 1][x], qf[i + 1][x], s1, 0, 0, 0);
      }
    load_keys(next, step + 4);
    f32x4_t s = s0 + s1;
    const int key = k0 + step * 16 + lg * 4;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (sight.cap > 0.f) s[r] = sight.cap * tanhf(s[r] / sight.cap);
      if (key + r > pos || key + r < first || key + r >= k1) s[r] = NEG_INF;
    }
    const float top = fmaxf(m, quad_rows_max(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
    const float at = top == NEG_INF ? 0.f : top;  // nothing seen yet: every weight is e^-inf = 0
    if (__any(top > m)) {
      const float keep = expf(m - at);
      l *= keep;
#pragma unroll
      for (int i = 0; i < DT; ++i) o[i] *= keep;
      m = top;
    }
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) p[r] = expf(s[r] - at);
    l += (p[0] + p[1]) + (p[2] + p[3]);
    if (__builtin_expect(k0 + step * 16 < seen || k0 + step * 16 + 16 > k1, 0)) {  // whatever lies where no key is seen: a weight of 0 is not enough
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (key + r < seen || key + r >= k1) {
#pragma unroll
          for (int i = 0; i < DT; ++i) vf[i][r] = 0.f;
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int i = 0; i < DT; ++i) o[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[i][r], p[r], o[i], 0, 0, 0);
    load_values(next, step + 4);
    next = page_of(step + 8);
  }
  l = quad_rows_sum(l);
  float* sm = smem;
  float* sl = smem + 64;
  float* so = smem + 128;
  if (lg == 0) { sm[wave * 16 + lr] = m; sl[wave * 16 + lr] = l; }
#pragma unroll
  for (int i = 0; i < DT; ++i) *reinterpret_cast<f32x4_t*>(so + (size_t)(wave * 16 + lr) * LD + i * 16 + lg * 4) = o[i];
  __syncthreads();
  for (int x = tid; x < count * G * D; x += 256) {
    const int c = x / D, d = x % D;
    float top = fmaxf(fmaxf(sm[c], sm[16 + c]), fmaxf(sm[32 + c], sm[48 + c])), num = 0.f, den = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float e = sm[w * 16 + c] == NEG_INF ? 0.f : expf(sm[w * 16 + c] - top);
      num += so[(size_t)(w * 16 + c) * LD + d] * e;
      den += sl[w * 16 + c] * e;
    }
    const int h = kvh * G + c % G;
    if (P == 1) {
      if (sight.sink) {
        const float sk = sink_score(1, sight.sinks, h), most = fmaxf(top, sk), e = expf(top - most);
        num *= e;
        den = den * e + expf(sk - most);
      }
      out[((size_t)(t0 + c / G) * H + h) * D + d] = num / den;
    } else {
      const size_t o = ((size_t)item * H + h) * P + part;
      part_acc[o * D + d] = num;
      if (d == 0) { part_m[o] = top; part_l[o] = den; }
    }
  }
}

// Which shapes it takes: heads of 64 or 128, at most 16 query heads to a kv head, pages of whole steps of 16 keys, no
// kept first keys (a second stretch of keys; the general kernel walks them).
static int launch_attn_f32(const FreshF32* fresh, const float* q, const float* k_pages, const float* v_pages, const int* tiles, int num_tiles,
                           int most, const int* items, int num_items, const int* positions, const int* tok_row,
                           const int* block_tables, int table_width, float* out, float* part_m, float* part_l,
                           float* part_acc, int H, int KV, int D, int bs, float scale, int window, int keep, int chunk,
                           float cap, int sink, const float* sinks, int wide, int part_size, int P, hipStream_t stream) {
  const Sight sight{window, keep, chunk, cap, sink, sinks, wide};
  const int blocks_of = tiles ? num_tiles : num_items;
  if (blocks_of <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || KV > 65535 || H % KV || H / KV > 16 || (D != 64 && D != 128) || bs <= 0 || bs % 16 || table_width <= 0 ||
      part_size <= 0 || part_size % 16 || P <= 0 || P > 65535 || !sight_ok(sight) || keep || wide)
    return AS_BAD_SHAPE;
  if ((tiles && (P != 1 || most <= 0)) || (P > 1 && (!part_m || !part_l || !part_acc))) return AS_BAD_SHAPE;
  const int per = tiles ? 16 / (H / KV) : 1, subs = tiles ? (most + per - 1) / per : 1;
  if ((long)blocks_of * subs > 0x7fffffffL) return AS_BAD_SHAPE;
  const dim3 grid(blocks_of * subs, KV, P);
  const size_t lds = (128 + (4 * 16 + (fresh ? H / KV : 0)) * (D + 4)) * sizeof(float);
  const FreshF32 none = {};
#define GO(DTV, FRESHV, PAGEV)                                                                                                           \
  attn_f32_kernel<DTV, FRESHV, PAGEV><<<grid, 256, lds, stream>>>(q, k_pages, v_pages, tiles, items, positions, tok_row, block_tables,    \
                                                                  table_width, out, part_m, part_l, part_acc, H, KV, bs, scale, sight,    \
                                                                  subs, part_size, P, blocks_of * subs, FRESHV ? *fresh : none)
#define GO_PAGES(DTV, FRESHV)           \
  if (bs == 16) GO(DTV, FRESHV, 16);    \
  else GO(DTV, FRESHV, 0)
  if (fresh) {
    if (D == 64) { GO_PAGES(4, true); }
    else { GO_PAGES(8, true); }
  } else if (D == 64) { GO_PAGES(4, false); }
  else { GO_PAGES(8, false); }
#undef GO_PAGES
#undef GO
  if (P > 1) {
    const int rc = launch_status();
    if (rc != AS_OK) return rc;
    attn_reduce_kernel<float><<<dim3(num_items, H), D, 0, stream>>>(items, part_m, part_l, part_acc, out, H, D, P, sight.sink, sight.sinks, 0);
  }
  return launch_status();
}

extern "C" int as_attn_f32(const float* q, const float* k_pages, const float* v_pages, const int* tiles, int num_tiles,
                           int most, const int* items, int num_items, const int* positions, const int* tok_row,
                           const int* block_tables, int table_width, float* out, float* part_m, float* part_l,
                           float* part_acc, int H, int KV, int D, int bs, float scale, int window, int keep, int chunk,
                           float cap, int sink, const float* sinks, int wide, int part_size, int P, hipStream_t stream) {
  return launch_attn_f32(nullptr, q, k_pages, v_pages, tiles, num_tiles, most, items, num_items, positions, tok_row, block_tables, table_width, out,
                         part_m, part_l, part_acc, H, KV, D, bs, scale, window, keep, chunk, cap, sink, sinks, wide, part_size, P, stream);
}

// The same for a decode step from the projection's output (see FreshF32): q is qkv [T, H + 2 KV, D]; token t is row t.  items
// [num_items] or null (all in order); slots may be null where store_kv is 0.
extern "C" int as_attn_f32_fresh(const float* qkv, const float* qw, const float* kw, const float* cs, const int* slots, float eps, int store_kv,
                                 float* k_pages, float* v_pages, const int* items, int num_items, const int* positions, const int* block_tables,
                                 int table_width, float* out, float* part_m, float* part_l, float* part_acc, int H, int KV, int D, int bs,
                                 float scale, int window, int part_size, int P, hipStream_t stream) {
  if (num_items <= 0) return AS_OK;
  if (!qkv || !qw || !kw || !cs || (store_kv && !slots) || (((uintptr_t)qkv | (uintptr_t)qw | (uintptr_t)kw | (uintptr_t)cs) & 15)) return AS_BAD_SHAPE;
  const FreshF32 fresh{qkv, qw, kw, (const float2*)cs, slots, k_pages, v_pages, eps, store_kv};
  return launch_attn_f32(&fresh, nullptr, k_pages, v_pages, nullptr, 0, 0, items, num_items, positions, nullptr, block_tables, table_width, out,
                         part_m, part_l, part_acc, H, KV, D, bs, scale, window, 0, 0, 0.f, 0, nullptr, 0, part_size, P, stream);
}

// ---- the same without scratch buffers from the caller ----------------------------------
//
// The partial results of a split context live in an array of the library's own; see no_alloc.h.
// In host code `scratch` is only a stand-in for the symbol: the address that kernels and copies
// use is the one hipGetSymbolAddress returns, and every GPU has its own.
static __device__ __align__(256) float scratch[AS_STATIC_SCRATCH_FLOATS];
static float* scratch_on_device[64] = {nullptr};

static int scratch_of_current_device(float** ptr) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return AS_LAUNCH_FAILED;
  if (scratch_on_device[dev] == nullptr) {
    void* found = nullptr;
    if (hipGetSymbolAddress(&found, HIP_SYMBOL(scratch)) != hipSuccess || found == nullptr) return AS_LAUNCH_FAILED;
    scratch_on_device[dev] = (float*)found;
  }
  *ptr = scratch_on_device[dev];
  return AS_OK;
}

extern "C" int as_attn_single_query_static(const void* q, const void* k_pages, const void* v_pages, int dtype,
                                           const int* items, int num_items, const int* positions,
                                           const int* tok_row, const int* block_tables, int table_width,
                                           void* out, int H, int KV, int D, int bs, float scale, int window,
                                           int part_size, int P, hipStream_t stream) {
  if (num_items <= 0) return AS_OK;
  if (H <= 0 || KV <= 0 || H % KV || D <= 0 || bs <= 0 || part_size <= 0 || P <= 0 || table_width <= 0)
    return AS_BAD_SHAPE;
  if (window > 0) {  // partitions cut the keys that the window shows: no more than these are ever filled
    const int most = (int)(((long)window + part_size - 1) / part_size);
    if (most < P) P = most;
  }
  float *part_m = nullptr, *part_l = nullptr, *part_acc = nullptr;
  if (P > 1) {
    const unsigned long long rows = (unsigned long long)num_items * (unsigned long long)H * (unsigned long long)P;
    if (rows > AS_STATIC_SCRATCH_FLOATS || rows * (unsigned long long)(D + 2) > AS_STATIC_SCRATCH_FLOATS)
      return AS_TOO_LARGE;
    float* base = nullptr;
    const int status = scratch_of_current_device(&base);
    if (status != AS_OK) return status;
    part_acc = base;  // [rows, D]: first, so that it keeps the array's alignment
    part_m = base + rows * D;
    part_l = part_m + rows;
  }
  return as_attn_single_query(q, k_pages, v_pages, dtype, items, num_items, positions, tok_row, block_tables,
                              table_width, out, part_m, part_l, part_acc, H, KV, D, bs, scale, window, 0, 0, 0.f, 0, nullptr, 0,
                              part_size, P, stream);
}
