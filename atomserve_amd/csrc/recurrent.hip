// Mixers that carry a fixed-size state from token to token: short causal convolutions, the gated
// delta rule and the gated linear recurrence.  Everything that enters a recurrence (decays, step
// sizes, gates, unit norms, the state itself) is fp32 in both precisions; only what the matrix
// products hand over (T) and the activations handed on to the next product are bf16 when serving.
//
// A step's rows are described as everywhere else: tok_row [T] (the row of a token), and per row its
// first flat token, its length, the position of its first token and its slot in the state tables.  A
// row that starts at position 0 starts from a zero state whatever its slot holds (slots are used
// again); a portion of a prompt goes on from what the portion before left.  State tables are fp32
// [slots, ...]; a row's state is written back only when `writes`.
#include "common.h"
#include "float_parts.h"
#include "rows.h"
#include <algorithm>
#include <climits>
#include <type_traits>

#define CONV_MAX_TAPS 8

__device__ __forceinline__ float sigmoidf_(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplusf_(float z) { return z > 20.f ? z : log1pf(expf(z)); }
__device__ __forceinline__ float siluf_(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float gelu_tanhf_(float z) {
  return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}

// ---- short causal convolution per channel ------------------------------------------------------
// in [T, ld]: the C channels start at column col0; in_bias [C] (or none) is added to every input that
// exists (the zeros before a sequence stay zeros).  w [C, taps], the last column multiplying the
// current token; bias [C] or none; act 1: silu.  history [slots, taps - 1, C]: the inputs of the last
// taps - 1 tokens before the row, oldest first.  out fp32 [T, C].
template <typename T, typename W>
__global__ void short_conv_kernel(const T* __restrict__ in, int ld, int col0, int C, const W* __restrict__ in_bias,
                                  const W* __restrict__ w, const W* __restrict__ bias, int taps, int act,
                                  const float* __restrict__ history, const int* __restrict__ tok_row,
                                  const int* __restrict__ row_first, const int* __restrict__ row_start,
                                  const int* __restrict__ row_slots, float* __restrict__ out) {
  const int t = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int r = tok_row ? tok_row[t] : t;
  const int first = row_first[r], j = t - first;
  const bool carried = row_start[r] > 0 && row_slots[r] >= 0;
  const float* old = history + (size_t)(carried ? row_slots[r] : 0) * (taps - 1) * C;
  const float ib = in_bias ? to_f32(in_bias[c]) : 0.f;
  float acc = 0.f;
  for (int i = 0; i < taps; ++i) {
    const int src = j - (taps - 1 - i);
    float v = 0.f;
    if (src >= 0) v = to_f32(in[(size_t)(first + src) * ld + col0 + c]) + ib;
    else if (carried) v = old[(size_t)(taps - 1 + src) * C + c];
    acc = fmaf(to_f32(w[(size_t)c * taps + i]), v, acc);
  }
  if (bias) acc += to_f32(bias[c]);
  out[(size_t)t * C + c] = act == 1 ? siluf_(acc) : acc;
}

// The same for many tokens, four neighbouring channels of CONV_TOKENS tokens in a row a thread: every input is read once for all
// its taps.  fp32 weights; C, col0 and ld multiples of four.
#define CONV_TOKENS 8
template <typename T> __device__ __forceinline__ float quick_silu(float z) { return siluf_(z); }
template <> __device__ __forceinline__ float quick_silu<bf16>(float z) { return z * __builtin_amdgcn_rcpf(1.0f + __expf(-z)); }

template <typename T, int TAPS>
__global__ __launch_bounds__(256) void short_conv_tile_kernel(const T* __restrict__ in, int ld, int col0, int C,
                                                              const float* __restrict__ in_bias, const float* __restrict__ w,
                                                              const float* __restrict__ bias, int act,
                                                              const float* __restrict__ history, const int* __restrict__ tok_row,
                                                              const int* __restrict__ row_first, const int* __restrict__ row_start,
                                                              const int* __restrict__ row_slots, float* __restrict__ out,
                                                              int num_tokens) {
  const int c = (blockIdx.y * 256 + threadIdx.x) * 4, t0 = blockIdx.x * CONV_TOKENS;
  if (c >= C) return;
  const int here = min(CONV_TOKENS, num_tokens - t0);
  const T* column = in + col0 + c;
  float now[CONV_TOKENS][4], wt[TAPS * 4], ib[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < CONV_TOKENS; ++i) load_vec<4>(column + (size_t)(t0 + min(i, here - 1)) * ld, now[i]);
#pragma unroll
  for (int i = 0; i < TAPS; ++i) load_vec<4>(w + (size_t)c * TAPS + 4 * i, wt + 4 * i);  // channel c + k, tap i: at k TAPS + i
  if (in_bias) load_vec<4>(in_bias + c, ib);
  if (bias) load_vec<4>(bias + c, b);
  float seen[TAPS][4];  // the last TAPS - 1 inputs, then the token's own
  int row = -1;
#pragma unroll
  for (int i = 0; i < CONV_TOKENS; ++i) {
    if (i < here) {
      const int t = t0 + i, r = tok_row[t];
      if (r != row) {  // a row's first token of this tile: what came before it in the row, or waits in the request's history
        row = r;
        const int first = row_first[r], j = t - first;
        const bool carried = row_start[r] > 0 && row_slots[r] >= 0;
        const float* old = history + (size_t)(carried ? row_slots[r] : 0) * (TAPS - 1) * C + c;
#pragma unroll
        for (int p = 0; p < TAPS - 1; ++p) {
          const int src = j - (TAPS - 1 - p);
#pragma unroll
          for (int k = 0; k < 4; ++k) seen[p][k] = 0.f;
          if (src >= 0) {
            load_vec<4>(column + (size_t)(first + src) * ld, seen[p]);
#pragma unroll
            for (int k = 0; k < 4; ++k) seen[p][k] += ib[k];
          } else if (carried) {
            load_vec<4>(old + (size_t)(TAPS - 1 + src) * C, seen[p]);
          }
        }
      }
      float v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        seen[TAPS - 1][k] = now[i][k] + ib[k];
        float acc = 0.f;
#pragma unroll
        for (int p = 0; p < TAPS; ++p) acc = fmaf(wt[k * TAPS + p], seen[p][k], acc);
        acc += b[k];
        v[k] = act == 1 ? quick_silu<T>(acc) : acc;
#pragma unroll
        for (int p = 0; p < TAPS - 1; ++p) seen[p][k] = seen[p + 1][k];
      }
      store_vec<4>(out + (size_t)t * C + c, v);
    }
  }
}

// After the convolution: the history of every row moves on by the row's tokens.
template <typename T, typename W>
__global__ void conv_history_kernel(const T* __restrict__ in, int ld, int col0, int C, const W* __restrict__ in_bias,
                                    int taps, float* __restrict__ history, const int* __restrict__ row_first,
                                    const int* __restrict__ row_len, const int* __restrict__ row_start,
                                    const int* __restrict__ row_slots) {
  const int r = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C || row_slots[r] < 0) return;
  const int first = row_first[r], len = row_len[r], keep = taps - 1;
  float* mine = history + (size_t)row_slots[r] * keep * C;
  const bool carried = row_start[r] > 0;
  const float ib = in_bias ? to_f32(in_bias[c]) : 0.f;
  float fresh[CONV_MAX_TAPS];
  for (int h = 0; h < keep; ++h) {
    const int src = len - keep + h;  // among the row's tokens; negative: among the old history
    if (src >= 0) fresh[h] = to_f32(in[(size_t)(first + src) * ld + col0 + c]) + ib;
    else fresh[h] = carried ? mine[(size_t)(keep + src) * C + c] : 0.f;
  }
  for (int h = 0; h < keep; ++h) mine[(size_t)h * C + c] = fresh[h];
}

// A decode step (every row one token: token t is row t): the convolution and the history's move in one
// kernel.  A thread owns a channel of a row, so it reads the old inputs before it writes the new ones.
template <typename T, typename W>
__global__ void short_conv_step_kernel(const T* __restrict__ in, int ld, int col0, int C, const W* __restrict__ in_bias,
                                       const W* __restrict__ w, const W* __restrict__ bias, int taps, int act,
                                       float* __restrict__ history, const int* __restrict__ row_start,
                                       const int* __restrict__ row_slots, int writes, float* __restrict__ out) {
  const int t = blockIdx.x, c = blockIdx.y * blockDim.x + threadIdx.x;
  if (c >= C) return;
  const int keep = taps - 1, slot = row_slots[t];
  const bool carried = row_start[t] > 0 && slot >= 0;
  float* mine = history + (size_t)(slot < 0 ? 0 : slot) * keep * C;
  float seen[CONV_MAX_TAPS];
  for (int i = 0; i < keep; ++i) seen[i] = carried ? mine[(size_t)i * C + c] : 0.f;
  seen[keep] = to_f32(in[(size_t)t * ld + col0 + c]) + (in_bias ? to_f32(in_bias[c]) : 0.f);
  float acc = 0.f;
  for (int i = 0; i < taps; ++i) acc = fmaf(to_f32(w[(size_t)c * taps + i]), seen[i], acc);
  if (bias) acc += to_f32(bias[c]);
  out[(size_t)t * C + c] = act == 1 ? siluf_(acc) : acc;
  if (writes && slot >= 0)
    for (int i = 0; i < keep; ++i) mine[(size_t)i * C + c] = seen[i + 1];
}

extern "C" int as_short_conv(const void* in, int dtype, int ld, int col0, int C, const void* in_bias, const void* w,
                             const void* bias, int w_dtype, int taps, int act, float* history, const int* tok_row,
                             const int* row_first, const int* row_len, const int* row_start, const int* row_slots,
                             float* out, int num_tokens, int num_rows, int writes, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (C <= 0 || taps < 1 || taps > CONV_MAX_TAPS || ld < col0 + C || num_rows <= 0) return AS_BAD_SHAPE;
  const int threads = C >= 256 ? 256 : 64;
  dim3 grid(num_tokens, (C + threads - 1) / threads), rows_grid(num_rows, (C + threads - 1) / threads);
  if (grid.y > 65535) return AS_BAD_SHAPE;
  const bool tiled = tok_row && num_tokens >= 64 && w_dtype == DT_F32 && taps >= 2 && taps <= 4 && ((C | col0 | ld) & 3) == 0;
  dim3 tiles((num_tokens + CONV_TOKENS - 1) / CONV_TOKENS, (C / 4 + 255) / 256);
#define TILE(T, TAPSV)                                                                                            \
  short_conv_tile_kernel<T, TAPSV><<<tiles, 256, 0, stream>>>((const T*)in, ld, col0, C, (const float*)in_bias, (const float*)w, \
                                                              (const float*)bias, act, history, tok_row, row_first, row_start,   \
                                                              row_slots, out, num_tokens)
#define LAUNCH(T, W)                                                                                              \
  do {                                                                                                            \
    if (!tok_row && num_rows == num_tokens) { /* every row one token */                                           \
      short_conv_step_kernel<T, W><<<grid, threads, 0, stream>>>((const T*)in, ld, col0, C, (const W*)in_bias,   \
                                                                 (const W*)w, (const W*)bias, taps, act, history, \
                                                                 row_start, row_slots, writes, out);             \
      break;                                                                                                      \
    }                                                                                                             \
    if (tiled) {                                                                                                  \
      if (taps == 2) TILE(T, 2);                                                                                  \
      else if (taps == 3) TILE(T, 3);                                                                             \
      else TILE(T, 4);                                                                                            \
    } else {                                                                                                      \
      short_conv_kernel<T, W><<<grid, threads, 0, stream>>>((const T*)in, ld, col0, C, (const W*)in_bias,        \
                                                            (const W*)w, (const W*)bias, taps, act, history,     \
                                                            tok_row, row_first, row_start, row_slots, out);      \
    }                                                                                                             \
    if (writes && taps > 1)                                                                                       \
      conv_history_kernel<T, W><<<rows_grid, threads, 0, stream>>>((const T*)in, ld, col0, C, (const W*)in_bias, \
                                                                   taps, history, row_first, row_len, row_start, \
                                                                   row_slots);                                    \
  } while (0)
  if (dtype == DT_F32 && w_dtype == DT_F32) LAUNCH(float, float);
  else if (dtype == DT_BF16 && w_dtype == DT_BF16) LAUNCH(bf16, bf16);
  else if (dtype == DT_BF16 && w_dtype == DT_F32) LAUNCH(bf16, float);
  else return AS_BAD_DTYPE;
#undef TILE
#undef LAUNCH
  return launch_status();
}

// ---- gated delta rule ----------------------------------------------------------------------------
// Before the scan, per token: the query and key heads (G of them, `dim` wide, in qkv [T, C] at columns
// 0 and G * dim) become unit vectors, x / sqrt(sum(x^2) + 1e-6), the query also times dim^(-1/2); per
// value head beta = sigmoid(b) and the decay g = exp(-exp(A_log) * softplus(a + dt_bias)), with b and a
// taken from the projection's output proj [T, ld] at columns b_off and a_off.
template <typename T, typename W>
__global__ __launch_bounds__(256) void delta_prepare_kernel(float* __restrict__ qkv, int C, int G, int dim, int H,
                                                            const T* __restrict__ proj, int ld, int b_off, int a_off,
                                                            const W* __restrict__ a_log, const W* __restrict__ dt_bias,
                                                            float* __restrict__ beta, float* __restrict__ decay) {
  // a workgroup of four waves per token and four heads (blockIdx.y), so that a decode step's few tokens are many workgroups
  const int t = blockIdx.x, lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
  float* row = qkv + (size_t)t * C;
  for (int head = blockIdx.y * waves + wave; head < 2 * G; head += gridDim.y * waves) {
    float* x = row + (size_t)head * dim;  // query heads first, then key heads
    float ss = 0.f;
    for (int d = lane; d < dim; d += WAVE) ss += x[d] * x[d];
    ss = wave_sum(ss);
    float f = 1.0f / sqrtf(ss + 1e-6f);
    if (head < G) f *= 1.0f / sqrtf((float)dim);
    for (int d = lane; d < dim; d += WAVE) x[d] *= f;
  }
  for (int h = blockIdx.y * blockDim.x + threadIdx.x; h < H; h += gridDim.y * blockDim.x) {
    const float b = to_f32(proj[(size_t)t * ld + b_off + h]), a = to_f32(proj[(size_t)t * ld + a_off + h]);
    beta[(size_t)t * H + h] = sigmoidf_(b);
    decay[(size_t)t * H + h] = expf(-expf(to_f32(a_log[h])) * softplusf_(a + to_f32(dt_bias[h])));
  }
}

// Sums over neighbouring lanes, 16, 32 or 64, in every one of them.
template <int LANES> __device__ __forceinline__ float lanes_sum(float v) {
  if constexpr (LANES == 64) return wave_sum(v);
  if constexpr (LANES == 32) v = plus_16(v);
  v += dpp<DPP_ROTATE(8)>(v);
  v += dpp<DPP_ROTATE(4)>(v);
  v += dpp<DPP_XOR_2>(v);
  return v + dpp<DPP_XOR_1>(v);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
template <typename T> struct Four;  // four neighbouring values
template <> struct Four<float> {
  static __device__ __forceinline__ f32x4 load(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
  static __device__ __forceinline__ void store(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
};
template <> struct Four<bf16> {
  typedef bf16 V __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ f32x4 load(const bf16* p) { return __builtin_convertvector(*reinterpret_cast<const V*>(p), f32x4); }
  static __device__ __forceinline__ void store(bf16* p, f32x4 v) { *reinterpret_cast<V*>(p) = __builtin_convertvector(v, V); }
};
// Whether p, and what lies `a` and `b` elements further, start on four elements of `size` bytes.
static bool on_four(const void* p, int size, long a, long b) { return ((uintptr_t)p & (4 * size - 1)) == 0 && ((a | b) & 3) == 0; }

// The same for heads of 64, 128 and 256 in rows on 16 bytes: a head is 16 to 64 lanes' work, four coordinates each, the heads of all tokens
// one after the other (1,500 tokens of 16 heads of 128, 24 MB: a token to a workgroup, one head of a wave after the other 10.5 us, now 7.3).
template <typename T, typename W, int LANES>
__global__ __launch_bounds__(256) void delta_prepare_four_kernel(float* __restrict__ qkv, int C, int G, int H, const T* __restrict__ proj,
                                                                 int ld, int b_off, int a_off, const W* __restrict__ a_log,
                                                                 const W* __restrict__ dt_bias, float* __restrict__ beta,
                                                                 float* __restrict__ decay, size_t units) {
  const size_t mine = ((size_t)blockIdx.x * 256 + threadIdx.x) / LANES, unit = mine < units ? mine : units - 1;
  const int l = threadIdx.x % LANES, head = (int)(unit % (2 * G));
  const size_t t = unit / (2 * G);
  float* x = qkv + t * C + (size_t)head * (4 * LANES) + 4 * l;
  const f32x4 v = Four<float>::load(x);
  const float ss = lanes_sum<LANES>((v[0] * v[0] + v[1] * v[1]) + (v[2] * v[2] + v[3] * v[3]));
  if (mine >= units) return;
  float f = 1.0f / sqrtf(ss + 1e-6f);
  if (head < G) f *= 1.0f / sqrtf((float)(4 * LANES));
  Four<float>::store(x, v * f);
  for (int h = head * LANES + l; h < H; h += 2 * G * LANES) {
    const float b = to_f32(proj[t * ld + b_off + h]), a = to_f32(proj[t * ld + a_off + h]);
    beta[t * H + h] = sigmoidf_(b);
    decay[t * H + h] = expf(-expf(to_f32(a_log[h])) * softplusf_(a + to_f32(dt_bias[h])));
  }
}

extern "C" int as_delta_prepare(float* qkv, int C, int G, int dim, int H, const void* proj, int dtype, int ld, int b_off,
                                int a_off, const void* a_log, const void* dt_bias, int w_dtype, float* beta,
                                float* decay, int num_tokens, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (G <= 0 || dim <= 0 || H <= 0 || C < 2 * G * dim) return AS_BAD_SHAPE;
  const int across = num_tokens >= 512 ? 1 : (2 * G + 3) / 4 > 64 ? 64 : (2 * G + 3) / 4;  // many tokens fill the GPU by themselves
  dim3 grid(num_tokens, across);
  const size_t units = (size_t)num_tokens * 2 * G, blocks = (units * (dim / 4) + 255) / 256;
  const bool four = (dim == 64 || dim == 128 || dim == 256) && on_four(qkv, 4, C, 0) && blocks <= 0x7fffffff;
#define FOUR(T, W, LANES)                                                                                          \
  delta_prepare_four_kernel<T, W, LANES><<<(int)blocks, 256, 0, stream>>>(                                         \
      qkv, C, G, H, (const T*)proj, ld, b_off, a_off, (const W*)a_log, (const W*)dt_bias, beta, decay, units)
#define LAUNCH(T, W)                                                                                               \
  if (four && dim == 64) FOUR(T, W, 16);                                                                           \
  else if (four && dim == 128) FOUR(T, W, 32);                                                                     \
  else if (four) FOUR(T, W, 64);                                                                                   \
  else delta_prepare_kernel<T, W><<<grid, 256, 0, stream>>>(qkv, C, G, dim, H, (const T*)proj, ld, b_off, a_off,        \
                                                       (const W*)a_log, (const W*)dt_bias, beta, decay)
  if (dtype == DT_F32 && w_dtype == DT_F32) { LAUNCH(float, float); }
  else if (dtype == DT_BF16 && w_dtype == DT_BF16) { LAUNCH(bf16, bf16); }
  else if (dtype == DT_BF16 && w_dtype == DT_F32) { LAUNCH(bf16, float); }
  else return AS_BAD_DTYPE;
#undef FOUR
#undef LAUNCH
  return launch_status();
}

// The scan.  Per head the state S [dim, vdim] moves on token by token:
//   S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q     (o sees the token's own write)
// The columns of S never meet, so a wave owns CJ columns of one head of one row and keeps them in
// registers for all the row's tokens: lane = column * SL + slice, a slice being RPL rows of S
// (SL = 64 / CJ slices cover dim; the slices of a column are neighbouring lanes, whose partial sums
// meet through DPP moves within a row of 16 lanes, not through LDS).  With p = S_old^T k and r = S_old^T q, both taken in one pass over the
// old state:  u = beta (v - g p),  S_new = g S_old + k u^T,  o = g r + u (k . q).
// Keys and queries of DELTA_TB tokens at a time go through LDS: a round's loads (16 bytes a lane, all asked
// for together, with the lanes' own values, betas and decays) are in flight while the round before is
// worked on, so the chain of dependent steps is the arithmetic alone.
#define DELTA_TB 8
#define DELTA_STAGE 8  // 16-byte pieces a lane brings per pass of a round's staging
template <int CTRL> __device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// The sum over SL neighbouring lanes (SL = 1, 2, 4, 8, 16), in every one of them: lane ^ 1, lane ^ 2, then
// the mirror image within eight lanes (which lies in the other four) and within sixteen (the other eight).
template <int SL> __device__ __forceinline__ float slices_sum(float v) {
  if (SL >= 2) v += dpp_move<0xB1>(v);   // quad_perm [1, 0, 3, 2]
  if (SL >= 4) v += dpp_move<0x4E>(v);   // quad_perm [2, 3, 0, 1]
  if (SL >= 8) v += dpp_move<0x141>(v);  // row_half_mirror
  if (SL >= 16) v += dpp_move<0x140>(v);  // row_mirror
  return v;
}

// MODE 0: the rule above.  MODE 1: a decay per head and key channel, chan [T, H, dim], on the rows of S:
//   S <- diag(g) S, then as above; with p = S_old^T (g k), r = S_old^T (g q): u = beta (v - p), S_new = g S_old + k u^T,
//   o = r + u (k . q).  The decays of a token go through LDS beside its key and query.
// MODE 2: a matrix memory with exponential gates: `beta` holds the logarithm of the input gate i, `decay` that of the
//   forget gate f, [T, H]; beside S the head keeps a normaliser n [dim] and a running maximum m (0 at the start):
//   m' = max(f + m, i);  S' = e^(f + m - m') S + e^(i - m') k v^T;  n' = e^(f + m - m') n + e^(i - m') k;
//   o = S'^T q / (max(|n' . q|, e^(-m')) + 1e-6).  norm_state [slots, H, dim], max_state [slots, H].
template <int RPL, int SL, int MODE>
__global__ __launch_bounds__(64) void delta_scan_kernel(const float* __restrict__ qkv, int C, int G, int dim, int H,
                                                        int vdim, const float* __restrict__ beta,
                                                        const float* __restrict__ decay,
                                                        const float* __restrict__ chan, float* __restrict__ state,
                                                        float* __restrict__ norm_state, float* __restrict__ max_state,
                                                        const int* __restrict__ row_first,
                                                        const int* __restrict__ row_len,
                                                        const int* __restrict__ row_start,
                                                        const int* __restrict__ row_slots, int writes, int most,
                                                        float* __restrict__ out) {
  constexpr int NV = MODE == 1 ? 3 : 2;  // vectors of a token that go through LDS: key, query (, decays)
  extern __shared__ __attribute__((aligned(16))) float lds[];  // [DELTA_TB][NV][dimp], dimp = SL * RPL
  const int r = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  constexpr int CJ = WAVE / SL;
  const int col = lane / SL, slice = lane % SL;
  constexpr int dimp = SL * RPL;
  const int j = blockIdx.z * CJ + col;
  const bool live = j < vdim;
  const int g = h / (H / G);
  const int first = row_first[r], len = row_len[r], slot = row_slots[r];
  if (most > 0 && len > most) return;  // the chunked form's
  const int i0 = slice * RPL;
  float S[RPL];
  float N[MODE == 2 ? RPL : 1];
  float m_run = 0.f;
  float* mine = state + ((size_t)(slot < 0 ? 0 : slot) * H + h) * dim * vdim;
  const bool carried = row_start[r] > 0 && slot >= 0;
#pragma unroll
  for (int i = 0; i < RPL; ++i) S[i] = (carried && live && i0 + i < dim) ? mine[(size_t)(i0 + i) * vdim + j] : 0.f;
  if (MODE == 2) {
    const float* n_mine = norm_state + ((size_t)(slot < 0 ? 0 : slot) * H + h) * dim;
#pragma unroll
    for (int i = 0; i < RPL; ++i) N[i] = (carried && i0 + i < dim) ? n_mine[i0 + i] : 0.f;
    m_run = carried ? max_state[(size_t)slot * H + h] : 0.f;
  }
  const int q_col = g * dim, k_col = (G + g) * dim, v_col = 2 * G * dim + h * vdim;
  // a round's keys and queries as 16-byte pieces: piece -> (token, which vector, four coordinates)
  const int quads = dimp >> 2, per_token = NV * quads, pieces = DELTA_TB * per_token;
  const int passes = (pieces + WAVE * DELTA_STAGE - 1) / (WAVE * DELTA_STAGE);
  float4 stage[DELTA_STAGE];
  float vj[DELTA_TB], bt[DELTA_TB], gt[DELTA_TB];
  const bool whole = ((dim | C) & 3) == 0;  // every key and query starts on 16 bytes
  auto fetch = [&](int t0, int pass) {
    const int nt = min(DELTA_TB, len - t0);
#pragma unroll
    for (int u = 0; u < DELTA_STAGE; ++u) {
      const int piece = (pass * DELTA_STAGE + u) * WAVE + lane;
      const int tt = piece / per_token, rest = piece - tt * per_token, which = rest / quads, i = (rest - which * quads) * 4;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (tt < nt && i < dim && piece < pieces) {
        const size_t t = (size_t)(first + t0 + tt);
        const float* src = which == 2 ? chan + (t * H + h) * dim + i : qkv + t * C + (which ? q_col : k_col) + i;
        if (whole) {
          v = *reinterpret_cast<const float4*>(src);
        } else {  // widths that are no multiples of 4: value by value
          v.x = src[0];
          if (i + 1 < dim) v.y = src[1];
          if (i + 2 < dim) v.z = src[2];
          if (i + 3 < dim) v.w = src[3];
        }
      }
      stage[u] = v;
    }
  };
  auto fetch_own = [&](int t0) {
    const int nt = min(DELTA_TB, len - t0);
#pragma unroll
    for (int tt = 0; tt < DELTA_TB; ++tt) {
      const size_t t = (size_t)first + t0 + (tt < nt ? tt : 0);
      vj[tt] = live ? qkv[t * C + v_col + j] : 0.f;
      bt[tt] = beta[t * H + h];
      gt[tt] = MODE == 1 ? 1.f : decay[t * H + h];
    }
  };
  auto put = [&](int pass) {
#pragma unroll
    for (int u = 0; u < DELTA_STAGE; ++u) {
      const int piece = (pass * DELTA_STAGE + u) * WAVE + lane;
      if (piece < pieces) *reinterpret_cast<float4*>(lds + (size_t)piece * 4) = stage[u];
    }
  };
  if (len > 0) {
    fetch(0, 0);
    fetch_own(0);
  }
  for (int t0 = 0; t0 < len; t0 += DELTA_TB) {
    const int nt = min(DELTA_TB, len - t0);
    __syncthreads();  // the round before has been read
    put(0);
    for (int pass = 1; pass < passes; ++pass) {  // heads wider than a pass brings: the rest, pass by pass
      fetch(t0, pass);
      put(pass);
    }
    float v_now[DELTA_TB], b_now[DELTA_TB], g_now[DELTA_TB];
#pragma unroll
    for (int tt = 0; tt < DELTA_TB; ++tt) { v_now[tt] = vj[tt]; b_now[tt] = bt[tt]; g_now[tt] = gt[tt]; }
    __syncthreads();
    if (t0 + DELTA_TB < len) {  // in flight while this round is worked on
      fetch(t0 + DELTA_TB, 0);
      fetch_own(t0 + DELTA_TB);
    }
#pragma unroll
    for (int tt = 0; tt < DELTA_TB; ++tt) {
      if (tt < nt) {
        // this lane's slice of the token's key and query, 16 bytes at a time (i0 is a multiple of 8)
        const float4* k4 = reinterpret_cast<const float4*>(lds + tt * NV * dimp + i0);
        const float4* q4 = reinterpret_cast<const float4*>(lds + tt * NV * dimp + dimp + i0);
        float kk[RPL], qq[RPL];
#pragma unroll
        for (int i = 0; i < RPL / 4; ++i) {
          const float4 a = k4[i], b = q4[i];
          kk[4 * i] = a.x; kk[4 * i + 1] = a.y; kk[4 * i + 2] = a.z; kk[4 * i + 3] = a.w;
          qq[4 * i] = b.x; qq[4 * i + 1] = b.y; qq[4 * i + 2] = b.z; qq[4 * i + 3] = b.w;
        }
        if (MODE == 2) {
          const float fl = g_now[tt], il = b_now[tt];
          const float m_new = fmaxf(fl + m_run, il);
          const float keep = expf(fl + m_run - m_new), take = expf(il - m_new);
          m_run = m_new;
          const float tv = take * v_now[tt];
          float num = 0.f, nq = 0.f, num2 = 0.f, nq2 = 0.f;
#pragma unroll
          for (int i = 0; i < RPL; i += 2) {
            S[i] = fmaf(kk[i], tv, keep * S[i]);
            N[i] = fmaf(kk[i], take, keep * N[i]);
            num = fmaf(S[i], qq[i], num);
            nq = fmaf(N[i], qq[i], nq);
            S[i + 1] = fmaf(kk[i + 1], tv, keep * S[i + 1]);
            N[i + 1] = fmaf(kk[i + 1], take, keep * N[i + 1]);
            num2 = fmaf(S[i + 1], qq[i + 1], num2);
            nq2 = fmaf(N[i + 1], qq[i + 1], nq2);
          }
          num = slices_sum<SL>(num + num2);
          nq = slices_sum<SL>(nq + nq2);
          if (live && slice == 0)
            out[((size_t)(first + t0 + tt) * H + h) * vdim + j] = num / (fmaxf(fabsf(nq), expf(-m_new)) + 1e-6f);
          continue;
        }
        if (MODE == 1) {  // the decays act on the rows of the old state
          const float4* g4 = reinterpret_cast<const float4*>(lds + tt * NV * dimp + 2 * dimp + i0);
#pragma unroll
          for (int i = 0; i < RPL / 4; ++i) {
            const float4 a = g4[i];
            S[4 * i] *= a.x; S[4 * i + 1] *= a.y; S[4 * i + 2] *= a.z; S[4 * i + 3] *= a.w;
          }
        }
        float p = 0.f, rr = 0.f, kq = 0.f, p2 = 0.f, rr2 = 0.f, kq2 = 0.f;  // two chains each: half the dependent steps
#pragma unroll
        for (int i = 0; i < RPL; i += 2) {
          p = fmaf(S[i], kk[i], p);
          rr = fmaf(S[i], qq[i], rr);
          kq = fmaf(kk[i], qq[i], kq);
          p2 = fmaf(S[i + 1], kk[i + 1], p2);
          rr2 = fmaf(S[i + 1], qq[i + 1], rr2);
          kq2 = fmaf(kk[i + 1], qq[i + 1], kq2);
        }
        p = slices_sum<SL>(p + p2);
        rr = slices_sum<SL>(rr + rr2);
        kq = slices_sum<SL>(kq + kq2);
        const float gg = g_now[tt];
        const float u = b_now[tt] * (v_now[tt] - gg * p);
#pragma unroll
        for (int i = 0; i < RPL; ++i) S[i] = fmaf(kk[i], u, gg * S[i]);
        if (live && slice == 0) out[((size_t)(first + t0 + tt) * H + h) * vdim + j] = fmaf(gg, rr, u * kq);
      }
    }
  }
  if (writes && live && slot >= 0) {
#pragma unroll
    for (int i = 0; i < RPL; ++i)
      if (i0 + i < dim) mine[(size_t)(i0 + i) * vdim + j] = S[i];
  }
  if (MODE == 2 && writes && slot >= 0 && blockIdx.z == 0 && col == 0) {  // every column group keeps the same n and m: one writes
    float* n_mine = norm_state + ((size_t)slot * H + h) * dim;
#pragma unroll
    for (int i = 0; i < RPL; ++i)
      if (i0 + i < dim) n_mine[i0 + i] = N[i];
    if (slice == 0) max_state[(size_t)slot * H + h] = m_run;
  }
}

template <int MODE>
static int launch_delta_scan(const float* qkv, int C, int G, int dim, int H, int vdim, const float* beta,
                             const float* decay, const float* chan, float* state, float* norm_state, float* max_state,
                             const int* row_first, const int* row_len, const int* row_start, const int* row_slots,
                             int writes, float* out, int num_rows, int force_slices, hipStream_t stream, int most = 0) {
  if (num_rows <= 0) return AS_OK;
  if (G <= 0 || H <= 0 || H % G || dim <= 0 || vdim <= 0 || C < 2 * G * dim + H * vdim || H > 65535)
    return AS_BAD_SHAPE;
  if (dim > 16 * 64) return AS_BAD_SHAPE;  // sixteen slices of 64 rows
  int slices = 1;
  while ((dim + slices - 1) / slices > 64) slices *= 2;  // a lane keeps at most 64 rows of its column
  if (MODE == 2)  // the normaliser's rows lie beside the state's: half as many to a lane
    while ((dim + slices - 1) / slices > 32) slices *= 2;
  // few rows and heads: narrower column groups (more slices of fewer rows) until the waves fill the GPU
  while (slices < 16 && (dim + 2 * slices - 1) / (2 * slices) >= 8 &&
         (long)num_rows * H * ((vdim + WAVE / slices - 1) / (WAVE / slices)) < 8L * compute_units())
    slices *= 2;
  if (force_slices > 0) {  // measurements and tests: 1, 2, 4, 8 or 16 slices, if a lane's share then fits
    if ((force_slices & (force_slices - 1)) || force_slices > 16 || (dim + force_slices - 1) / force_slices > 64)
      return AS_BAD_SHAPE;
    slices = force_slices;
  }
  if (slices > 16) return AS_BAD_SHAPE;
  const int rows_per_lane = (dim + slices - 1) / slices;
  const int RPL = rows_per_lane <= 8 ? 8 : rows_per_lane <= 16 ? 16 : rows_per_lane <= 32 ? 32 : 64;
  const int CJ = WAVE / slices;
  dim3 grid(num_rows, H, (vdim + CJ - 1) / CJ);
  const size_t lds = (size_t)DELTA_TB * (MODE == 1 ? 3 : 2) * slices * RPL * sizeof(float);
  if (lds > 64 * 1024) return AS_BAD_SHAPE;
#define LAUNCH(R, SLV)                                                                                            \
  delta_scan_kernel<R, SLV, MODE><<<grid, 64, lds, stream>>>(qkv, C, G, dim, H, vdim, beta, decay, chan, state,   \
                                                             norm_state, max_state, row_first, row_len, row_start, \
                                                             row_slots, writes, most, out)
#define LAUNCH_SL(R)              \
  do {                            \
    if (slices == 1) LAUNCH(R, 1);      \
    else if (slices == 2) LAUNCH(R, 2); \
    else if (slices == 4) LAUNCH(R, 4); \
    else if (slices == 8) LAUNCH(R, 8); \
    else LAUNCH(R, 16);                 \
  } while (0)
  if (RPL == 8) LAUNCH_SL(8);
  else if (RPL == 16) LAUNCH_SL(16);
  else if (RPL == 32) LAUNCH_SL(32);
  else LAUNCH_SL(64);
#undef LAUNCH_SL
#undef LAUNCH
  return launch_status();
}

// most > 0: rows of more tokens are left out (`as_delta_chunks` takes them).
extern "C" int as_delta_scan(const float* qkv, int C, int G, int dim, int H, int vdim, const float* beta,
                             const float* decay, float* state, const int* row_first, const int* row_len,
                             const int* row_start, const int* row_slots, int writes, float* out, int num_rows,
                             int force_slices, int most, hipStream_t stream) {
  return launch_delta_scan<0>(qkv, C, G, dim, H, vdim, beta, decay, nullptr, state, nullptr, nullptr, row_first, row_len,
                              row_start, row_slots, writes, out, num_rows, force_slices, stream, most);
}

// The rule in chunks of 64 tokens (long rows).  With D[t, j] = g_{j+1} .. g_t, P_t = g_1 .. g_t within the chunk and S the state
// before it, the updates of a chunk solve a triangular system:
//   u_t = beta_t (v_t - P_t S^T k_t - sum_{j<t} D[t, j] (k_t . k_j) u_j),  so  U = (I + A)^-1 diag(beta) (V - P K S)
// with A[t, j] = beta_t D[t, j] k_t . k_j below the diagonal;
//   o_t = P_t S^T q_t + sum_{j<=t} D[t, j] (q_t . k_j) u_j,   S <- P_64 S + sum_j D[64, j] k_j u_j^T.
// delta_pairs (a workgroup a chunk and head, all side by side) makes (I + A)^-1 diag(beta) and D (Q K^T); delta_chunks (a
// workgroup a row, head and 16 columns of the state) walks the chunks.  All of it in 32 bits: products by
// v_mfma_f32_16x16x4_f32, the decays by multiplication in the order of the scan (no logarithms, so none is lost to a
// strong decay before a weak one).  A chunk whose updates u are not all finite (a number that is not came in, or one grew beyond
// 32 bits), or that has a query that is not, is walked token by token by one wave instead, as the scan does, from the state before
// it: 0 times such a number is NaN, and in the matrix form it would reach the tokens before it, where the scan keeps a query's
// to its own token and a value's to its column of the state.
// Bound by the chain of a chunk (128 matrix instructions of a workgroup's last wave, which take 1.9 us, and three barriers: 4.1 us a
// chunk) and by the fill of the GPU (rows x heads x column groups workgroups).  One prompt of 1,500 tokens, 16 heads of 128 x 128:
// 25 + 98 us; token by token (0.4 us a token, the scan above) 619; with every chunk walked by token (its values NaN from the first
// on) 1,360.  The triangle inverted by one wave, a column to a lane from the top down, took the first kernel 33 us.  The state
// before a chunk stays in LDS for that walk: kept in registers, heads of 128 exceed what two workgroups on a compute unit leave.
typedef float floatx4 __attribute__((ext_vector_type(4)));
#define DC 64                            // tokens of a chunk
#define DC_SCRATCH (2 * DC * DC + 3 * DC)  // floats per chunk and head: the inverse, the pairs, P, D[64, :], whether a query is not finite

__device__ __forceinline__ int delta_chunks_of(int len, int most) { return len > most ? (len + DC - 1) / DC : 0; }
__device__ __forceinline__ bool finite4(floatx4 v) {
  const float s = (v[0] - v[0]) + (v[1] - v[1]) + (v[2] - v[2]) + (v[3] - v[3]);  // 0, or NaN if one is not finite
  return s == 0.f;
}

template <int DT>
__global__ __launch_bounds__(256) void delta_pairs_kernel(const float* __restrict__ qkv, int C, int G, int H, int vdim,
                                                          const float* __restrict__ beta, const float* __restrict__ decay,
                                                          const int* __restrict__ row_first, const int* __restrict__ row_len,
                                                          int num_rows, int most, float* __restrict__ scratch) {
  constexpr int dim = 16 * DT, LA = DC + 4, LDD = DC + 1;
  __shared__ __attribute__((aligned(16))) float A[DC * LA];
  __shared__ float D[DC * LDD];
  __shared__ __attribute__((aligned(16))) float sg[DC], sb[DC];
  __shared__ floatx4 inv[4][4][64];
  __shared__ __attribute__((aligned(16))) float rows[4][16 * 20];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4, h = blockIdx.y, g = h / (H / G);
  int chunk = blockIdx.x, r = 0;
  for (; r < num_rows; ++r) {
    const int n = delta_chunks_of(row_len[r], most);
    if (chunk < n) break;
    chunk -= n;
  }
  if (r == num_rows) return;
  const int first = row_first[r] + chunk * DC, n = min(DC, row_len[r] - chunk * DC);
  float* mine = scratch + ((size_t)blockIdx.x * H + h) * DC_SCRATCH;
  const int q_col = g * dim, k_col = (G + g) * dim, v_col = 2 * G * dim + h * vdim;
  auto row_of = [&](int tile, int col) { return qkv + (size_t)(first + min(tile * 16 + lr, n - 1)) * C + col + lg * 4; };
  floatx4 q[DT], kk[4][DT];  // this wave's 16 queries, and the keys of every token up to its own: all asked for at once
  {
    const float* qp = row_of(wave, q_col);
#pragma unroll
    for (int j = 3; j >= 0; --j) {
      if (j <= wave) {
        const float* kp = row_of(j, k_col);
#pragma unroll
        for (int i = 0; i < DT; ++i) kk[j][i] = *reinterpret_cast<const floatx4*>(kp + i * 16);
      }
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) q[i] = *reinterpret_cast<const floatx4*>(qp + i * 16);
    if (tid < DC) {
      const size_t at = (size_t)(first + min(tid, n - 1)) * H + h;
      sg[tid] = tid < n ? decay[at] : 1.f;
      sb[tid] = tid < n ? beta[at] : 0.f;
    }
  }
  bool finite = true;
#pragma unroll
  for (int i = 0; i < DT; ++i) finite = finite && finite4(q[i]);
  const int by_token = __syncthreads_or(!finite);
  {  // column `lane` of D: this wave keeps its 16 rows
    float cur = 0.f;
    for (int t4 = 0; t4 < DC; t4 += 16) {
#pragma unroll
      for (int i = 0; i < 16; i += 4) {
        const floatx4 gg = *reinterpret_cast<const floatx4*>(sg + t4 + i);
#pragma unroll
        for (int x = 0; x < 4; ++x) {
          cur = t4 + i + x == lane ? 1.f : cur * gg[x];  // 0 above the diagonal
          if (t4 >> 4 == wave) D[(t4 + i + x) * LDD + lane] = cur;
        }
      }
    }
  }
  __syncthreads();
  floatx4 own[DT];  // the keys of this wave's own tokens
#pragma unroll
  for (int i = 0; i < DT; ++i) own[i] = wave == 0 ? kk[0][i] : wave == 1 ? kk[1][i] : wave == 2 ? kk[2][i] : kk[3][i];
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {
    if (jt <= wave) {
      floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(own[i][x], kk[jt][i][x], acc, 0, 0, 0);
      const int j = jt * 16 + lr;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int t = wave * 16 + lg * 4 + x;
        A[t * LA + j] = j < t ? sb[t] * D[t * LDD + j] * acc[x] : 0.f;
      }
    }
  }
  // The inverse in blocks of 16: a wave inverts its block on the diagonal, column by column from the top down, then the
  // blocks below, one diagonal after the other: T_ij = -T_ii sum_k A_ik T_kj.  A block lies as a product leaves it (lane:
  // column lr, rows 4 lg + x), which is how the next product takes it as its right operand.
  // A wave reads what its own lanes have written: LDS answers a wave in order, and the fences keep the compiler from
  // moving the reads before the writes (a lane's own addresses differ, so nothing else would).
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  floatx4 diag, left;  // T_ww as a right and as a left operand
  {
    const float* block = A + (wave * 16) * LA + wave * 16;
    float x[16];
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      float v = t == lr ? 1.f : 0.f;
#pragma unroll
      for (int i = 0; i < t; i += 4) {
        const floatx4 row = *reinterpret_cast<const floatx4*>(block + t * LA + i);
#pragma unroll
        for (int y = 0; y < 4; ++y)
          if (i + y < t) v = fmaf(-row[y], x[i + y], v);
      }
      x[t] = v;
    }
#pragma unroll
    for (int y = 0; y < 4; ++y) diag[y] = lg == 0 ? x[y] : lg == 1 ? x[4 + y] : lg == 2 ? x[8 + y] : x[12 + y];
    if (lg == 0) {
#pragma unroll
      for (int t = 0; t < 16; ++t) rows[wave][t * 20 + lr] = x[t];
    }
    inv[wave][wave][lane] = diag;
  }
  __syncthreads();
  left = *reinterpret_cast<const floatx4*>(rows[wave] + lr * 20 + lg * 4);
#pragma unroll
  for (int d = 1; d < 4; ++d) {
    if (wave >= d) {
      const int j = wave - d;
      floatx4 m = floatx4{0.f, 0.f, 0.f, 0.f}, t = m;
      for (int k = j; k < wave; ++k) {
        const floatx4 l = *reinterpret_cast<const floatx4*>(A + (wave * 16 + lr) * LA + k * 16 + lg * 4), r = inv[k][j][lane];
#pragma unroll
        for (int x = 0; x < 4; ++x) m = __builtin_amdgcn_mfma_f32_16x16x4f32(l[x], r[x], m, 0, 0, 0);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) t = __builtin_amdgcn_mfma_f32_16x16x4f32(-left[x], m[x], t, 0, 0, 0);
      inv[wave][j][lane] = t;
    }
    __syncthreads();
  }
  for (int j = 0; j <= wave; ++j) {
    const floatx4 t = inv[wave][j][lane];
    const float bj = sb[j * 16 + lr];
#pragma unroll
    for (int x = 0; x < 4; ++x) mine[(wave * 16 + lg * 4 + x) * DC + j * 16 + lr] = t[x] * bj;
  }
#pragma unroll
  for (int jt = 0; jt < 4; ++jt) {  // queries and keys
    if (jt <= wave) {
      floatx4 acc = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < DT; ++i)
#pragma unroll
        for (int x = 0; x < 4; ++x) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(q[i][x], kk[jt][i][x], acc, 0, 0, 0);
      const int j = jt * 16 + lr;
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int t = wave * 16 + lg * 4 + x;
        mine[DC * DC + t * DC + j] = j <= t ? D[t * LDD + j] * acc[x] : 0.f;
      }
    }
  }
  if (wave == 0) {
    mine[2 * DC * DC + lane] = D[lane * LDD] * sg[0];
    mine[2 * DC * DC + DC + lane] = D[(DC - 1) * LDD + lane];
    if (lane == 0) reinterpret_cast<int*>(mine)[2 * DC * DC + 2 * DC] = by_token;
  }
}

template <int DT>
__global__ __launch_bounds__(256) void delta_chunks_kernel(const float* __restrict__ qkv, int C, int G, int H, int vdim,
                                                           const float* __restrict__ beta, const float* __restrict__ decay,
                                                           float* __restrict__ state, const int* __restrict__ row_first,
                                                           const int* __restrict__ row_len, const int* __restrict__ row_start,
                                                           const int* __restrict__ row_slots, int writes, int most,
                                                           const float* __restrict__ scratch, int per_xcd, int total,
                                                           float* __restrict__ out) {
  constexpr int dim = 16 * DT, LK = dim + 4;
  __shared__ __attribute__((aligned(16))) float keys[DC * LK];
  __shared__ floatx4 sy[4 * 64], su[4 * 64], se[4 * 64], ss[2][DT * 64];  // ss: the states before and after a chunk
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lr = lane & 15, lg = lane >> 4;
  // a head's column groups side by side on one XCD (workgroups are dealt to the eight in turn): they read the same
  const int item = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
  if (item >= total) return;
  const int groups = vdim / 16, c0 = item % groups * 16, h = item / groups % H, r = item / groups / H, g = h / (H / G);
  const int len = row_len[r], chunks = delta_chunks_of(len, most);
  if (chunks == 0) return;
  int before = 0;
  for (int i = 0; i < r; ++i) before += delta_chunks_of(row_len[i], most);
  const int first = row_first[r], slot = row_slots[r];
  const bool carried = row_start[r] > 0 && slot >= 0;
  float* kept = state + ((size_t)(slot < 0 ? 0 : slot) * H + h) * dim * vdim + c0 + lr;
  const int q_col = g * dim, k_col = (G + g) * dim, v_col = 2 * G * dim + h * vdim + c0 + lr;

  // S: tile i holds rows 16 i + 4 lg + x of column c0 + lr, the layout of a product's result, which is also what a product
  // takes as its right operand when the left one brings its four columns 16 i + 4 lg + x the same way
  floatx4 S[DT], kf[DT], qf[DT], tf[4], pf[4], vv, P, E;
#pragma unroll
  for (int i = 0; i < DT; ++i) {
#pragma unroll
    for (int x = 0; x < 4; ++x) S[i][x] = carried ? kept[(size_t)(16 * i + 4 * lg + x) * vdim] : 0.f;
    if (wave == 0) ss[0][i * 64 + lane] = S[i];
  }
  int by_token = 0;
  float last_P = 1.f;
  auto token = [&](int n, int t) { return qkv + (size_t)(first + min(n * DC + t, len - 1)) * C; };
  auto load_rows = [&](int n) {
    const float* p = token(n, wave * 16 + lr) + lg * 4;
#pragma unroll
    for (int i = 0; i < DT; ++i) kf[i] = *reinterpret_cast<const floatx4*>(p + k_col + i * 16);
#pragma unroll
    for (int i = 0; i < DT; ++i) qf[i] = *reinterpret_cast<const floatx4*>(p + q_col + i * 16);
  };
  auto load_rest = [&](int n) {
    const float* mine = scratch + ((size_t)(before + n) * H + h) * DC_SCRATCH;
    const float* p = mine + (wave * 16 + lr) * DC + lg * 4;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j <= wave) {
        tf[j] = *reinterpret_cast<const floatx4*>(p + j * 16);
        pf[j] = *reinterpret_cast<const floatx4*>(p + DC * DC + j * 16);
      }
    }
#pragma unroll
    for (int x = 0; x < 4; ++x) vv[x] = token(n, wave * 16 + lg * 4 + x)[v_col];
    P = *reinterpret_cast<const floatx4*>(mine + 2 * DC * DC + wave * 16 + lg * 4);
    E = *reinterpret_cast<const floatx4*>(mine + 2 * DC * DC + DC + wave * 16 + lg * 4);
    last_P = mine[2 * DC * DC + DC - 1];
    by_token = reinterpret_cast<const int*>(mine)[2 * DC * DC + 2 * DC];
  };
  load_rows(0);
  load_rest(0);
  for (int n = 0; n < chunks; ++n) {
    floatx4 *const old = ss[n & 1], *const now = ss[(n + 1) & 1];
#pragma unroll
    for (int i = 0; i < DT; ++i) *reinterpret_cast<floatx4*>(keys + (wave * 16 + lr) * LK + i * 16 + lg * 4) = kf[i];
    floatx4 xk = floatx4{0.f, 0.f, 0.f, 0.f}, xq = xk;
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        xk = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][x], S[i][x], xk, 0, 0, 0);
        xq = __builtin_amdgcn_mfma_f32_16x16x4f32(qf[i][x], S[i][x], xq, 0, 0, 0);
      }
    const int ahead = min(n + 1, chunks - 1);
    load_rows(ahead);
    const floatx4 y = vv - P * xk;
    sy[wave * 64 + lane] = y;
    __syncthreads();
    floatx4 u = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j <= wave) {
        const floatx4 yj = sy[j * 64 + lane];
#pragma unroll
        for (int x = 0; x < 4; ++x) u = __builtin_amdgcn_mfma_f32_16x16x4f32(tf[j][x], yj[x], u, 0, 0, 0);
      }
    }
    su[wave * 64 + lane] = u;
    se[wave * 64 + lane] = u * E;
    __syncthreads();
    floatx4 o = P * xq;
    // the state first (the next chunk waits for it), then the outputs
    floatx4 next[DT / 4];
    bool finite = true;
#pragma unroll
    for (int m = 0; m < DT / 4; ++m) {
      const int i = wave * (DT / 4) + m;
      next[m] = old[i * 64 + lane] * last_P;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const floatx4 uj = se[j * 64 + lane];
        if (m == 0) finite = finite && finite4(uj);
#pragma unroll
        for (int x = 0; x < 4; ++x)
          next[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(keys[(j * 16 + lg * 4 + x) * LK + i * 16 + lr], uj[x], next[m], 0, 0, 0);
      }
      now[i * 64 + lane] = next[m];
    }
    const bool lost = by_token || __any(!finite);  // the same in all four waves: each has looked at every update
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      if (j <= wave) {
        const floatx4 uj = su[j * 64 + lane];
#pragma unroll
        for (int x = 0; x < 4; ++x) o = __builtin_amdgcn_mfma_f32_16x16x4f32(pf[j][x], uj[x], o, 0, 0, 0);
      }
    }
    load_rest(ahead);  // before the stores: who waits for it does not wait for them
#pragma unroll
    for (int x = 0; x < 4; ++x) {
      const int t = wave * 16 + lg * 4 + x;
      if (!lost && n * DC + t < len) out[((size_t)(first + n * DC + t) * H + h) * vdim + c0 + lr] = o[x];
    }
    __syncthreads();
    if (lost) {
      if (wave == 0) {
#pragma unroll
        for (int i = 0; i < DT; ++i) S[i] = old[i * 64 + lane];
        for (int t = 0; t < min(DC, len - n * DC); ++t) {
          const size_t at = (size_t)(first + n * DC + t) * H + h;
          const float* row = qkv + (size_t)(first + n * DC + t) * C;
          const float g_now = decay[at], b_now = beta[at], v_now = row[v_col];
          float p = 0.f, r = 0.f, kq = 0.f;
#pragma unroll
          for (int i = 0; i < DT; ++i) {
            const floatx4 k = *reinterpret_cast<const floatx4*>(keys + t * LK + i * 16 + lg * 4);
            const floatx4 q = *reinterpret_cast<const floatx4*>(row + q_col + i * 16 + lg * 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              p = fmaf(S[i][x], k[x], p);
              r = fmaf(S[i][x], q[x], r);
              kq = fmaf(k[x], q[x], kq);
            }
          }
          p += __shfl_xor(p, 16, WAVE);
          r += __shfl_xor(r, 16, WAVE);
          kq += __shfl_xor(kq, 16, WAVE);
          p += __shfl_xor(p, 32, WAVE);
          r += __shfl_xor(r, 32, WAVE);
          kq += __shfl_xor(kq, 32, WAVE);
          const float u_now = b_now * (v_now - g_now * p);
#pragma unroll
          for (int i = 0; i < DT; ++i) {
            const floatx4 k = *reinterpret_cast<const floatx4*>(keys + t * LK + i * 16 + lg * 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) S[i][x] = fmaf(k[x], u_now, g_now * S[i][x]);
          }
          if (lg == 0) out[at * vdim + c0 + lr] = fmaf(g_now, r, u_now * kq);
        }
#pragma unroll
        for (int i = 0; i < DT; ++i) now[i * 64 + lane] = S[i];
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < DT; ++i) S[i] = now[i * 64 + lane];
  }
  if (writes && slot >= 0 && wave == 0) {
#pragma unroll
    for (int i = 0; i < DT; ++i)
#pragma unroll
      for (int x = 0; x < 4; ++x) kept[(size_t)(16 * i + 4 * lg + x) * vdim] = S[i][x];
  }
}

// Rows of more than `most` tokens.  Heads of 64 or 128 keys, values in whole tiles of 16, every key, query and value on 16
// bytes.  scratch: most_chunks x H x (2 x 64 x 64 + 3 x 64) floats, most_chunks at least the chunks of 64 tokens that these rows have.
extern "C" int as_delta_chunks(const float* qkv, int C, int G, int dim, int H, int vdim, const float* beta, const float* decay,
                               float* state, const int* row_first, const int* row_len, const int* row_start,
                               const int* row_slots, int writes, float* out, int num_rows, int most, float* scratch,
                               int most_chunks, hipStream_t stream) {
  if (num_rows <= 0 || most_chunks <= 0) return AS_OK;
  if (G <= 0 || H <= 0 || H % G || H > 65535 || (dim != 64 && dim != 128) || vdim <= 0 || vdim % 16 || C % 4 || most < 0 ||
      C < 2 * G * dim + H * vdim || ((uintptr_t)qkv & 15) || ((uintptr_t)scratch & 15) || !scratch)
    return AS_BAD_SHAPE;
  const long total = (long)num_rows * H * (vdim / 16);
  if (total > 0x3fffffff) return AS_BAD_SHAPE;
  const int per_xcd = (int)((total + 7) / 8);
#define LAUNCH(DT)                                                                                                             \
  do {                                                                                                                         \
    delta_pairs_kernel<DT><<<dim3(most_chunks, H), 256, 0, stream>>>(qkv, C, G, H, vdim, beta, decay, row_first, row_len,      \
                                                                     num_rows, most, scratch);                                 \
    delta_chunks_kernel<DT><<<per_xcd * 8, 256, 0, stream>>>(qkv, C, G, H, vdim, beta, decay, state, row_first, row_len, row_start,         \
                                                             row_slots, writes, most, scratch, per_xcd, (int)total, out);      \
  } while (0)
  if (dim == 64) LAUNCH(4);
  else LAUNCH(8);
#undef LAUNCH
  return launch_status();
}

// The same rule with a decay per head and key channel: chan [T, H, dim].
extern "C" int as_delta_scan_channels(const float* qkv, int C, int G, int dim, int H, int vdim, const float* beta,
                                      const float* chan, float* state, const int* row_first, const int* row_len,
                                      const int* row_start, const int* row_slots, int writes, float* out,
                                      int num_rows, int force_slices, hipStream_t stream) {
  if (!chan) return AS_BAD_SHAPE;
  return launch_delta_scan<1>(qkv, C, G, dim, H, vdim, beta, nullptr, chan, state, nullptr, nullptr, row_first, row_len,
                              row_start, row_slots, writes, out, num_rows, force_slices, stream);
}

// The matrix memory: qkv [T, C] holds H query heads (already times dim^(-1/2)), H key heads and H value heads.
extern "C" int as_memory_scan(const float* qkv, int C, int dim, int H, int vdim, const float* i_log, const float* f_log,
                              float* state, float* norm_state, float* max_state, const int* row_first,
                              const int* row_len, const int* row_start, const int* row_slots, int writes, float* out,
                              int num_rows, int force_slices, hipStream_t stream) {
  if (!norm_state || !max_state) return AS_BAD_SHAPE;
  return launch_delta_scan<2>(qkv, C, H, dim, H, vdim, i_log, f_log, nullptr, state, norm_state, max_state, row_first,
                              row_len, row_start, row_slots, writes, out, num_rows, force_slices, stream);
}

// After the scan: every head's output over its root mean square (over vdim, eps inside the root), times
// a weight (w [vdim] shared by the heads with w_stride 0, w [H, vdim] with w_stride vdim), times silu (gate_act 0)
// or sigmoid (1) of a gate projection's output (gate [T, ld] at g_off, laid out heads x vdim), times scale: the
// input of the output projection, act [T, ld_out] from column out_off on.
template <typename T, typename W>
__global__ __launch_bounds__(64) void delta_finish_kernel(const float* __restrict__ o, int H, int vdim,
                                                          const W* __restrict__ w, int w_stride, float eps,
                                                          const T* __restrict__ gate, int ld, int g_off, int gate_act,
                                                          float scale, T* __restrict__ act, int ld_out, int out_off) {
  const int t = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const float* x = o + ((size_t)t * H + h) * vdim;
  float ss = 0.f;
  for (int d = lane; d < vdim; d += WAVE) ss += x[d] * x[d];
  ss = wave_sum(ss);
  const float inv = scale / sqrtf(ss / (float)vdim + eps);
  for (int d = lane; d < vdim; d += WAVE) {
    const float z = to_f32(gate[(size_t)t * ld + g_off + h * vdim + d]);
    const float gv = gate_act == 1 ? sigmoidf_(z) : siluf_(z);
    act[(size_t)t * ld_out + out_off + h * vdim + d] = from_f32<T>(x[d] * inv * to_f32(w[(size_t)h * w_stride + d]) * gv);
  }
}

// The same for heads of 64, 128 and 256 on pieces of four values, as in delta_prepare (1,500 tokens of 16 heads of 128, 24 MB: a workgroup of
// 64 threads a head 10.5 us, now 7.6).
template <typename T, typename W, int LANES>
__global__ __launch_bounds__(256) void delta_finish_four_kernel(const float* __restrict__ o, int H, const W* __restrict__ w, int w_stride,
                                                                float eps, const T* __restrict__ gate, int ld, int g_off, int gate_act,
                                                                float scale, T* __restrict__ act, int ld_out, int out_off, size_t units) {
  const size_t mine = ((size_t)blockIdx.x * 256 + threadIdx.x) / LANES, unit = mine < units ? mine : units - 1;
  const int d = 4 * (threadIdx.x % LANES), h = (int)(unit % H);
  const size_t t = unit / H;
  const f32x4 x = Four<float>::load(o + unit * (4 * LANES) + d), z = Four<T>::load(gate + t * ld + g_off + (size_t)h * (4 * LANES) + d),
              g = Four<W>::load(w + (size_t)h * w_stride + d);
  const float ss = lanes_sum<LANES>((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]));
  const float inv = scale / sqrtf(ss / (float)(4 * LANES) + eps);
  f32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = x[i] * inv * g[i] * (gate_act == 1 ? sigmoidf_(z[i]) : siluf_(z[i]));
  if (mine < units) Four<T>::store(act + t * ld_out + out_off + (size_t)h * (4 * LANES) + d, r);
}

extern "C" int as_delta_finish(const float* o, int H, int vdim, const void* w, int w_dtype, int w_per_head, float eps,
                               const void* gate, int dtype, int ld, int g_off, int gate_act, float scale, void* act,
                               int ld_out, int out_off, int num_tokens, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (H <= 0 || H > 65535 || vdim <= 0 || gate_act < 0 || gate_act > 1 || ld < g_off + H * vdim ||
      ld_out < out_off + H * vdim)
    return AS_BAD_SHAPE;
  dim3 grid(num_tokens, H);
  const int w_stride = w_per_head ? vdim : 0, size = dtype == DT_F32 ? 4 : 2;
  const size_t units = (size_t)num_tokens * H, blocks = (units * (vdim / 4) + 255) / 256;
  const bool four = (vdim == 64 || vdim == 128 || vdim == 256) && on_four(o, 4, 0, 0) && on_four(gate, size, ld, g_off) &&
                    on_four(act, size, ld_out, out_off) && on_four(w, w_dtype == DT_F32 ? 4 : 2, 0, 0) && blocks <= 0x7fffffff;
#define FOUR(T, W, LANES)                                                                                          \
  delta_finish_four_kernel<T, W, LANES><<<(int)blocks, 256, 0, stream>>>(                                          \
      o, H, (const W*)w, w_stride, eps, (const T*)gate, ld, g_off, gate_act, scale, (T*)act, ld_out, out_off, units)
#define LAUNCH(T, W)                                                                                               \
  if (four && vdim == 64) FOUR(T, W, 16);                                                                          \
  else if (four && vdim == 128) FOUR(T, W, 32);                                                                    \
  else if (four) FOUR(T, W, 64);                                                                                   \
  else delta_finish_kernel<T, W><<<grid, 64, 0, stream>>>((const float*)o, H, vdim, (const W*)w, w_stride, eps,     \
                                                          (const T*)gate, ld, g_off, gate_act, scale, (T*)act,     \
                                                          ld_out, out_off)
  if (dtype == DT_F32 && w_dtype == DT_F32) { LAUNCH(float, float); }
  else if (dtype == DT_BF16 && w_dtype == DT_BF16) { LAUNCH(bf16, bf16); }
  else if (dtype == DT_BF16 && w_dtype == DT_F32) { LAUNCH(bf16, float); }
  else return AS_BAD_DTYPE;
#undef FOUR
#undef LAUNCH
  return launch_status();
}

// Before the scan with a decay per channel: unit vectors as in delta_prepare; beta = sigmoid(proj[t, b_off + h]);
// chan[t, h, d] = exp(-exp(a_log[h]) * softplus(steps[t, a_off + h * dim + d] + dt_bias[h * dim + d])), `steps` being
// the output of the step sizes' second projection, [T, ld_s].  a_log and dt_bias fp32.
template <typename T>
__global__ __launch_bounds__(256) void delta_prepare_channels_kernel(float* __restrict__ qkv, int C, int G, int dim, int H,
                                                                     const T* __restrict__ proj, int ld, int b_off,
                                                                     const T* __restrict__ steps, int ld_s, int a_off,
                                                                     const float* __restrict__ a_log,
                                                                     const float* __restrict__ dt_bias,
                                                                     float* __restrict__ beta, float* __restrict__ chan) {
  const int t = blockIdx.x, lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, waves = blockDim.x / WAVE;
  float* row = qkv + (size_t)t * C;
  for (int head = blockIdx.y * waves + wave; head < 2 * G; head += gridDim.y * waves) {
    float* x = row + (size_t)head * dim;  // query heads first, then key heads
    float ss = 0.f;
    for (int d = lane; d < dim; d += WAVE) ss += x[d] * x[d];
    ss = wave_sum(ss);
    float f = 1.0f / sqrtf(ss + 1e-6f);
    if (head < G) f *= 1.0f / sqrtf((float)dim);
    for (int d = lane; d < dim; d += WAVE) x[d] *= f;
  }
  for (int h = blockIdx.y * blockDim.x + threadIdx.x; h < H; h += gridDim.y * blockDim.x)
    beta[(size_t)t * H + h] = sigmoidf_(to_f32(proj[(size_t)t * ld + b_off + h]));
  const int HD = H * dim;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < HD; c += gridDim.y * blockDim.x) {
    const float a = to_f32(steps[(size_t)t * ld_s + a_off + c]);
    chan[(size_t)t * HD + c] = expf(-expf(a_log[c / dim]) * softplusf_(a + dt_bias[c]));
  }
}

extern "C" int as_delta_prepare_channels(float* qkv, int C, int G, int dim, int H, const void* proj, int dtype, int ld,
                                         int b_off, const void* steps, int ld_s, int a_off, const float* a_log,
                                         const float* dt_bias, float* beta, float* chan, int num_tokens,
                                         hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (G <= 0 || dim <= 0 || H <= 0 || C < 2 * G * dim || ld < b_off + H || ld_s < a_off + H * dim) return AS_BAD_SHAPE;
  int across = num_tokens >= 512 ? 1 : (H * dim + 255) / 256;
  if (across > 64) across = 64;
  dim3 grid(num_tokens, across);
  if (dtype == DT_F32)
    delta_prepare_channels_kernel<float><<<grid, 256, 0, stream>>>(qkv, C, G, dim, H, (const float*)proj, ld, b_off,
                                                                   (const float*)steps, ld_s, a_off, a_log, dt_bias,
                                                                   beta, chan);
  else if (dtype == DT_BF16)
    delta_prepare_channels_kernel<bf16><<<grid, 256, 0, stream>>>(qkv, C, G, dim, H, (const bf16*)proj, ld, b_off,
                                                                  (const bf16*)steps, ld_s, a_off, a_log, dt_bias, beta,
                                                                  chan);
  else return AS_BAD_DTYPE;
  return launch_status();
}

// Before the scan of a matrix memory: proj [T, ld] holds H query heads at q_off, H key heads at k_off (`dim` wide) and
// H value heads at v_off (`vdim` wide), and the gates' logits at i_off and f_off [H].  qkv fp32 [T, 2 H dim + H vdim]
// receives the queries times dim^(-1/2), the keys and the values; i_log = cap tanh((z_i + b_i) / cap), f_log =
// logsigmoid(cap tanh((z_f + b_f) / cap)), both [T, H]; biases fp32 [H].
__device__ __forceinline__ float log_sigmoidf_(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

template <typename T>
__global__ __launch_bounds__(256) void memory_prepare_kernel(const T* __restrict__ proj, int ld, int q_off, int k_off,
                                                             int v_off, int i_off, int f_off, int H, int dim, int vdim,
                                                             const float* __restrict__ i_bias,
                                                             const float* __restrict__ f_bias, float cap,
                                                             float* __restrict__ qkv, float* __restrict__ i_log,
                                                             float* __restrict__ f_log) {
  const int t = blockIdx.x;
  const T* row = proj + (size_t)t * ld;
  const int HD = H * dim, C = 2 * HD + H * vdim;
  const float qs = 1.0f / sqrtf((float)dim);
  float* dst = qkv + (size_t)t * C;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < C; c += gridDim.y * blockDim.x) {
    float v;
    if (c < HD) v = to_f32(row[q_off + c]) * qs;
    else if (c < 2 * HD) v = to_f32(row[k_off + c - HD]);
    else v = to_f32(row[v_off + c - 2 * HD]);
    dst[c] = v;
  }
  for (int h = blockIdx.y * blockDim.x + threadIdx.x; h < H; h += gridDim.y * blockDim.x) {
    const float zi = to_f32(row[i_off + h]) + i_bias[h], zf = to_f32(row[f_off + h]) + f_bias[h];
    i_log[(size_t)t * H + h] = cap * tanhf(zi / cap);
    f_log[(size_t)t * H + h] = log_sigmoidf_(cap * tanhf(zf / cap));
  }
}

extern "C" int as_memory_prepare(const void* proj, int dtype, int ld, int q_off, int k_off, int v_off, int i_off,
                                 int f_off, int H, int dim, int vdim, const float* i_bias, const float* f_bias,
                                 float cap, float* qkv, float* i_log, float* f_log, int num_tokens,
                                 hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (H <= 0 || dim <= 0 || vdim <= 0 || !(cap > 0.f) || ld < q_off + H * dim || ld < k_off + H * dim ||
      ld < v_off + H * vdim || ld < i_off + H || ld < f_off + H)
    return AS_BAD_SHAPE;
  int across = num_tokens >= 512 ? 1 : ((2 * dim + vdim) * H + 255) / 256;
  if (across > 64) across = 64;
  dim3 grid(num_tokens, across);
  if (dtype == DT_F32)
    memory_prepare_kernel<float><<<grid, 256, 0, stream>>>((const float*)proj, ld, q_off, k_off, v_off, i_off, f_off, H,
                                                           dim, vdim, i_bias, f_bias, cap, qkv, i_log, f_log);
  else if (dtype == DT_BF16)
    memory_prepare_kernel<bf16><<<grid, 256, 0, stream>>>((const bf16*)proj, ld, q_off, k_off, v_off, i_off, f_off, H,
                                                          dim, vdim, i_bias, f_bias, cap, qkv, i_log, f_log);
  else return AS_BAD_DTYPE;
  return launch_status();
}

// ---- gated linear recurrence ----------------------------------------------------------------------
// The gates.  u fp32 [T, width] is cut into `blocks` parts of bw channels; in part b
//   r = sigmoid(ra[b] u_b + ra_b[b]),  i = sigmoid(ri[b] u_b + ri_b[b])     (ra, ri [blocks, bw, bw], out x in)
//   a = exp(-c r softplus(lam));  a_out = a,  x_out = sqrt(1 - a^2) i u.
// A workgroup takes 64 tokens by 64 outputs of one part and a thread four by four of them for both gates;
// tokens and weights meet in LDS in pieces of 32 inputs, laid out input-major so that a thread reads its
// four tokens and its four outputs 16 bytes at a time; every output is one fma chain over its inputs in
// order, whatever shares the launch.
#define GATE_TT 64
#define GATE_TO 64
#define GATE_KC 32
template <typename W>
__global__ __launch_bounds__(256) void rglru_gates_kernel(const float* __restrict__ u, int width, int bw,
                                                          const W* __restrict__ ra, const W* __restrict__ ra_b,
                                                          const W* __restrict__ ri, const W* __restrict__ ri_b,
                                                          const W* __restrict__ lam, float c, float* __restrict__ a_out,
                                                          float* __restrict__ x_out, int num_tokens) {
  __shared__ __attribute__((aligned(16))) float us[GATE_KC][GATE_TT + 4];
  __shared__ __attribute__((aligned(16))) float wr[GATE_KC][GATE_TO + 4];
  __shared__ __attribute__((aligned(16))) float wi[GATE_KC][GATE_TO + 4];
  const int b = blockIdx.y, t0 = blockIdx.x * GATE_TT, o0 = blockIdx.z * GATE_TO;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;  // outputs o0 + 4 tx .., tokens t0 + 4 ty ..
  float accr[4][4] = {}, acci[4][4] = {};
  const W* rab = ra + (size_t)b * bw * bw;
  const W* rib = ri + (size_t)b * bw * bw;
  const int lk = threadIdx.x & 31, lrow = threadIdx.x >> 5;  // loads: input k0 + lk of rows lrow + 8 i
  for (int k0 = 0; k0 < bw; k0 += GATE_KC) {
    float uu[8], rr[8], ii[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int row = lrow + 8 * i, k = k0 + lk;
      uu[i] = (t0 + row < num_tokens && k < bw) ? u[(size_t)(t0 + row) * width + b * bw + k] : 0.f;
      const bool in = o0 + row < bw && k < bw;
      rr[i] = in ? to_f32(rab[(size_t)(o0 + row) * bw + k]) : 0.f;
      ii[i] = in ? to_f32(rib[(size_t)(o0 + row) * bw + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      us[lk][lrow + 8 * i] = uu[i];
      wr[lk][lrow + 8 * i] = rr[i];
      wi[lk][lrow + 8 * i] = ii[i];
    }
    __syncthreads();
#pragma unroll 8
    for (int kk = 0; kk < GATE_KC; ++kk) {
      const float4 u4 = *reinterpret_cast<const float4*>(&us[kk][4 * ty]);
      const float4 r4 = *reinterpret_cast<const float4*>(&wr[kk][4 * tx]);
      const float4 i4 = *reinterpret_cast<const float4*>(&wi[kk][4 * tx]);
      const float uv[4] = {u4.x, u4.y, u4.z, u4.w}, rv[4] = {r4.x, r4.y, r4.z, r4.w}, iv[4] = {i4.x, i4.y, i4.z, i4.w};
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int oo = 0; oo < 4; ++oo) {
          accr[tt][oo] = fmaf(rv[oo], uv[tt], accr[tt][oo]);
          acci[tt][oo] = fmaf(iv[oo], uv[tt], acci[tt][oo]);
        }
    }
  }
#pragma unroll
  for (int oo = 0; oo < 4; ++oo) {
    const int o = o0 + 4 * tx + oo;
    if (o >= bw) continue;
    const int ch = b * bw + o;
    const float rb = to_f32(ra_b[ch]), ib = to_f32(ri_b[ch]), sp = softplusf_(to_f32(lam[ch]));
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      const int t = t0 + 4 * ty + tt;
      if (t >= num_tokens) continue;
      const float rg = sigmoidf_(accr[tt][oo] + rb), ig = sigmoidf_(acci[tt][oo] + ib);
      const float log_a = -c * rg * sp;
      a_out[(size_t)t * width + ch] = expf(log_a);
      x_out[(size_t)t * width + ch] = sqrtf(-expm1f(2.0f * log_a)) * ig * u[(size_t)t * width + ch];
    }
  }
}

// The same on the matrix cores, for parts of whole steps of 32 inputs: u and 32-bit weights as three bf16 parts each (six products
// of a pair), bf16 weights as they are (three).  A workgroup takes 64 tokens by 64 outputs of both gates of one part and a
// wave 16 of the outputs; every value is taken apart once a workgroup, on its way into LDS, and the next step's are loaded
// while this one's are multiplied.  Three workgroups fit a compute unit (37 KB of LDS): they fill one another's waits, for a
// workgroup's few steps (eight of a part of 256) end before a deep pipeline would have paid.  An output's sum is one pair of
// chains over the steps in order, so it does not depend on what shares the launch.  A sum that is not finite is computed
// again by multiply-adds (an infinity has no parts).  What bounds it: the
// exponentials and divisions of the way out, about as much as the products and the taking apart.  1,500 tokens of 8 parts of
// 256: 79 -> 38 us (bf16 weights 27), 2,048 of 16: 179 -> 99 (65), 20 of 8: 43 -> 14; the error of a against 64 bits 1.3e-7
// -> 0.66e-7.
// Places of 16 bytes (8 inputs of a row) in LDS as in the 32-bit products: row * 4 + (c ^ f(row / 4 % 4)), f = 0, 2, 3, 1.
#define GATE_ROWS (GATE_TT + 2 * GATE_TO)
__device__ __forceinline__ int gate_place(int row, int c) { return row * 4 + (c ^ (0x78 >> (row >> 1 & 6) & 3)); }

template <typename W> __device__ float plain_dot(const float* u, const W* w, int n) {
  float s = 0.f;
  for (int k = 0; k < n; ++k) s = fmaf(to_f32(w[k]), u[k], s);
  return s;
}

template <typename W>
__global__ __launch_bounds__(256, 3) void rglru_gates_mfma_kernel(const float* __restrict__ u, int width, int bw,
                                                               const W* __restrict__ ra, const W* __restrict__ ra_b,
                                                               const W* __restrict__ ri, const W* __restrict__ ri_b,
                                                               const W* __restrict__ lam, float c,
                                                               float* __restrict__ a_out, float* __restrict__ x_out,
                                                               int num_tokens) {
  constexpr bool PARTED = sizeof(W) == 4;
  __shared__ bf16x8 lds[3][GATE_ROWS * 4];
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE, lr = lane & 15, lg = lane >> 4;
  const int b = blockIdx.y, t0 = blockIdx.x * GATE_TT, o0 = blockIdx.z * GATE_TO;
  const int row = threadIdx.x >> 2, piece = threadIdx.x & 3;  // this thread brings 8 inputs of a token and of two outputs
  const float* src_u = u + (size_t)min(t0 + row, num_tokens - 1) * width + b * bw + piece * 8;
  const size_t at_w = ((size_t)b * bw + min(o0 + row, bw - 1)) * bw + piece * 8;
  const W* src_w[2] = {ra + at_w, ri + at_w};
  floatx4 au[2], aw[2][2];
  bf16x8 whole[2];
  auto load = [&](int k) {
#pragma unroll
    for (int h = 0; h < 2; ++h) au[h] = *reinterpret_cast<const floatx4*>(src_u + k + 4 * h);
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      if constexpr (PARTED) {
#pragma unroll
        for (int h = 0; h < 2; ++h) aw[g][h] = *reinterpret_cast<const floatx4*>(src_w[g] + k + 4 * h);
      } else {
        whole[g] = *reinterpret_cast<const bf16x8*>(src_w[g] + k);
      }
    }
  };
  auto place = [&](int to, const Parts& s) {
    lds[0][to] = s.h;
    lds[1][to] = s.m;
    lds[2][to] = s.l;
  };
  floatx4 acc[2][4], low[2][4];
#pragma unroll
  for (int g = 0; g < 2; ++g)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[g][j] = low[g][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  load(0);
  for (int k = 0; k < bw; k += 32) {
    __syncthreads();  // the step before has been read
    place(gate_place(row, piece), parts(au[0], au[1]));
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int to = gate_place(GATE_TT + g * GATE_TO + row, piece);
      if constexpr (PARTED) place(to, parts(aw[g][0], aw[g][1]));
      else lds[0][to] = whole[g];
    }
    __syncthreads();
    if (k + 32 < bw) load(k + 32);
    Parts ws[2];
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      const int from = gate_place(GATE_TT + g * GATE_TO + wave * 16 + lr, lg);
      ws[g].h = lds[0][from];
      if constexpr (PARTED) { ws[g].m = lds[1][from]; ws[g].l = lds[2][from]; }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int from = gate_place(j * 16 + lr, lg);
      const Parts us = {lds[0][from], lds[1][from], lds[2][from]};
#pragma unroll
      for (int x = 0; x < 6; ++x) {
        if (!PARTED && PART_W[x] != 0) continue;
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          floatx4& to = x == 5 ? acc[g][j] : low[g][j];
          to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(part(ws[g], PART_W[x]), part(us, PART_A[x]), to, 0, 0, 0);
        }
      }
    }
  }
  // a lane holds outputs o .. o+3 of token t0 + 16 j + lr
  const int o = o0 + wave * 16 + 4 * lg, ch = b * bw + o;
  if (o >= bw) return;  // bw is a multiple of 4
  float rb[4], ib[4], sp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) { rb[i] = to_f32(ra_b[ch + i]); ib[i] = to_f32(ri_b[ch + i]); sp[i] = softplusf_(to_f32(lam[ch + i])); }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int t = t0 + j * 16 + lr;
    if (t >= num_tokens) continue;
    floatx4 r = acc[0][j] + low[0][j], g = acc[1][j] + low[1][j], av, xv;
    if (!finite(r) || !finite(g)) {
      for (int i = 0; i < 4; ++i) {
        r[i] = plain_dot(u + (size_t)t * width + b * bw, ra + (size_t)(ch + i) * bw, bw);
        g[i] = plain_dot(u + (size_t)t * width + b * bw, ri + (size_t)(ch + i) * bw, bw);
      }
    }
    const floatx4 uu = *reinterpret_cast<const floatx4*>(u + (size_t)t * width + ch);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float log_a = -c * sigmoidf_(r[i] + rb[i]) * sp[i];
      av[i] = expf(log_a);
      xv[i] = sqrtf(-expm1f(2.0f * log_a)) * sigmoidf_(g[i] + ib[i]) * uu[i];
    }
    *reinterpret_cast<floatx4*>(a_out + (size_t)t * width + ch) = av;
    *reinterpret_cast<floatx4*>(x_out + (size_t)t * width + ch) = xv;
  }
}

// The same for a few tokens (a decode step): the two matrices are streamed once.  Sixteen lanes share an
// output channel (a wave four channels): each takes four inputs in sixteen (16-byte loads, a row of the
// matrix read in whole lines), and their sums meet through DPP moves within the sixteen; eight tokens at a
// time.  Blocks whose rows do not start on 16 bytes are read value by value.
template <typename W>
__global__ __launch_bounds__(256) void rglru_gates_few_kernel(const float* __restrict__ u, int width, int bw,
                                                              const W* __restrict__ ra, const W* __restrict__ ra_b,
                                                              const W* __restrict__ ri, const W* __restrict__ ri_b,
                                                              const W* __restrict__ lam, float c,
                                                              float* __restrict__ a_out, float* __restrict__ x_out,
                                                              int num_tokens) {
  const int part = threadIdx.x & 15, ch = blockIdx.x * (blockDim.x / 16) + threadIdx.x / 16;
  const bool mine = ch < width;  // lanes without a channel walk an existing one and store nothing
  const int chc = mine ? ch : width - 1;
  const int b = chc / bw, o = chc - b * bw;
  const W* wr = ra + ((size_t)b * bw + o) * bw;
  const W* wi = ri + ((size_t)b * bw + o) * bw;
  const float rb = to_f32(ra_b[chc]), ib = to_f32(ri_b[chc]), sp = softplusf_(to_f32(lam[chc]));
  const bool quads = (bw & 3) == 0 && (width & 3) == 0 && sizeof(W) == 4;  // rows start on 16 bytes: four inputs a load
  for (int t0 = 0; t0 < num_tokens; t0 += 8) {
    float accr[8] = {}, acci[8] = {};
    if (quads) {
      for (int k = 4 * part; k < bw; k += 64) {
        const float4 a4 = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(wr) + k);
        const float4 b4 = *reinterpret_cast<const float4*>(reinterpret_cast<const float*>(wi) + k);
        float4 u4[8];
#pragma unroll
        for (int tt = 0; tt < 8; ++tt)
          u4[tt] = t0 + tt < num_tokens ? *reinterpret_cast<const float4*>(u + (size_t)(t0 + tt) * width + b * bw + k)
                                        : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) {
          accr[tt] = fmaf(a4.w, u4[tt].w, fmaf(a4.z, u4[tt].z, fmaf(a4.y, u4[tt].y, fmaf(a4.x, u4[tt].x, accr[tt]))));
          acci[tt] = fmaf(b4.w, u4[tt].w, fmaf(b4.z, u4[tt].z, fmaf(b4.y, u4[tt].y, fmaf(b4.x, u4[tt].x, acci[tt]))));
        }
      }
    } else {
      for (int k = part; k < bw; k += 16) {
        const float a = to_f32(wr[k]), bb = to_f32(wi[k]);
#pragma unroll
        for (int tt = 0; tt < 8; ++tt) {
          const float uu = t0 + tt < num_tokens ? u[(size_t)(t0 + tt) * width + b * bw + k] : 0.f;
          accr[tt] = fmaf(a, uu, accr[tt]);
          acci[tt] = fmaf(bb, uu, acci[tt]);
        }
      }
    }
#pragma unroll
    for (int tt = 0; tt < 8; ++tt) {
      const float sr = slices_sum<16>(accr[tt]), si = slices_sum<16>(acci[tt]);
      const int t = t0 + tt;
      if (mine && part == 0 && t < num_tokens) {
        const float rg = sigmoidf_(sr + rb), ig = sigmoidf_(si + ib);
        const float log_a = -c * rg * sp;
        a_out[(size_t)t * width + ch] = expf(log_a);
        x_out[(size_t)t * width + ch] = sqrtf(-expm1f(2.0f * log_a)) * ig * u[(size_t)t * width + ch];
      }
    }
  }
}

#define GATE_FEW_TOKENS 16
extern "C" int as_rglru_gates(const float* u, int width, int blocks, const void* ra, const void* ra_b, const void* ri,
                              const void* ri_b, const void* lam, int w_dtype, float c, float* a_out, float* x_out,
                              int num_tokens, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (width <= 0 || blocks <= 0 || width % blocks || blocks > 65535) return AS_BAD_SHAPE;
  const int bw = width / blocks;
  if (num_tokens <= GATE_FEW_TOKENS) {
    const int blocks_few = (width + 15) / 16;  // sixteen channels a workgroup of 256
    if (w_dtype == DT_F32)
      rglru_gates_few_kernel<float><<<blocks_few, 256, 0, stream>>>(u, width, bw, (const float*)ra, (const float*)ra_b,
                                                                   (const float*)ri, (const float*)ri_b,
                                                                   (const float*)lam, c, a_out, x_out, num_tokens);
    else if (w_dtype == DT_BF16)
      rglru_gates_few_kernel<bf16><<<blocks_few, 256, 0, stream>>>(u, width, bw, (const bf16*)ra, (const bf16*)ra_b,
                                                                  (const bf16*)ri, (const bf16*)ri_b, (const bf16*)lam,
                                                                  c, a_out, x_out, num_tokens);
    else return AS_BAD_DTYPE;
    return launch_status();
  }
  dim3 grid((num_tokens + GATE_TT - 1) / GATE_TT, blocks, (bw + GATE_TO - 1) / GATE_TO);
  if (grid.z > 65535) return AS_BAD_SHAPE;
  const uintptr_t starts = (uintptr_t)u | (uintptr_t)ra | (uintptr_t)ri | (uintptr_t)a_out | (uintptr_t)x_out;
  if (bw % 32 == 0 && (starts & 15) == 0 && (w_dtype == DT_F32 || w_dtype == DT_BF16)) {  // whole steps of 16-byte pieces
    if (w_dtype == DT_F32)
      rglru_gates_mfma_kernel<float><<<grid, 256, 0, stream>>>(u, width, bw, (const float*)ra, (const float*)ra_b, (const float*)ri,
                                                              (const float*)ri_b, (const float*)lam, c, a_out, x_out, num_tokens);
    else
      rglru_gates_mfma_kernel<bf16><<<grid, 256, 0, stream>>>(u, width, bw, (const bf16*)ra, (const bf16*)ra_b, (const bf16*)ri,
                                                             (const bf16*)ri_b, (const bf16*)lam, c, a_out, x_out, num_tokens);
    return launch_status();
  }
  if (w_dtype == DT_F32)
    rglru_gates_kernel<float><<<grid, 256, 0, stream>>>(u, width, bw, (const float*)ra, (const float*)ra_b,
                                                        (const float*)ri, (const float*)ri_b, (const float*)lam, c,
                                                        a_out, x_out, num_tokens);
  else if (w_dtype == DT_BF16)
    rglru_gates_kernel<bf16><<<grid, 256, 0, stream>>>(u, width, bw, (const bf16*)ra, (const bf16*)ra_b,
                                                       (const bf16*)ri, (const bf16*)ri_b, (const bf16*)lam, c, a_out,
                                                       x_out, num_tokens);
  else return AS_BAD_DTYPE;
  return launch_status();
}

// The scan: S = a S + x per channel, from zero at the start of a sequence; what leaves is
// scale * S * gelu_tanh(y + y_bias) with y from proj [T, ld] at y_off, into out [T, ld_out] at out_off.
// Three ways to walk a row:
// a row of one token (a decode step): a thread a channel.
// middle: a workgroup 64 channels, its 16 waves a sixteenth of the tokens each: every wave composes its stretch from the identity (the
//   product of the decays and what the stretch ends with), the stretches are chained in LDS in order, and every wave runs its
//   stretch again from its true start, now writing.  Every input is read twice.
// long: a workgroup 16 channels, 1,024 tokens at a time, a thread up to 16 neighbouring ones of one channel: it loads them all at once,
//   composes them, the stretches are chained (four of a wave by lane moves, the waves' through LDS), and the thread runs its
//   tokens again, out of its registers.  Every input is read once and the chain of dependent steps is 16 + 2 + 16 a thousand tokens, but it
//   takes four times the workgroups, of which a compute unit holds one and of the middle way's two: only while the step's rows of more
//   than SCAN_LONG tokens fit two rounds of them (every other row stays with the middle way, or goes along where all rows of more than
//   one token fit four: 32, 100 and 168 tokens at 4,096 channels in two kernels 14.7 us, in one 10), in a kernel of its own.
// The rows of a way are dealt to lines of workgroups by their place among them, so that no row costs workgroups that find
// nothing to do.  Neighbouring workgroups of an XCD take neighbouring channels, so that a 128-byte line of two workgroups'
// channels enters one L2.
// us: every row the middle way, one workgroup of 64 channels a row / every row the long way, workgroups of every row / now.  4,096 channels:
// 255 rows of one token beside one of 512 79 120 19, 200 beside one of two 38 93 5.8, 128 rows of 4 26 228 26, 64 of 16 27 118 26, 16 of 128 26 45 26,
// 4 of 250 15 19 15, one of 2,048 81 27 26; 2,048 channels: one of 1,500 55 18 17 (45 MB: 2.6 TB/s; half of the compute units hold a
// workgroup), 8 of one beside 512 17 8.6 8.1; 1,024 channels: one of 300 11.3 5.8 6.1, 4 of 250 10.2 5.5 5.7.
template <typename T, typename W> struct Scan {
  const float *a, *x;
  const T* proj;
  const W* y_bias;
  float* state;
  const int *row_first, *row_len, *row_start, *row_slots;
  T* out;
  int width, ld, y_off, ld_out, out_off, writes, num_rows;
  float scale;
};

struct ScanRow { int first, len, start, slot; };
template <typename T, typename W> __device__ __forceinline__ ScanRow scan_row(const Scan<T, W>& p, int r) {
  return {p.row_first[r], p.row_len[r], p.row_start[r], p.row_slots[r]};
}

// Channel c of a row, token by token.
template <typename T, typename W>
__device__ __forceinline__ void rglru_step(const Scan<T, W>& p, const ScanRow& row, int c) {
  const int first = row.first, len = row.len, slot = row.slot;
  float* held = p.state + (size_t)(slot < 0 ? 0 : slot) * p.width + c;
  float S = (row.start > 0 && slot >= 0) ? *held : 0.f;
  const float yb = p.y_bias ? to_f32(p.y_bias[c]) : 0.f;
  for (int j = 0; j < len; ++j) {
    const size_t t = (size_t)first + j;
    S = fmaf(p.a[t * p.width + c], S, p.x[t * p.width + c]);
    p.out[t * p.ld_out + p.out_off + c] = from_f32<T>(p.scale * S * gelu_tanhf_(to_f32(p.proj[t * p.ld + p.y_off + c]) + yb));
  }
  if (p.writes && slot >= 0) *held = S;
}

#define SCAN_TOKENS 16   // a thread's, the long way
#define SCAN_CHANNELS 16
#define SCAN_WAVES 16
#define SCAN_THREADS (WAVE * SCAN_WAVES)
#define SCAN_LONG 64     // more tokens than this may go the long way
#define SCAN_ONLY 32     // so may a row that is the step's only one

template <typename T, typename W>
__device__ __forceinline__ void rglru_middle(const Scan<T, W>& p, float (&ends)[2][SCAN_WAVES][WAVE], const ScanRow& row, int group) {
  const int lane = threadIdx.x & (WAVE - 1), seg = threadIdx.x / WAVE;
  const int first = row.first, len = row.len, slot = row.slot, c = min(group * WAVE + lane, p.width - 1);
  const int per = (len + SCAN_WAVES - 1) / SCAN_WAVES, lo = min(len, seg * per), hi = min(len, lo + per);
  float A = 1.f, B = 0.f;
#pragma unroll 4
  for (int j = lo; j < hi; ++j) {
    const size_t t = (size_t)first + j;
    const float av = p.a[t * p.width + c];
    B = fmaf(av, B, p.x[t * p.width + c]);
    A *= av;
  }
  float* held = p.state + (size_t)(slot < 0 ? 0 : slot) * p.width + c;
  float S = (row.start > 0 && slot >= 0) ? *held : 0.f;
  const float yb = p.y_bias ? to_f32(p.y_bias[c]) : 0.f;
  ends[0][seg][lane] = A;
  ends[1][seg][lane] = B;
  __syncthreads();
  for (int s = 0; s < seg; ++s) S = fmaf(ends[0][s][lane], S, ends[1][s][lane]);
  if (group * WAVE + lane >= p.width) return;
#pragma unroll 4
  for (int j = lo; j < hi; ++j) {
    const size_t t = (size_t)first + j;
    S = fmaf(p.a[t * p.width + c], S, p.x[t * p.width + c]);
    p.out[t * p.ld_out + p.out_off + c] = from_f32<T>(p.scale * S * gelu_tanhf_(to_f32(p.proj[t * p.ld + p.y_off + c]) + yb));
  }
  if (p.writes && slot >= 0 && seg == SCAN_WAVES - 1) *held = S;  // the last stretch ends where the row ends
}

// `buf`: the half of `ends` whose turn it is, from round to round and from row to row
template <typename T, typename W>
__device__ __forceinline__ void rglru_long(const Scan<T, W>& p, float (&ends)[2][2][SCAN_WAVES][SCAN_CHANNELS], int& buf, const ScanRow& row, int tile) {
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int ch = lane & (SCAN_CHANNELS - 1), sub = lane / SCAN_CHANNELS;  // four stretches a wave
  const int mine = tile * SCAN_CHANNELS + ch, c = min(mine, p.width - 1);
  const int first = row.first, len = row.len, slot = row.slot;
  float* held = p.state + (size_t)(slot < 0 ? 0 : slot) * p.width + c;
  float S = (row.start > 0 && slot >= 0) ? *held : 0.f;  // the state where the round begins
  const float yb = p.y_bias ? to_f32(p.y_bias[c]) : 0.f;
  const int per = min(SCAN_TOKENS, (len + 4 * SCAN_WAVES - 1) / (4 * SCAN_WAVES));
  // a thread's tokens in a straight line, as many as the row's length asks for (tests between them would make every load wait)
  auto walk = [&](auto most) {
    constexpr int N = decltype(most)::value;
    for (int base = 0; base < len; base += SCAN_TOKENS * 4 * SCAN_WAVES, buf ^= 1) {
      const int lo = base + (wave * 4 + sub) * per, mine_n = min(per, len - lo);  // tokens of this stretch, if any
      float av[N], xv[N], yv[N];
      if (mine_n > 0) {  // places beyond the row repeat its last token and count as the identity
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const size_t t = (size_t)first + lo + min(i, mine_n - 1);
          av[i] = p.a[t * p.width + c];
          xv[i] = p.x[t * p.width + c];
          yv[i] = to_f32(p.proj[t * p.ld + p.y_off + c]);
        }
      }
      float A = 1.f, B = 0.f;
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if (i < mine_n) {
          B = fmaf(av[i], B, xv[i]);
          A *= av[i];
        }
      }
#pragma unroll
      for (int off = SCAN_CHANNELS; off < WAVE; off *= 2) {  // with the stretches before it in the wave
        const float Ab = __shfl_up(A, off, WAVE), Bb = __shfl_up(B, off, WAVE);
        if (lane >= off) {
          B = fmaf(A, Bb, B);
          A *= Ab;
        }
      }
      if (sub == 3) {
        ends[buf][0][wave][ch] = A;
        ends[buf][1][wave][ch] = B;
      }
      float Ae = __shfl_up(A, SCAN_CHANNELS, WAVE), Be = __shfl_up(B, SCAN_CHANNELS, WAVE);
      if (sub == 0) { Ae = 1.f; Be = 0.f; }
      __syncthreads();  // the next round writes the other half; the one after it comes behind the next round's barrier
      float s = S;
#pragma unroll
      for (int w = 0; w < SCAN_WAVES; ++w) {
        if (w == wave) s = S;
        S = fmaf(ends[buf][0][w][ch], S, ends[buf][1][w][ch]);
      }
      s = fmaf(Ae, s, Be);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        if (i < mine_n) {
          s = fmaf(av[i], s, xv[i]);
          if (mine < p.width)
            p.out[((size_t)first + lo + i) * p.ld_out + p.out_off + c] = from_f32<T>(p.scale * s * gelu_tanhf_(yv[i] + yb));
        }
      }
    }
  };
  if (per > 8) walk(std::integral_constant<int, 16>{});
  else if (per > 4) walk(std::integral_constant<int, 8>{});
  else walk(std::integral_constant<int, 4>{});
  if (p.writes && slot >= 0 && threadIdx.x < SCAN_CHANNELS && mine < p.width) *held = S;
}

// f(row) for the rows of low < length <= high in the places line, line + lines, ... among them; the whole workgroup together.  A
// lane to a row: 16 waves that count one by one take longer than the rows.
template <typename T, typename W, typename F>
__device__ __forceinline__ void scan_rows(const Scan<T, W>& p, int low, int high, int line, int lines, F f) {
  const int lane = threadIdx.x & (WAVE - 1);
  for (int base = 0, before = 0; base < p.num_rows; base += WAVE) {
    const ScanRow row = scan_row(p, min(base + lane, p.num_rows - 1));
    const bool one = base + lane < p.num_rows && row.len > low && row.len <= high;
    const unsigned long long found = __ballot(one);
    const int place = before + __popcll(found & ((1ull << lane) - 1));
    before += __popcll(found);
    for (; line < before; line += lines) {
      const int l = __ffsll((unsigned long long)__ballot(one && place == line)) - 1;
      f(ScanRow{__builtin_amdgcn_readlane(row.first, l), __builtin_amdgcn_readlane(row.len, l), __builtin_amdgcn_readlane(row.start, l),
                __builtin_amdgcn_readlane(row.slot, l)});
    }
  }
}

// Workgroup `at` of those that take rows of one token, a thousand channels each
template <typename T, typename W> __device__ __forceinline__ void scan_ones(const Scan<T, W>& p, int at) {
  const int chunks = (p.width + SCAN_THREADS - 1) / SCAN_THREADS, r = at / chunks, c = at % chunks * SCAN_THREADS + (int)threadIdx.x;
  if (r >= p.num_rows) return;
  const ScanRow row = scan_row(p, r);
  if (c < p.width && row.len <= 1) rglru_step(p, row, c);
}

#define SCAN_PARAMS                                                                                                                     \
  const float *__restrict__ a, const float *__restrict__ x, int width, const T *__restrict__ proj, int ld, int y_off,                   \
      const W *__restrict__ y_bias, float scale, float *__restrict__ state, const int *__restrict__ row_first,                          \
      const int *__restrict__ row_len, const int *__restrict__ row_start, const int *__restrict__ row_slots, int writes,                \
      T *__restrict__ out, int ld_out, int out_off, int num_rows
#define SCAN_STRUCT                                                                                                                     \
  const Scan<T, W> p = {a, x, proj, y_bias, state, row_first, row_len, row_start, row_slots, out, width, ld, y_off, ld_out, out_off,     \
                        writes, num_rows, scale}

// blockIdx.y < lines: rows of more than `low` tokens; beyond: rows of one token
template <typename T, typename W>
__global__ __launch_bounds__(SCAN_THREADS) void rglru_long_kernel(SCAN_PARAMS, int lines, int per_xcd, int low) {
  SCAN_STRUCT;
  __shared__ float ends[2][2][SCAN_WAVES][SCAN_CHANNELS];  // [round % 2][decays, ends]
  if ((int)blockIdx.y >= lines) return scan_ones(p, ((int)blockIdx.y - lines) * per_xcd * 8 + (int)blockIdx.x);
  const int tile = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if (tile * SCAN_CHANNELS >= width) return;
  int buf = 0;
  if (lines == num_rows) rglru_long(p, ends, buf, scan_row(p, blockIdx.y), tile);  // all of them
  else scan_rows(p, low, INT_MAX, blockIdx.y, lines, [&](const ScanRow& row) { rglru_long(p, ends, buf, row, tile); });
}

// BY_ROW: row blockIdx.y, whatever its length.  Else `lines` times the groups of 64 channels workgroups: rows of 2 to `high` tokens; the
// others: rows of one token
template <typename T, typename W, bool BY_ROW>
__global__ __launch_bounds__(SCAN_THREADS, 8) void rglru_scan_kernel(SCAN_PARAMS, int lines, int groups, int high) {
  SCAN_STRUCT;
  __shared__ float ends[2][SCAN_WAVES][WAVE];
  if constexpr (BY_ROW) {
    rglru_middle(p, ends, scan_row(p, blockIdx.y), blockIdx.x);
  } else {
    if ((int)blockIdx.x >= lines * groups) return scan_ones(p, (int)blockIdx.x - lines * groups);
    const int line = (int)blockIdx.x / groups, group = (int)blockIdx.x % groups;
    scan_rows(p, 1, high, line, lines, [&](const ScanRow& row) {
      __syncthreads();  // the row before has been read
      rglru_middle(p, ends, row, group);
    });
  }
}

template <typename T, typename W> __global__ __launch_bounds__(WAVE) void rglru_step_kernel(SCAN_PARAMS) {
  SCAN_STRUCT;
  const int c = blockIdx.x * WAVE + threadIdx.x;
  if (c < width) rglru_step(p, scan_row(p, blockIdx.y), c);
}

// num_tokens: of the whole step; as many as rows: every row has one.  several, many: rows of more than one token, of more than SCAN_LONG
// (< 0: not known), by which workgroups are dealt out.
extern "C" int as_rglru_scan(const float* a, const float* x, int width, const void* proj, int dtype, int ld, int y_off,
                             const void* y_bias, int w_dtype, float scale, float* state, const int* row_first,
                             const int* row_len, const int* row_start, const int* row_slots, int writes, void* out,
                             int ld_out, int out_off, int num_rows, int num_tokens, int several, int many, hipStream_t stream) {
  if (num_rows <= 0) return AS_OK;
  if (width <= 0 || num_rows > 65535 || ld < y_off + width || ld_out < out_off + width) return AS_BAD_SHAPE;
  const int tiles = (width + SCAN_CHANNELS - 1) / SCAN_CHANNELS, per_xcd = (tiles + 7) / 8, all = per_xcd * 8;
  const int groups = (width + WAVE - 1) / WAVE, chunks = (width + SCAN_THREADS - 1) / SCAN_THREADS, cus = compute_units();
  const bool only = num_rows == 1, known = several >= 0 && many >= 0;
  if (!known) several = num_rows, many = 0;
  // two rounds of workgroups of either way at most; a line a row where few rows or none have one token
  const bool long_way = only ? num_tokens > SCAN_ONLY : many > 0 && many <= std::max(1, 2 * cus / tiles);
  const bool by_row = !long_way && (only || (known && several == num_rows) || (long)num_rows * groups <= 2 * cus);
  const int low = several <= std::max(1, 4 * cus / tiles) ? 1 : SCAN_LONG;  // a few middle rows go with the long ones: a launch less
  const int longs = only ? 1 : low == 1 ? several : many, middle = only ? 0 : several - (long_way ? longs : 0);
  const int lines = by_row ? 0 : std::min(middle, std::max(1, 4 * cus / groups));
  const long ones = by_row || only || (known && several == num_rows) ? 0 : (long)num_rows * chunks;
  const long blocks = (long)lines * groups + (long_way ? 0 : ones);
  if (blocks > 0x3fffff) return AS_BAD_SHAPE;
#define ARGS(T, W)                                                                                                       \
  a, x, width, (const T*)proj, ld, y_off, (const W*)y_bias, scale, state, row_first, row_len, row_start, row_slots, writes, \
      (T*)out, ld_out, out_off, num_rows
#define LAUNCH(T, W)                                                                                                     \
  do {                                                                                                                   \
    if (num_tokens == num_rows) {                                                                                        \
      rglru_step_kernel<T, W><<<dim3(groups, num_rows), WAVE, 0, stream>>>(ARGS(T, W));                                  \
      break;                                                                                                             \
    }                                                                                                                    \
    if (long_way)                                                                                                        \
      rglru_long_kernel<T, W><<<dim3(all, longs + (int)((ones + all - 1) / all)), SCAN_THREADS, 0, stream>>>(ARGS(T, W), longs, per_xcd, low); \
    if (by_row)                                                                                                          \
      rglru_scan_kernel<T, W, true><<<dim3(groups, num_rows), SCAN_THREADS, 0, stream>>>(ARGS(T, W), 0, groups, 0);       \
    else if (blocks > 0)                                                                                                 \
      rglru_scan_kernel<T, W, false><<<(int)blocks, SCAN_THREADS, 0, stream>>>(ARGS(T, W), lines, groups, long_way ? SCAN_LONG : INT_MAX); \
  } while (0)
  if (dtype == DT_F32 && w_dtype == DT_F32) LAUNCH(float, float);
  else if (dtype == DT_BF16 && w_dtype == DT_BF16) LAUNCH(bf16, bf16);
  else if (dtype == DT_BF16 && w_dtype == DT_F32) LAUNCH(bf16, float);
  else return AS_BAD_DTYPE;
#undef ARGS
#undef LAUNCH
  return launch_status();
}
