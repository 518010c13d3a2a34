// Feed-forward layers made of several small experts, of which every token uses a few.
//
// Which experts a token uses is decided on the GPU (a table indexed by the token id here), so a step
// never waits for the host and can be replayed as a graph.  A (token, chosen expert) is a "pair":
// pair p = token * top + choice.  `moe_route` sorts the pairs by expert and cuts every expert's run
// into tiles of up to 128; the two grouped products then take one workgroup per (tile or half of it, strip of outputs): the first
// applies act(gate) * up on the way out, the second writes every pair's output where the pair stands
// (so the outputs of a token's experts lie side by side), and `moe_combine` adds them up with their
// weights.  A pair's result does not depend on what else is in the step: every output is a dot product
// over the whole width in a fixed order.
#include "wide_tile.h"

#define MOE_TILE 128     // pairs of one expert that a tile holds at most (eight column tiles of 16); a route has tiles of 64 or 128
#define MOE_HALF 64      // four column tiles
#define MOE_KC 128       // inputs per round: the tile's activations of a round meet in LDS
#define MOE_STRIP 64     // outputs that a workgroup takes: four waves of 16
#define MOE_MAX_EXPERTS 1024

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));  // 16 bytes as they are moved, whatever they hold

// ---- routing ------------------------------------------------------------------------------------
// table [vocab, top] int32: the experts of every token id.  order [P]: the pairs sorted by expert;
// tiles [max_tiles, 3]: (expert, first place in `order`, count <= `size`, 64 or 128); counts[0] = number of tiles.
// One workgroup; the order of pairs within an expert is whatever the atomics make it, which no
// result depends on.
// With token_ids null, `table` is [P]: the expert of every pair as a router's kernel left it.  identity > 0: the numbers
// experts .. experts + identity - 1 are experts without matrices; their pairs (-1 here) stand in no tile and nowhere in `order`.
__device__ __forceinline__ int expert_of_pair(const int* token_ids, const int* table, int vocab, int top, int experts,
                                              int identity, int p) {
  int e;
  if (token_ids) {
    int id = token_ids[p / top];
    id = id < 0 ? 0 : (id >= vocab ? vocab - 1 : id);
    e = table[(size_t)id * top + p % top];
  } else {
    e = table[p];
  }
  if (identity > 0 && e >= experts) return -1;
  return e < 0 ? 0 : (e >= experts ? experts - 1 : e);
}

__global__ __launch_bounds__(1024) void moe_route_table_kernel(const int* __restrict__ token_ids,
                                                               const int* __restrict__ table, int vocab, int top,
                                                               int experts, int num_tokens, int* __restrict__ order,
                                                               int* __restrict__ tiles, int* __restrict__ counts,
                                                               int max_tiles, int identity, int size) {
  __shared__ int hist[MOE_MAX_EXPERTS];
  __shared__ int cursor[MOE_MAX_EXPERTS];
  const int P = num_tokens * top;
  // A thread's first pairs stay in registers between the two passes: their loads, one behind the other, are asked for together
  // (3,000 pairs of 16 experts: each pass by itself 11.4 us, now 8.3).
  constexpr int HELD = 4;
  int mine[HELD];
#pragma unroll
  for (int i = 0; i < HELD; ++i) {
    const int p = threadIdx.x + i * blockDim.x;
    mine[i] = p < P ? expert_of_pair(token_ids, table, vocab, top, experts, identity, p) : -1;
  }
  for (int e = threadIdx.x; e < experts; e += blockDim.x) hist[e] = 0;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HELD; ++i)
    if (mine[i] >= 0) atomicAdd(&hist[mine[i]], 1);
  for (int p = threadIdx.x + HELD * blockDim.x; p < P; p += blockDim.x) {
    const int e = expert_of_pair(token_ids, table, vocab, top, experts, identity, p);
    if (e >= 0) atomicAdd(&hist[e], 1);
  }
  __syncthreads();
  if (threadIdx.x < WAVE) {  // a lane an expert, 64 at a time: where its pairs and its tiles start
    int at = 0, n = 0;
    for (int e0 = 0; e0 < experts; e0 += WAVE) {
      const int e = e0 + threadIdx.x, pairs = e < experts ? hist[e] : 0, parts = (pairs + size - 1) / size;
      int pairs_to = pairs, parts_to = parts;  // of the experts up to this one
#pragma unroll
      for (int d = 1; d < WAVE; d <<= 1) {
        const int a = __shfl_up(pairs_to, d), b = __shfl_up(parts_to, d);
        if ((int)threadIdx.x >= d) { pairs_to += a; parts_to += b; }
      }
      const int first = at + pairs_to - pairs, tile = n + parts_to - parts;
      if (e < experts) cursor[e] = first;
      for (int i = 0; i < parts && tile + i < max_tiles; ++i) {
        tiles[3 * (tile + i)] = e;
        tiles[3 * (tile + i) + 1] = first + i * size;
        tiles[3 * (tile + i) + 2] = min(size, pairs - i * size);
      }
      at += __shfl(pairs_to, WAVE - 1);
      n += __shfl(parts_to, WAVE - 1);
    }
    if (threadIdx.x == 0) counts[0] = min(n, max_tiles);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < HELD; ++i)
    if (mine[i] >= 0) order[atomicAdd(&cursor[mine[i]], 1)] = threadIdx.x + i * blockDim.x;
  for (int p = threadIdx.x + HELD * blockDim.x; p < P; p += blockDim.x) {
    const int e = expert_of_pair(token_ids, table, vocab, top, experts, identity, p);
    if (e >= 0) order[atomicAdd(&cursor[e], 1)] = p;
  }
}

// ---- a router that scores every expert ---------------------------------------------------------------
// z = router h (+ bias [experts] fp32) in fp32 (router [experts, K], h [T, K], both T-typed).  mode 0: s = sigmoid(z); a
// token's `top` experts are those with the largest s (of equal ones the lower number first); their weights are
// s / (sum of the chosen + 1e-20).  mode 1: the experts with the largest z, weighing the softmax over the chosen z alone.
// mode 2: s = softmax(z) over all experts; the experts form `groups` equal groups of neighbours, a group scores its
// largest s, and only experts of the `keep` best groups (of equal ones the lower number first) can be chosen; the `top`
// largest s among them weigh s * scale, not renormalised.  correction [experts] (mode 2 with one group; null: none) is
// added to s for the choice alone: the `top` largest s + correction are chosen and weigh s * scale.
// pair_expert, pair_weight [T * top].  A workgroup per token: its waves take the experts four at a time, a lane 16 bytes
// of the token's row and of the four router rows at a time (the rows stream once, coalesced), the sums meet by lane swaps
// and the scores in LDS, where the first wave makes the choice.
template <typename T> struct RoutePiece;
template <> struct RoutePiece<float> {
  static constexpr int N = 4;
  static __device__ __forceinline__ void load(const float* p, float* v) {
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
  }
};
template <> struct RoutePiece<bf16> {
  static constexpr int N = 8;
  static __device__ __forceinline__ void load(const bf16* p, float* v) {
    const bf16x8 x = *reinterpret_cast<const bf16x8*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = (float)x[i];
  }
};

template <typename T>
__global__ __launch_bounds__(256) void moe_route_scores_kernel(const T* __restrict__ h, const T* __restrict__ router,
                                                                const float* __restrict__ bias, int mode,
                                                                const float* __restrict__ correction, int groups,
                                                                int keep, float scale,
                                                                int K, int experts, int top, int num_tokens,
                                                                int* __restrict__ pair_expert,
                                                                float* __restrict__ pair_weight) {
  extern __shared__ float scores[];  // [experts], then [groups] group scores and [groups] marks of the kept ones, or [experts] weights
  constexpr int N = RoutePiece<T>::N;
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int t = blockIdx.x;
  const T* row = h + (size_t)t * K;
  const bool whole = K % N == 0;  // rows start on 16 bytes
  // a wave takes four experts at a time: the token's piece is loaded once for the four rows' pieces, and four
  // rows' loads are in flight together
  for (int e0 = wave * 4; e0 < experts; e0 += 16) {
    float z[4] = {0.f, 0.f, 0.f, 0.f};
    if (whole) {
      for (int k = lane * N; k < K; k += WAVE * N) {
        float hv[N], wv[4][N];
        RoutePiece<T>::load(row + k, hv);
#pragma unroll
        for (int j = 0; j < 4; ++j) RoutePiece<T>::load(router + (size_t)min(e0 + j, experts - 1) * K + k, wv[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int i = 0; i < N; ++i) z[j] = fmaf(hv[i], wv[j][i], z[j]);
      }
    } else {
      for (int k = lane; k < K; k += WAVE) {
        const float hv = to_f32(row[k]);
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = fmaf(hv, to_f32(router[(size_t)min(e0 + j, experts - 1) * K + k]), z[j]);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float zs = wave_sum(z[j]);
      if (lane == 0 && e0 + j < experts) {
        if (bias) zs += bias[e0 + j];
        scores[e0 + j] = mode >= 1 ? zs : 1.0f / (1.0f + expf(-zs));
      }
    }
  }
  __syncthreads();
  if (wave) return;
  float* mine = scores;
  if (mode == 2) {
    float mx = -INFINITY, sum = 0.f;
    for (int e = lane; e < experts; e += WAVE) mx = fmaxf(mx, mine[e]);
    mx = wave_max(mx);
    for (int e = lane; e < experts; e += WAVE) sum += expf(mine[e] - mx);
    sum = wave_sum(sum);
    for (int e = lane; e < experts; e += WAVE) mine[e] = expf(mine[e] - mx) / sum;
    __builtin_amdgcn_wave_barrier();
    if (correction) {  // what is chosen by, and beside it what a chosen one weighs
      for (int e = lane; e < experts; e += WAVE) {
        scores[experts + e] = mine[e];
        mine[e] += correction[e];
      }
      __builtin_amdgcn_wave_barrier();
    } else if (groups > 1 && keep < groups) {
      float* gscore = scores + experts;
      float* gkept = gscore + groups;
      const int per = experts / groups;
      for (int g = lane; g < groups; g += WAVE) {
        float m = -INFINITY;
        for (int e = g * per; e < (g + 1) * per; ++e) m = fmaxf(m, mine[e]);
        gscore[g] = m;
        gkept[g] = 0.f;
      }
      __builtin_amdgcn_wave_barrier();
      for (int j = 0; j < keep; ++j) {
        float best = -INFINITY;
        int at = 0x7fffffff;
        for (int g = lane; g < groups; g += WAVE) {
          const float v = gscore[g];
          if (gkept[g] == 0.f && (v > best || at == 0x7fffffff)) { best = v; at = g; }
        }
#pragma unroll
        for (int off = WAVE / 2; off > 0; off >>= 1) {
          const float ob = __shfl_xor(best, off, WAVE);
          const int oa = __shfl_xor(at, off, WAVE);
          if (oa != 0x7fffffff && (at == 0x7fffffff || ob > best || (ob == best && oa < at))) { best = ob; at = oa; }
        }
        if (lane == 0 && at < groups) gkept[at] = 1.f;
        __builtin_amdgcn_wave_barrier();
      }
      for (int e = lane; e < experts; e += WAVE)
        if (gkept[e / per] == 0.f) mine[e] = -INFINITY;
      __builtin_amdgcn_wave_barrier();
    }
  }
  float total = 0.f, my_score = 0.f, largest = 0.f;
  int my_expert = 0;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < experts; e += WAVE) {
      const float v = mine[e];
      if (v > best) { best = v; at = e; }
    }
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) {
      const float ob = __shfl_xor(best, off, WAVE);
      const int oa = __shfl_xor(at, off, WAVE);
      if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
    }
    if (at >= experts) { at = 0; best = 0.f; }  // nothing left to choose (scores that are not numbers)
    else if (correction) best = scores[experts + at];
    if (mode == 1) {  // the first found is the largest: weights are exponentials of the distance to it
      if (j == 0) largest = best;
      best = expf(best - largest);
    }
    if (lane == j % WAVE && j / WAVE == 0) { my_score = best; my_expert = at; }
    if (j >= WAVE && lane == 0) {  // more than 64 experts a token: written as they are found, weighed below
      pair_expert[(size_t)t * top + j] = at;
      pair_weight[(size_t)t * top + j] = best;
    }
    total += best;
    if (lane == 0) mine[at] = -INFINITY;
    __builtin_amdgcn_wave_barrier();
  }
  const float inv = mode == 2 ? scale : 1.0f / (total + (mode == 1 ? 0.f : 1e-20f));
  if (lane < top && lane < WAVE) {
    pair_expert[(size_t)t * top + lane] = my_expert;
    pair_weight[(size_t)t * top + lane] = my_score * inv;
  }
  if (lane == 0)
    for (int j = WAVE; j < top; ++j) pair_weight[(size_t)t * top + j] *= inv;
}

extern "C" int as_moe_route_scores(const void* h, const void* router, const float* bias, int mode,
                                   const float* correction, int groups, int keep, float scale, int dtype, int K,
                                   int experts, int top, int num_tokens, int* pair_expert, float* pair_weight,
                                   hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (K <= 0 || experts <= 0 || experts > MOE_MAX_EXPERTS || top <= 0 || top > experts || mode < 0 || mode > 2) return AS_BAD_SHAPE;
  if (mode == 2 && (groups < 1 || experts % groups || keep < 1 || keep > groups || keep * (experts / groups) < top)) return AS_BAD_SHAPE;
  if (correction && (mode != 2 || groups > 1)) return AS_BAD_SHAPE;
  const int blocks = num_tokens;
  const size_t lds = (size_t)(correction ? 2 * experts : experts + 2 * (groups > 0 ? groups : 0)) * sizeof(float);
  if (dtype == DT_F32)
    moe_route_scores_kernel<float><<<blocks, 256, lds, stream>>>((const float*)h, (const float*)router, bias, mode, correction, groups, keep, scale, K, experts, top,
                                                                  num_tokens, pair_expert, pair_weight);
  else if (dtype == DT_BF16)
    moe_route_scores_kernel<bf16><<<blocks, 256, lds, stream>>>((const bf16*)h, (const bf16*)router, bias, mode, correction, groups, keep, scale, K, experts, top,
                                                                 num_tokens, pair_expert, pair_weight);
  else return AS_BAD_DTYPE;
  return launch_status();
}

extern "C" int as_moe_route_table(const int* token_ids, const int* table, int vocab, int top, int experts,
                                  int num_tokens, int* order, int* tiles, int* counts, int max_tiles, int identity,
                                  int size, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (top <= 0 || experts <= 0 || experts > MOE_MAX_EXPERTS || (token_ids && vocab <= 0)) return AS_BAD_SHAPE;
  if (size != MOE_HALF && size != MOE_TILE) return AS_BAD_SHAPE;
  if (max_tiles < (num_tokens * top + size - 1) / size + experts) return AS_BAD_SHAPE;
  moe_route_table_kernel<<<1, 1024, 0, stream>>>(token_ids, table, vocab, top, experts, num_tokens, order, tiles,
                                                 counts, max_tiles, identity, size);
  return launch_status();
}

// ---- the grouped products -------------------------------------------------------------------------
// a: the inputs, a row per token (pair p reads row p / a_div: a_div = top for the first product, 1 for
// the second, whose inputs are the first one's outputs, a row per pair).  w [experts, N_w, K].
// GATED: N_w = 2 N, rows 0..N-1 the gate, N..2N-1 the up projection; out[p, n] = silu(gate) * up.
// else:  out[p, n] = the product.  out has a row per pair.
//
// bf16: v_mfma_f32_16x16x32_bf16 with the weights as the A operand (16 rows of w) and 16 of the tile's
// pairs as the B operand.  A wave owns 16 outputs (and their up rows) for all of the tile's pairs (up to
// four column tiles of 16).  Per round of 128 inputs the workgroup brings the tile's activations and its 64
// (gated: 128) weight rows into LDS, whole 256-byte runs of a row per 16 lanes, rows padded by 16 bytes
// against bank conflicts; the next round's loads are in flight while this round is multiplied.  Few pairs
// (a decode step) cost few products: column tiles beyond the tile's count are skipped.  Rows of any width (16-byte loads where K % 8 == 0, single values else).
// Eight inputs of a row from column k on, one by one, zeros beyond the row's end (rows that do not start on
// 16 bytes, and a round that reaches beyond K).
__device__ __forceinline__ bf16x8 row_piece(const bf16* row, int k, int K) {
  bf16x8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = k + i < K ? row[k + i] : (bf16)0.f;
  return v;
}

// silu(g) * u, or with limits (limit > 0): g = min(g, limit), u = clamp(u, -limit, limit): g sigmoid(1.702 g) (u + 1)
#define CLAMPED_GATE_ALPHA 1.702f
__device__ __forceinline__ float gate_times_up(float g, float u, float limit) {
  if (limit > 0.f) {
    g = fminf(g, limit);
    u = fminf(fmaxf(u, -limit), limit);
    return g / (1.0f + expf(-CLAMPED_GATE_ALPHA * g)) * (u + 1.0f);
  }
  return g / (1.0f + expf(-g)) * u;
}

template <bool GATED, typename OutT, bool RELU2 = false>
__global__ __launch_bounds__(256) void moe_gemm_bf16_kernel(const bf16* __restrict__ a, int a_div,
                                                            const bf16* __restrict__ w, int N, int K,
                                                            const int* __restrict__ order,
                                                            const int* __restrict__ tiles,
                                                            const int* __restrict__ counts, OutT* __restrict__ out,
                                                            float limit) {
  constexpr int WROWS = GATED ? 2 * MOE_STRIP : MOE_STRIP;  // weight rows of a round: the strip's, then their up rows
  constexpr int WLOADS = WROWS * (MOE_KC / 8) / 256;        // 16-byte pieces of them per thread
  __shared__ __attribute__((aligned(16))) bf16 acts[MOE_HALF][MOE_KC + 8];
  __shared__ __attribute__((aligned(16))) bf16 wts[WROWS][MOE_KC + 8];
  __shared__ int pair_of[MOE_HALF];
  const int tile = blockIdx.y, skip = blockIdx.z * MOE_HALF;  // a tile of 128 in halves
  if (tile >= counts[0]) return;
  const int e = tiles[3 * tile], at = tiles[3 * tile + 1] + skip, cnt = min(tiles[3 * tile + 2] - skip, MOE_HALF);
  if (cnt <= 0) return;
  const int lane = threadIdx.x & (WAVE - 1), wave = threadIdx.x / WAVE;
  const int lr = lane & 15, lg = lane >> 4;
  const int nb = blockIdx.x * MOE_STRIP, n0 = nb + wave * 16;
  const int col_tiles = (cnt + 15) >> 4;
  if (threadIdx.x < MOE_HALF) pair_of[threadIdx.x] = threadIdx.x < cnt ? order[at + threadIdx.x] : -1;
  __syncthreads();
  const int NW = GATED ? 2 * N : N;
  const bf16* wbase = w + (size_t)e * NW * K;
  floatx4 acc[4], acc_up[4];
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) { acc[ct] = floatx4{0.f, 0.f, 0.f, 0.f}; acc_up[ct] = floatx4{0.f, 0.f, 0.f, 0.f}; }
  const bool whole = (K & 7) == 0;
  // thread -> (row, 16-byte piece of the round): 16 pieces a row, so 16 lanes read 256 bytes of a row in a run.
  // Rows that stand for no pair or no output read a row that exists (their products are never stored); only a
  // round that reaches beyond K, or rows that do not start on 16 bytes, take the careful way.
  const int piece_k = (threadIdx.x & 15) * 8, piece_row = threadIdx.x >> 4;  // rows piece_row + 16 i
  const bf16* arow[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = piece_row + 16 * i;
    const int pair = row < col_tiles * 16 ? pair_of[row] : -1;
    arow[i] = a + (size_t)(pair >= 0 ? pair / a_div : 0) * K;
  }
  const bf16* wrow[WLOADS];
#pragma unroll
  for (int i = 0; i < WLOADS; ++i) {
    const int row = piece_row + 16 * i;                                        // of the round's weight rows
    const int n = min(nb + (row & (MOE_STRIP - 1)), N - 1);                    // the output it belongs to
    wrow[i] = wbase + (size_t)((GATED && row >= MOE_STRIP) ? N + n : n) * K;
  }
  u32x4 staged[4], wstaged[WLOADS];
  auto fetch = [&](int k0) {
    const int k = k0 + piece_k;
    if (whole && k0 + MOE_KC <= K) {
#pragma unroll
      for (int i = 0; i < 4; ++i) staged[i] = *reinterpret_cast<const u32x4*>(arow[i] + k);
#pragma unroll
      for (int i = 0; i < WLOADS; ++i) wstaged[i] = *reinterpret_cast<const u32x4*>(wrow[i] + k);
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) staged[i] = __builtin_bit_cast(u32x4, row_piece(arow[i], k, K));
#pragma unroll
      for (int i = 0; i < WLOADS; ++i) wstaged[i] = __builtin_bit_cast(u32x4, row_piece(wrow[i], k, K));
    }
  };
  fetch(0);
  for (int k0 = 0; k0 < K; k0 += MOE_KC) {
    __syncthreads();  // the round before has been read
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (piece_row + 16 * i < col_tiles * 16) *reinterpret_cast<u32x4*>(&acts[piece_row + 16 * i][piece_k]) = staged[i];
#pragma unroll
    for (int i = 0; i < WLOADS; ++i) *reinterpret_cast<u32x4*>(&wts[piece_row + 16 * i][piece_k]) = wstaged[i];
    __syncthreads();
    if (k0 + MOE_KC < K) fetch(k0 + MOE_KC);  // in flight while this round is multiplied
    // the round's products in a straight line for the tile's number of column tiles (a test between the
    // products makes the compiler move the accumulators about: three times the kernel's time)
    auto multiply = [&](auto count) {
      constexpr int CT = decltype(count)::value;
#pragma unroll
      for (int s = 0; s < MOE_KC / 32; ++s) {
        const bf16x8 wv = *reinterpret_cast<const bf16x8*>(&wts[wave * 16 + lr][s * 32 + lg * 8]);
        bf16x8 uv = wv;
        if (GATED) uv = *reinterpret_cast<const bf16x8*>(&wts[MOE_STRIP + wave * 16 + lr][s * 32 + lg * 8]);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const bf16x8 av = *reinterpret_cast<const bf16x8*>(&acts[ct * 16 + lr][s * 32 + lg * 8]);
          acc[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, av, acc[ct], 0, 0, 0);
          if (GATED) acc_up[ct] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(uv, av, acc_up[ct], 0, 0, 0);
        }
      }
    };
    if (n0 < N) {
      if (col_tiles == 4) multiply(std::integral_constant<int, 4>{});
      else if (col_tiles == 3) multiply(std::integral_constant<int, 3>{});
      else if (col_tiles == 2) multiply(std::integral_constant<int, 2>{});
      else multiply(std::integral_constant<int, 1>{});
    }
  }
  // a lane holds outputs n0 + 4 lg + i (i < 4) of the pair in column lr of each column tile
  if (n0 >= N) return;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct) {
    if (ct >= col_tiles) continue;
    const int pair = pair_of[ct * 16 + lr];
    if (pair < 0) continue;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = n0 + 4 * lg + i;
      if (n >= N) continue;
      float v = acc[ct][i];
      if (GATED) {
        const float g = to_f32((bf16)acc[ct][i]), u = to_f32((bf16)acc_up[ct][i]);  // the two products rounded as if stored
        v = gate_times_up(g, u, limit);
      }
      if (RELU2) {
        const float u = fmaxf(to_f32((bf16)v), 0.f);  // the product rounded as if stored
        v = u * u;
      }
      out[(size_t)pair * N + n] = from_f32<OutT>(v);
    }
  }
}

// The same where K comes in whole blocks of 128 columns and outputs in strips of 16 (and everything on 16 bytes): the weights go
// straight from memory into registers, for no wave needs another's rows; only the tile's activations, which all waves multiply
// with, meet in LDS (a chunk in use and the one before, through registers one chunk ahead).  A wave owns two strips of 16 weight
// rows (GATED: a gate strip and its up strip; few pairs of a product without a gate: one).  A lane takes 32 neighbouring
// bytes of its row, the two halves of a step of 64 columns (the columns of a step permuted alike for both operands), so that a
// wave's two loads use whole lines.  Weights' loads go through a buffer descriptor of the expert's matrix: those for chunks past
// the last are sent beyond its end, where they move nothing, and the number of loads in flight is the same everywhere.
// Workgroups start at different blocks of columns and wrap round, so that they do not all ask for the same memory channels.
// An output's products are added up in one order, which depends on the output and its expert alone.
// Two of 16 experts, both products of a layer, us before (every operand through LDS, tiles of 64 x 64) and now: width 4,096, 8 tokens
// 155 and 144, 32 255 and 207 (6.0 and 5.5 TB/s of weights); more pairs: below.
enum { MOE_PLAIN, MOE_GATED, MOE_RELU2 };

template <int MODE, typename OutT>
__global__ __launch_bounds__(256, 2) void moe_gemm_stream_kernel(
    const bf16* __restrict__ a, int a_div, const bf16* __restrict__ w, int N, int K, const int* __restrict__ order,
    const int* __restrict__ tiles, const int* __restrict__ counts, OutT* __restrict__ out, float limit) {
  constexpr bool GATED = MODE == MOE_GATED;
  constexpr int WAVES = 4, S = GATED ? 2 : 1;  // waves, strips of weight rows a wave
  constexpr int ACROSS = WAVES * 16;           // outputs a workgroup
  constexpr int KC = 128, STEPS = KC / 64, PIECES = KC / 8;
  constexpr int MOST = MOE_HALF, PASS = WAVES * 64 / PIECES;  // pairs; rows the threads bring at once
  constexpr unsigned BEYOND = 0xfffffff0u;
  __shared__ u32x4 lds[2][MOST * PIECES];
  const int strip = blockIdx.x, tile = blockIdx.y;
  if (tile >= counts[0]) return;
  const int e = tiles[3 * tile], at = tiles[3 * tile + 1], cnt = min(tiles[3 * tile + 2], MOST);
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lr = lane & 15, lg = lane >> 4;
  const int n0 = strip * ACROSS + wave * 16;
  const int nchunks = K / KC, turn = (int)((strip * ACROSS / (GATED ? 128 : 256) * 5u + (unsigned)e * 3u) % (unsigned)(K / 128)) * (128 / KC);
  const unsigned NW = GATED ? 2 * N : N;
  const __amdgpu_buffer_rsrc_t w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w) + (size_t)e * NW * K, 0,
                                                                        (int)(NW * (unsigned)K * 2u), 0x00020000);
  unsigned w_off[S];  // this lane's first byte of its row of either strip (rows beyond N repeat the last one)
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const unsigned row = GATED ? (unsigned)min(n0 + lr, N - 1) + s * (unsigned)N : (unsigned)min(n0 + s * 16 + lr, N - 1);
    w_off[s] = (row * (unsigned)K + lg * 16) * 2u;
  }
  auto where = [&](int j) { const int c = j + turn; return c >= nchunks ? c - nchunks : c; };
  // LDS place (16 bytes) of block c (8 columns) of pair row r: the hardware reads 16-byte operands in the lane groups
  // {0-3, 12-15, 20-27}, {4-11, 16-19, 28-31} and the same above 32, which so touch every bank once
  auto place_of = [](int r, int c) { return r * 16 + (c ^ (r & 15)); };

  auto run = [&](auto count) {
    constexpr int CT = decltype(count)::value, TIMES = (CT * 16 + PASS - 1) / PASS;
    const int piece = threadIdx.x % PIECES, prow = threadIdx.x / PIECES;  // this thread brings 16 bytes of rows prow + PASS i
    int pair[TIMES];
    const bf16* arow[TIMES];
#pragma unroll
    for (int i = 0; i < TIMES; ++i) pair[i] = order[at + min(prow + PASS * i, cnt - 1)];
    u32x4 wa[STEPS][S][2], wb[STEPS][S][2], wc[STEPS][S][2], held[TIMES];
    auto fetch = [&](u32x4 (&into)[STEPS][S][2], int j) {
      const unsigned col = (unsigned)where(j) * (KC * 2u);
#pragma unroll
      for (int t = 0; t < STEPS; ++t)
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            into[t][s][h] = __builtin_amdgcn_raw_buffer_load_b128(w_buf, j < nchunks ? w_off[s] + col + t * 128u + h * 16u : BEYOND, 0, 0);
    };
    auto request = [&](int j) {  // past the last: the last again
      const int k = where(min(j, nchunks - 1)) * KC;
#pragma unroll
      for (int i = 0; i < TIMES; ++i) held[i] = *reinterpret_cast<const u32x4*>(arow[i] + k);
    };
    floatx4 acc[S][CT];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int i = 0; i < CT; ++i) acc[s][i] = floatx4{0.f, 0.f, 0.f, 0.f};
    // One chunk: its activations go to LDS, whose half everyone left before the barrier of the chunk before; what comes next is
    // requested; a bare barrier (a fence would wait for every load in flight); the products.
    auto chunk = [&](int j, u32x4 (&now)[STEPS][S][2], u32x4 (&later)[STEPS][S][2]) {
#pragma unroll
      for (int i = 0; i < TIMES; ++i) lds[j & 1][place_of(prow + PASS * i, piece)] = held[i];
      request(j + 1);
      fetch(later, j + 2);
      __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0): this wave's LDS writes have landed
      __builtin_amdgcn_s_barrier();
#pragma unroll
      for (int t = 0; t < STEPS; ++t)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < CT; ++i) {
            const bf16x8 av = __builtin_bit_cast(bf16x8, lds[j & 1][place_of(i * 16 + lr, t * 8 + lg * 2 + h)]);
#pragma unroll
            for (int s = 0; s < S; ++s)
              acc[s][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, now[t][s][h]), av, acc[s][i], 0, 0, 0);
          }
    };
    fetch(wa, 0);
    fetch(wb, 1);
    __builtin_amdgcn_sched_barrier(0);  // the first weights are asked for before the pairs' numbers are waited for
#pragma unroll
    for (int i = 0; i < TIMES; ++i) arow[i] = a + (size_t)(pair[i] / a_div) * K + piece * 8;
    request(0);
    const int rounds = nchunks / 3;
    for (int it = 0; it < rounds; ++it) {  // three chunks: the roles of the weights' registers come round
      chunk(3 * it, wa, wc);
      chunk(3 * it + 1, wb, wa);
      chunk(3 * it + 2, wc, wb);
    }
    if (nchunks - 3 * rounds >= 1) chunk(3 * rounds, wa, wc);
    if (nchunks - 3 * rounds == 2) chunk(3 * rounds + 1, wb, wa);
    // a lane holds outputs n .. n+3 of either strip for the pair in column lr of each column tile
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      if (i * 16 + lr >= cnt) continue;
      OutT* to = out + (size_t)order[at + i * 16 + lr] * N;
#pragma unroll
      for (int s = 0; s < (GATED ? 1 : S); ++s) {
        const int n = n0 + s * 16 + 4 * lg;
        if (n >= N) continue;  // N % 4 == 0
        __attribute__((aligned(16))) OutT v[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float z = acc[s][i][r];
          if (GATED) z = gate_times_up(to_f32((bf16)z), to_f32((bf16)acc[S - 1][i][r]), limit);  // the two products rounded as if stored
          if (MODE == MOE_RELU2) { z = fmaxf(to_f32((bf16)z), 0.f); z *= z; }
          v[r] = from_f32<OutT>(z);
        }
        if constexpr (sizeof(OutT) == 4) *reinterpret_cast<float4*>(to + n) = *reinterpret_cast<const float4*>(v);
        else *reinterpret_cast<uint2*>(to + n) = *reinterpret_cast<const uint2*>(v);
      }
    }
  };
  const int col_tiles = (cnt + 15) >> 4;
  if (col_tiles == 4) run(std::integral_constant<int, 4>{});
  else if (col_tiles == 3) run(std::integral_constant<int, 3>{});
  else if (col_tiles == 2) run(std::integral_constant<int, 2>{});
  else run(std::integral_constant<int, 1>{});
}

// Tiles of 128 pairs: the same products, the same bits, with both operands in LDS by copies that pass no register (`wide_tile.h`); the
// pairs' rows of a are where the copies' lanes find them.  A tile's first 64 pairs are the first four waves', whose neighbours on their
// SIMDs are the other four: where a tile has no more, those only copy.
template <int MODE, typename OutT, int FN, int RA, int RW>
__global__ __launch_bounds__(512, 2) void moe_gemm_tile_kernel(const bf16* __restrict__ a, int a_div, const bf16* __restrict__ w, int N, int K,
                                                               const int* __restrict__ order, const int* __restrict__ tiles,
                                                               const int* __restrict__ counts, OutT* __restrict__ out, float limit, int strips) {
  using T = wide::Tile<2, 4, 4, FN, RA, RW, true>;
  static_assert(T::TM == MOE_TILE, "a tile's pairs");
  constexpr bool GATED = MODE == MOE_GATED;
  constexpr int ACROSS = GATED ? T::TN / 2 : T::TN;  // outputs of a workgroup
  extern __shared__ __attribute__((aligned(128))) char tile_lds[];
  const int live = counts[0], total = live * strips, per_xcd = (total + 7) >> 3;
  const int place = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
  if ((int)(blockIdx.x >> 3) >= per_xcd || place >= total) return;
  const int strip = place / live, tile = place - strip * live;
  const int e = tiles[3 * tile], at = tiles[3 * tile + 1], cnt = min(tiles[3 * tile + 2], MOE_TILE);
  const int lane = threadIdx.x & (WAVE - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const int lr = lane & 15, lg = lane >> 4, wm = wave >> 2, wn = wave & 3;
  const int n0 = strip * ACROSS;
  const int units = K / wide::UNIT, turn = (int)((unsigned)(n0 / (GATED ? 128 : 256) * 5 + e * 3) % (unsigned)(K / 128)) * 2;
  auto column = [&](int t) { const int u = min(t, units - 1) + turn; return (unsigned)(u >= units ? u - units : u) * wide::ROW_BYTES; };

  const unsigned pitch = (unsigned)K * 2u, NW = GATED ? 2 * N : N;
  const __amdgpu_buffer_rsrc_t a_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(a), 0, (int)0xfffffff0u, 0x00020000);
  const __amdgpu_buffer_rsrc_t w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(w) + (size_t)e * NW * K, 0, (int)(NW * pitch), 0x00020000);
  unsigned a_at[T::A_COPIES], w_at[T::W_COPIES];
#pragma unroll
  for (int i = 0; i < T::A_COPIES; ++i) {  // rows beyond the tile's pairs repeat its last
    const int row = T::row_of(i, wave, lane);
    a_at[i] = (unsigned)(order[at + min(row, cnt - 1)] / a_div) * pitch + T::piece_of(row, lane);
  }
#pragma unroll
  for (int i = 0; i < T::W_COPIES; ++i) {  // rows beyond N repeat the last; which row lies where: so that a lane's sums are neighbours
    const int row = T::row_of(i, wave, lane);
    const int column_of_waves = row / (16 * FN), q = row % (16 * FN), f = q >> 4, g = (q >> 2) & 3, r = q & 3;
    int n;
    if constexpr (GATED) n = min(n0 + column_of_waves * 8 * FN + g * 2 * FN + 2 * f + (r & 1), N - 1) + (r >> 1) * N;
    else if constexpr (sizeof(OutT) == 4) n = min(n0 + row, N - 1);
    else n = min(n0 + column_of_waves * 16 * FN + (f & ~1) * 16 + 8 * g + 4 * (f & 1) + r, N - 1);
    w_at[i] = (unsigned)n * pitch + T::piece_of(row, lane);
  }
  floatx4 acc[4][FN];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
  const bool idle = wm * 64 >= cnt;
  T::run(tile_lds, a_buf, w_buf, a_at, w_at, wave, wm, wn, lane, units, column, acc, idle);
  if (idle) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = wm * 64 + i * 16 + lr;
    if (row >= cnt) continue;
    OutT* to = out + (size_t)order[at + row] * N;
    if constexpr (GATED) {
      const int n = n0 + wn * 8 * FN + lg * 2 * FN;
      alignas(16) bf16 v[2 * FN];
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int r = 0; r < 2; ++r) v[2 * j + r] = (bf16)gate_times_up(to_f32((bf16)acc[i][j][r]), to_f32((bf16)acc[i][j][2 + r]), limit);
      if (n >= N) continue;  // N % 16 == 0
      if constexpr (FN == 4) *reinterpret_cast<u32x4*>(to + n) = *reinterpret_cast<const u32x4*>(v);
      else *reinterpret_cast<uint2*>(to + n) = *reinterpret_cast<const uint2*>(v);
    } else if constexpr (sizeof(OutT) == 4) {
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + wn * 16 * FN + j * 16 + 4 * lg;
        if (n < N) *reinterpret_cast<floatx4*>(to + n) = acc[i][j];
      }
    } else {
#pragma unroll
      for (int j = 0; j < FN; j += 2) {
        const int n = n0 + wn * 16 * FN + j * 16 + 8 * lg;
        alignas(16) bf16 v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          float z = acc[i][j + (r >> 2)][r & 3];
          if (MODE == MOE_RELU2) { z = fmaxf(to_f32((bf16)z), 0.f); z *= z; }
          v[r] = (bf16)z;
        }
        if (n < N) *reinterpret_cast<u32x4*>(to + n) = *reinterpret_cast<const u32x4*>(v);
      }
    }
  }
}

template <int MODE, typename OutT, int FN, int RA, int RW>
static int launch_moe_tile(const void* a, int a_div, const void* w, int N, int K, const int* order, const int* tiles, const int* counts,
                           int max_tiles, void* out, float limit, hipStream_t stream) {
  using T = wide::Tile<2, 4, 4, FN, RA, RW, true>;
  const int across = MODE == MOE_GATED ? T::TN / 2 : T::TN, strips = (N + across - 1) / across;
  if ((long long)strips * max_tiles > 0x7ffff8ll) return AS_BAD_SHAPE;
  auto kernel = moe_gemm_tile_kernel<MODE, OutT, FN, RA, RW>;
  static bool raised = false;
  if (!raised) {
    if (hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, T::LDS) != hipSuccess) return AS_LAUNCH_FAILED;
    raised = true;
  }
  kernel<<<(strips * max_tiles + 7) / 8 * 8, 512, T::LDS, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (OutT*)out,
                                                                    limit, strips);
  return launch_status();
}

// fp32: plain multiply-add, every output one chain over k in order.  A thread owns an output and, of every
// sixteen of the tile's pairs in turn, four.
template <bool GATED, bool RELU2 = false>
__global__ __launch_bounds__(256) void moe_gemm_f32_kernel(const float* __restrict__ a, int a_div,
                                                           const float* __restrict__ w, int N, int K,
                                                           const int* __restrict__ order,
                                                           const int* __restrict__ tiles,
                                                           const int* __restrict__ counts, float* __restrict__ out,
                                                           float limit) {
  const int tile = blockIdx.y;
  if (tile >= counts[0]) return;
  const int e = tiles[3 * tile], at = tiles[3 * tile + 1], cnt = tiles[3 * tile + 2];
  const int n = blockIdx.x * MOE_STRIP + (threadIdx.x & 63), quarter = threadIdx.x >> 6;
  if (n >= N) return;
  const int NW = GATED ? 2 * N : N;
  const float* wrow = w + ((size_t)e * NW + n) * K;
  const float* urow = w + ((size_t)e * NW + N + n) * K;
  for (int base = 0; base < cnt; base += 16) {
    int pairs[4];
    const float* arow[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int place = base + quarter * 4 + i;
      pairs[i] = place < cnt ? order[at + place] : -1;
      arow[i] = a + (size_t)(pairs[i] < 0 ? 0 : pairs[i] / a_div) * K;
    }
    if (pairs[0] < 0) continue;
    float acc[4] = {0.f, 0.f, 0.f, 0.f}, acc_up[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k = 0; k < K; ++k) {
      const float wv = wrow[k], uv = GATED ? urow[k] : 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float av = arow[i][k];
        acc[i] = fmaf(wv, av, acc[i]);
        if (GATED) acc_up[i] = fmaf(uv, av, acc_up[i]);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (pairs[i] < 0) continue;
      float v = acc[i];
      if (GATED) v = gate_times_up(v, acc_up[i], limit);
      if (RELU2) v = fmaxf(v, 0.f) * fmaxf(v, 0.f);
      out[(size_t)pairs[i] * N + n] = v;
    }
  }
}

// out_dtype: DT_BF16 or DT_F32 for the bf16 product's results (fp32 where several experts' outputs
// are still to be added up); the fp32 product writes fp32.
// gated: 0: the product; 1: act(gate) * up (limit 0: silu(gate) * up; > 0: the gated activation with limits);
// 2: relu(product)^2 (an expert without a gate).
// size: of the route's tiles, 64 or 128.  across: weight rows that a tile of 128 pairs is multiplied with in a workgroup, 256 or 128.
extern "C" int as_moe_gemm(const void* a, int dtype, int a_div, const void* w, int N, int K, int gated, const int* order,
                           const int* tiles, const int* counts, int max_tiles, void* out, int out_dtype, float limit,
                           int size, int across, hipStream_t stream) {
  if (max_tiles <= 0) return AS_OK;
  if (N <= 0 || K <= 0 || a_div <= 0 || max_tiles > 65535 || (size != MOE_HALF && size != MOE_TILE) || (across != 128 && across != 256)) return AS_BAD_SHAPE;
  dim3 grid((N + MOE_STRIP - 1) / MOE_STRIP, max_tiles);
  if (dtype == DT_F32) {
    if (out_dtype != DT_F32) return AS_BAD_DTYPE;
    if (gated == 2) moe_gemm_f32_kernel<false, true><<<grid, 256, 0, stream>>>((const float*)a, a_div, (const float*)w, N, K, order, tiles, counts, (float*)out, limit);
    else if (gated) moe_gemm_f32_kernel<true><<<grid, 256, 0, stream>>>((const float*)a, a_div, (const float*)w, N, K, order, tiles, counts, (float*)out, limit);
    else moe_gemm_f32_kernel<false><<<grid, 256, 0, stream>>>((const float*)a, a_div, (const float*)w, N, K, order, tiles, counts, (float*)out, limit);
    return launch_status();
  }
  if (dtype != DT_BF16) return AS_BAD_DTYPE;
  const unsigned long long expert_bytes = (unsigned long long)(gated == 1 ? 2 : 1) * N * K * 2ull;  // 32-bit offsets within an expert
  if (K % 128 == 0 && N % 16 == 0 && (((uintptr_t)a | (uintptr_t)w | (uintptr_t)out) & 15) == 0 && expert_bytes <= 0xf0000000ull &&
      (gated ? out_dtype == DT_BF16 : out_dtype == DT_BF16 || out_dtype == DT_F32)) {
    if (size == MOE_TILE && (unsigned long long)max_tiles * MOE_TILE * K * 2 <= 0xf0000000ull) {  // 32-bit offsets among the pairs' rows, too
#define TILED(MODE, T)                                                                                                                       \
  return across == 256 ? launch_moe_tile<MODE, T, 4, 3, 3>(a, a_div, w, N, K, order, tiles, counts, max_tiles, out, limit, stream)            \
                       : launch_moe_tile<MODE, T, 2, 4, 4>(a, a_div, w, N, K, order, tiles, counts, max_tiles, out, limit, stream)
      if (gated == 1) TILED(MOE_GATED, bf16);
      if (gated) TILED(MOE_RELU2, bf16);
      if (out_dtype == DT_BF16) TILED(MOE_PLAIN, bf16);
      TILED(MOE_PLAIN, float);
#undef TILED
    }
    if (size == MOE_HALF) {
      const dim3 half_grid((N + 63) / 64, max_tiles);
#define STREAM(MODE, T) \
  moe_gemm_stream_kernel<MODE, T><<<half_grid, 256, 0, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (T*)out, limit)
      if (gated == 1) STREAM(MOE_GATED, bf16);
      else if (gated) STREAM(MOE_RELU2, bf16);
      else if (out_dtype == DT_BF16) STREAM(MOE_PLAIN, bf16);
      else STREAM(MOE_PLAIN, float);
#undef STREAM
      return launch_status();
    }
  }
  grid.z = size / MOE_HALF;
  if (gated == 2) {
    if (out_dtype != DT_BF16) return AS_BAD_DTYPE;
    moe_gemm_bf16_kernel<false, bf16, true><<<grid, 256, 0, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (bf16*)out, limit);
  } else if (gated) {
    if (out_dtype != DT_BF16) return AS_BAD_DTYPE;
    moe_gemm_bf16_kernel<true, bf16><<<grid, 256, 0, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (bf16*)out, limit);
  } else if (out_dtype == DT_BF16) {
    moe_gemm_bf16_kernel<false, bf16><<<grid, 256, 0, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (bf16*)out, limit);
  } else if (out_dtype == DT_F32) {
    moe_gemm_bf16_kernel<false, float><<<grid, 256, 0, stream>>>((const bf16*)a, a_div, (const bf16*)w, N, K, order, tiles, counts, (float*)out, limit);
  } else {
    return AS_BAD_DTYPE;
  }
  return launch_status();
}

// out[t, n] = sum over a token's `top` pairs of weight * pair_weight[t * top + j] * pair_out[t * top + j, n]
// (+ add[t, n]); fp32 in, T out.  pair_weight null: every pair weighs `weight`; add (T) null: nothing is added.
// same [T, N] (null: none) with pair_expert: a pair whose expert is numbered `experts` or more has same[t] as its output.
template <typename T>
__global__ void moe_combine_kernel(const float* __restrict__ pair_out, int top, float weight, int N,
                                   T* __restrict__ out, size_t total, const float* __restrict__ pair_weight,
                                   const T* __restrict__ add, const T* __restrict__ same,
                                   const int* __restrict__ pair_expert, int experts) {
  const size_t stride = (size_t)gridDim.x * blockDim.x;
  for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total; idx += stride) {
    const size_t t = idx / N;
    const int n = (int)(idx % N);
    float s = 0.f;
    for (int j = 0; j < top; ++j) {
      const bool is_same = same && pair_expert[t * top + j] >= experts;
      s += weight * (pair_weight ? pair_weight[t * top + j] : 1.f) * (is_same ? to_f32(same[idx]) : pair_out[(t * top + j) * N + n]);
    }
    if (add) s += to_f32(add[idx]);
    out[idx] = from_f32<T>(s);
  }
}

// The same for rows of whole pieces of four values on 16 (outputs, 8 in bf16) bytes: a workgroup a token and 1,024 of its columns (3,000 pairs of
// 2,048 for 1,500 tokens, 31 MB: value by value 10.5 us, now 6.6).
template <typename T>
__global__ __launch_bounds__(256) void moe_combine_four_kernel(const float* __restrict__ pair_out, int top, float weight, int N,
                                                               T* __restrict__ out, const float* __restrict__ pair_weight,
                                                               const T* __restrict__ add, const T* __restrict__ same,
                                                               const int* __restrict__ pair_expert, int experts) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  typedef T tx4 __attribute__((ext_vector_type(4)));
  const size_t t = blockIdx.x;
  const int n = (blockIdx.y * 256 + threadIdx.x) * 4;
  if (n >= N) return;
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
  for (int j = 0; j < top; ++j) {
    const size_t pair = t * top + j;
    const bool is_same = same && pair_expert[pair] >= experts;
    const f32x4 v = is_same ? __builtin_convertvector(*reinterpret_cast<const tx4*>(same + t * N + n), f32x4)
                            : *reinterpret_cast<const f32x4*>(pair_out + pair * N + n);
    s += weight * (pair_weight ? pair_weight[pair] : 1.f) * v;
  }
  if (add) s += __builtin_convertvector(*reinterpret_cast<const tx4*>(add + t * N + n), f32x4);
  *reinterpret_cast<tx4*>(out + t * N + n) = __builtin_convertvector(s, tx4);
}

extern "C" int as_moe_combine(const float* pair_out, int top, float weight, int N, void* out, int out_dtype,
                              int num_tokens, const float* pair_weight, const void* add, const void* same,
                              const int* pair_expert, int experts, hipStream_t stream) {
  if (num_tokens <= 0) return AS_OK;
  if (top <= 0 || N <= 0 || (same && !pair_expert)) return AS_BAD_SHAPE;
  const size_t total = (size_t)num_tokens * N, want = (total + 255) / 256;
  const int blocks = (int)(want > 8192 ? 8192 : want);
  const uintptr_t typed = (uintptr_t)out | (uintptr_t)add | (uintptr_t)same;
  if ((N & 3) == 0 && ((uintptr_t)pair_out & 15) == 0 && (typed & (out_dtype == DT_F32 ? 15 : 7)) == 0 && (N + 1023) / 1024 <= 65535 &&
      (out_dtype == DT_F32 || out_dtype == DT_BF16)) {
    const dim3 grid(num_tokens, (N + 1023) / 1024);
    if (out_dtype == DT_F32) moe_combine_four_kernel<float><<<grid, 256, 0, stream>>>(pair_out, top, weight, N, (float*)out, pair_weight, (const float*)add, (const float*)same, pair_expert, experts);
    else moe_combine_four_kernel<bf16><<<grid, 256, 0, stream>>>(pair_out, top, weight, N, (bf16*)out, pair_weight, (const bf16*)add, (const bf16*)same, pair_expert, experts);
    return launch_status();
  }
  if (out_dtype == DT_F32) moe_combine_kernel<float><<<blocks, 256, 0, stream>>>(pair_out, top, weight, N, (float*)out, total, pair_weight, (const float*)add, (const float*)same, pair_expert, experts);
  else if (out_dtype == DT_BF16) moe_combine_kernel<bf16><<<blocks, 256, 0, stream>>>(pair_out, top, weight, N, (bf16*)out, total, pair_weight, (const bf16*)add, (const bf16*)same, pair_expert, experts);
  else return AS_BAD_DTYPE;
  return launch_status();
}
