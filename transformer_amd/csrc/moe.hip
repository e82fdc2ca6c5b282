// Routed feed-forward: every token is sent to `top` of E small feed-forward layers.
//
//   moe_route   : scores = f(router logits) per token (sigmoid, or softmax over the experts),
//                 the `top` largest (lowest index among equals), optionally renormalised
//   moe_plan    : the (token, choice) pairs ordered by expert: each expert's pairs take a run
//                 of rows that starts on a multiple of 16, so a tile of 16 rows belongs to one
//                 expert; the row count is bounded by pairs + 15 * min(pairs, E) whatever the routing is,
//                 so a step's launches do not depend on the data
//   moe_gather  : the ordered rows of activations, each times its pair's weight when the weight
//                 acts on the expert's input
//   moe_gemm    : C[rows of a tile] = A[rows] * W[expert of the tile]^T for all tiles, with an
//                 optional activation; float32 chains on the vector ALU, or the matrix cores
//                 (v_mfma_f32_16x16x32_bf16) for bfloat16: operands through LDS for the many
//                 tiles of a prompt, K divided among the waves for the few of a single-token step
//   moe_combine : delta[t] = sum of the token's pairs' rows (times the weight when it acts on
//                 the output) + sigmoid(shared gate) * the shared expert's rows
//
// Choices from E on are identity experts: they have no rows and no matrices, and moe_combine adds the
// token's own row times the pair's weight for them.
//
// Router scores, weights and all sums are float32.
#include "common.h"

#define MOE_TILE 16

// ------------------------------------------------------------------ routing
// logits: [nt, ld] float32, the first E columns of a row are the router's. mode 0: sigmoid
// scores; 1: softmax over the experts. renorm: the chosen weights are divided by their sum
// (with mode 1 that is the softmax over the chosen logits alone). bias [E] or null: added to
// the logits first. groups > 1: the experts form that many equal groups of neighbours, a group
// counts as its largest score, and only experts of the `keep` best groups (the lowest index
// among equals) can be chosen. correction [E] or null: the choice compares score + correction, the
// weights are the scores without it. factor: the weights are multiplied by it last.
struct MoeRoute {
  const float* logits;
  int ld, E, top, mode, renorm;
  const float* bias;
  int groups, keep;
  const float* correction;
  float factor;
  // floats of LDS that a token takes: a score per expert, one per group, and with a correction the plain scores
  __host__ __device__ int lds() const { return E + groups + (correction ? E : 0); }
};

// the wave's LDS writes before this are seen by its reads behind it
__device__ __forceinline__ void moe_wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// the scores of groups that do not stay, in the wave's LDS, become -inf
__device__ __forceinline__ void moe_keep_groups(const MoeRoute& p, float* sc, int lane) {
  const int E = p.E, groups = p.groups, keep = p.keep;
  float* gs = sc + E;
  const int size = E / groups;
  for (int g = lane; g < groups; g += 64) {
    float best = -INFINITY;
    for (int e = g * size; e < (g + 1) * size; ++e) best = fmaxf(best, sc[e]);
    gs[g] = best;
  }
  moe_wave_sync();
  // a group stays when fewer than `keep` groups come before it in the order (score down, index up)
  for (int g = lane; g < groups; g += 64) {
    const float mine = gs[g];
    int ahead = 0;
    for (int o = 0; o < groups; ++o) ahead += (gs[o] > mine || (gs[o] == mine && o < g)) ? 1 : 0;
    if (ahead >= keep)
      for (int e = g * size; e < (g + 1) * size; ++e) sc[e] = -INFINITY;
  }
  moe_wave_sync();
}

// the largest of 64 lanes' numbers, in every lane; NaN is no number
__device__ __forceinline__ float moe_max(float v) {
  v = fmaxf(v, ta_dpp<0xB1>(v));
  v = fmaxf(v, ta_dpp<0x4E>(v));
  v = fmaxf(v, ta_dpp<0x141>(v));
  v = fmaxf(v, ta_dpp<0x140>(v));
  auto row = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
  return fmaxf(fmaxf(row(0), row(16)), fmaxf(row(32), row(48)));
}

// One wave routes token t; chosen and weight are the token's own `top` places. 64 R scores and 64 choices or fewer: the scores
// stay in registers, a choice is a maximum over the lanes without LDS and a look at who has it, and its weight waits in lane j
// instead of going to memory and back before it is divided by the sum. What bounds it: the chain of `top` choices. us in LDS /
// so, with the plan: 4 tokens, 4 of 32 6.4 / 3.8; 2, 6 of 64 7.6 / 4.1; 16, 8 of 256 in eight groups 18.7 / 13.1; the routing alone of
// 2,943 tokens, 6 of 64, 8.0 / 4.3.
template <int R>
__device__ __forceinline__ void moe_route_few(const MoeRoute& p, size_t t, float* sc, int* chosen, float* weight) {
  const int lane = threadIdx.x % TA_WAVE;
  float s[R], plain[R];
  float mx = -INFINITY;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int e = lane + 64 * k;
    s[k] = e < p.E ? p.logits[t * p.ld + e] + (p.bias ? p.bias[e] : 0.f) : -INFINITY;
    mx = fmaxf(mx, s[k]);
  }
  mx = moe_max(mx);
  float sum = 0.f;
#pragma unroll
  for (int k = 0; k < R; ++k) {
    if (lane + 64 * k >= p.E) continue;
    s[k] = p.mode == 0 ? 1.0f / (1.0f + expf(-s[k])) : expf(s[k] - mx);
    sum += s[k];
  }
  sum = wave_sum(sum);
#pragma unroll
  for (int k = 0; k < R; ++k) {
    const int e = lane + 64 * k;
    plain[k] = s[k];
    if (p.correction && e < p.E) {
      plain[k] = p.mode == 0 ? s[k] : s[k] / sum;
      s[k] = plain[k] + p.correction[e];
    }
  }
  if (p.groups > 1) {
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (lane + 64 * k < p.E) sc[lane + 64 * k] = s[k];
    moe_wave_sync();
    moe_keep_groups(p, sc, lane);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (lane + 64 * k < p.E) s[k] = sc[lane + 64 * k];
  }
  float total = 0.f, my_weight = 0.f;
  int my_choice = 0;
  for (int j = 0; j < p.top; ++j) {
    float best = -INFINITY;
#pragma unroll
    for (int k = 0; k < R; ++k) best = fmaxf(best, s[k]);
    best = moe_max(best);
    // the lowest index among equals; scores of a token that are all NaN choose nobody
    int at = 0x7fffffff;
    float w = p.correction ? 0.f : best;
#pragma unroll
    for (int k = R - 1; k >= 0; --k) {
      const unsigned long long who = __ballot(s[k] == best && best > -INFINITY);
      if (who) {
        const int l = __builtin_amdgcn_readfirstlane(__ffsll(who) - 1);
        at = 64 * k + l;
        w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(p.correction ? plain[k] : s[k]), l));
      }
    }
    if (!p.correction && p.mode != 0) w = w / sum;
    total += w;
    if (lane == j) my_choice = at, my_weight = w;
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (lane + 64 * k == at) s[k] = -INFINITY;
  }
  if (lane < p.top) {
    chosen[lane] = my_choice;
    weight[lane] = p.renorm ? my_weight / total * p.factor : my_weight * p.factor;
  }
}

// the same of any number of scores, in LDS
__device__ void moe_route_token(const MoeRoute& p, size_t t, float* sc, int* chosen, float* weight) {
  const float *logits = p.logits, *bias = p.bias, *correction = p.correction;
  const int ld = p.ld, E = p.E, top = p.top, mode = p.mode, groups = p.groups;
  float* plain = sc + E + groups;
  const int lane = threadIdx.x % TA_WAVE;
  float mx = -INFINITY;
  for (int e = lane; e < E; e += 64) mx = fmaxf(mx, logits[t * ld + e] + (bias ? bias[e] : 0.f));
  mx = wave_max(mx);
  float sum = 0.f;
  for (int e = lane; e < E; e += 64) {
    const float z = logits[t * ld + e] + (bias ? bias[e] : 0.f);
    const float s = mode == 0 ? 1.0f / (1.0f + expf(-z)) : expf(z - mx);
    sc[e] = s;
    sum += s;
  }
  sum = wave_sum(sum);
  if (correction) {                       // (a lane meets the entries that it wrote itself)
    for (int e = lane; e < E; e += 64) {
      const float s = mode == 0 ? sc[e] : sc[e] / sum;
      plain[e] = s;
      sc[e] = s + correction[e];
    }
  }
  moe_wave_sync();
  if (groups > 1) moe_keep_groups(p, sc, lane);
  float total = 0.f;
  for (int j = 0; j < top; ++j) {
    float best = -INFINITY;
    int at = 0x7fffffff;
    for (int e = lane; e < E; e += 64) {
      const float s = sc[e];
      if (s > best) { best = s; at = e; }       // ascending e: the lowest index among equals
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      const float ob = __shfl_xor(best, o, TA_WAVE);
      const int oa = __shfl_xor(at, o, TA_WAVE);
      if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
    }
    // scores of a token that are all NaN choose nobody: such a token touches no LDS but its own
    const float w = correction ? (at < E ? plain[at] : 0.f) : mode == 0 ? best : best / sum;
    if (lane == 0) {
      chosen[j] = at;
      weight[j] = p.renorm ? w : w * p.factor;
    }
    total += w;
    moe_wave_sync();
    if (lane == 0 && at < E) sc[at] = -INFINITY;
    moe_wave_sync();
  }
  if (p.renorm) {
    moe_wave_sync();
    for (int j = lane; j < top; j += 64) weight[j] = weight[j] / total * p.factor;
  }
}

// R: 64 R scores in registers, or 0
template <int R>
__global__ __launch_bounds__(64) void moe_route_kernel(MoeRoute p, int* __restrict__ chosen, float* __restrict__ weight) {
  extern __shared__ float sc[];
  const size_t t = blockIdx.x;
  if constexpr (R > 0) moe_route_few<R>(p, t, sc, chosen + t * p.top, weight + t * p.top);
  else moe_route_token(p, t, sc, chosen + t * p.top, weight + t * p.top);
}

extern "C" int ta_moe_route(hipStream_t stream, const float* logits, const float* bias, int ld, int nt, int E,
                            int top, int mode, int renorm, int groups, int keep, const float* correction,
                            float factor, int* chosen, float* weight) {
  TA_REQUIRE(nt >= 0 && E >= 1 && E <= 8192 && top >= 1 && top <= E && ld >= E && (mode == 0 || mode == 1),
             "ta_moe_route: bad sizes nt=%d experts=%d top=%d ld=%d", nt, E, top, ld);
  TA_REQUIRE(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (E / groups),
             "ta_moe_route: %d experts in %d groups of which %d stay do not hold %d choices", E, groups, keep, top);
  if (nt == 0) return 0;
  const size_t lds = ((size_t)E + groups + (correction ? E : 0)) * sizeof(float);
  TA_REQUIRE(lds <= 65536, "ta_moe_route: %d experts in %d groups do not fit the LDS", E, groups);
  const MoeRoute p = {logits, ld, E, top, mode, renorm, bias, groups, keep, correction, factor};
  if (E <= 64 && top <= 64) moe_route_kernel<1><<<nt, 64, lds, stream>>>(p, chosen, weight);
  else if (E <= 256 && top <= 64) moe_route_kernel<4><<<nt, 64, lds, stream>>>(p, chosen, weight);
  else moe_route_kernel<0><<<nt, 64, lds, stream>>>(p, chosen, weight);
  return ta_check_launch("ta_moe_route");
}

// ------------------------------------------------------------------ ordering the pairs by expert
// One workgroup. row_pair: [max_rows] pair index of every ordered row, -1 for a row that only
// fills a tile; tile_expert: [max_rows / 16], -1 for a tile past the last; pair_row: [pairs],
// -1 for a pair whose choice is no expert with matrices (E or more).
__global__ __launch_bounds__(1024) void moe_plan_kernel(const int* __restrict__ chosen, int pairs, int E,
                                                        int max_rows, int* __restrict__ row_pair,
                                                        int* __restrict__ tile_expert, int* __restrict__ pair_row) {
  extern __shared__ int sh[];             // count [E], start [E + 1]
  int* count = sh;
  int* start = sh + E;
  for (int e = threadIdx.x; e < E; e += 1024) count[e] = 0;
  for (int i = threadIdx.x; i < max_rows; i += 1024) row_pair[i] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += 1024)
    if (chosen[i] < E) atomicAdd(&count[chosen[i]], 1);
  __syncthreads();
  if (threadIdx.x == 0) {
    int at = 0;
    for (int e = 0; e < E; ++e) {
      start[e] = at;
      at += (count[e] + MOE_TILE - 1) / MOE_TILE * MOE_TILE;
    }
    start[E] = at;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < max_rows / MOE_TILE; i += 1024) {
    const int r = i * MOE_TILE;
    int e = -1;
    if (r < start[E]) {                   // the last expert whose run starts at or before r
      int lo = 0, hi = E - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= r) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    tile_expert[i] = e;
  }
  for (int e = threadIdx.x; e < E; e += 1024) count[e] = 0;
  __syncthreads();
  // the order of an expert's rows among themselves does not matter: every row is computed alone
  for (int i = threadIdx.x; i < pairs; i += 1024) {
    const int e = chosen[i];
    if (e >= E) {
      pair_row[i] = -1;
      continue;
    }
    const int r = start[e] + atomicAdd(&count[e], 1);
    row_pair[r] = i;
    pair_row[i] = r;
  }
}

extern "C" int ta_moe_max_rows(int pairs, int E) {
  const long long n = (long long)pairs + (long long)(MOE_TILE - 1) * (pairs < E ? pairs : E);
  const long long r = (n + MOE_TILE - 1) / MOE_TILE * MOE_TILE;
  return r > 2147483647ll ? -1 : (int)r;
}

extern "C" int ta_moe_plan(hipStream_t stream, const int* chosen, int pairs, int E, int max_rows, int* row_pair,
                           int* tile_expert, int* pair_row) {
  TA_REQUIRE(pairs >= 0 && E >= 1 && E <= 8192, "ta_moe_plan: bad sizes pairs=%d experts=%d", pairs, E);
  TA_REQUIRE(max_rows == ta_moe_max_rows(pairs, E), "ta_moe_plan: %d rows for %d pairs of %d experts", max_rows, pairs, E);
  moe_plan_kernel<<<1, 1024, (size_t)(2 * E + 1) * sizeof(int), stream>>>(chosen, pairs, E, max_rows, row_pair,
                                                                        tile_expert, pair_row);
  return ta_check_launch("ta_moe_plan");
}

// Routing and ordering for a step of few tokens in one launch: a workgroup of 16 waves, a wave a token, then the
// plan as above with the experts' runs added up by one wave: one launch and no trip between the two.
#define MOE_FEW_TOKENS 16
#define MOE_FEW_EXPERTS 256
template <int R>
__global__ __launch_bounds__(1024) void moe_route_plan_kernel(MoeRoute p, int nt, int experts, int max_rows,
                                                              int* __restrict__ chosen, float* __restrict__ weight,
                                                              int* __restrict__ row_pair, int* __restrict__ tile_expert,
                                                              int* __restrict__ pair_row) {
  extern __shared__ float moe_few[];      // a token's scores for every wave, then count [experts], start [experts + 1], chosen [pairs]
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE, pairs = nt * p.top;
  int* count = reinterpret_cast<int*>(moe_few + MOE_FEW_TOKENS * p.lds());
  int* start = count + experts;
  int* mine = start + experts + 1;
  for (int e = threadIdx.x; e < experts; e += 1024) count[e] = 0;
  for (int i = threadIdx.x; i < max_rows; i += 1024) row_pair[i] = -1;
  if (wave < nt) {
    moe_route_few<R>(p, wave, moe_few + wave * p.lds(), mine + wave * p.top, weight + wave * p.top);
    moe_wave_sync();
    for (int j = lane; j < p.top; j += TA_WAVE) chosen[wave * p.top + j] = mine[wave * p.top + j];
  }
  __syncthreads();
  for (int i = threadIdx.x; i < pairs; i += 1024)
    if (mine[i] < experts) atomicAdd(&count[mine[i]], 1);
  __syncthreads();
  if (wave == 0) {
    int run = 0;
    for (int e0 = 0; e0 < experts; e0 += TA_WAVE) {
      const int e = e0 + lane;
      const int n = e < experts ? (count[e] + MOE_TILE - 1) / MOE_TILE * MOE_TILE : 0;
      int inc = n;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const int up = __shfl_up(inc, o, TA_WAVE);
        if (lane >= o) inc += up;
      }
      if (e < experts) {
        start[e] = run + inc - n;
        count[e] = 0;
      }
      run += __shfl(inc, TA_WAVE - 1, TA_WAVE);
    }
    if (lane == 0) start[experts] = run;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < max_rows / MOE_TILE; i += 1024) {
    const int r = i * MOE_TILE;
    int e = -1;
    if (r < start[experts]) {
      int lo = 0, hi = experts - 1;
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (start[mid] <= r) lo = mid; else hi = mid - 1;
      }
      e = lo;
    }
    tile_expert[i] = e;
  }
  for (int i = threadIdx.x; i < pairs; i += 1024) {
    const int e = mine[i];
    int r = -1;
    if (e < experts) {
      r = start[e] + atomicAdd(&count[e], 1);
      row_pair[r] = i;
    }
    pair_row[i] = r;
  }
}

// Whether ta_moe_route_plan takes a step of this many tokens.
extern "C" int ta_moe_few_tokens(int nt, int E, int top) {
  return nt >= 1 && nt <= MOE_FEW_TOKENS && E <= MOE_FEW_EXPERTS && top <= 32;
}

// ta_moe_route over E scores a token, then ta_moe_plan for `experts` experts with matrices (E or fewer).
extern "C" int ta_moe_route_plan(hipStream_t stream, const float* logits, const float* bias, int ld, int nt, int E,
                                 int top, int mode, int renorm, int groups, int keep, const float* correction,
                                 float factor, int* chosen, float* weight, int experts, int max_rows, int* row_pair,
                                 int* tile_expert, int* pair_row) {
  TA_REQUIRE(ta_moe_few_tokens(nt, E, top) && E >= 1 && top >= 1 && top <= E && ld >= E && (mode == 0 || mode == 1),
             "ta_moe_route_plan: bad sizes nt=%d experts=%d top=%d ld=%d", nt, E, top, ld);
  TA_REQUIRE(groups >= 1 && E % groups == 0 && keep >= 1 && keep <= groups && top <= keep * (E / groups),
             "ta_moe_route_plan: %d experts in %d groups of which %d stay do not hold %d choices", E, groups, keep, top);
  TA_REQUIRE(experts >= 1 && experts <= E && max_rows == ta_moe_max_rows(nt * top, experts),
             "ta_moe_route_plan: %d rows for %d pairs of %d experts", max_rows, nt * top, experts);
  const MoeRoute p = {logits, ld, E, top, mode, renorm, bias, groups, keep, correction, factor};
  const size_t lds = ((size_t)MOE_FEW_TOKENS * p.lds() + 2 * experts + 1 + nt * top) * sizeof(float);
  static_assert(MOE_FEW_EXPERTS <= 256, "what a wave's registers hold");
  auto kern = E <= 64 ? moe_route_plan_kernel<1> : moe_route_plan_kernel<4>;
  kern<<<1, 1024, lds, stream>>>(p, nt, experts, max_rows, chosen, weight, row_pair, tile_expert, pair_row);
  return ta_check_launch("ta_moe_route_plan");
}

// ------------------------------------------------------------------ gathering the rows
template <typename T>
__global__ __launch_bounds__(256) void moe_gather_kernel(const T* __restrict__ h, int d, int top,
                                                         const int* __restrict__ row_pair,
                                                         const float* __restrict__ weight, T* __restrict__ out) {
  const size_t r = blockIdx.x;
  const int pair = row_pair[r];
  T* dst = out + r * d;
  if (pair < 0) {
    for (int c = threadIdx.x; c < d; c += 256) dst[c] = from_f32<T>(0.f);
    return;
  }
  const T* src = h + (size_t)(pair / top) * d;
  if (weight) {
    const float w = weight[pair];
    for (int c = threadIdx.x; c < d; c += 256) dst[c] = from_f32<T>(to_f32(src[c]) * w);
  } else {
    for (int c = threadIdx.x; c < d; c += 256) dst[c] = src[c];
  }
}

// out[r] = h[token of row r] (* weight of its pair; weight null: as it is); filling rows are zero.
extern "C" int ta_moe_gather(hipStream_t stream, int dtype, const void* h, int d, int top, const int* row_pair,
                             const float* weight, void* out, int max_rows) {
  TA_REQUIRE(d > 0 && top >= 1 && max_rows >= 0, "ta_moe_gather: bad sizes");
  if (max_rows == 0) return 0;
  if (dtype == TA_F32)
    moe_gather_kernel<float><<<max_rows, 256, 0, stream>>>((const float*)h, d, top, row_pair, weight, (float*)out);
  else if (dtype == TA_BF16)
    moe_gather_kernel<bf16_t><<<max_rows, 256, 0, stream>>>((const bf16_t*)h, d, top, row_pair, weight, (bf16_t*)out);
  else
    return ta_fail("ta_moe_gather: unknown dtype %d", dtype);
  return ta_check_launch("ta_moe_gather");
}

// ------------------------------------------------------------------ the experts' products
__device__ __forceinline__ float moe_act(int act, float z) {
  switch (act) {
    case 1: return 0.5f * z * (1.0f + erff(z * 0.7071067811865476f));
    case 2: return 0.5f * z * (1.0f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
    case 3: { const float r = fmaxf(z, 0.f); return r * r; }
    case 4: return z / (1.0f + expf(-z));
    default: return z;
  }
}

// float32 chains: a workgroup owns a tile of 16 rows and 64 columns; a thread 1 row x 4 columns.
// Every element is one ascending-k chain of fused multiply-adds.
template <typename T, typename TC>
__global__ __launch_bounds__(256) void moe_gemm_fma_kernel(const T* __restrict__ A, const T* __restrict__ W,
                                                           const int* __restrict__ tile_expert, TC* __restrict__ C,
                                                           int N, int K, int act) {
  __shared__ float As[16][MOE_TILE + 1];
  __shared__ float Ws[16][64 + 1];
  const int e = tile_expert[blockIdx.y];
  if (e < 0) return;
  const size_t r0 = (size_t)blockIdx.y * MOE_TILE;
  const int n0 = blockIdx.x * 64;
  const T* We = W + (size_t)e * N * K;
  const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
  float acc[4] = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 16) {
    {
      const int r = threadIdx.x / 16, k = k0 + threadIdx.x % 16;
      As[threadIdx.x % 16][r] = k < K ? to_f32(A[(r0 + r) * K + k]) : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int idx = threadIdx.x + 256 * i, n = idx / 16, k = k0 + idx % 16;
      Ws[idx % 16][n] = (n0 + n < N && k < K) ? to_f32(We[(size_t)(n0 + n) * K + k]) : 0.f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const float a = As[kk][tr];
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[j] = fmaf(a, Ws[kk][tc * 4 + j], acc[j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int n = n0 + tc * 4 + j;
    if (n < N) C[(r0 + tr) * N + n] = from_f32<TC>(moe_act(act, acc[j]));
  }
}

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 moe_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float moe_floatx4;
typedef uint32_t moe_u32x4 __attribute__((ext_vector_type(4)));
union MoeFrag {
  moe_bf16x8 v;
  moe_u32x4 q;
};
static __device__ __forceinline__ moe_u32x4 moe_zero4() { return moe_u32x4{0, 0, 0, 0}; }

// Matrix cores: a workgroup of 4 waves owns four neighbouring tiles of 16 rows, a wave 64
// columns of them (four 16 x 16 tiles). Neighbouring tiles of one expert form a run; a wave
// walks K once per run, in steps of 32 (a lane holds 8 consecutive k of row lane % 16 of its
// operand), and every piece of the expert's matrix that it loads serves all tiles of the run:
// a prompt's rows, of which an expert gets many, read the matrix a quarter as often; a step of
// few tokens has runs of one tile and reads every chosen expert's matrix once. The operands of
// the next step are asked for before the products of this one. K % 8 == 0; the last step's
// missing k are zero.
template <typename TC, int RUN>
__device__ __forceinline__ void moe_run(const bf16_t* __restrict__ A, const bf16_t* __restrict__ We,
                                        TC* __restrict__ C, size_t r0, int n0, int N, int K, int act, int lane) {
  const int r = lane % 16, kb = lane / 16;
  const bf16_t* arow[RUN];
#pragma unroll
  for (int u = 0; u < RUN; ++u) arow[u] = A + (r0 + 16 * u + r) * K + kb * 8;
  const bf16_t* wrow[4];
  bool wok[4];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int n = n0 + 16 * t + r;
    wok[t] = n < N;
    wrow[t] = We + (size_t)(wok[t] ? n : 0) * K + kb * 8;
  }
  moe_floatx4 acc[RUN][4];
#pragma unroll
  for (int u = 0; u < RUN; ++u)
#pragma unroll
    for (int t = 0; t < 4; ++t) acc[u][t] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
  // Three steps of 32 k are on their way while one is multiplied: a trip to memory takes several
  // times as long as a step's products. The whole steps load without a condition (a column past
  // N reads row 0 of the matrix and is never stored): a value chosen after its load would be
  // waited for where the load is issued.
  struct Step {
    MoeFrag a[RUN], w[4];
  };
  auto load = [&](Step& s, int k0) {
#pragma unroll
    for (int u = 0; u < RUN; ++u) s.a[u].q = *reinterpret_cast<const moe_u32x4*>(arow[u] + k0);
#pragma unroll
    for (int t = 0; t < 4; ++t) s.w[t].q = *reinterpret_cast<const moe_u32x4*>(wrow[t] + k0);   // other tiles read it again: it stays cached
  };
  auto mma = [&](const Step& s) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int u = 0; u < RUN; ++u)
        // register j of a lane: W row 4 * (lane / 16) + j of the tile, activation row lane % 16
        acc[u][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s.w[t].v, s.a[u].v, acc[u][t], 0, 0, 0);
  };
  const int KF = K / 32 * 32;                           // whole steps
  Step s0, s1, s2;
  if (KF > 0) load(s0, 0);
  if (KF > 32) load(s1, 32);
  for (int k0 = 0; k0 < KF; k0 += 96) {
    if (k0 + 64 < KF) load(s2, k0 + 64);
    mma(s0);
    if (k0 + 32 >= KF) break;
    if (k0 + 96 < KF) load(s0, k0 + 96);
    mma(s1);
    if (k0 + 64 >= KF) break;
    if (k0 + 128 < KF) load(s1, k0 + 128);
    mma(s2);
  }
  if (KF < K) {                                         // the last, partial step
    const bool kok = KF + kb * 8 < K;
#pragma unroll
    for (int u = 0; u < RUN; ++u) s0.a[u].q = kok ? *reinterpret_cast<const moe_u32x4*>(arow[u] + KF) : moe_zero4();
#pragma unroll
    for (int t = 0; t < 4; ++t) s0.w[t].q = kok ? *reinterpret_cast<const moe_u32x4*>(wrow[t] + KF) : moe_zero4();
    mma(s0);
  }
#pragma unroll
  for (int u = 0; u < RUN; ++u)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = n0 + 16 * t + 4 * kb + j;
        if (n < N) C[(r0 + 16 * u + r) * N + n] = from_f32<TC>(moe_act(act, acc[u][t][j]));
      }
}

template <typename TC>
__global__ __launch_bounds__(256) void moe_gemm_mfma_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                            const int* __restrict__ tile_expert, int tiles,
                                                            TC* __restrict__ C, int N, int K, int act) {
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int n0 = (blockIdx.x * 4 + wave) * 64;
  if (n0 >= N) return;
  int t = blockIdx.y * 4;
  const int t_end = t + 4 < tiles ? t + 4 : tiles;
  while (t < t_end) {
    const int e = tile_expert[t];
    if (e < 0) return;                                  // tiles past the last expert's rows
    int run = 1;
    while (t + run < t_end && tile_expert[t + run] == e) ++run;
    const bf16_t* We = W + (size_t)e * N * K;
    const size_t r0 = (size_t)t * MOE_TILE;
    if (run == 4) moe_run<TC, 4>(A, We, C, r0, n0, N, K, act, lane);
    else if (run == 3) moe_run<TC, 3>(A, We, C, r0, n0, N, K, act, lane);
    else if (run == 2) moe_run<TC, 2>(A, We, C, r0, n0, N, K, act, lane);
    else moe_run<TC, 1>(A, We, C, r0, n0, N, K, act, lane);
    t += run;
  }
}

__device__ uint4 moe_zeros;             // where a piece past K is read from (never written: zero)

// Few tiles (a step of few tokens), bound by reading the chosen experts' matrices: a workgroup owns ONE tile of 16
// rows and 16 NT rows of the matrix and its four waves divide K; the partial tiles are added in wave order through
// LDS. While 128 k are multiplied the next are on their way (16 KB a wave). The matrix comes in whole lines, sixteen lanes a
// row's 256 bytes, and takes the operands' layout in the wave's own LDS: read in that layout straight from memory, 16 bytes of
// sixteen rows at a time, it is the lines a CU touches that bind. 2 tokens of six of 64 experts of 1,408 x 4,096 (gate and up,
// then down) 49.8 -> 35 and 29.9 -> 22.4 us; 4 of four of 32 of 1,024 x 2,048 16.3 -> 14.0 and 16.2 -> 12.2.
// row_pair (or null: A holds the ordered rows): the tile's rows are read from the tokens' rows h, each times its
// pair's weight, rounded as moe_gather rounds it: a step of few tokens needs no ordered copy.
// GLU: the matrix holds gate rows, then up rows; the workgroup takes 8 NT of each and joins them.
struct MoeRows {
  const bf16_t* A;
  const int* row_pair;
  const float* weight;
  int top;
};
template <typename TC, bool GLU, int NT>
__global__ __launch_bounds__(256) void moe_gemm_mfma_splitk_kernel(MoeRows rows, const bf16_t* __restrict__ W,
                                                                   const int* __restrict__ tile_expert,
                                                                   TC* __restrict__ C, int N, int K, int act, TaGlu glu) {
  static_assert(NT == 1 || NT == 2 || NT == 4, "tiles of 16 rows of the matrix");
  static_assert(!GLU || NT > 1, "gates and ups");
  // a wave's 16 NT rows x 128 k of the matrix on their way from whole lines to the operands' layout, then its sums
  __shared__ __attribute__((aligned(16))) uint32_t stage[4][NT][1024];
  typedef float Sums[16][16 * NT + 1];
  Sums* red = reinterpret_cast<Sums*>(&stage[0][0][0]);
  const int e = tile_expert[blockIdx.y];
  if (e < 0) return;                                    // the whole workgroup: tiles past the last expert's rows
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int r = lane % 16, kb = lane / 16;
  constexpr int COLS = GLU ? 8 * NT : 16 * NT, HALF = NT / 2;     // of C
  const int n0 = blockIdx.x * COLS;
  const size_t r0 = (size_t)blockIdx.y * MOE_TILE;
  const bf16_t* We = W + (size_t)e * (GLU ? 2 : 1) * N * K;
  const int steps = (K + 31) / 32;
  const int kbeg = __builtin_amdgcn_readfirstlane(32 * (steps * wave / 4));
  const int kend = __builtin_amdgcn_readfirstlane(32 * (steps * (wave + 1) / 4));
  const int pair = rows.row_pair ? rows.row_pair[r0 + r] : 0;    // asked for before the matrix, needed behind it
  // loading: instruction i of tile t brings rows 4 i + lane / 16; a row's sixteen lanes bring its 256 bytes, permuted by the
  // row's number so that the operands' reads meet no bank twice
  const int lrow = lane / 16, lpiece = lane % 16;
  const bf16_t* wbase[2] = {We + (size_t)n0 * K, We + (size_t)(GLU ? N + n0 : n0) * K};
  uint32_t woff[NT][4];                                  // rows past N: another row, whose products are not stored
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = (GLU ? 16 * (t % HALF) : 16 * t) + 4 * i + lrow;
      woff[t][i] = (uint32_t)(n0 + n < N ? n : N - 1 - n0) * (uint32_t)K + (uint32_t)((lpiece ^ (4 * i + lrow)) * 8);
    }
  moe_floatx4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
  constexpr int DEPTH = 4;                              // steps of 32 k asked for together
  MoeFrag af[2][DEPTH], wf[2][NT][4];
  auto load_matrix = [&](int set, int k0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int k = k0 + (lpiece ^ (4 * i + lrow)) * 8;
      const bool kok = k < kend && k < K;
#pragma unroll
      for (int t = 0; t < NT; ++t)
        wf[set][t][i].q = __builtin_nontemporal_load(
            reinterpret_cast<const moe_u32x4*>(kok ? (const void*)(wbase[GLU && t >= HALF] + k0 + woff[t][i]) : (const void*)&moe_zeros));
    }
  };
  load_matrix(0, kbeg);
  __builtin_amdgcn_sched_barrier(0);
  const bf16_t* arow = rows.A + (r0 + r) * K + kb * 8;
  float factor = 1.f;
  if (rows.row_pair) {                                  // a row that only fills the tile: any token's, never read again
    arow = rows.A + (size_t)(pair >= 0 ? pair / rows.top : 0) * K + kb * 8;
    if (rows.weight) factor = pair >= 0 ? rows.weight[pair] : 0.f;
  }
  const bool weighs = rows.row_pair && rows.weight;
  auto load_rows = [&](int set, int k0) {
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      const int k = k0 + 32 * u;
      const bool kok = k < kend && k + kb * 8 < K;
      af[set][u].q = *reinterpret_cast<const moe_u32x4*>(kok ? (const void*)(arow + k) : (const void*)&moe_zeros);
    }
  };
  auto multiply = [&](int set) {
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<moe_u32x4*>(&stage[wave][t][(4 * i + lrow) * 64 + lpiece * 4]) = wf[set][t][i].q;
    // the wave reads what its other lanes wrote: LDS serves a wave's requests in order
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int u = 0; u < DEPTH; ++u) {
      if (weighs) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint32_t x = af[set][u].q[i];
          af[set][u].q[i] = f32x2_to_bf16x2_bits(__uint_as_float(x << 16) * factor, __uint_as_float(x & 0xffff0000u) * factor);
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        MoeFrag w;
        w.q = *reinterpret_cast<const moe_u32x4*>(&stage[wave][t][r * 64 + ((4 * u + kb) ^ r) * 4]);
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w.v, af[set][u].v, acc[t], 0, 0, 0);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };
  load_rows(0, kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += 64 * DEPTH) {
    const bool second = k0 + 32 * DEPTH < kend, third = k0 + 64 * DEPTH < kend;   // nothing is asked for past the wave's k
    if (second) {
      load_matrix(1, k0 + 32 * DEPTH);
      load_rows(1, k0 + 32 * DEPTH);
    }
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    __builtin_amdgcn_sched_barrier(0);
    if (third) {
      load_matrix(0, k0 + 64 * DEPTH);
      load_rows(0, k0 + 64 * DEPTH);
    }
    __builtin_amdgcn_sched_barrier(0);
    if (second) multiply(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  __syncthreads();                                      // (the waves' sums lie where the others' rows were)
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int j = 0; j < 4; ++j) red[wave][r][16 * t + 4 * kb + j] = acc[t][j];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (COLS + 15) / 16; ++i) {
    const int idx = threadIdx.x + 256 * i, row = idx / COLS, col = idx % COLS;
    if (idx >= 16 * COLS) break;
    float v = (red[0][row][col] + red[1][row][col]) + (red[2][row][col] + red[3][row][col]);
    if (GLU) {
      const int up = col + 16 * HALF;
      const float u = (red[0][row][up] + red[1][row][up]) + (red[2][row][up] + red[3][row][up]);
      // the product of its own stores gate and up in the engine's type
      v = ta_glu(glu, to_f32(from_f32<bf16_t>(v)), to_f32(from_f32<bf16_t>(u)));
    } else {
      v = moe_act(act, v);
    }
    if (n0 + col < N) C[(r0 + row) * N + n0 + col] = from_f32<TC>(v);
  }
}

// 16 NT rows of the matrix a workgroup: fewer where the tiles of 64 would leave CUs with one workgroup or none. us with 64 / 32 / 16
// rows, by tiles times blocks of 64: 4 tokens of four of 32 experts 1,024 x 2,048 (256) 13.8 / 12.6 / 10.5, 2,048 x 1,024 (512) 12.9 / 11.9 /
// 13.0, one token (64, 128) 12.2 / 8.9 / 6.7 and 8.9 / 7.6 / 7.1, 8 tokens (512, 1,024) 22.4 / 19.1 / 18.4 and 21.9 / 21.6 / 23.5; of six
// of 64 experts of 1,408 x 4,096, gated, and 4,096 x 1,408 one token (264, 384) 34.8 / 30.1 and 20.0 / 18.2 / 21.7, two (528, 768)
// 43.8 / 44.8 and 30.5 / 31.8 / 35.8.
template <typename TC, bool GLU>
static void moe_splitk(hipStream_t stream, const MoeRows& rows, const void* W, const int* tile_expert, void* C, int tiles, int N, int K,
                       int act, const TaGlu& glu) {
  const long long blocks = (long long)tiles * ((N + (GLU ? 31 : 63)) / (GLU ? 32 : 64));
#define SPLITK(NT)                                                                                                            \
  moe_gemm_mfma_splitk_kernel<TC, GLU, NT><<<dim3((N + (GLU ? 8 : 16) * NT - 1) / ((GLU ? 8 : 16) * NT), tiles), 256, 0, stream>>>( \
      rows, (const bf16_t*)W, tile_expert, (TC*)C, N, K, act, glu)
  if constexpr (!GLU)
    if (blocks <= 256) {
      SPLITK(1);
      return;
    }
  if (blocks <= 512) SPLITK(2); else SPLITK(4);
#undef SPLITK
}

// Many tiles (a prompt): operands through LDS. An expert's tiles of 16 rows are cut, from its first one on, into
// blocks of up to 16, so that its matrix is read once for every 256 rows. A workgroup of eight waves owns 256 columns
// of the blocks that begin at four neighbouring tiles (one block where the experts have four tiles or more), and what is
// sent for runs on from one block into the next. The operands go from memory to LDS without passing through registers, 64 k of
// a step at a time and so whole lines of 128 bytes: with 32 k a CU takes in 27 bytes a clock, with 64 36, and alone the loads of
// 64 experts of 2,816 x 4,096 with 256 rows each take 433 us and 368 (the load of half lines was what bounded this
// kernel). The columns, from HBM, go two steps ahead into three buffers, the rows, which other workgroups read too, one step
// into two (160 KB). A row's eight pieces of 16 bytes are permuted by the row number, so that eight rows' reads meet no bank
// twice. The waves stand in 2 x 4; each multiplies half of the block's tiles by 64 columns, and reads the operands of the
// next 32 k meanwhile, which also frees a step's buffers before its last products: one barrier every 64 k. What bounds it: few
// rows an expert, the experts' matrices from memory (4.1 TB/s); many, the loads into LDS (0.78 to 0.98 PFLOP/s).
// us with steps of 32 k, operands read when they are due / so: 64 experts of 2,816 x 4,096 at 2,943 tokens of six, unevenly routed
// 622 / 558, evenly 774 / 673, at 1,200 402 / 364; of 4,096 x 1,408 366 / 328 and 237 / 209; 32 experts of 2,048 x 1,408 at 8,000 of
// four 309 / 272, of 1,024 x 4,096 404 / 345, at 2,000 of 1,024 x 2,048 99 / 91; 8 of 28,672 x 4,096 at 4,096 of two 2,116 / 1,968;
// 8 of 1,024 x 4,096 174 / 147 and 64 of 384 x 2,048 at 6,000 of six 142 / 134. Loads for the rows of a block only, by the
// exec mask, cost more than they saved (592 against 558); an XCD's workgroups on neighbouring blocks gained where experts are
// evenly used (629) and lost where not (571, 2,210).
// Workgroups are numbered by the blocks there are: with one for every four tiles, most of them empty, the blocks of long
// runs fell on every fourth workgroup and so on a part of the XCDs and shader engines (32 experts of 2,048 x 1,408 at
// 8,000 tokens of four twice the time). Finding its number costs a workgroup some 2 us.
#define ML_BM 256
#define ML_BN 256
#define ML_BK 64
#define ML_TILES (ML_BM / MOE_TILE)
#define ML_OWN 4

static __device__ const moe_u32x4 ml_zeros = {0, 0, 0, 0};

// Multiplies 32 k of a block, UU tiles of rows from As on by 64 columns from Ws on, and while it does reads the next 32 k's: the
// columns' into the other set, a tile's rows into the registers that its last product has just left. `at`: the lane's piece.
template <int UU>
static __device__ __forceinline__ void ml_multiply(moe_floatx4 (&acc)[UU][4], MoeFrag (&af)[UU], const MoeFrag (&wf)[4], MoeFrag (&wn)[4],
                                                   const moe_u32x4* As, const moe_u32x4* Ws, int at) {
#pragma unroll
  for (int v = 0; v < 4; ++v) wn[v].q = Ws[16 * 8 * v + at];
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int u = 0; u < UU; ++u) {
#pragma unroll
    for (int v = 0; v < 4; ++v)
      // register j of a lane: column 4 * (lane / 16) + j of the tile, row lane % 16
      acc[u][v] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[v].v, af[u].v, acc[u][v], 0, 0, 0);
    af[u].q = As[16 * 8 * u + at];
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Of the windows of ML_OWN tiles in which a block begins, number `want`: its first tile, or -1 if there are fewer, and in
// `first` the first tile of that tile's run. A run's blocks begin at every `most` tiles (a power of two) from its first
// on. All eight waves, 4,096 tiles at a time: one trip to memory, three barriers. `lds`: 1.5 KB.
static __device__ __forceinline__ int ml_find(const int* __restrict__ tile_expert, int tiles, int most, int want, unsigned char* lds, int& first) {
  unsigned long long* starts_of = reinterpret_cast<unsigned long long*>(lds);            // of 64 chunks of 64 tiles: where runs start
  unsigned long long* windows_of = starts_of + 64;                                        // the windows with a block's beginning
  int* last_of = reinterpret_cast<int*>(windows_of + 64);                                 // the last start in them, or -1
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
  int begun = 0;                                        // the start of the run that reaches into these 4,096
  for (int base = 0, seen = 0; base < tiles; base += 4096) {
    int here[8];
    unsigned long long starts[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int t = base + (wave + 8 * k) * 64 + lane;
      here[k] = tile_expert[t < tiles ? t : tiles - 1];
      const int before = tile_expert[t == 0 ? 0 : t <= tiles ? t - 1 : tiles - 1];
      here[k] = t < tiles ? here[k] : -1;
      starts[k] = __ballot(t == 0 || here[k] != before);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (lane == 0) {
        starts_of[wave + 8 * k] = starts[k];
        last_of[wave + 8 * k] = starts[k] ? base + (wave + 8 * k) * 64 + 63 - __clzll((long long)starts[k]) : -1;
      }
    __syncthreads();
    int reach = last_of[lane];                          // lane c: the last start up to and with chunk c
#pragma unroll
    for (int o = 1; o < TA_WAVE; o <<= 1) {
      const int up = __shfl_up(reach, o, TA_WAVE);
      if (lane >= o && up > reach) reach = up;
    }
    const int before_ = __shfl_up(reach, 1, TA_WAVE), into = lane && before_ >= 0 ? before_ : begun;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = wave + 8 * k, t = base + c * 64 + lane;
      const unsigned long long mine = starts[k] & ((2ull << lane) - 1);
      const int carried = __builtin_amdgcn_readlane(into, c);              // by all lanes, whichever needs it
      const int from = mine ? base + c * 64 + 63 - __clzll((long long)mine) : carried;
      unsigned long long begins = __ballot(here[k] >= 0 && ((t - from) & (most - 1)) == 0);
      begins |= begins >> 2;
      if (lane == 0) windows_of[c] = (begins | begins >> 1) & 0x1111111111111111ull;
    }
    __syncthreads();
    const unsigned long long windows = windows_of[lane], runs = starts_of[lane];
    const int n = __popcll(windows);
    int upto = n;
#pragma unroll
    for (int o = 1; o < TA_WAVE; o <<= 1) {
      const int up = __shfl_up(upto, o, TA_WAVE);
      if (lane >= o) upto += up;
    }
    __syncthreads();                                    // everyone has read before the LDS is written again
    const unsigned long long there = __ballot(want - seen < upto);
    if (there) {
      const int who = __ffsll(there) - 1;               // the chunk's lane
      unsigned long long left = windows;
      for (int k = lane == who ? want - seen - (upto - n) : 0; k > 0; --k) left &= left - 1;
      const int at = left ? __ffsll(left) - 1 : 0;
      const unsigned long long mine = runs & ((2ull << at) - 1);
      const int from = mine ? base + lane * 64 + 63 - __clzll((long long)mine) : into;
      first = __builtin_amdgcn_readlane(from, who);
      return __builtin_amdgcn_readlane(base + lane * 64 + at, who);
    }
    seen += __builtin_amdgcn_readlane(upto, 63);
    const int end = __builtin_amdgcn_readlane(reach, 63);
    if (end >= 0) begun = end;
  }
  return -1;
}

// a barrier for LDS alone: what is on its way from memory stays on its way
static __device__ __forceinline__ void ml_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <typename TC, bool ACT>
__global__ __launch_bounds__(512, 2) void moe_gemm_lds_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W,
                                                           const int* __restrict__ tile_expert, int tiles, int most,
                                                           TC* __restrict__ C, int N, int K, int act) {
  extern __shared__ __attribute__((aligned(16))) unsigned char ml_lds[];
  moe_u32x4* As = reinterpret_cast<moe_u32x4*>(ml_lds);                 // [2][ML_BM * 8]
  moe_u32x4* Ws = As + 2 * ML_BM * 8;                                   // [3][ML_BN * 8]
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x / 64), lane = threadIdx.x % 64;
  const int r = lane % 16, kb = lane / 16, wr = wave / 4, wc = wave % 4;
  const int ncol = (N + ML_BN - 1) / ML_BN;
  const int want = __builtin_amdgcn_readfirstlane((int)(blockIdx.x / (unsigned)ncol));
  const int n0 = ((int)blockIdx.x - want * ncol) * ML_BN;
  // Windows without a block have no workgroup: a long run's blocks begin at every fourth window, and with a workgroup each
  // those would all be the same XCD's or shader engine's.
  int first;
  const int t0 = ml_find(tile_expert, tiles, most, want, ml_lds, first);
  if (t0 < 0) return;
  int e = tile_expert[t0];
  // The blocks that begin at this workgroup's tiles: five bits each, their tiles (none: 0)
  unsigned blocks = 0;
#pragma unroll
  for (int i = 0; i < ML_OWN; ++i) {
    const int t = t0 + i, here = t < tiles ? tile_expert[t] : -1;
    if (here != e) e = here, first = t;
    if (here >= 0 && ((t - first) & (most - 1)) == 0) {
      const int ahead = t + lane;
      const unsigned long long other = __ballot(lane >= most || ahead >= tiles || tile_expert[ahead < tiles ? ahead : t] != e);
      blocks |= (unsigned)(__ffsll(other) - 1) << (5 * i);
    }
  }
  blocks = __builtin_amdgcn_readfirstlane(blocks);
  if (blocks == 0) return;
  auto next_block = [&](int i) {                        // the first one from i on, or ML_OWN
    const unsigned left = blocks >> (5 * i);
    return __builtin_amdgcn_readfirstlane(left ? i + (__ffs(left) - 1) / 5 : ML_OWN);
  };
  auto run_of = [&](int i) { return (int)(blocks >> (5 * i) & 31u); };
  const int nk = (K + ML_BK - 1) / ML_BK;

  // The senders, of rows and of columns: a block and a step of it each. A wave brings 8 rows at a time, 128 bytes of each: rows
  // 8 (wave + 8 i).
  const int srow = lane / 8, piece = lane % 8 ^ srow;
  const bf16_t *abase, *wbase;                          // of the block, at the step
  uint32_t aoff[4], woff[4];                            // bytes from there on
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * (wave + 8 * i) + srow;
    woff[i] = ((uint32_t)(n0 + row < N ? row : N - 1 - n0) * K + piece * 8) * 2;   // columns past N: read again, never stored
  }
  int asent = next_block(0), wsent = asent, aks = 0, wks = 0;
  auto aim_rows = [&]() {
    const int R = run_of(asent) * MOE_TILE;
    abase = A + (size_t)(t0 + asent) * MOE_TILE * K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = 8 * (wave + 8 * i) + srow;
      aoff[i] = ((uint32_t)(row < R ? row : R - 1) * K + piece * 8) * 2;           // rows past the block likewise
    }
  };
  auto aim_columns = [&]() { wbase = W + ((size_t)__builtin_amdgcn_readfirstlane(tile_expert[t0 + wsent]) * N + n0) * K; };
  auto bring = [&](const bf16_t* base, const uint32_t (&off)[4], int ks, moe_u32x4* to) {
    if (ks + 1 < nk || K % ML_BK == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) ta_load_to_lds16(base, off[i], &to[64 * (wave + 8 * i)]);
    } else {                                                            // the last, partial step: past K zeros
      const bool in = ks * ML_BK + piece * 8 < K;
#pragma unroll
      for (int i = 0; i < 4; ++i) ta_load_to_lds16(in ? (const char*)base + off[i] : (const char*)&ml_zeros, &to[64 * (wave + 8 * i)]);
    }
  };
  // the next step, on into the next block; after the last one the last step again, unused
  auto send_rows = [&](int buf) {
    bring(abase, aoff, aks, As + buf * ML_BM * 8);
    if (aks + 1 < nk) {
      ++aks;
      abase += ML_BK;
    } else if (next_block(asent + 1) < ML_OWN) {
      asent = next_block(asent + 1);
      aks = 0;
      aim_rows();
    }
  };
  auto send_columns = [&](int buf) {
    bring(wbase, woff, wks, Ws + buf * ML_BN * 8);
    if (wks + 1 < nk) {
      ++wks;
      wbase += ML_BK;
    } else if (next_block(wsent + 1) < ML_OWN) {
      wsent = next_block(wsent + 1);
      wks = 0;
      aim_columns();
    }
  };
  aim_rows();
  aim_columns();
  send_rows(0);
  send_columns(0);
  send_columns(1);
  send_rows(1);
  send_columns(2);
  ta_wait_loads<12>();                                  // the first step
  ml_barrier();

  const int at = r * 8 + (kb ^ (r & 7));                // a lane's piece of a step's first 32 k; the others': ^ 4
  int abuf = 0, wbuf = 0;
  for (int i = next_block(0); i < ML_OWN; i = next_block(i + 1)) {
    const int run = run_of(i), half = (run + 1) / 2;
    auto block = [&](auto width) {
      constexpr int U = decltype(width)::value;         // tiles of a wave
      // all of a wave's, which the compiler no longer sees behind the stores of the block before
      auto same = [](uint64_t x) {
        const uint32_t high = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32)), low = __builtin_amdgcn_readfirstlane((uint32_t)x);
        return (uint64_t)high << 32 | low;
      };
      asent = __builtin_amdgcn_readfirstlane(asent);
      wsent = __builtin_amdgcn_readfirstlane(wsent);
      aks = __builtin_amdgcn_readfirstlane(aks);
      wks = __builtin_amdgcn_readfirstlane(wks);
      abuf = __builtin_amdgcn_readfirstlane(abuf);
      wbuf = __builtin_amdgcn_readfirstlane(wbuf);
      abase = reinterpret_cast<const bf16_t*>(same((uint64_t)abase));
      wbase = reinterpret_cast<const bf16_t*>(same((uint64_t)wbase));
      moe_floatx4 acc[U][4];
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[u][v] = moe_floatx4{0.f, 0.f, 0.f, 0.f};
      // 32 k's operands are read while the 32 before are multiplied, so that a step's buffers are free when its second half is.
      const moe_u32x4 *ar = As + 16 * U * wr * 8, *wr_ = Ws + 64 * wc * 8;
      MoeFrag af[U], wf[2][4];
#pragma unroll
      for (int v = 0; v < 4; ++v) wf[0][v].q = wr_[wbuf * ML_BN * 8 + 16 * 8 * v + at];
#pragma unroll
      for (int u = 0; u < U; ++u) af[u].q = ar[abuf * ML_BM * 8 + 16 * 8 * u + at];
      for (int step = 0; step < nk; ++step) {
        ml_multiply<U>(acc, af, wf[0], wf[1], ar + abuf * ML_BM * 8, wr_ + wbuf * ML_BN * 8, at ^ 4);
        ta_wait_loads<4>();                             // the next step's rows and columns; C's stores, if any, only make it wait longer
        ml_barrier();                                   // everyone's; and everyone has this step's operands in registers
        send_rows(abuf);
        send_columns(wbuf);
        abuf ^= 1;
        wbuf = wbuf == 2 ? 0 : wbuf + 1;
        ml_multiply<U>(acc, af, wf[1], wf[0], ar + abuf * ML_BM * 8, wr_ + wbuf * ML_BN * 8, at);   // a last step's: the next block's, read again
      }
      TC* out = C + ((size_t)(t0 + i) * MOE_TILE + r) * N;
      const bool whole = N % 4 == 0 && (uintptr_t)C % (4 * sizeof(TC)) == 0;   // a lane's four columns are stored at once
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int tile = U * wr + u;
        if (tile >= run) break;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const int n = n0 + 64 * wc + 16 * v + 4 * kb;
          TC x[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) x[j] = from_f32<TC>(ACT ? moe_act(act, acc[u][v][j]) : acc[u][v][j]);
          TC* o = out + (size_t)tile * MOE_TILE * N + n;
          if (whole) {
            struct alignas(4 * sizeof(TC)) Four { TC x[4]; };
            if (n < N) *reinterpret_cast<Four*>(o) = Four{{x[0], x[1], x[2], x[3]}};
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j)
              if (n + j < N) o[j] = x[j];
          }
        }
      }
    };
    switch (half) {
      case 1: block(std::integral_constant<int, 1>{}); break;
      case 2: block(std::integral_constant<int, 2>{}); break;
      case 3:
      case 4: block(std::integral_constant<int, 4>{}); break;
      case 5:
      case 6: block(std::integral_constant<int, 6>{}); break;
      default: block(std::integral_constant<int, 8>{}); break;
    }
  }
  ta_wait_loads<0>();                                   // what was sent for and not used has landed before the LDS is given back
}

// A: [max_rows, K] ordered rows; W: [E, N, K]; C: [max_rows, N], float32 or the type of A;
// act: 0 none, 1 gelu, 2 gelu (tanh), 3 relu squared, 4 silu. Tiles past the last expert's
// rows are skipped and their rows of C keep what they held.
static int moe_gemm_lds_launch(hipStream_t stream, int out_dtype, const void* A, const void* W, const int* tile_expert,
                               void* C, int tiles, int N, int K, int act) {
  const size_t lds = (size_t)(2 * ML_BM + 3 * ML_BN) * ML_BK * sizeof(bf16_t);
  const int ncol = (N + ML_BN - 1) / ML_BN;
  const unsigned g = (unsigned)ncol * (unsigned)((tiles + ML_OWN - 1) / ML_OWN);
  // Blocks of 8 where they give every CU one at most (8 experts, tiles x columns x k: 133 x 2,048 x 1,408 71 us by 16 and
  // 56 by 8, 520 x 512 x 2,048 95 and 77, 258 x 1,408 x 2,048 95 and 77); beyond, a block of 16 costs less than two of 8
  // (520 x 2,048 x 1,408 84 against 99).
  const int most = (long long)((tiles + 7) / 8) * ncol <= 256 ? 8 : ML_TILES;
#define ML_RUN(TC, ACT)                                                                                          \
  do {                                                                                                           \
    auto kern = moe_gemm_lds_kernel<TC, ACT>;                                                                    \
    static bool allowed = false;                        /* asked for once, not at every launch */                \
    if (!allowed) {                                                                                              \
      const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),                            \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);          \
      if (err != hipSuccess) return ta_fail("ta_moe_gemm: %zu bytes of LDS refused (%s)", lds, hipGetErrorString(err)); \
      allowed = true;                                                                                            \
    }                                                                                                            \
    kern<<<g, 512, lds, stream>>>((const bf16_t*)A, (const bf16_t*)W, tile_expert, tiles, most, (TC*)C, N, K, act); \
  } while (0)
  if (out_dtype == TA_BF16) {
    if (act) ML_RUN(bf16_t, true); else ML_RUN(bf16_t, false);
  } else {
    if (act) ML_RUN(float, true); else ML_RUN(float, false);
  }
#undef ML_RUN
  return ta_check_launch("ta_moe_gemm");
}

// Whether the experts' product of this many ordered rows takes the form for few tiles (bfloat16). Below the line the
// blocks of the other form leave CUs idle, above it this one reads an expert's matrix once for every tile; the larger the matrices,
// the longer the other's few workgroups walk. Tiles by blocks of 256 columns, us few / LDS: 4,096 x 2,048 1,120 126 / 128,
// 1,280 143 / 157, 1,600 178 / 152; 4,096 x 1,408 1,328 150 / 175, 1,760 188 / 180; 2,816 x 4,096 1,210 330 / 416, 1,430 379 / 407, 1,650
// 423 / 353; 28,672 x 4,096 1,344 384 / 444; smaller ones 4,096 x 1,024 960 55 / 67, 1,120 61 / 50; 2,048 x 2,048 560 60 / 65, 800 77 / 68;
// 2,048 x 1,024 480 31 / 51, 800 43 / 38 (and a first product through LDS wants its rows ordered, some 5 us).
extern "C" int ta_moe_few_rows(int max_rows, int N, int K) {
  const long long size = (long long)N * K, line = size < 5 << 20 ? 1024 : 1400;
  return K % 8 == 0 && (long long)(max_rows / MOE_TILE) * ((N + 255) / 256) < line;
}

// The first product of the experts of a step of few tokens, from the tokens' rows h [nt, K]: C [max_rows, N] in
// bfloat16. glu: W is [E, 2 N, K], gate rows then up rows, joined by silu (limit 0) or the limited form; else W is
// [E, N, K] and `act` as in ta_moe_gemm. weight (or null): of the pairs, acts on the rows.
extern "C" int ta_moe_gemm_tokens(hipStream_t stream, const void* h, int nt, const int* row_pair, const float* weight, int top,
                                  const void* W, const int* tile_expert, void* C, int max_rows, int N, int K, int act, int glu,
                                  float limit, float slope, float shift) {
  TA_REQUIRE(nt >= 1 && top >= 1 && max_rows >= 0 && max_rows % MOE_TILE == 0 && N > 0 && K > 0 && K % 8 == 0 && act >= 0 && act <= 4 &&
                 (uintptr_t)h % 16 == 0 && (uintptr_t)W % 16 == 0,
             "ta_moe_gemm_tokens: bad sizes rows=%d N=%d K=%d act=%d", max_rows, N, K, act);
  if (max_rows == 0) return 0;
  const MoeRows rows = {(const bf16_t*)h, row_pair, weight, top};
  const TaGlu g = {limit, slope, shift};
  const int tiles = max_rows / MOE_TILE;
  if (glu) moe_splitk<bf16_t, true>(stream, rows, W, tile_expert, C, tiles, N, K, 0, g);
  else moe_splitk<bf16_t, false>(stream, rows, W, tile_expert, C, tiles, N, K, act, g);
  return ta_check_launch("ta_moe_gemm_tokens");
}

// form: 0 = chosen by the shape; 1 = the waves divide K (few tiles); 2 = runs of tiles with operands
// straight from memory; 3 = operands through LDS (many tiles). 1 to 3 take bfloat16 with K % 8 == 0.
extern "C" int ta_moe_gemm_form(hipStream_t stream, int dtype, int out_dtype, const void* A, const void* W,
                                const int* tile_expert, void* C, int max_rows, int N, int K, int act, int form) {
  TA_REQUIRE(max_rows >= 0 && max_rows % MOE_TILE == 0 && N > 0 && K > 0 && act >= 0 && act <= 4,
             "ta_moe_gemm: bad sizes rows=%d N=%d K=%d act=%d", max_rows, N, K, act);
  TA_REQUIRE(form >= 0 && form <= 3 && (form == 0 || (dtype == TA_BF16 && K % 8 == 0)),
             "ta_moe_gemm: form %d needs bfloat16 and K %% 8 == 0", form);
  if (max_rows == 0) return 0;
  const int tiles = max_rows / MOE_TILE;
  if (dtype == TA_BF16 && K % 8 == 0) {
    if (out_dtype != TA_BF16 && out_dtype != TA_F32) return ta_fail("ta_moe_gemm: unknown output type %d", out_dtype);
    const bool few = ta_moe_few_rows(max_rows, N, K);
    const bool aligned = ((uintptr_t)A | (uintptr_t)W) % 16 == 0;   // else operands straight from memory
    if ((form == 3 || (form == 0 && !few)) && aligned)
      return moe_gemm_lds_launch(stream, out_dtype, A, W, tile_expert, C, tiles, N, K, act);
    if (form == 1 || (form == 0 && few)) {   // too few workgroups to fill the CUs: the waves divide K
      const MoeRows rows = {(const bf16_t*)A, nullptr, nullptr, 1};
      const TaGlu none = {0.f, 1.f, 0.f};
      if (out_dtype == TA_BF16) moe_splitk<bf16_t, false>(stream, rows, W, tile_expert, C, tiles, N, K, act, none);
      else moe_splitk<float, false>(stream, rows, W, tile_expert, C, tiles, N, K, act, none);
      return ta_check_launch("ta_moe_gemm");
    }
    dim3 g((N + 255) / 256, (tiles + 3) / 4);
    if (out_dtype == TA_BF16)
      moe_gemm_mfma_kernel<bf16_t><<<g, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, tile_expert, tiles, (bf16_t*)C, N, K, act);
    else if (out_dtype == TA_F32)
      moe_gemm_mfma_kernel<float><<<g, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, tile_expert, tiles, (float*)C, N, K, act);
    else
      return ta_fail("ta_moe_gemm: unknown output type %d", out_dtype);
    return ta_check_launch("ta_moe_gemm");
  }
  dim3 g((N + 63) / 64, tiles);
  if (dtype == TA_F32 && out_dtype == TA_F32)
    moe_gemm_fma_kernel<float, float><<<g, 256, 0, stream>>>((const float*)A, (const float*)W, tile_expert, (float*)C, N, K, act);
  else if (dtype == TA_BF16 && out_dtype == TA_BF16)
    moe_gemm_fma_kernel<bf16_t, bf16_t><<<g, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, tile_expert, (bf16_t*)C, N, K, act);
  else if (dtype == TA_BF16 && out_dtype == TA_F32)
    moe_gemm_fma_kernel<bf16_t, float><<<g, 256, 0, stream>>>((const bf16_t*)A, (const bf16_t*)W, tile_expert, (float*)C, N, K, act);
  else
    return ta_fail("ta_moe_gemm: unsupported types %d -> %d", dtype, out_dtype);
  return ta_check_launch("ta_moe_gemm");
}

extern "C" int ta_moe_gemm(hipStream_t stream, int dtype, int out_dtype, const void* A, const void* W,
                           const int* tile_expert, void* C, int max_rows, int N, int K, int act) {
  return ta_moe_gemm_form(stream, dtype, out_dtype, A, W, tile_expert, C, max_rows, N, K, act, 0);
}

// ------------------------------------------------------------------ putting the rows back
// A thread V columns of a token. V 4: rows of whole 16-byte pieces; the rows of up to four pairs are asked for together
// and a token's columns are dealt out to several workgroups, so that a step of few tokens is one trip to memory and
// not `top` times the columns of a thread (2 tokens, 4,096 columns, top 6: 20 us in one workgroup a token, 5 now).
template <typename T, int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(const float* __restrict__ rows, int d, int top,
                                                          const int* __restrict__ pair_row,
                                                          const float* __restrict__ weight,
                                                          const float* __restrict__ shared, int planes, size_t plane,
                                                          const float* __restrict__ shared_gate, int gate_ld,
                                                          float* __restrict__ delta,
                                                          const float* __restrict__ extra, int xplanes, size_t xplane,
                                                          const T* __restrict__ h) {
  typedef float vec __attribute__((ext_vector_type(V)));
  const size_t t = blockIdx.x;
  const int c = (blockIdx.y * 256 + threadIdx.x) * V;
  if (c >= d) return;
  const size_t at = t * d + c;
  float sg = 1.f;
  if (shared && shared_gate) sg = 1.0f / (1.0f + expf(-shared_gate[t * gate_ld]));
  vec s, own;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    s[i] = 0.f;
    own[i] = h ? to_f32(h[at + i]) : 0.f;                    // what an identity expert gives
  }
  for (int j0 = 0; j0 < top; j0 += 4) {
    vec y[4];
    float w[4];
    int r[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const size_t pair = t * top + (j0 + j < top ? j0 + j : j0);
      r[j] = pair_row[pair];
      w[j] = weight ? weight[pair] : 1.f;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) y[j] = *reinterpret_cast<const vec*>(rows + (size_t)(r[j] >= 0 ? r[j] : 0) * d + c);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (j0 + j < top) {
#pragma unroll
        for (int i = 0; i < V; ++i) s[i] = fmaf(r[j] >= 0 ? y[j][i] : own[i], w[j], s[i]);
      }
  }
  if (shared) {
    vec v = *reinterpret_cast<const vec*>(shared + at);
    for (int p = 1; p < planes; ++p) v += *reinterpret_cast<const vec*>(shared + at + p * plane);
#pragma unroll
    for (int i = 0; i < V; ++i) s[i] = fmaf(sg, v[i], s[i]);
  }
  if (extra)      // what another sublayer adds to the stream beside this one, planes in order
    for (int p = 0; p < xplanes; ++p) s += *reinterpret_cast<const vec*>(extra + at + p * xplane);
  *reinterpret_cast<vec*>(delta + at) = s;
}

// rows: [max_rows, d] float32, the experts' results in the planned order. weight: null when it
// has acted on the inputs. shared (or null): [planes, nt, d] float32 planes that add up to the
// shared expert's result; shared_gate (or null): its gate's pre-activation, one number per
// token, element 0 of a row of gate_ld float32. delta: [nt, d] float32.
// extra (or null): [xplanes, nt, d] float32 planes, ``xplane`` elements apart, added as they are.
// h (or null; float32 or bfloat16 by h_dtype): [nt, d] the rows that identity experts (pairs without a row)
// hand back.
extern "C" int ta_moe_combine(hipStream_t stream, const float* rows, int d, int top, const int* pair_row,
                              const float* weight, const float* shared, int planes, long long plane,
                              const float* shared_gate, int gate_ld, const float* extra, int xplanes,
                              long long xplane, int h_dtype, const void* h, float* delta, int nt) {
  TA_REQUIRE(h_dtype == TA_F32 || h_dtype == TA_BF16, "ta_moe_combine: unknown dtype %d", h_dtype);
  TA_REQUIRE(nt >= 0 && d > 0 && top >= 1 && planes >= 1 && planes <= TA_MAX_PLANES, "ta_moe_combine: bad sizes");
  TA_REQUIRE(!extra || (xplanes >= 1 && xplanes <= TA_MAX_PLANES && (xplanes == 1 || xplane > 0)),
             "ta_moe_combine: %d planes of the further addend", xplanes);
  if (nt == 0) return 0;
#define MOE_COMBINE(T)                                                                                          \
  do {                                                                                                          \
    if (vec)                                                                                                    \
      moe_combine_kernel<T, 4><<<dim3(nt, (d / 4 + 255) / 256), 256, 0, stream>>>(                              \
          rows, d, top, pair_row, weight, shared, planes, (size_t)plane, shared_gate, gate_ld, delta, extra, xplanes, \
          (size_t)xplane, (const T*)h);                                                                         \
    else                                                                                                        \
      moe_combine_kernel<T, 1><<<dim3(nt, (d + 255) / 256), 256, 0, stream>>>(                                  \
          rows, d, top, pair_row, weight, shared, planes, (size_t)plane, shared_gate, gate_ld, delta, extra, xplanes, \
          (size_t)xplane, (const T*)h);                                                                         \
  } while (0)
  const bool vec = d % 4 == 0 && plane % 4 == 0 && xplane % 4 == 0 &&
                   ((uintptr_t)rows | (uintptr_t)shared | (uintptr_t)extra | (uintptr_t)delta) % 16 == 0;
  TA_REQUIRE((d + 255) / 256 <= 65535, "ta_moe_combine: rows of %d", d);
  if (h_dtype == TA_F32) MOE_COMBINE(float); else MOE_COMBINE(bf16_t);
#undef MOE_COMBINE
  return ta_check_launch("ta_moe_combine");
}

// ------------------------------------------------------------------ the limited gated activation
// Rows of [gate | up] (``di`` columns each, ``ld`` elements between rows): g = min(gate, limit),
// u = clamp(up, -limit, limit), out = g * sigmoid(slope * g) * (u + shift). float32 inside.
template <typename T>
__global__ __launch_bounds__(256) void glu_limit_kernel(const T* __restrict__ gu, int ld, T* __restrict__ out, int di,
                                                        float limit, float slope, float shift) {
  const size_t t = blockIdx.y;
  const T* g = gu + t * (size_t)ld;
  T* o = out + t * (size_t)di;
  auto unit = [&](T gate, T up) {
    const float a = fminf(to_f32(gate), limit);
    const float u = fminf(fmaxf(to_f32(up), -limit), limit);
    return from_f32<T>(a / (1.0f + expf(-slope * a)) * (u + shift));
  };
  constexpr int V = 4;
  struct alignas(V * sizeof(T)) Piece { T x[V]; };
  if (di % V == 0 && ld % V == 0 && ((uintptr_t)gu | (uintptr_t)out) % sizeof(Piece) == 0) {
    for (int i = V * (blockIdx.x * 256 + threadIdx.x); i < di; i += V * gridDim.x * 256) {
      const Piece a = *reinterpret_cast<const Piece*>(g + i), u = *reinterpret_cast<const Piece*>(g + di + i);
      Piece r;
#pragma unroll
      for (int e = 0; e < V; ++e) r.x[e] = unit(a.x[e], u.x[e]);
      *reinterpret_cast<Piece*>(o + i) = r;
    }
    return;
  }
  for (int i = blockIdx.x * 256 + threadIdx.x; i < di; i += gridDim.x * 256) o[i] = unit(g[i], g[di + i]);
}

extern "C" int ta_glu_limit(hipStream_t stream, int dtype, const void* gate_up, int ld, void* out, int nt, int di,
                            float limit, float slope, float shift) {
  TA_REQUIRE(nt >= 0 && di > 0 && ld >= 2 * di, "ta_glu_limit: bad sizes nt=%d di=%d ld=%d", nt, di, ld);
  TA_REQUIRE(limit > 0.f, "ta_glu_limit: the limit must be positive, got %g", (double)limit);
  for (int t0 = 0; t0 < nt; t0 += 65535) {
    const int rows = nt - t0 < 65535 ? nt - t0 : 65535;
    dim3 g((di + 1023) / 1024 < 64 ? (di + 1023) / 1024 : 64, rows);
    if (dtype == TA_F32)
      glu_limit_kernel<float><<<g, 256, 0, stream>>>((const float*)gate_up + (size_t)t0 * ld, ld,
                                                    (float*)out + (size_t)t0 * di, di, limit, slope, shift);
    else if (dtype == TA_BF16)
      glu_limit_kernel<bf16_t><<<g, 256, 0, stream>>>((const bf16_t*)gate_up + (size_t)t0 * ld, ld,
                                                     (bf16_t*)out + (size_t)t0 * di, di, limit, slope, shift);
    else
      return ta_fail("ta_glu_limit: unknown dtype %d", dtype);
  }
  return ta_check_launch("ta_glu_limit");
}
