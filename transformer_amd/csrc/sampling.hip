// Next-token choice from float32 logits: argmax, and sampling from
// softmax(logits / temperature) restricted by top-k and top-p.
//
// Sampling works on fixed-point probabilities q_i = floor(2^40 * exp2((l_i - max) / T * log2 e)),
// so every sum is an integer sum: the kept set and the drawn token do not depend
// on the order in which threads add, and a row gives the same token in any batch.
// Order of preference: higher logit first, lower index first among equals. Kept
// are the first top_k tokens of that order, cut after the token with which the
// kept probability reaches top_p. The token drawn for a uniform u in [0,1) is the
// first kept token, in index order, whose running sum exceeds floor(u * kept sum).
#include "common.h"

#define SAMPLE_THREADS 1024
#define SAMPLE_WAVES (SAMPLE_THREADS / TA_WAVE)
typedef unsigned long long u64;

__device__ __forceinline__ uint32_t order_key(float l) {
  const uint32_t b = __float_as_uint(l);
  return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}
// floor(2^40 * exp((l - m) / T)) from the hardware's exp2 and two 32-bit conversions: the
// library's expf and a float-to-64-bit conversion are some fifty instructions, and sampling is
// bound by what it does for each token, whether a row is one workgroup's or dealt out in parts
__device__ __forceinline__ u64 fixed_mass(float l, float m, float inv_t) {
  const float w = __builtin_amdgcn_exp2f((l - m) * inv_t * 1.44269504088896341f);   // in [0, 1]
  const float upper = w * 1048576.0f;                    // 2^20; exact, as is what follows
  const uint32_t hi = (uint32_t)upper;
  const uint32_t lo = (uint32_t)((upper - (float)hi) * 1048576.0f);
  return ((u64)hi << 20) + lo;
}
__device__ __forceinline__ u64 shfl_xor_u64(u64 v, int o) {
  uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
  lo = __shfl_xor(lo, o, TA_WAVE);
  hi = __shfl_xor(hi, o, TA_WAVE);
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 shfl_up_u64(u64 v, int o) {
  uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
  lo = __shfl_up(lo, o, TA_WAVE);
  hi = __shfl_up(hi, o, TA_WAVE);
  return ((u64)hi << 32) | lo;
}

// ------------------------------------------------------------------ argmax
// Highest logit; among equals the lowest index.
__global__ __launch_bounds__(SAMPLE_THREADS) void argmax_kernel(const float* __restrict__ logits,
                                                                 size_t ld, int vocab,
                                                                 int* __restrict__ out) {
  const float* row = logits + (size_t)blockIdx.x * ld;
  float best = -INFINITY;
  int bi = 0x7fffffff;
  // a thread meets its indices in ascending order, so among equals the first one stays
#define CONSIDER(v_, i_)                                          \
  do {                                                            \
    const float cv_ = (v_);                                       \
    if (cv_ > best || bi == 0x7fffffff) {                         \
      if (!(cv_ < best)) { /* NaN never wins over a number already held */ \
        best = cv_;                                               \
        bi = (i_);                                                \
      }                                                           \
    }                                                             \
  } while (0)
  int done = 0;
  if (((uintptr_t)row % 16) == 0) {
    // sixteen bytes per lane; a single workgroup per row is bound by what one CU can load
    const float4* row4 = reinterpret_cast<const float4*>(row);
    const int n4 = vocab / 4;
    // eight loads on their way per thread: with one, a row of 128 K logits took 22 us
    constexpr int AHEAD = 8;
    int j = threadIdx.x;
    for (; j + (AHEAD - 1) * SAMPLE_THREADS < n4; j += AHEAD * SAMPLE_THREADS) {
      float4 v[AHEAD];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) v[u] = row4[j + u * SAMPLE_THREADS];
#pragma unroll
      for (int u = 0; u < AHEAD; ++u) {
        const int jj = j + u * SAMPLE_THREADS;
        CONSIDER(v[u].x, 4 * jj);
        CONSIDER(v[u].y, 4 * jj + 1);
        CONSIDER(v[u].z, 4 * jj + 2);
        CONSIDER(v[u].w, 4 * jj + 3);
      }
    }
    for (; j < n4; j += SAMPLE_THREADS) {
      const float4 v = row4[j];
      CONSIDER(v.x, 4 * j);
      CONSIDER(v.y, 4 * j + 1);
      CONSIDER(v.z, 4 * j + 2);
      CONSIDER(v.w, 4 * j + 3);
    }
    done = n4 * 4;
  }
  for (int i = done + threadIdx.x; i < vocab; i += SAMPLE_THREADS) CONSIDER(row[i], i);
#undef CONSIDER
#pragma unroll
  for (int o = TA_WAVE / 2; o > 0; o >>= 1) {
    const float ov = __shfl_xor(best, o, TA_WAVE);
    const int oi = __shfl_xor(bi, o, TA_WAVE);
    if (ov > best || (ov == best && oi < bi)) {
      best = ov;
      bi = oi;
    }
  }
  __shared__ float sv[SAMPLE_WAVES];
  __shared__ int si[SAMPLE_WAVES];
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  if (lane == 0) {
    sv[wave] = best;
    si[wave] = bi;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < SAMPLE_WAVES; ++w)
      if (sv[w] > best || (sv[w] == best && si[w] < bi)) {
        best = sv[w];
        bi = si[w];
      }
    out[blockIdx.x] = bi == 0x7fffffff ? 0 : bi;
  }
}

extern "C" int ta_argmax(hipStream_t stream, const float* logits, long long ld, int n, int vocab,
                         int* out) {
  TA_REQUIRE(n >= 0 && vocab > 0 && ld >= vocab, "ta_argmax: bad sizes n=%d vocab=%d ld=%lld", n, vocab, ld);
  if (n == 0) return 0;
  argmax_kernel<<<n, SAMPLE_THREADS, 0, stream>>>(logits, (size_t)ld, vocab, out);
  return ta_check_launch("ta_argmax");
}

// ------------------------------------------------------------------ sampling
struct SelectState {
  uint32_t prefix, mask;
  uint32_t count_above;
  u64 mass_above;
  uint32_t tie_count;
  u64 tie_mass;
};

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_kernel(
    const float* __restrict__ logits, size_t ld, int vocab, float inv_t, int top_k, float top_p,
    const float* __restrict__ uniform, int* __restrict__ out) {
  const float* row = logits + (size_t)blockIdx.x * ld;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  __shared__ float s_f[SAMPLE_WAVES];
  __shared__ u64 s_q[SAMPLE_WAVES];
  __shared__ uint32_t s_c[SAMPLE_WAVES];
  __shared__ uint32_t h_cnt[256];
  __shared__ u64 h_mass[256];
  __shared__ SelectState st;
  __shared__ float s_max;
  __shared__ u64 s_total;
  __shared__ int s_pick;

  // ---- max
  float m = -INFINITY;
  {
    int done = 0;
    if (((uintptr_t)row % 16) == 0) {
      const float4* row4 = reinterpret_cast<const float4*>(row);
      const int n4 = vocab / 4;
      for (int j = threadIdx.x; j < n4; j += SAMPLE_THREADS) {
        const float4 v = row4[j];
        m = fmaxf(fmaxf(m, v.x), fmaxf(fmaxf(v.y, v.z), v.w));
      }
      done = n4 * 4;
    }
    for (int i = done + threadIdx.x; i < vocab; i += SAMPLE_THREADS) m = fmaxf(m, row[i]);
  }
  m = wave_max(m);
  if (lane == 0) s_f[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float mm = s_f[0];
    for (int w = 1; w < SAMPLE_WAVES; ++w) mm = fmaxf(mm, s_f[w]);
    s_max = mm;
  }
  __syncthreads();
  m = s_max;

  // ---- total mass (only the cuts need it; without them the sweeps below sum what is kept)
  const bool cut = top_k < vocab || top_p < 1.0f;
  u64 tot = 0;
  if (cut)
    for (int i = threadIdx.x; i < vocab; i += SAMPLE_THREADS) tot += fixed_mass(row[i], m, inv_t);
#pragma unroll
  for (int o = TA_WAVE / 2; o > 0; o >>= 1) tot += shfl_xor_u64(tot, o);
  if (lane == 0) s_q[wave] = tot;
  __syncthreads();
  if (threadIdx.x == 0) {
    u64 t = 0;
    for (int w = 0; w < SAMPLE_WAVES; ++w) t += s_q[w];
    s_total = t;
    st.prefix = 0;
    st.mask = 0;
    st.count_above = 0;
    st.mass_above = 0;
    st.tie_count = 0xffffffffu;   // "every token of the threshold value is kept"
    st.tie_mass = 0;
    s_pick = 0;
  }
  __syncthreads();
  const u64 total = s_total;

  // ---- threshold of the kept set (only when top-k or top-p cut anything)
  if (cut) {
    const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
    u64 p_lim = (u64)ceil((double)top_p * (double)total);
    if (p_lim < 1) p_lim = 1;
    if (p_lim > total) p_lim = total;
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      for (int i = threadIdx.x; i < 256; i += SAMPLE_THREADS) {
        h_cnt[i] = 0;
        h_mass[i] = 0;
      }
      __syncthreads();
      const uint32_t prefix = st.prefix, mask = st.mask;
      for (int i = threadIdx.x; i < vocab; i += SAMPLE_THREADS) {
        const float l = row[i];
        const uint32_t key = order_key(l);
        if ((key & mask) == prefix) {
          const int bin = (key >> shift) & 255;
          atomicAdd(&h_cnt[bin], 1u);
          atomicAdd(&h_mass[bin], fixed_mass(l, m, inv_t));
        }
      }
      __syncthreads();
      if (threadIdx.x == 0) {
        uint32_t ca = st.count_above;
        u64 ma = st.mass_above;
        int chosen = -1;
        for (int bin = 255; bin >= 0; --bin) {
          if (h_cnt[bin] == 0) continue;
          if (ca + h_cnt[bin] >= k_lim || ma + h_mass[bin] >= p_lim) {
            chosen = bin;
            break;
          }
          ca += h_cnt[bin];
          ma += h_mass[bin];
        }
        // p_lim <= total, so the lowest non-empty bin reaches it at the latest
        if (chosen < 0) chosen = 0;
        st.count_above = ca;
        st.mass_above = ma;
        st.prefix = prefix | ((uint32_t)chosen << shift);
        st.mask = mask | (255u << shift);
        if (pass == 3) {
          const uint32_t c_t = h_cnt[chosen];
          const u64 q_t = c_t ? h_mass[chosen] / c_t : 0;
          uint32_t n = k_lim - ca;                       // >= 1
          if (q_t > 0) {
            const u64 need = (p_lim - ma + q_t - 1) / q_t;  // >= 1
            if (need < n) n = (uint32_t)need;
          }
          if (n > c_t) n = c_t;
          st.tie_count = n;
          st.tie_mass = q_t;
        }
      }
      __syncthreads();
    }
  }
  const uint32_t thr = st.prefix;          // 0 when nothing is cut: every key is > 0
  const uint32_t n_tie = st.tie_count;

  // ---- ordered sweeps: wave w owns the contiguous indices [w*span, (w+1)*span)
  const int span = ((vocab + SAMPLE_WAVES - 1) / SAMPLE_WAVES + TA_WAVE - 1) / TA_WAVE * TA_WAVE;
  const int lo = wave * span;
  const int hi = (lo + span < vocab) ? lo + span : vocab;
  const u64 lanes_below = ((u64)1 << lane) - 1;

  // sweep 1: threshold-valued tokens per wave -> rank base of each wave
  uint32_t ties = 0;
  for (int i0 = lo; i0 < hi; i0 += TA_WAVE) {
    const int i = i0 + lane;
    const bool tie = cut && i < hi && order_key(row[i]) == thr;
    ties += __popcll(__ballot(tie));
  }
  if (lane == 0) s_c[wave] = ties;
  __syncthreads();
  uint32_t tie_base = 0;
  for (int w = 0; w < wave; ++w) tie_base += s_c[w];
  __syncthreads();

  // sweep 2: kept mass per wave -> mass base of each wave
  u64 kept = 0;
  {
    uint32_t rank = tie_base;
    for (int i0 = lo; i0 < hi; i0 += TA_WAVE) {
      const int i = i0 + lane;
      bool keep = false, tie = false;
      float l = 0.f;
      if (i < hi) {
        l = row[i];
        const uint32_t key = order_key(l);
        tie = cut && key == thr;
        keep = !cut || key > thr;
      }
      const u64 b = __ballot(tie);
      if (tie && rank + __popcll(b & lanes_below) < n_tie) keep = true;
      rank += __popcll(b);
      if (keep) kept += fixed_mass(l, m, inv_t);
    }
  }
#pragma unroll
  for (int o = TA_WAVE / 2; o > 0; o >>= 1) kept += shfl_xor_u64(kept, o);
  if (lane == 0) s_q[wave] = kept;
  __syncthreads();
  u64 mass_base = 0, kept_total = 0;
  for (int w = 0; w < SAMPLE_WAVES; ++w) {
    if (w < wave) mass_base += s_q[w];
    kept_total += s_q[w];
  }
  u64 target = (u64)((double)uniform[blockIdx.x] * (double)kept_total);
  if (kept_total > 0 && target >= kept_total) target = kept_total - 1;

  // sweep 3: the wave whose range holds the target finds the token
  if (kept_total > 0 && target >= mass_base && target < mass_base + s_q[wave]) {
    uint32_t rank = tie_base;
    u64 run = mass_base;
    for (int i0 = lo; i0 < hi; i0 += TA_WAVE) {
      const int i = i0 + lane;
      bool keep = false, tie = false;
      float l = 0.f;
      if (i < hi) {
        l = row[i];
        const uint32_t key = order_key(l);
        tie = cut && key == thr;
        keep = !cut || key > thr;
      }
      const u64 b = __ballot(tie);
      if (tie && rank + __popcll(b & lanes_below) < n_tie) keep = true;
      rank += __popcll(b);
      const u64 q = keep ? fixed_mass(l, m, inv_t) : 0;
      u64 inc = q;                                   // inclusive scan over the wave
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const u64 up = shfl_up_u64(inc, o);
        if (lane >= o) inc += up;
      }
      const bool hit = q > 0 && run + inc > target && run + inc - q <= target;
      const u64 hb = __ballot(hit);
      if (hb) {
        if (hit) s_pick = i;
        break;
      }
      {  // the last lane holds the sum of this group of 64
        uint32_t lo32 = (uint32_t)inc, hi32 = (uint32_t)(inc >> 32);
        lo32 = __shfl(lo32, TA_WAVE - 1, TA_WAVE);
        hi32 = __shfl(hi32, TA_WAVE - 1, TA_WAVE);
        run += ((u64)hi32 << 32) | lo32;
      }
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = s_pick;
}

// Sum over the 64 lanes, the same in every lane, without going through the LDS crossbar:
// DPP moves inside a row of 16 lanes (1 apart, 2 apart, mirrored within 8, mirrored within 16),
// then the lane swaps of gfx950 across rows. A shuffle costs over a hundred cycles in a chain
// of its own; this is a dozen vector operations.
template <int CTRL>
__device__ __forceinline__ u64 dpp_move_u64(u64 v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)v, CTRL, 0xf, 0xf, true);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(v >> 32), CTRL, 0xf, 0xf, true);
  return ((u64)hi << 32) | lo;
}
__device__ __forceinline__ u64 wave_sum_u64(u64 v) {
  v += dpp_move_u64<0xB1>(v);
  v += dpp_move_u64<0x4E>(v);
  v += dpp_move_u64<0x141>(v);
  v += dpp_move_u64<0x140>(v);
  {
    const auto lo = __builtin_amdgcn_permlane16_swap((uint32_t)v, (uint32_t)v, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
    v = (((u64)hi[0] << 32) | lo[0]) + (((u64)hi[1] << 32) | lo[1]);
  }
  {
    const auto lo = __builtin_amdgcn_permlane32_swap((uint32_t)v, (uint32_t)v, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((uint32_t)(v >> 32), (uint32_t)(v >> 32), false, false);
    v = (((u64)hi[0] << 32) | lo[0]) + (((u64)hi[1] << 32) | lo[1]);
  }
  return v;
}

// a mass no row reaches (2^17 tokens of 2^40 each are 2^57), with room to add to it
#define NO_MASS_LIMIT ((u64)1 << 62)
#define STEPS 128          // steps of 1/8 of a unit of logit / T that a part counts one by one: 16 units down from its largest
#define STEPS_PER_UNIT 8.0f
#define PART 4096          // tokens of a row that one workgroup looks at
#define PART_THREADS 256
#define MAX_PARTS 256       // of a row: a million tokens
#define PART_CAND 512      // tokens of the steps that hold the threshold, per part
#define ROW_CAND 4096      // and per row
#define MASS_MARGIN 1e-4   // sums relative to a part's maximum are this close to the row's own (3e-6 measured from the formats)

// The step a logit lies in, counted up from 0 at logit 0: a rising function of the logit.
__device__ __forceinline__ int step_of(float l, float inv_t) {
  return (int)floorf(fminf(fmaxf(l * inv_t * STEPS_PER_UNIT, -1e9f), 1e9f));
}

// One digit of the threshold key, by one wave (a lane four bins): the highest bin with which the count
// reaches k_lim or the mass p_lim. The last digit also settles how many tokens of the threshold value are
// kept (the lower indices among equals).
__device__ void choose_digit(SelectState& st, const uint32_t* h_cnt, const u64* h_mass, int shift,
                             bool last, uint32_t k_lim, u64 p_lim) {
  const int lane = threadIdx.x % TA_WAVE;
  uint32_t c[4], cs = 0;
  u64 q[4], qs = 0;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    c[i] = h_cnt[255 - 4 * lane - i];
    q[i] = h_mass[255 - 4 * lane - i];
    cs += c[i];
    qs += q[i];
  }
  u64 ci = cs, qi = qs;                            // sums up to and with this lane
#pragma unroll
  for (int o = 1; o < TA_WAVE; o <<= 1) {
    const u64 cu = shfl_up_u64(ci, o), qu = shfl_up_u64(qi, o);
    if (lane >= o) {
      ci += cu;
      qi += qu;
    }
  }
  uint32_t ca = st.count_above + (uint32_t)ci - cs;
  u64 ma = st.mass_above + qi - qs;
  int hit = -1;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (hit < 0) {
      if (c[i] && (ca + c[i] >= k_lim || ma + q[i] >= p_lim)) hit = i;
      else {
        ca += c[i];
        ma += q[i];
      }
    }
  const u64 found = __ballot(hit >= 0);
  // p_lim <= total, so the lowest non-empty bin reaches it at the latest
  const int who = found ? __ffsll((unsigned long long)found) - 1 : TA_WAVE - 1;
  if (lane != who) return;
  const int chosen = hit >= 0 ? 255 - 4 * lane - hit : 0;
  st.count_above = ca;
  st.mass_above = ma;
  st.prefix |= (uint32_t)chosen << shift;
  st.mask |= 255u << shift;
  if (last) {
    const uint32_t c_t = h_cnt[chosen];
    const u64 q_t = c_t ? h_mass[chosen] / c_t : 0;
    uint32_t n = k_lim - ca;                       // >= 1
    if (q_t > 0) {
      const u64 need = (p_lim - ma + q_t - 1) / q_t;  // >= 1
      if (need < n) n = (uint32_t)need;
    }
    if (n > c_t) n = c_t;
    st.tie_count = n;
    st.tie_mass = q_t;
  }
}

#define CAND_PER_WAVE 256  // tokens near the maximum that a wave's share of the row may hold
#define NEAR_BINS 96       // steps of 1/9 counted one by one: down to e^-10.7 of the largest probability

// distance from the maximum in steps of 1/9 of (max - logit) / T; 255 holds all that is further
__device__ __forceinline__ int near_bin(float l, float m, float inv_t) {
  const float d = (m - l) * inv_t * 9.0f;
  return d < 255.0f ? (int)d : 255;
}

// The same choice by one workgroup for a row that starts on a 16-byte boundary, every pass over the row bringing
// sixteen bytes per lane. GATHER: the kept tokens, where they are few, go through LDS and the row is read three times;
// without it (rows whose threshold the parts below cannot enclose: more than PART_CAND tokens of a part within a step
// of it, as when thousands are equal, or a threshold more than 16 units of logit / T under the maximum) up to nine
// times. All sums are integer sums and the sweeps keep the order of the indices, so every way chooses the same token.
#define VEC_STEPS 64      // steps of 256 tokens whose sums a wave remembers (16 waves: 262,144 tokens)
struct Four {
  float v[4];
  bool ok[4];
};
// group j of the row: tokens 4j .. 4j+3. The row's stride is a multiple of four, so the last
// group may be read whole; what lies past the vocabulary is marked and reads as -inf. No
// branch: a loop can ask for several groups before it looks at the first.
__device__ __forceinline__ Four load_four(const float* __restrict__ row, int j, int vocab) {
  Four f;
  const float4 x = *reinterpret_cast<const float4*>(row + 4 * j);
  const float in[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    f.ok[e] = 4 * j + e < vocab;
    f.v[e] = f.ok[e] ? in[e] : -INFINITY;
  }
  return f;
}
// the same for a group that may lie past the row: then nothing of it is there
__device__ __forceinline__ Four load_four_if(const float* __restrict__ row, int j, int groups, int vocab) {
  return load_four(row, j < groups ? j : 0, j < groups ? vocab : 0);
}

template <bool GATHER>
__device__ void sample_whole_row(const float* __restrict__ row, int vocab, float inv_t, int top_k, float top_p,
                                 float uniform, int* __restrict__ out) {
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  const int groups = (vocab + 3) / 4;                  // runs of four tokens
  __shared__ float s_f[SAMPLE_WAVES];
  __shared__ u64 s_q[SAMPLE_WAVES];
  __shared__ uint32_t s_c[SAMPLE_WAVES];
  __shared__ uint32_t h_cnt[256];
  __shared__ u64 h_mass[256];
  __shared__ SelectState st;
  __shared__ float s_max;
  __shared__ u64 s_total;
  __shared__ int s_pick;
  __shared__ u64 s_step[SAMPLE_WAVES][VEC_STEPS];      // kept mass of each step of a wave's range
  // tokens near the maximum, gathered in index order: wave w's share of the row in cand_*[w]
  __shared__ float cand_l[GATHER ? SAMPLE_WAVES : 1][GATHER ? CAND_PER_WAVE : 1];
  __shared__ int cand_i[GATHER ? SAMPLE_WAVES : 1][GATHER ? CAND_PER_WAVE : 1];
  __shared__ int s_ccnt[SAMPLE_WAVES];
  __shared__ int s_small;

  // ---- max
  float m = -INFINITY;
  // four groups are asked for before the first is looked at: one CU pulls what its loads in
  // flight allow, and a pass over the row is this kernel's unit of cost
  for (int j = threadIdx.x; j < groups; j += 4 * SAMPLE_THREADS) {
    Four f[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) f[u] = load_four_if(row, j + u * SAMPLE_THREADS, groups, vocab);
#pragma unroll
    for (int u = 0; u < 4; ++u)
      m = fmaxf(fmaxf(m, f[u].v[0]), fmaxf(fmaxf(f[u].v[1], f[u].v[2]), f[u].v[3]));
  }
  m = wave_max(m);
  if (lane == 0) s_f[wave] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    float mm = s_f[0];
    for (int w = 1; w < SAMPLE_WAVES; ++w) mm = fmaxf(mm, s_f[w]);
    s_max = mm;
  }
  __syncthreads();
  m = s_max;

  const bool cut = top_k < vocab || top_p < 1.0f;
  if (threadIdx.x == 0) {
    s_total = 0;
    st.prefix = 0;
    st.mask = 0;
    st.count_above = 0;
    st.mass_above = 0;
    st.tie_count = 0xffffffffu;   // "every token of the threshold value is kept"
    st.tie_mass = 0;
    s_pick = 0;
    s_small = 0;
  }
  for (int i = threadIdx.x; i < 256; i += SAMPLE_THREADS) {
    h_cnt[i] = 0;
    h_mass[i] = 0;
  }
  __syncthreads();

  // ---- with a cut: the tokens by their distance from the maximum, in steps of 1/9 of a
  // unit of (max - logit) / T. The sums give the total mass, and the step in which the count
  // reaches top_k or the mass reaches top_p bounds the kept set: usually a few hundred
  // tokens, which are then gathered into LDS and cut and drawn from there, so the row is
  // read three times in all instead of nine. When that step lies far from the maximum or
  // the tokens do not fit, the digits of the threshold are found over the whole row.
  if (GATHER && cut) {
    // steps from NEAR_BINS on are lumped into the last one, summed in registers: most tokens
    // lie there, and the cut almost never does
    uint32_t far_cnt = 0;
    u64 far_mass = 0;
    const bool need_total = top_p < 1.0f;    // top-k alone never asks for the mass of the far tokens
    for (int j = threadIdx.x; j < groups; j += 4 * SAMPLE_THREADS) {
      Four f[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) f[u] = load_four_if(row, j + u * SAMPLE_THREADS, groups, vocab);
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (!f[u].ok[e]) continue;
          const int bin = near_bin(f[u].v[e], m, inv_t);
          if (bin < NEAR_BINS) {             // such a token has mass left by a wide margin
            atomicAdd(&h_cnt[bin], 1u);
            atomicAdd(&h_mass[bin], fixed_mass(f[u].v[e], m, inv_t));
          } else {
            ++far_cnt;
            if (need_total) far_mass += fixed_mass(f[u].v[e], m, inv_t);
          }
        }
    }
    far_cnt = (uint32_t)wave_sum_u64(far_cnt);
    far_mass = wave_sum_u64(far_mass);
    if (lane == 0 && far_cnt) {
      atomicAdd(&h_cnt[255], far_cnt);
      atomicAdd(&h_mass[255], far_mass);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      u64 t = 0;
      for (int bin = 0; bin < 256; ++bin) t += h_mass[bin];
      s_total = t;
      const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
      u64 p_lim = (u64)ceil((double)top_p * (double)t);
      if (p_lim < 1) p_lim = 1;
      if (p_lim > t) p_lim = t;
      if (top_p >= 1.0f) p_lim = NO_MASS_LIMIT;   // the far tokens' mass was not summed; nothing is cut by mass
      uint32_t ca = 0;
      u64 ma = 0;
      int last = 255;
      for (int bin = 0; bin < 256; ++bin) {
        ca += h_cnt[bin];
        ma += h_mass[bin];
        if (ca >= k_lim || ma >= p_lim) {
          last = bin;
          break;
        }
      }
      s_pick = last;                          // borrowed until the draw: the last step that matters
      s_small = t > 0 && last < NEAR_BINS && ca <= (uint32_t)(SAMPLE_WAVES * CAND_PER_WAVE);
    }
    __syncthreads();
  }
  // ---- total mass, which only the cut by mass asks for
  if (!GATHER && cut) {
    u64 tot = 0;
    if (top_p < 1.0f)
      for (int j = threadIdx.x; j < groups; j += SAMPLE_THREADS) {
        const Four f = load_four(row, j, vocab);
#pragma unroll
        for (int e = 0; e < 4; ++e) tot += f.ok[e] ? fixed_mass(f.v[e], m, inv_t) : 0;
      }
    tot = wave_sum_u64(tot);
    if (lane == 0) atomicAdd(&s_total, tot);
    __syncthreads();
  }
  const u64 total = s_total;
  const int near_last = GATHER ? s_pick : 0;
  if (GATHER) {
    __syncthreads();
    if (threadIdx.x == 0) s_pick = 0;
  }

  const int span = ((groups + SAMPLE_WAVES - 1) / SAMPLE_WAVES + TA_WAVE - 1) / TA_WAVE * TA_WAVE;
  const int lo = wave * span;
  const int hi = (lo + span < groups) ? lo + span : groups;
  const u64 lanes_below = ((u64)1 << lane) - 1;

  // ---- gather the tokens of the steps up to that one, wave by wave in index order
  if (GATHER && cut && s_small) {
    int have = 0;
    for (int j0 = lo; j0 < hi; j0 += TA_WAVE) {
      const int j = j0 + lane;
      Four f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f.v[e] = -INFINITY;
        f.ok[e] = false;
      }
      if (j < hi) f = load_four(row, j, vocab);
      bool take[4];
      int before = 0, all = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        take[e] = f.ok[e] && near_bin(f.v[e], m, inv_t) <= near_last;
        const u64 b = __ballot(take[e]);
        before += __popcll(b & lanes_below);
        all += __popcll(b);
      }
      int at = have + before;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (take[e]) {
          if (at < CAND_PER_WAVE) {
            cand_l[wave][at] = f.v[e];
            cand_i[wave][at] = 4 * j + e;
          }
          ++at;
        }
      have += all;
    }
    if (lane == 0) s_ccnt[wave] = have;
    __syncthreads();
    if (threadIdx.x == 0) {
      int ok = 1;
      for (int w = 0; w < SAMPLE_WAVES; ++w)
        if (s_ccnt[w] > CAND_PER_WAVE) ok = 0;         // a wave's share did not fit: the long way
      s_small = ok;
    }
    __syncthreads();
  }

  if (GATHER && cut && s_small) {
    // ---- the cut among the gathered tokens (they hold every token at or above the threshold)
    const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
    u64 p_lim = (u64)ceil((double)top_p * (double)total);
    if (p_lim < 1) p_lim = 1;
    if (p_lim > total) p_lim = total;
    if (top_p >= 1.0f) p_lim = NO_MASS_LIMIT;      // see above: only top_k cuts
    const int mine = s_ccnt[wave];
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      for (int i = threadIdx.x; i < 256; i += SAMPLE_THREADS) {
        h_cnt[i] = 0;
        h_mass[i] = 0;
      }
      __syncthreads();
      const uint32_t prefix = st.prefix, mask = st.mask;
      for (int c = lane; c < mine; c += TA_WAVE) {
        const float l = cand_l[wave][c];
        const uint32_t key = order_key(l);
        if ((key & mask) == prefix) {
          const int bin = (key >> shift) & 255;
          atomicAdd(&h_cnt[bin], 1u);
          atomicAdd(&h_mass[bin], fixed_mass(l, m, inv_t));
        }
      }
      __syncthreads();
      if (wave == 0) choose_digit(st, h_cnt, h_mass, shift, pass == 3, k_lim, p_lim);
      __syncthreads();
    }
    const uint32_t thr = st.prefix;
    const uint32_t n_tie = st.tie_count;
    // ---- the draw, in index order: wave by wave, and inside a wave as gathered
    uint32_t ties = 0;
    for (int c0 = 0; c0 < mine; c0 += TA_WAVE) {
      const int c = c0 + lane;
      ties += __popcll(__ballot(c < mine && order_key(cand_l[wave][c]) == thr));
    }
    if (lane == 0) s_c[wave] = ties;
    __syncthreads();
    uint32_t tie_base = 0;
    for (int w = 0; w < wave; ++w) tie_base += s_c[w];
    u64 kept = 0;
    {
      uint32_t rank = tie_base;
      for (int c0 = 0; c0 < mine; c0 += TA_WAVE) {
        const int c = c0 + lane;
        bool keep = false, tie = false;
        float l = 0.f;
        if (c < mine) {
          l = cand_l[wave][c];
          const uint32_t key = order_key(l);
          tie = key == thr;
          keep = key > thr;
        }
        const u64 b = __ballot(tie);
        if (tie && rank + __popcll(b & lanes_below) < n_tie) keep = true;
        rank += __popcll(b);
        if (keep) kept += fixed_mass(l, m, inv_t);
      }
    }
    kept = wave_sum_u64(kept);
    if (lane == 0) s_q[wave] = kept;
    __syncthreads();
    u64 mass_base = 0, kept_total = 0;
    for (int w = 0; w < SAMPLE_WAVES; ++w) {
      if (w < wave) mass_base += s_q[w];
      kept_total += s_q[w];
    }
    u64 target = (u64)((double)uniform * (double)kept_total);
    if (kept_total > 0 && target >= kept_total) target = kept_total - 1;
    if (kept_total > 0 && target >= mass_base && target < mass_base + s_q[wave]) {
      uint32_t rank = tie_base;
      u64 run = mass_base;
      for (int c0 = 0; c0 < mine; c0 += TA_WAVE) {
        const int c = c0 + lane;
        bool keep = false, tie = false;
        float l = 0.f;
        if (c < mine) {
          l = cand_l[wave][c];
          const uint32_t key = order_key(l);
          tie = key == thr;
          keep = key > thr;
        }
        const u64 b = __ballot(tie);
        if (tie && rank + __popcll(b & lanes_below) < n_tie) keep = true;
        rank += __popcll(b);
        const u64 q = keep ? fixed_mass(l, m, inv_t) : 0;
        u64 inc = q;
#pragma unroll
        for (int o = 1; o < TA_WAVE; o <<= 1) {
          const u64 up = shfl_up_u64(inc, o);
          if (lane >= o) inc += up;
        }
        const bool hit = q > 0 && run + inc > target && run + inc - q <= target;
        if (__ballot(hit)) {
          if (hit) s_pick = cand_i[wave][c];
          break;
        }
        uint32_t lo32 = (uint32_t)inc, hi32 = (uint32_t)(inc >> 32);
        lo32 = __shfl(lo32, TA_WAVE - 1, TA_WAVE);
        hi32 = __shfl(hi32, TA_WAVE - 1, TA_WAVE);
        run += ((u64)hi32 << 32) | lo32;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0) *out = s_pick;
    return;
  }

  // ---- threshold of the kept set (only when top-k or top-p cut anything)
  if (cut) {
    const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
    u64 p_lim = (u64)ceil((double)top_p * (double)total);
    if (p_lim < 1) p_lim = 1;
    if (p_lim > total) p_lim = total;
    if (top_p >= 1.0f) p_lim = NO_MASS_LIMIT;      // the mass was not summed: only top_k cuts
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      for (int i = threadIdx.x; i < 256; i += SAMPLE_THREADS) {
        h_cnt[i] = 0;
        h_mass[i] = 0;
      }
      __syncthreads();
      const uint32_t prefix = st.prefix, mask = st.mask;
      for (int j = threadIdx.x; j < groups; j += SAMPLE_THREADS) {
        const Four f = load_four(row, j, vocab);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint32_t key = order_key(f.v[e]);
          if (f.ok[e] && (key & mask) == prefix) {
            const int bin = (key >> shift) & 255;
            atomicAdd(&h_cnt[bin], 1u);
            atomicAdd(&h_mass[bin], fixed_mass(f.v[e], m, inv_t));
          }
        }
      }
      __syncthreads();
      if (wave == 0) choose_digit(st, h_cnt, h_mass, shift, pass == 3, k_lim, p_lim);
      __syncthreads();
    }
  }
  const uint32_t thr = st.prefix;          // 0 when nothing is cut: every key is > 0
  const uint32_t n_tie = st.tie_count;

  // ---- ordered sweeps: wave w owns the contiguous groups [lo, hi); inside a step of 64
  // groups the order of the indices is lane by lane, and inside a lane element by element

  // which of a lane's four tokens are kept, given the ties counted before this step
#define KEEP_FOUR(f_, rank_, keep_, q_)                                                   \
  do {                                                                                    \
    bool tie_[4];                                                                         \
    uint32_t before_ = 0, all_ = 0;                                                       \
    _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                       \
      const uint32_t key_ = order_key(f_.v[e]);                                           \
      tie_[e] = cut && f_.ok[e] && key_ == thr;                                           \
      keep_[e] = f_.ok[e] && (!cut || key_ > thr);                                        \
      const u64 b_ = __ballot(tie_[e]);                                                   \
      before_ += __popcll(b_ & lanes_below);                                              \
      all_ += __popcll(b_);                                                               \
    }                                                                                     \
    uint32_t mine_ = rank_ + before_;            /* ties in the lanes before this one */  \
    _Pragma("unroll") for (int e = 0; e < 4; ++e) {                                       \
      if (tie_[e]) {                                                                      \
        if (mine_ < n_tie) keep_[e] = true;                                               \
        ++mine_;                                                                          \
      }                                                                                   \
      q_[e] = keep_[e] ? fixed_mass(f_.v[e], m, inv_t) : 0;                               \
    }                                                                                     \
    rank_ += all_;                                                                        \
  } while (0)

  // sweep 1: threshold-valued tokens per wave -> rank base of each wave
  uint32_t ties = 0;
  if (cut)
    for (int j0 = lo; j0 < hi; j0 += TA_WAVE) {
      const int j = j0 + lane;
      Four f;
      if (j < hi) f = load_four(row, j, vocab);
#pragma unroll
      for (int e = 0; e < 4; ++e) ties += __popcll(__ballot(j < hi && f.ok[e] && order_key(f.v[e]) == thr));
    }
  if (lane == 0) s_c[wave] = ties;
  __syncthreads();
  uint32_t tie_base = 0;
  for (int w = 0; w < wave; ++w) tie_base += s_c[w];
  __syncthreads();

  // sweep 2: kept mass per wave -> mass base of each wave
  u64 kept = 0;
  {
    uint32_t rank = tie_base;
    for (int j0 = lo; j0 < hi; j0 += TA_WAVE) {
      const int j = j0 + lane;
      Four f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f.v[e] = -INFINITY;
        f.ok[e] = false;
      }
      if (j < hi) f = load_four(row, j, vocab);
      bool keep[4];
      u64 q[4];
      if (cut) {
        KEEP_FOUR(f, rank, keep, q);
      } else {                                   // temperature alone: every token is kept
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = f.ok[e] ? fixed_mass(f.v[e], m, inv_t) : 0;
      }
      const u64 here = wave_sum_u64(q[0] + q[1] + q[2] + q[3]);
      const int step = (j0 - lo) / TA_WAVE;
      if (lane == 0 && step < VEC_STEPS) s_step[wave][step] = here;
      kept += here;
    }
  }
  if (lane == 0) s_q[wave] = kept;
  __syncthreads();
  u64 mass_base = 0, kept_total = 0;
  for (int w = 0; w < SAMPLE_WAVES; ++w) {
    if (w < wave) mass_base += s_q[w];
    kept_total += s_q[w];
  }
  u64 target = (u64)((double)uniform * (double)kept_total);
  if (kept_total > 0 && target >= kept_total) target = kept_total - 1;

  // sweep 3: the wave whose range holds the target finds the token
  if (kept_total > 0 && target >= mass_base && target < mass_base + s_q[wave]) {
    uint32_t rank = tie_base;
    u64 run = mass_base;
    for (int j0 = lo; j0 < hi; j0 += TA_WAVE) {
      const int j = j0 + lane;
      Four f;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f.v[e] = -INFINITY;
        f.ok[e] = false;
      }
      if (j < hi) f = load_four(row, j, vocab);
      const int step = (j0 - lo) / TA_WAVE;
      if (step < VEC_STEPS && run + s_step[wave][step] <= target) {
        // the target lies behind this step: only its ties have to be counted
        run += s_step[wave][step];
        if (cut) {
#pragma unroll
          for (int e = 0; e < 4; ++e) rank += __popcll(__ballot(f.ok[e] && order_key(f.v[e]) == thr));
        }
        continue;
      }
      bool keep[4];
      u64 q[4];
      if (cut) {
        KEEP_FOUR(f, rank, keep, q);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) q[e] = f.ok[e] ? fixed_mass(f.v[e], m, inv_t) : 0;
      }
      const u64 mine = q[0] + q[1] + q[2] + q[3];
      u64 inc = mine;                                // inclusive scan over the wave
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const u64 up = shfl_up_u64(inc, o);
        if (lane >= o) inc += up;
      }
      const bool hit = mine > 0 && run + inc > target && run + inc - mine <= target;
      if (__ballot(hit)) {
        if (hit) {
          u64 at = run + inc - mine;                 // mass before this lane's four tokens
          int pick = 4 * j;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (q[e] > 0 && at + q[e] > target && at <= target) pick = 4 * j + e;
            at += q[e];
          }
          s_pick = pick;
        }
        break;
      }
      {  // the last lane holds the sum of this step
        uint32_t lo32 = (uint32_t)inc, hi32 = (uint32_t)(inc >> 32);
        lo32 = __shfl(lo32, TA_WAVE - 1, TA_WAVE);
        hi32 = __shfl(hi32, TA_WAVE - 1, TA_WAVE);
        run += ((u64)hi32 << 32) | lo32;
      }
    }
  }
#undef KEEP_FOUR
  __syncthreads();
  if (threadIdx.x == 0) *out = s_pick;
}

// Rows that start on a 16-byte boundary are dealt out in parts of 4,096 tokens, one workgroup each, so that eight rows
// keep 256 CUs busy and not eight: a row is bound by instructions per token, not by memory. Three kernels:
//   parts   each part's maximum, and its tokens and their mass (relative to that maximum) by steps of 1/8 of a
//           unit of logit / T;
//   gather  from all parts' steps the step that holds the threshold, or the two between which the margin of the
//           relative masses leaves it; what lies above it is kept: its mass and count, exactly; what lies in
//           it is gathered in index order;
//   draw    one workgroup a row: the threshold among the gathered tokens by the digits of their keys, the part that
//           holds the drawn mass, the token in it.
// 8 rows of 128,256 tokens, top-k 40 and top-p 0.95: 125 us by one workgroup a row (which gathered whole kept sets of a
// few thousand tokens), 27 us in parts
// (5 + 10 + 12, the draw asking for all it needs of the records at once); 64 rows 50 us, 256 rows 125, one row without a cut 16. Cuts at
// few tokens go by the two kernels below.
struct PartRecord {
  float2 mass[STEPS / 2];    // of two steps each, relative to the part's maximum
  uint32_t cnt[STEPS / 2];   // tokens of two steps each, 16 bits of them (a part has 4,096)
  u64 above, total;          // exact: of the tokens above the steps in question; of all
  double rest;               // of all its tokens, relative to the part's maximum
  float max;
  uint32_t above_n;
  int lo, hi;                // the steps in question, counted down from the row's largest; lo < 0: not enclosed
  int n;                     // gathered
  float cand_l[PART_CAND];   // in index order
};

// The rows' random numbers in the launch's arguments: the first of the three kernels puts them where the last reads them.
#define SAMPLE_IN_ARGS 64
struct SampleUniforms {
  float u[SAMPLE_IN_ARGS];
};

// group u (of four) of this thread in its part
__device__ __forceinline__ int part_group(int part, int u) { return part * (PART / 4) + u * PART_THREADS + (int)threadIdx.x; }

__global__ __launch_bounds__(PART_THREADS) void sample_parts_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                    float inv_t, int cut, int by_mass,
                                                                    PartRecord* __restrict__ records, SampleUniforms given,
                                                                    int n_given, float* __restrict__ uniform) {
  const float* row = logits + (size_t)blockIdx.y * ld;
  if (blockIdx.x == 0 && blockIdx.y == 0 && (int)threadIdx.x < n_given) uniform[threadIdx.x] = given.u[threadIdx.x];
  PartRecord& rec = records[(size_t)blockIdx.y * gridDim.x + blockIdx.x];
  const int groups = (vocab + 3) / 4, wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  __shared__ float s_f[PART_THREADS / TA_WAVE];
  __shared__ uint32_t cnt[STEPS];
  __shared__ u64 mass[STEPS], rest;
  for (int i = threadIdx.x; i < STEPS; i += PART_THREADS) {
    cnt[i] = 0;
    mass[i] = 0;
  }
  if (threadIdx.x == 0) rest = 0;
  Four f[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) f[u] = load_four_if(row, part_group(blockIdx.x, u), groups, vocab);
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(m, f[u].v[e]);
  m = wave_max(m);
  if (lane == 0) s_f[wave] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < PART_THREADS / TA_WAVE; ++w) m = fmaxf(m, s_f[w]);
  if (threadIdx.x == 0) rec.max = m;
  if (!cut) return;
  const int top = step_of(m, inv_t);
  u64 all = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (!f[u].ok[e]) continue;
      const int at = top - step_of(f[u].v[e], inv_t);
      const u64 q = by_mass ? fixed_mass(f[u].v[e], m, inv_t) : 0;
      all += q;
      if (at < STEPS) {
        atomicAdd(&cnt[at], 1u);
        if (by_mass) atomicAdd(&mass[at], q);
      }
    }
  if (by_mass) {
    all = wave_sum_u64(all);
    if (lane == 0) atomicAdd(&rest, all);
  }
  __syncthreads();
  if (threadIdx.x < STEPS / 2) {
    const int i = 2 * threadIdx.x;
    rec.cnt[threadIdx.x] = cnt[i] | (cnt[i + 1] << 16);
    rec.mass[threadIdx.x] = float2{(float)mass[i], (float)mass[i + 1]};
  }
  if (threadIdx.x == 0) rec.rest = (double)rest;
}

// the row's maximum from its parts'
__device__ __forceinline__ float row_max(const PartRecord* rec, int parts) {
  float m = -INFINITY;
  for (int p = threadIdx.x % TA_WAVE; p < parts; p += TA_WAVE) m = fmaxf(m, rec[p].max);
  return wave_max(m);
}

__global__ __launch_bounds__(PART_THREADS) void sample_gather_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                     float inv_t, int top_k, float top_p, int cut,
                                                                     PartRecord* __restrict__ records) {
  const float* row = logits + (size_t)blockIdx.y * ld;
  PartRecord* all = records + (size_t)blockIdx.y * gridDim.x;
  PartRecord& rec = all[blockIdx.x];
  const int parts = gridDim.x, groups = (vocab + 3) / 4;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  constexpr int WAVES = PART_THREADS / TA_WAVE;
  __shared__ u64 s_c[WAVES][TA_WAVE][3];
  __shared__ double s_q[WAVES][TA_WAVE][3], s_rest[WAVES];
  __shared__ int s_lo, s_hi, s_n[4][WAVES];
  __shared__ u64 s_above[WAVES], s_total[WAVES];
  __shared__ uint32_t s_above_n[WAVES];
  Four f[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) f[u] = load_four_if(row, part_group(blockIdx.x, u), groups, vocab);
  const float m = row_max(all, parts);
  const int top = step_of(m, inv_t);
  const bool by_mass = top_p < 1.0f;
  if (cut) {
    // the row's steps from the parts': a step is the same interval of logits in all of them, so a part's are
    // moved by the difference of the largest ones. A wave takes every fourth part, a lane two steps; where a part
    // is moved by an odd number its pairs fall on two lanes' steps
    u64 c[3] = {0, 0, 0};                            // this lane's steps 2 lane, 2 lane + 1, and what belongs one further
    double q[3] = {0.0, 0.0, 0.0}, t = 0.0;
    for (int p0 = wave; p0 < parts; p0 += 8 * WAVES) {
      uint32_t cn[8];
      float2 qn[8];
      float pm[8];
      double rest[8];
      int off[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) pm[i] = all[p0 + i * WAVES < parts ? p0 + i * WAVES : p0].max;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const PartRecord& r = all[p0 + i * WAVES < parts ? p0 + i * WAVES : p0];
        off[i] = top - step_of(pm[i], inv_t);
        const int at = lane - off[i] / 2;            // pair of the part whose first step is 2 lane (or one further)
        const bool in = p0 + i * WAVES < parts && at >= 0;
        cn[i] = r.cnt[in ? at : 0];
        qn[i] = r.mass[in ? at : 0];
        rest[i] = r.rest;
        if (!in) {
          cn[i] = 0;
          qn[i] = float2{0.f, 0.f};
        }
        if (p0 + i * WAVES >= parts) rest[i] = 0.0;
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float w = __builtin_amdgcn_exp2f((pm[i] - m) * inv_t * 1.44269504088896341f);
        const bool odd = off[i] & 1;
        const uint32_t ca = cn[i] & 0xffffu, cb = cn[i] >> 16;
        c[0] += odd ? 0 : ca;
        c[1] += odd ? ca : cb;
        c[2] += odd ? cb : 0;
        if (by_mass) {
          const double qa = (double)qn[i].x * w, qb = (double)qn[i].y * w;
          q[0] += odd ? 0.0 : qa;
          q[1] += odd ? qa : qb;
          q[2] += odd ? qb : 0.0;
          t += rest[i] * w;
        }
      }
    }
    s_c[wave][lane][0] = c[0];
    s_c[wave][lane][1] = c[1];
    s_c[wave][lane][2] = c[2];
    s_q[wave][lane][0] = q[0];
    s_q[wave][lane][1] = q[1];
    s_q[wave][lane][2] = q[2];
    if (lane == 0) s_rest[wave] = t;                 // the same in all lanes
    __syncthreads();
    if (wave == 0) {                                 // a lane two steps
      u64 c0 = 0, c = 0;
      double q0 = 0.0, q = 0.0;
      t = 0.0;
#pragma unroll
      for (int w = 0; w < WAVES; ++w) {
        c0 += s_c[w][lane][0] + (lane ? s_c[w][lane - 1][2] : 0);
        c += s_c[w][lane][1];
        q0 += s_q[w][lane][0] + (lane ? s_q[w][lane - 1][2] : 0.0);
        q += s_q[w][lane][1];
        t += s_rest[w];
      }
      const u64 c1 = c;
      const double q1 = q;
      c += c0;
      q += q0;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const u64 cu = shfl_up_u64(c, o);
        const double qu = __shfl_up(q, o, TA_WAVE);
        if (lane >= o) {
          c += cu;
          q += qu;
        }
      }
      const double want = (double)top_p * t;
      auto reaches = [&](u64 cn, double qn, double factor) {
        return cn >= (u64)top_k || (by_mass && qn >= want * factor);
      };
      c0 = c - c1;                                   // up to and with the first of the two
      q0 = q - q1;
      auto first = [&](double factor) {
        const u64 b0 = __ballot(reaches(c0, q0, factor)), b1 = __ballot(reaches(c, q, factor));
        const u64 any = b0 | b1;
        if (!any) return STEPS;
        const int who = __ffsll((unsigned long long)any) - 1;
        return 2 * who + ((b0 >> who) & 1 ? 0 : 1);
      };
      const int lo = first(1.0 - MASS_MARGIN), hi = first(1.0 + MASS_MARGIN);
      if (lane == 0) {
        s_lo = hi < STEPS && m > -INFINITY && m < INFINITY ? lo : -1;
        s_hi = hi;
      }
    }
    __syncthreads();
  }
  const int lo = cut ? s_lo : STEPS, hi = cut ? s_hi : STEPS;
  // this part: what is kept for certain, and what is in question
  u64 above = 0, total = 0;
  uint32_t above_n = 0;
  int before[4], mine[4];
  u64 take[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int all_ = 0;
    before[u] = mine[u] = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool ok = f[u].ok[e];
      const u64 q = ok ? fixed_mass(f[u].v[e], m, inv_t) : 0;
      const int at = top - step_of(f[u].v[e], inv_t);
      total += q;
      const bool keep = ok && (!cut || at < lo);
      above += keep ? q : 0;
      above_n += keep;
      take[u][e] = __ballot(ok && cut && at >= lo && at <= hi);
      before[u] += __popcll(take[u][e] & (((u64)1 << lane) - 1));
      all_ += __popcll(take[u][e]);
    }
    if (lane == 0) s_n[u][wave] = all_;
  }
  above = wave_sum_u64(above);
  total = wave_sum_u64(total);
  above_n = (uint32_t)wave_sum_u64(above_n);
  if (lane == 0) {
    s_above[wave] = above;
    s_total[wave] = total;
    s_above_n[wave] = above_n;
  }
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w == wave) {
        int at = base + before[u];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if ((take[u][e] >> lane) & 1) {
            if (at < PART_CAND) rec.cand_l[at] = f[u].v[e];
            ++at;
          }
      }
      base += s_n[u][w];
    }
  if (threadIdx.x == 0) {
    u64 a = 0, t = 0;
    uint32_t n = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      a += s_above[w];
      t += s_total[w];
      n += s_above_n[w];
    }
    rec.above = a;
    rec.total = t;
    rec.above_n = n;
    rec.lo = lo;
    rec.hi = hi;
    rec.n = base;
  }
}

// The first part with which the running sum of what the parts keep exceeds target (-1: none), the sum in front of it in
// *base. By a whole wave.
__device__ __forceinline__ int find_part(const u64* kept, int parts, u64 target, u64* base) {
  const int lane = threadIdx.x % TA_WAVE;
  u64 run = 0;
  for (int p0 = 0; p0 < parts; p0 += TA_WAVE) {
    const u64 mine = p0 + lane < parts ? kept[p0 + lane] : 0;
    u64 inc = mine;
#pragma unroll
    for (int o = 1; o < TA_WAVE; o <<= 1) {
      const u64 up = shfl_up_u64(inc, o);
      if (lane >= o) inc += up;
    }
    const u64 hit = __ballot(target < run + inc);
    if (hit) {
      const int who = __ffsll((unsigned long long)hit) - 1;
      if (lane == who) *base = run + inc - mine;
      return p0 + who;
    }
    run += (u64)__shfl((unsigned long long)inc, TA_WAVE - 1, TA_WAVE);
  }
  return -1;
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_draw_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                     float inv_t, int top_k, float top_p, int cut, int parts,
                                                                     const PartRecord* __restrict__ records,
                                                                     const float* __restrict__ uniform, int* __restrict__ out,
                                                                     int* __restrict__ out_host) {
  const float* row = logits + (size_t)blockIdx.x * ld;
  const PartRecord* all = records + (size_t)blockIdx.x * parts;
  const int groups = (vocab + 3) / 4;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  const u64 lanes_below = ((u64)1 << lane) - 1;
  __shared__ float cand_l[ROW_CAND];
  __shared__ uint32_t s_ties[SAMPLE_WAVES];
  __shared__ uint32_t h_cnt[256];
  __shared__ u64 h_mass[256];
  __shared__ SelectState st;
  __shared__ int s_ok, s_cands, s_part, s_pick, s_lo, s_hi;
  __shared__ u64 s_total, s_target, s_base, s_wave[SAMPLE_WAVES];
  __shared__ uint32_t s_tie_base;
  __shared__ float s_max;
  __shared__ int s_first[MAX_PARTS], s_n[MAX_PARTS]; // first gathered token of a part, its number of them
  __shared__ u64 s_kept[MAX_PARTS];                  // mass that a part keeps

  // ---- what the parts say: everything that is needed of the records is asked for at once, before it is known how many
  // tokens a part has gathered; a wave adds up
  const float uni = uniform[blockIdx.x];
  constexpr int AHEAD = 2;                           // parts of a wave whose first 64 gathered tokens are on their way
  float ahead[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    const int p = wave + i * SAMPLE_WAVES;
    ahead[i] = cut ? all[p < parts ? p : 0].cand_l[lane] : 0.f;
  }
  if (wave == 0) {
    int run = 0;
    u64 total = 0, above = 0;
    uint32_t above_n = 0;
    bool ok = true;
    float m = -INFINITY;
    const int lo0 = all[0].lo, hi0 = all[0].hi;
    for (int p0 = 0; p0 < parts; p0 += TA_WAVE) {
      const int p = p0 + lane;
      const bool in = p < parts;
      const PartRecord& r = all[in ? p : 0];
      const int n = in ? r.n : 0;
      m = fmaxf(m, r.max);
      total += in ? r.total : 0;
      above += in ? r.above : 0;
      above_n += in ? r.above_n : 0;
      ok = ok && n <= PART_CAND;
      int inc = n;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const int up = __shfl_up(inc, o, TA_WAVE);
        if (lane >= o) inc += up;
      }
      if (in) {
        s_first[p] = run + inc - n;
        s_n[p] = n;
        s_kept[p] = r.above;
      }
      run += __shfl(inc, TA_WAVE - 1, TA_WAVE);
    }
    m = wave_max(m);
    total = wave_sum_u64(total);
    above = wave_sum_u64(above);
    above_n = (uint32_t)wave_sum_u64(above_n);
    ok = __ballot(!ok) == 0;
    if (lane == 0) {
      s_max = m;
      s_lo = lo0;
      s_hi = hi0;
      s_total = total;
      s_cands = run;
      s_ok = ok && run <= ROW_CAND && total > 0 && lo0 >= 0;
      st.prefix = 0;
      st.mask = 0;
      st.count_above = above_n;
      st.mass_above = above;
      st.tie_count = 0xffffffffu;
      st.tie_mass = 0;
      s_pick = 0;
      s_part = -1;
      s_tie_base = 0;
    }
  }
  __syncthreads();
  if (!s_ok) {
    sample_whole_row<false>(row, vocab, inv_t, top_k, top_p, uni, out + blockIdx.x);
    __syncthreads();
    if (threadIdx.x == 0 && out_host) out_host[blockIdx.x] = out[blockIdx.x];
    return;
  }
  const float m = s_max;
  const int cands = s_cands, lo = s_lo, hi = s_hi, top = step_of(m, inv_t);
  if (cut) {
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const int p = wave + i * SAMPLE_WAVES;
      if (p < parts && lane < s_n[p]) cand_l[s_first[p] + lane] = ahead[i];
    }
    for (int p = wave; p < parts; p += SAMPLE_WAVES)
      for (int c = lane + (p < AHEAD * SAMPLE_WAVES ? TA_WAVE : 0); c < s_n[p]; c += TA_WAVE) cand_l[s_first[p] + c] = all[p].cand_l[c];
    // ---- the threshold among the gathered tokens
    const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
    u64 p_lim = (u64)ceil((double)top_p * (double)s_total);
    if (p_lim < 1) p_lim = 1;
    if (p_lim > s_total) p_lim = s_total;
    if (top_p >= 1.0f) p_lim = NO_MASS_LIMIT;
    for (int pass = 0; pass < 4; ++pass) {
      const int shift = 24 - 8 * pass;
      if (threadIdx.x < 256) {
        h_cnt[threadIdx.x] = 0;
        h_mass[threadIdx.x] = 0;
      }
      __syncthreads();
      const uint32_t prefix = st.prefix, mask = st.mask;
      for (int c = threadIdx.x; c < cands; c += SAMPLE_THREADS) {
        const float l = cand_l[c];
        const uint32_t key = order_key(l);
        if ((key & mask) == prefix) {
          atomicAdd(&h_cnt[(key >> shift) & 255], 1u);
          atomicAdd(&h_mass[(key >> shift) & 255], fixed_mass(l, m, inv_t));
        }
      }
      __syncthreads();
      if (wave == 0) choose_digit(st, h_cnt, h_mass, shift, pass == 3, k_lim, p_lim);
      __syncthreads();
    }
  }
  const uint32_t thr = st.prefix, n_tie = st.tie_count;
  // ---- what every part keeps of its gathered tokens. Waves take the parts in turn; the ties of a row are
  // ranked in index order, so their numbers per part come first
  if (cut) {
    __shared__ uint32_t s_part_ties[MAX_PARTS];
    for (int p = wave; p < parts; p += SAMPLE_WAVES) {
      const int n = s_n[p];
      uint32_t ties = 0;
      u64 kept = 0;
      for (int c0 = 0; c0 < n; c0 += TA_WAVE) {
        const bool in = c0 + lane < n;
        const float l = in ? cand_l[s_first[p] + c0 + lane] : 0.f;
        const uint32_t key = order_key(l);
        ties += __popcll(__ballot(in && key == thr));
        if (in && key > thr) kept += fixed_mass(l, m, inv_t);
      }
      kept = wave_sum_u64(kept);
      if (lane == 0) {
        s_part_ties[p] = ties;
        s_kept[p] += kept;
      }
    }
    __syncthreads();
    // ranks of the ties, then sums of what is kept, in the parts' order: a wave, 64 parts at a time
    if (wave == 0) {
      uint32_t rank = 0;
      u64 sum = 0;
      for (int p0 = 0; p0 < parts; p0 += TA_WAVE) {
        const int p = p0 + lane;
        const uint32_t t = p < parts ? s_part_ties[p] : 0;
        uint32_t inc = t;
#pragma unroll
        for (int o = 1; o < TA_WAVE; o <<= 1) {
          const uint32_t up = __shfl_up(inc, o, TA_WAVE);
          if (lane >= o) inc += up;
        }
        const uint32_t before = rank + inc - t, room = n_tie > before ? n_tie - before : 0;
        const u64 kept = p < parts ? s_kept[p] + (u64)(t < room ? t : room) * st.tie_mass : 0;
        if (p < parts) {
          s_kept[p] = kept;
          s_part_ties[p] = before;
        }
        rank += __shfl(inc, TA_WAVE - 1, TA_WAVE);
        sum += wave_sum_u64(kept);
      }
      u64 target = (u64)((double)uni * (double)sum);
      if (sum > 0 && target >= sum) target = sum - 1;
      const int p = find_part(s_kept, parts, target, &s_base);
      if (lane == 0) {
        s_total = sum;
        s_target = target;
        s_part = p;
        if (p >= 0) s_tie_base = s_part_ties[p];
      }
    }
  } else if (wave == 0) {
    u64 target = (u64)((double)uni * (double)s_total);
    if (target >= s_total) target = s_total - 1;
    const int p = find_part(s_kept, parts, target, &s_base);
    if (lane == 0) {
      s_part = p;
      s_target = target;
    }
  }
  __syncthreads();
  if (s_part < 0) {
    if (threadIdx.x == 0) {
      out[blockIdx.x] = 0;
      if (out_host) out_host[blockIdx.x] = 0;
    }
    return;
  }
  // ---- the token in that part: one group of four a thread, in index order
  const int j = s_part * (PART / 4) + (int)threadIdx.x;
  const Four f = load_four_if(row, j, groups, vocab);
  bool keep[4], tie[4];
  uint32_t ties_before = 0, ties_all = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int at = top - step_of(f.v[e], inv_t);
    const bool asked = cut && f.ok[e] && at >= lo && at <= hi;
    const uint32_t key = order_key(f.v[e]);
    tie[e] = asked && key == thr;
    keep[e] = f.ok[e] && (!cut || at < lo || (asked && key > thr));
    const u64 b = __ballot(tie[e]);
    ties_before += __popcll(b & lanes_below);
    ties_all += __popcll(b);
  }
  if (lane == 0) s_ties[wave] = ties_all;
  __syncthreads();
  uint32_t rank = s_tie_base + ties_before;
  for (int w = 0; w < wave; ++w) rank += s_ties[w];
  u64 q[4], mine = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (tie[e]) {
      keep[e] = rank < n_tie;
      ++rank;
    }
    q[e] = keep[e] ? fixed_mass(f.v[e], m, inv_t) : 0;
    mine += q[e];
  }
  u64 inc = mine;
#pragma unroll
  for (int o = 1; o < TA_WAVE; o <<= 1) {
    const u64 up = shfl_up_u64(inc, o);
    if (lane >= o) inc += up;
  }
  if (lane == TA_WAVE - 1) s_wave[wave] = inc;
  __syncthreads();
  u64 run = s_base;
  for (int w = 0; w < wave; ++w) run += s_wave[w];
  const u64 target = s_target;
  if (mine > 0 && run + inc > target && run + inc - mine <= target) {
    u64 at = run + inc - mine;
    int pick = 4 * j;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if (q[e] > 0 && at + q[e] > target && at <= target) pick = 4 * j + e;
      at += q[e];
    }
    s_pick = pick;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    out[blockIdx.x] = s_pick;
    if (out_host) out_host[blockIdx.x] = s_pick;
  }
}

// ------------------------------------------------------------------ few tokens kept at most
// A cut at top_k <= TOP_MOST_K in two kernels. A row keeps no token that top_k others of its own part go before, so
//   top     a part hands on its tokens down to the step (1/16 of a unit of logit / T, counted from its largest) with which
//           it has top_k of them (of the last one, where it holds too many, those down to one of its 256 equal pieces), and
//           the mass of all its tokens relative to its own largest;
//   draw    one workgroup a row: of these some 40 to 100 tokens a part the step that holds the threshold (the steps cut into as
//           many as there is room for), the order of the few tokens in it one against the other, and the token drawn, all from LDS.
// What is not handed on has top_k tokens of its own part in front of it, all of them handed on, so that neither counts nor sums
// down to the threshold miss anything.
// The cut by mass wants a share of the row's exact mass, which no part knows; the sum of the parts' is within MASS_ERROR of it,
// and where the two ends of that interval keep different tokens, the row is added up exactly. A row whose threshold lies
// below what some part has handed on (its largest tokens 16 units and more above the threshold), or with more tokens within
// 1/4,096 of a unit than there is room for, is one workgroup's from the start. (Whole steps alone left flat rows to it: 8 rows of
// 128,256 of deviation 0.05 206 us, by the three kernels above 30, in pieces 17; of 0.003 204, 208 and 21.) 8 rows of 128,256,
// top-k 40 and top-p 0.95: 27 us in the three kernels above, 15 in these two; 64 rows 50 and 24, 128 rows 75 and 34, 8 rows of
// 32,000 with top-k 50 24 and 13. Bound by the two kernels' chains: a trip to memory and a histogram each, then one scan, the order
// in the step and a scan for the token.
#define TOP_MOST_K 128
#define TOP_STEPS 256
#define TOP_PER_UNIT 16.0f
#define TOP_CAND 384       // handed on by a part
#define TOP_TIES 1024      // in the step that holds the threshold
#define MASS_ERROR 2e-5    // three roundings of at most 40 in the exponent on either way: 1e-5
#define NO_STEP (-2000000000)
struct TopRecord {
  double rest;             // mass of all its tokens, relative to its largest
  float max;
  int floor;               // what is left out lies in this step, behind top_k others, or below; NO_STEP: nothing is left out
  int n, unused;
  float l[TOP_CAND];       // in index order
  uint16_t i[TOP_CAND];
};
static_assert(sizeof(TopRecord) <= sizeof(PartRecord), "either records fit the scratch");

__device__ __forceinline__ int top_step(float l, float inv_t) {
  return (int)floorf(fminf(fmaxf(l * inv_t * TOP_PER_UNIT, -1e9f), 1e9f));
}

__global__ __launch_bounds__(PART_THREADS) void sample_top_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                  float inv_t, int top_k, int by_mass, int most,
                                                                  TopRecord* __restrict__ records) {
  constexpr int WAVES = PART_THREADS / TA_WAVE;
  const float* row = logits + (size_t)blockIdx.y * ld;
  TopRecord& rec = records[(size_t)blockIdx.y * gridDim.x + blockIdx.x];
  const int groups = (vocab + 3) / 4, wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  const int live = vocab - (int)blockIdx.x * PART < PART ? vocab - (int)blockIdx.x * PART : PART;
  __shared__ float s_f[WAVES];
  __shared__ uint32_t cnt[TOP_STEPS];
  __shared__ u64 s_rest[WAVES];
  __shared__ int s_low, s_got, s_before, s_n[4][WAVES];
  static_assert(TOP_STEPS == PART_THREADS, "a thread a step");
  cnt[threadIdx.x] = 0;
  Four f[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) f[u] = load_four_if(row, part_group(blockIdx.x, u), groups, vocab);
  float m = -INFINITY;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) m = fmaxf(m, f[u].v[e]);
  m = wave_max(m);
  if (lane == 0) s_f[wave] = m;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < WAVES; ++w) m = fmaxf(m, s_f[w]);
  if (m == -INFINITY) {                            // nothing here to be kept before anything of another part
    if (threadIdx.x == 0) {
      rec.rest = 0.0;
      rec.max = m;
      rec.floor = 1 - 1000000000;
      rec.n = 0;
    }
    return;
  }
  const int top = top_step(m, inv_t);
  int at[4][4];
  u64 all = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      at[u][e] = f[u].ok[e] ? top - top_step(f[u].v[e], inv_t) : TOP_STEPS;
      if (at[u][e] < TOP_STEPS) atomicAdd(&cnt[at[u][e]], 1u);
      if (by_mass && f[u].ok[e]) all += fixed_mass(f[u].v[e], m, inv_t);
    }
  if (by_mass) {
    all = wave_sum_u64(all);
    if (lane == 0) s_rest[wave] = all;
  }
  __syncthreads();
  // the step with which there are k tokens (the last one if there are not): how many with it, and how many in front of it
  auto reach = [&](uint32_t k) {
    if (wave == 0) {                               // a lane four steps
      const uint4 c = *reinterpret_cast<const uint4*>(&cnt[4 * lane]);
      const uint32_t mine = c.x + c.y + c.z + c.w;
      uint32_t inc = mine;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const uint32_t up = __shfl_up(inc, o, TA_WAVE);
        if (lane >= o) inc += up;
      }
      const u64 found = __ballot(inc >= k);
      const int who = found ? __ffsll((unsigned long long)found) - 1 : TA_WAVE - 1;
      if (lane == who) {
        const uint32_t run = inc - mine;
        int step = 4 * lane + 3;
        uint32_t n = inc, last = c.w;
        if (found) {
          if (run + c.x >= k) { step = 4 * lane; n = run + c.x; last = c.x; }
          else if (run + c.x + c.y >= k) { step = 4 * lane + 1; n = run + c.x + c.y; last = c.y; }
          else if (run + c.x + c.y + c.z >= k) { step = 4 * lane + 2; n = run + c.x + c.y + c.z; last = c.z; }
        }
        s_low = step;
        s_got = (int)n;
        s_before = (int)(n - last);
      }
    }
    __syncthreads();
  };
  reach((uint32_t)top_k);
  const int low = s_low;
  int n = s_got;
  if (n > most) {                                  // more than top_k, then: of the last step the pieces that it takes from above
    const int in_front = s_before;
    auto piece = [&](float l) {                    // the fraction is exact
      const float x = fminf(fmaxf(l * inv_t * TOP_PER_UNIT, -1e9f), 1e9f);
      return TOP_STEPS - 1 - (int)((x - floorf(x)) * (float)TOP_STEPS);
    };
    cnt[threadIdx.x] = 0;
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (at[u][e] == low) atomicAdd(&cnt[piece(f[u].v[e])], 1u);
    __syncthreads();
    reach((uint32_t)(top_k - in_front));
    const int fine = s_low;
    n = in_front + s_got;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (at[u][e] == low && piece(f[u].v[e]) > fine) at[u][e] = TOP_STEPS;
  }
  if (threadIdx.x == 0) {
    u64 rest = 0;
    if (by_mass)
#pragma unroll
      for (int w = 0; w < WAVES; ++w) rest += s_rest[w];
    rec.rest = (double)rest;
    rec.max = m;
    rec.floor = n < live ? top - low : NO_STEP;
    rec.n = n;
  }
  int before[4];
  u64 take[4][4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    int sum = 0;
    before[u] = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      take[u][e] = __ballot(at[u][e] <= low);
      before[u] += __popcll(take[u][e] & (((u64)1 << lane) - 1));
      sum += __popcll(take[u][e]);
    }
    if (lane == 0) s_n[u][wave] = sum;
  }
  __syncthreads();
  int base = 0;
#pragma unroll
  for (int u = 0; u < 4; ++u)
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      if (w == wave) {
        int to = base + before[u];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if ((take[u][e] >> lane) & 1) {
            if (to < TOP_CAND) {
              rec.l[to] = f[u].v[e];
              rec.i[to] = (uint16_t)(4 * (u * PART_THREADS + (int)threadIdx.x) + e);
            }
            ++to;
          }
      }
      base += s_n[u][w];
    }
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_top_draw_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                         float inv_t, int top_k, float top_p, int parts,
                                                                         const TopRecord* __restrict__ records,
                                                                         const float* __restrict__ uniform, SampleUniforms given,
                                                                         int row0, int* __restrict__ out, int* __restrict__ out_host) {
  const float* row = logits + (size_t)blockIdx.x * ld;
  const TopRecord* all = records + (size_t)blockIdx.x * parts;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  __shared__ float cand_l[ROW_CAND];
  __shared__ uint32_t cand_i[ROW_CAND];
  __shared__ uint8_t keep[ROW_CAND];
  __shared__ uint32_t h_cnt[TOP_STEPS], tie_key[TOP_TIES], tie_at[TOP_TIES];
  __shared__ u64 h_mass[TOP_STEPS], tie_q[TOP_TIES], s_wave[SAMPLE_WAVES];
  __shared__ int s_first[MAX_PARTS], s_n[MAX_PARTS];
  __shared__ int s_ok, s_cands, s_floor, s_bin, s_ties, s_unsure;
  __shared__ uint32_t s_count;
  __shared__ u64 s_mass, s_p[2];
  __shared__ float s_max;
  const bool by_mass = top_p < 1.0f;
  const float uni = uniform ? uniform[blockIdx.x] : given.u[row0 + blockIdx.x];
  // the first 64 tokens of a wave's parts are on their way before it is known how many there are
  constexpr int AHEAD = 2;
  float ahead_l[AHEAD];
  uint32_t ahead_i[AHEAD];
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    const int p = wave + i * SAMPLE_WAVES;
    ahead_l[i] = all[p < parts ? p : 0].l[lane];
    ahead_i[i] = all[p < parts ? p : 0].i[lane];
  }
  if (threadIdx.x < TOP_STEPS) {
    h_cnt[threadIdx.x] = 0;
    h_mass[threadIdx.x] = 0;
  }
  if (wave == 0) {
    float m = -INFINITY;
    for (int p = lane; p < parts; p += TA_WAVE) m = fmaxf(m, all[p].max);
    m = wave_max(m);
    int run = 0, floor = NO_STEP;
    bool ok = true;
    double t = 0.0;
    for (int p0 = 0; p0 < parts; p0 += TA_WAVE) {
      const int p = p0 + lane;
      const bool in = p < parts;
      const TopRecord& r = all[in ? p : 0];
      const int n = in ? r.n : 0;
      ok = ok && n <= TOP_CAND;
      if (in) floor = r.floor > floor ? r.floor : floor;
      if (in && by_mass) t += r.rest * (double)__builtin_amdgcn_exp2f((r.max - m) * inv_t * 1.44269504088896341f);
      int inc = n;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const int up = __shfl_up(inc, o, TA_WAVE);
        if (lane >= o) inc += up;
      }
      if (in) {
        s_first[p] = run + inc - n;
        s_n[p] = n;
      }
      run += __shfl(inc, TA_WAVE - 1, TA_WAVE);
    }
#pragma unroll
    for (int o = 1; o < TA_WAVE; o <<= 1) {
      t += __shfl_xor(t, o, TA_WAVE);
      const int other = __shfl_xor(floor, o, TA_WAVE);
      floor = other > floor ? other : floor;
    }
    ok = __ballot(!ok) == 0;
    if (lane == 0) {
      s_max = m;
      s_floor = floor;
      s_cands = run;
      s_ok = ok && run <= ROW_CAND && m > -INFINITY && m < INFINITY;
      s_ties = 0;
      s_unsure = 0;
      // the mass with which the cut is reached lies between these
      const double want = (double)top_p * t;
      s_p[0] = by_mass ? (u64)fmax(ceil(want * (1.0 - MASS_ERROR)), 1.0) : NO_MASS_LIMIT;
      s_p[1] = by_mass ? (u64)fmax(ceil(want * (1.0 + MASS_ERROR)), 1.0) : NO_MASS_LIMIT;
    }
  }
  __syncthreads();
  auto whole = [&]() {
    sample_whole_row<false>(row, vocab, inv_t, top_k, top_p, uni, out + blockIdx.x);
    __syncthreads();
    if (threadIdx.x == 0 && out_host) out_host[blockIdx.x] = out[blockIdx.x];
  };
  if (!s_ok) return whole();
  const float m = s_max;
  const int cands = s_cands;
  // the threshold lies in the steps from s_floor on: each is cut into as many as all 256 allow
  int finer = 0;
  const int span = s_floor > NO_STEP ? top_step(m, inv_t) - s_floor + 1 : TOP_STEPS;
  if (fabsf(m * inv_t * TOP_PER_UNIT) < (float)(1 << 21))
    while (finer < 7 && span <= (TOP_STEPS - 1) >> (finer + 1)) ++finer;
  const float per_unit = TOP_PER_UNIT * (float)(1 << finer);
  auto fine_step = [&](float l) { return (int)floorf(fminf(fmaxf(l * inv_t * per_unit, -1e9f), 1e9f)); };
  const int top = fine_step(m);
#pragma unroll
  for (int i = 0; i < AHEAD; ++i) {
    const int p = wave + i * SAMPLE_WAVES;
    if (p < parts && lane < s_n[p]) {
      cand_l[s_first[p] + lane] = ahead_l[i];
      cand_i[s_first[p] + lane] = p * PART + ahead_i[i];
    }
  }
  for (int p = wave; p < parts; p += SAMPLE_WAVES)
    for (int c = lane + (p < AHEAD * SAMPLE_WAVES ? TA_WAVE : 0); c < s_n[p]; c += TA_WAVE) {
      cand_l[s_first[p] + c] = all[p].l[c];
      cand_i[s_first[p] + c] = p * PART + all[p].i[c];
    }
  __syncthreads();
  auto step = [&](float l) {
    const int at = top - fine_step(l);
    return at < TOP_STEPS - 1 ? at : TOP_STEPS - 1;
  };
  for (int c = threadIdx.x; c < cands; c += SAMPLE_THREADS) {
    const float l = cand_l[c];
    const int at = step(l);
    atomicAdd(&h_cnt[at], 1u);
    atomicAdd(&h_mass[at], fixed_mass(l, m, inv_t));
  }
  __syncthreads();
  const uint32_t k_lim = (uint32_t)(top_k < vocab ? top_k : vocab);
  for (int exact = 0;; exact = 1) {
    // ---- the step that holds the threshold: with it the count reaches k_lim or the mass its share
    if (wave == 0) {
      uint32_t c[4], cs = 0;
      u64 q[4], qs = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        cs += c[i] = h_cnt[4 * lane + i];
        qs += q[i] = h_mass[4 * lane + i];
      }
      uint32_t ci = cs;
      u64 qi = qs;
#pragma unroll
      for (int o = 1; o < TA_WAVE; o <<= 1) {
        const uint32_t cu = __shfl_up(ci, o, TA_WAVE);
        const u64 qu = shfl_up_u64(qi, o);
        if (lane >= o) {
          ci += cu;
          qi += qu;
        }
      }
      const u64 p0 = s_p[0], p1 = s_p[1];
      const u64 at_least = __ballot(ci >= k_lim || qi >= p0), surely = __ballot(ci >= k_lim || qi >= p1);
      if (!surely) {
        if (lane == 0) s_bin = at_least && !exact ? -2 : -1;
      } else if (lane == __ffsll((unsigned long long)surely) - 1) {
        uint32_t ca = ci - cs;
        u64 ma = qi - qs;
        int hit = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
          if (hit == i && !(ca + c[i] >= k_lim || ma + q[i] >= p1)) {
            ca += c[i];
            ma += q[i];
            hit = i + 1;
          }
        // reached before at the lower end of the interval: it matters which it is
        s_bin = ma >= p0 ? -2 : 4 * lane + hit;
        s_count = ca;
        s_mass = ma;
      }
    }
    __syncthreads();
    const int bin = s_bin;
    if (bin == -1 || bin == TOP_STEPS - 1 || (bin >= 0 && (top - bin) >> finer < s_floor)) return whole();
    if (bin >= 0) {
      for (int c = threadIdx.x; c < cands; c += SAMPLE_THREADS) {
        const float l = cand_l[c];
        const int at = step(l);
        keep[c] = at < bin;
        if (at == bin) {
          const int to = atomicAdd(&s_ties, 1);
          if (to < TOP_TIES) {
            tie_key[to] = order_key(l);
            tie_at[to] = c;
            tie_q[to] = fixed_mass(l, m, inv_t);
          }
        }
      }
      __syncthreads();
      const int ties = s_ties;
      if (ties > TOP_TIES) return whole();
      // ---- what goes before each of them: higher logits, lower indices among equals
      if ((int)threadIdx.x < ties) {
        const uint32_t key = tie_key[threadIdx.x], place = tie_at[threadIdx.x];
        uint32_t n = s_count;
        u64 q = s_mass;
        for (int j = 0; j < ties; ++j) {
          const bool first = tie_key[j] > key || (tie_key[j] == key && tie_at[j] < place);
          n += first;
          q += first ? tie_q[j] : 0;
        }
        const bool low = n < k_lim && q < s_p[0], high = n < k_lim && q < s_p[1];
        keep[place] = low;
        if (low != high) s_unsure = 1;
      }
      __syncthreads();
      if (!s_unsure) break;
    }
    // ---- the row's mass itself
    u64 sum = 0;
    const int groups = (vocab + 3) / 4;
    for (int j = threadIdx.x; j < groups; j += SAMPLE_THREADS) {
      const Four f = load_four(row, j, vocab);
#pragma unroll
      for (int e = 0; e < 4; ++e) sum += f.ok[e] ? fixed_mass(f.v[e], m, inv_t) : 0;
    }
    sum = wave_sum_u64(sum);
    if (lane == 0) s_wave[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0) {
      u64 total = 0;
      for (int w = 0; w < SAMPLE_WAVES; ++w) total += s_wave[w];
      u64 p_lim = (u64)ceil((double)top_p * (double)total);
      if (p_lim < 1) p_lim = 1;
      if (p_lim > total) p_lim = total;
      s_p[0] = s_p[1] = p_lim;
      s_ties = 0;
      s_unsure = 0;
    }
    __syncthreads();
  }
  // ---- the token: the running sum of the kept ones in index order, four neighbours a thread
  u64 q[ROW_CAND / SAMPLE_THREADS], mine = 0;
  constexpr int EACH = ROW_CAND / SAMPLE_THREADS;
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int c = EACH * (int)threadIdx.x + i;
    q[i] = c < cands && keep[c < cands ? c : 0] ? fixed_mass(cand_l[c], m, inv_t) : 0;
    mine += q[i];
  }
  u64 inc = mine;
#pragma unroll
  for (int o = 1; o < TA_WAVE; o <<= 1) {
    const u64 up = shfl_up_u64(inc, o);
    if (lane >= o) inc += up;
  }
  if (lane == TA_WAVE - 1) s_wave[wave] = inc;
  __syncthreads();
  u64 sum = 0, run = 0;
#pragma unroll
  for (int w = 0; w < SAMPLE_WAVES; ++w) {
    if (w == wave) run = sum;
    sum += s_wave[w];
  }
  u64 target = (u64)((double)uni * (double)sum);
  if (sum > 0 && target >= sum) target = sum - 1;
  if (mine > 0 && run + inc > target && run + inc - mine <= target) {
    u64 at = run + inc - mine;
    int pick = 0;
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      if (q[i] > 0 && at + q[i] > target && at <= target) pick = (int)cand_i[EACH * (int)threadIdx.x + i];
      at += q[i];
    }
    out[blockIdx.x] = pick;
    if (out_host) out_host[blockIdx.x] = pick;
  }
}

__global__ __launch_bounds__(SAMPLE_THREADS) void sample_rows_kernel(const float* __restrict__ logits, size_t ld, int vocab,
                                                                     float inv_t, int top_k, float top_p,
                                                                     const float* __restrict__ uniform, int* __restrict__ out) {
  sample_whole_row<true>(logits + (size_t)blockIdx.x * ld, vocab, inv_t, top_k, top_p, uniform[blockIdx.x], out + blockIdx.x);
}

static int sample_parts(int vocab) { return (vocab + PART - 1) / PART; }

// Rows that are dealt out in parts at a time, so that the records stay within 24 MB (8,600 rows of one part); more go
// through in turns.
static int rows_at_a_time(int vocab) {
  const long long rows = (24ll << 20) / (sample_parts(vocab) * (long long)sizeof(PartRecord));
  return rows < 1 ? 1 : rows > 65535 ? 65535 : (int)rows;
}

// Whether rows are better dealt out in parts than given to a workgroup each (GPU time of a call, us, parts against whole):
// - nothing is cut: three launches, which pay while few workgroups would walk long rows. 8 x 1,000 13 against 5; 8 x
//   32,000 14.5 against 14.5; 8 x 128,256 16 against 44; 64 x 128,256 29 against 48; 512 x 128,256 148 against 104. A row
//   alone costs 5 + 3e-4 a token, parts 12 + 2.1e-6 a token of all rows.
// - else a workgroup gathers the kept tokens where they are few, and with every CU busy its three passes are cheaper than
//   the parts' two with the exponential in both. k 200, p 0.95: 100 x 128,256 70 against 74, 187 105 against 81, 512 263 against 144;
//   k 300: 750 x 32,000 122 against 74.
//   Kept tokens that don't fit (a cut by mass alone can keep thousands) are walked nine times: 188 x 128,256,
//   p 0.9, 109 against 286, 512 257 against 451, but 235 against 129 where dozens are kept: such cuts stay in parts a little
//   longer. Cuts at few tokens share the line, although their two kernels stay ahead beyond it: k 40, 187 x 128,256 43 against
//   80, 512 110 against 142, 2,048 448 against 489, 750 x 32,000 54 against 71; with k 128 1,500 x 32,000 125 against 124.
static bool in_parts(int n, int vocab, int top_k, float top_p) {
  if (sample_parts(vocab) > MAX_PARTS) return false;
  const long long all = (long long)n * vocab;
  if (top_k >= vocab && top_p >= 1.0f) return all < 145ll * vocab - 3500000;
  return vocab <= 16384 || all <= (top_k <= 1024 ? 24000000 : 35000000);
}

// Bytes of scratch that lets ta_sample_parts deal rows out in parts (0: rows of this vocabulary are not).
extern "C" long long ta_sample_scratch(int n, int vocab) {
  if (n <= 0 || vocab <= 0 || sample_parts(vocab) > MAX_PARTS) return 0;
  const int rows = n < rows_at_a_time(vocab) ? n : rows_at_a_time(vocab);
  return (long long)rows * sample_parts(vocab) * (long long)sizeof(PartRecord);
}
// The same for these cuts: 0 also where a workgroup a row is the better way.
extern "C" long long ta_sample_scratch_for(int n, int vocab, int top_k, float top_p) {
  return n > 0 && vocab > 0 && in_parts(n, vocab, top_k, top_p) ? ta_sample_scratch(n, vocab) : 0;
}

// given: null, or the n random numbers on the host, which then reach ``uniform`` in the launch's arguments; out_host: null, or
// where the tokens go as well.
static int sample_launch(hipStream_t stream, const float* logits, long long ld, int n, int vocab, float temperature, int top_k,
                         float top_p, float* uniform, int* out, void* scratch, long long scratch_bytes, const float* given,
                         int* out_host) {
  TA_REQUIRE(n >= 0 && vocab > 0 && ld >= vocab, "ta_sample: bad sizes n=%d vocab=%d ld=%lld", n, vocab, ld);
  TA_REQUIRE(temperature > 0.f, "ta_sample: temperature %g must be > 0 (0 means argmax)", (double)temperature);
  TA_REQUIRE(top_k >= 1, "ta_sample: top_k %d < 1", top_k);
  TA_REQUIRE(top_p >= 0.f && top_p <= 1.f, "ta_sample: top_p %g outside [0, 1]", (double)top_p);
  TA_REQUIRE((uintptr_t)scratch % 8 == 0, "ta_sample: scratch does not start on 8 bytes");
  if (n == 0) return 0;
  const float inv_t = 1.0f / temperature;
  const bool whole = ((uintptr_t)logits % 16) != 0 || ld % 4 != 0 || scratch == nullptr || !in_parts(n, vocab, top_k, top_p);
  TA_REQUIRE(!given || (!whole && n <= SAMPLE_IN_ARGS), "ta_sample_given: %d rows that are not dealt out in parts, or more than %d", n,
             SAMPLE_IN_ARGS);
  if (((uintptr_t)logits % 16) != 0 || ld % 4 != 0) {
    sample_kernel<<<n, SAMPLE_THREADS, 0, stream>>>(logits, (size_t)ld, vocab, inv_t, top_k, top_p, uniform, out);
  } else if (whole) {
    sample_rows_kernel<<<n, SAMPLE_THREADS, 0, stream>>>(logits, (size_t)ld, vocab, inv_t, top_k, top_p, uniform, out);
  } else {
    TA_REQUIRE(scratch_bytes >= ta_sample_scratch(n, vocab), "ta_sample: %lld bytes of scratch, %lld are needed", scratch_bytes,
               ta_sample_scratch(n, vocab));
    const int parts = sample_parts(vocab), cut = top_k < vocab || top_p < 1.0f;
    // half as many again as top_k, with room to spare, are what a part hands on
    const bool few = top_k < vocab && top_k <= TOP_MOST_K && parts * top_k <= ROW_CAND / 2;
    PartRecord* rec = (PartRecord*)scratch;
    const int turn = rows_at_a_time(vocab);
    SampleUniforms args = {};
    if (given)
      for (int i = 0; i < n; ++i) args.u[i] = given[i];
    for (int r0 = 0; r0 < n; r0 += turn) {
      const int rows = n - r0 < turn ? n - r0 : turn;
      const float* from = logits + (size_t)r0 * ld;
      const dim3 g(parts, rows);
      if (few) {
        TopRecord* tops = (TopRecord*)scratch;
        sample_top_kernel<<<g, PART_THREADS, 0, stream>>>(from, (size_t)ld, vocab, inv_t, top_k, top_p < 1.0f,
                                                          ROW_CAND / parts < TOP_CAND ? ROW_CAND / parts : TOP_CAND, tops);
        sample_top_draw_kernel<<<rows, SAMPLE_THREADS, 0, stream>>>(from, (size_t)ld, vocab, inv_t, top_k, top_p, parts, tops,
                                                                    given ? nullptr : uniform + r0, args, r0, out + r0,
                                                                    out_host ? out_host + r0 : nullptr);
        continue;
      }
      sample_parts_kernel<<<g, PART_THREADS, 0, stream>>>(from, (size_t)ld, vocab, inv_t, cut, top_p < 1.0f, rec, args,
                                                      given && r0 == 0 ? n : 0, uniform);
      sample_gather_kernel<<<g, PART_THREADS, 0, stream>>>(from, (size_t)ld, vocab, inv_t, top_k, top_p, cut, rec);
      sample_draw_kernel<<<rows, SAMPLE_THREADS, 0, stream>>>(from, (size_t)ld, vocab, inv_t, top_k, top_p, cut, parts, rec,
                                                              uniform + r0, out + r0, out_host ? out_host + r0 : nullptr);
    }
  }
  return ta_check_launch("ta_sample");
}

// scratch: scratch_bytes on an 8-byte boundary, ta_sample_scratch_for of them or more, or null: one workgroup takes a
// row then.
extern "C" int ta_sample_parts(hipStream_t stream, const float* logits, long long ld, int n, int vocab,
                               float temperature, int top_k, float top_p, const float* uniform,
                               int* out, void* scratch, long long scratch_bytes) {
  return sample_launch(stream, logits, ld, n, vocab, temperature, top_k, top_p, const_cast<float*>(uniform), out, scratch,
                       scratch_bytes, nullptr, nullptr);
}

// Rows that are dealt out in parts, at most ta_sample_given_rows of them, without a copy to the GPU in front or one back behind:
// given [n] random numbers on the host (read before the call returns), uniform [n] floats of scratch on the GPU, out_host [n]:
// pinned host memory that receives the tokens beside out. A copy of a few bytes costs 3 us on the GPU and 5 to ask for:
// 8 rows of 128,256 through Sampler 40 us a choice with them, 30 to 34 without (42 and 35 of which the host works).
extern "C" int ta_sample_given_rows() { return SAMPLE_IN_ARGS; }
extern "C" int ta_sample_given(hipStream_t stream, const float* logits, long long ld, int n, int vocab, float temperature,
                               int top_k, float top_p, const float* given, float* uniform, int* out, int* out_host,
                               void* scratch, long long scratch_bytes) {
  TA_REQUIRE(given && uniform && out_host, "ta_sample_given: the random numbers, their place and the host's tokens are needed");
  void* seen = nullptr;                              // the GPU's address of the host memory; not pinned: refused here
  const hipError_t e = hipHostGetDevicePointer(&seen, out_host, 0);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return ta_fail("ta_sample_given: the host's tokens are not in pinned memory: %s", hipGetErrorString(e));
  }
  return sample_launch(stream, logits, ld, n, vocab, temperature, top_k, top_p, uniform, out, scratch, scratch_bytes, given, (int*)seen);
}

// Without scratch: one workgroup a row.
extern "C" int ta_sample(hipStream_t stream, const float* logits, long long ld, int n, int vocab,
                         float temperature, int top_k, float top_p, const float* uniform, int* out) {
  return ta_sample_parts(stream, logits, ld, n, vocab, temperature, top_k, top_p, uniform, out, nullptr, 0);
}
