// Matrix states of long steps on the 32-bit matrix instructions: gated linear attention (a decay per key channel), the
// same with a bonus for the current token, and states with one decay per token (or per head), 16 tokens at a time.
//
// With P_t the product of a chunk's decays up to token t and S the state in front of the chunk,
//     o_t = S^T (P_t q_t) + sum_{s <= t} A[t][s] v_s,   A[t][s] = sum_i q_t[i] k_s[i] prod_{s < u <= t} a_u[i]
//     S'  = diag(P_16) S + sum_s (k_s prod_{u > s} a_u) v_s^T
// which is two products of 16 x dk x dv and one of 16 x 16 x dv where the walk token by token has 16 updates one behind
// the other. Every factor is a product of decays (no logarithm, no quotient), so none overflows and a decay of 0 is a decay
// of 0.
//
// Rounding: sixteen factors in a row add up sixteen roundings, which the walk spreads over S, and a readout that is one chain
// over a head's channels is twice as far off as the walk's sum over lanes. So products of decays are carried in two numbers,
// S takes in a chunk as one group of tokens before and one behind its own product, and readouts are chains of four added
// in pairs. Relative errors against 64 bits, walk / chunks / chunks without that care, in 1e-7: readouts of 32 heads of
// 128 x 128 1.16 / 1.09 / 2.16, their states 0.86 / 0.76 / 1.16; the bonus form of 64 x 64 0.89 / 0.87 / 1.61 and 0.54 / 0.55 /
// 0.76; matrix memory of 256 x 512 1.18 / 1.15 / 2.16 and 0.89 / 0.82 / 1.13.
//
// A workgroup owns CT value columns of one (sequence, head). Eight waves prepare the next chunk (P_t q_t, the decayed
// keys, A) on the vector ALU and leave it in LDS in the matrix instructions' order while the other waves, 16 columns each
// (and half of the key channels where there are more than 128), take this chunk; the accumulators' layout of S is the
// operands' layout of the readout, so S never leaves its registers.
//
// A chunk takes 4 to 8 us (1 to 8 sequences of 32 heads of 128 x 128), of which the matrix instructions need 1.8 at the
// most: bound by the preparation's chain of reads from LDS, products and sums over lanes. 8 x 656 tokens of 32 heads of
// 128 x 128, decays included: 829 us token by token, 336 in chunks (287 with products of decays in one number), and the norm
// reads one plane of readouts instead of four; the matrix memory of 2 x 1,536 tokens, 8 heads of 256 x 512: 730 -> 390. Half
// as many preparing waves cost 1.5 times as much; reading a group of tokens ahead of the branches, for every wave, 10 to 30 %
// more.
#include "chunked.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));

#define CH_PRODUCERS 512    // threads that prepare: 16 tokens x 32 groups of channels

enum { CH_CHANNEL = 0, CH_BONUS = 1, CH_SCALAR = 2 };

template <typename T, int N>
struct alignas(N * sizeof(T)) ChRun { T x[N]; };

__device__ float ch_one = 1.f;      // the factor of keys that have none (chosen by its address: no load waits for a branch)

// N values from c on of the row at p + off, of which n exist (c past them reads what is there and is not used)
template <int N, bool VEC, typename T>
__device__ __forceinline__ ChRun<T, N> ch_load(const T* p, uint32_t off, int c, int n) {
  if (VEC) return *reinterpret_cast<const ChRun<T, N>*>(p + (off + (uint32_t)(c < n ? c : 0)));
  ChRun<T, N> r;
#pragma unroll
  for (int e = 0; e < N; ++e) r.x[e] = p[off + (uint32_t)(c + e < n ? c + e : 0)];
  return r;
}

// Where the piece of tokens g, g + 4, g + 8, g + 12 lies in a row of 16 (rows of keys, values and A), so that the matrix
// instructions take the tokens in their order, four at a time: sixteen lanes that ask for 16 bytes
// each, of neighbouring rows and either of two pieces, meet every bank once.
__device__ __forceinline__ int ch_place(int row, int g) {
  return 4 * (g ^ ((0x78 >> (2 * ((row >> 2) & 3))) & 3));       // rows in fours: 0, 2, 3, 1
}

// Where channel c of token t lies in a row of queries, for the same reason
__device__ __forceinline__ int ch_query(int t, int c) { return (c & ~63) + 4 * (((c >> 2) & 15) ^ t) + (c & 3); }

// x is formed here. (Sums of what the matrix instructions left would else be put off to where they are stored, and what they
// are made of kept in registers until then.)
__device__ __forceinline__ void ch_now(f32x4_t& x) { asm volatile("" : "+v"(x)); }

// hi + lo, a product of decays to twice 24 bits, times one more. (A sum of hi and lo must not take the product along.)
__device__ __forceinline__ void ch_fall(float& hi, float& lo, float d) {
#pragma clang fp contract(off)
  const float p = hi * d, e = fmaf(hi, d, -p);
  lo = fmaf(lo, d, e);
  hi = p;
}
// x times such a product, rounded once; xl is x, or 0 for an infinite x, which lo would turn into an undefined one
__device__ __forceinline__ float ch_times(float x, float xl, float hi, float lo) { return fmaf(x, hi, xl * lo); }
__device__ __forceinline__ float ch_finite(float x) { return fabsf(x) < INFINITY ? x : 0.f; }

// VEC: known when the kernel is chosen, since a load inside a branch is waited for where the branch ends
template <typename T, int DK, int CT, int MODE, bool VEC>
__global__ __launch_bounds__(CH_PRODUCERS + CT / 16 * (DK > 128 ? 2 : 1) * TA_WAVE) void chunked_kernel(TaChunked p) {
  constexpr bool SCALAR = MODE == CH_SCALAR, BONUS = MODE == CH_BONUS;
  constexpr int RS = DK > 128 ? 2 : 1, ROWS = DK / RS, TILES = ROWS / 16, CW = CT / 16;
  constexpr int PC = DK / 32, RN = PC < 4 ? PC : 4, RUNS = PC / RN, VC = CT / 32;   // a producer's channels and columns
  typedef float run_t __attribute__((ext_vector_type(RN)));
  __shared__ __attribute__((aligned(16))) float s_q[2][16][DK], s_k[2][DK][16], s_v[2][CT][16], s_a[2][16][16];
  __shared__ __attribute__((aligned(16))) float s_p[2][SCALAR ? 4 : DK];          // P_16
  __shared__ __attribute__((aligned(16))) float r_q[2][16][DK], r_a[2][SCALAR ? 1 : 16][SCALAR ? 16 : DK];
  __shared__ float s_n[2][SCALAR ? DK : 1], s_red[2][RS > 1 ? CW : 1][16][17];
  __shared__ int s_odd[2][8];                      // a producer wave has seen an infinite or undefined value
  const int b = blockIdx.x, h = blockIdx.y, col0 = blockIdx.z * CT;
  const int start = p.cu_q[b], end = p.cu_q[b + 1];
  if (start >= end) return;
  const int tid = threadIdx.x, lane = tid % TA_WAVE;
  const bool producer = tid < CH_PRODUCERS;
  const int chunks = (end - start + TA_CHUNK - 1) / TA_CHUNK;
  const size_t head = (size_t)p.slots[b] * p.H + h;
  const T* proj = (const T*)p.proj;

  if (producer) {
    const int tt = tid / 32, ig = tid % 32, wave = __builtin_amdgcn_readfirstlane(tid / TA_WAVE), own = tt % 2;
    const int hq = h / p.qk_share, dk = p.dk, dv = p.dv;
    const bool norm = SCALAR && p.den_out != nullptr && blockIdx.z == 0;
    auto chan = [&](int r) { return 32 * RN * r + RN * ig; };       // run r of this thread's channels
    ChRun<T, RN> q[RUNS], k[RUNS];
    ChRun<T, VC> v;
    ChRun<float, RN> a[SCALAR ? 1 : RUNS];
    float ks = 1.f, as = 1.f;
    const float* decays = p.head_decay ? p.head_decay + h : p.tok_decay;
    const float* factors = p.tok_kscale ? p.tok_kscale : &ch_one;
    const int dstep = p.head_decay ? 0 : 1, kstep = p.tok_kscale ? 1 : 0;
    // the chunk's first row is the wave's address, a thread's place in it an offset of 32 bits: few registers
    auto fetch = [&](int c) {
      const int t0 = start + TA_CHUNK * (c < chunks ? c : chunks - 1), left = end - 1 - t0, at = tt < left ? tt : left;
      const T* pr = proj + (size_t)t0 * p.stride;
      const uint32_t off = (uint32_t)at * (uint32_t)p.stride;
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        q[r] = ch_load<RN, VEC>(pr + p.qoff + hq * dk, off, chan(r), dk);
        k[r] = ch_load<RN, VEC>(pr + p.koff + hq * dk, off, chan(r), dk);
        if (!SCALAR)
          a[r] = ch_load<RN, VEC>(p.alpha + (size_t)t0 * ((size_t)p.H * dk) + h * dk, (uint32_t)at * (uint32_t)(p.H * dk), chan(r), dk);
      }
      v = ch_load<VC, VEC>(pr + p.voff + h * dv, off, col0 + ig * VC, dv);      // (columns past dv: those of the head's start)
      if (SCALAR) {
        const size_t th = (size_t)(t0 + at) * p.H + h;
        as = decays[th * dstep];
        ks = factors[th * kstep];
      }
    };
    // what fetch(c) brought: queries and decays to LDS for the other threads, keys and values kept
    float kf[PC], vf[VC];
    auto take = [&](int c) {
      const bool on = start + TA_CHUNK * c + tt < end;
      const int at = c & 1;
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        run_t x, y;
#pragma unroll
        for (int e = 0; e < RN; ++e) {
          const bool ok = on && chan(r) + e < dk;
          x[e] = ok ? to_f32(q[r].x[e]) * p.qscale : 0.f;
          kf[RN * r + e] = ok ? to_f32(k[r].x[e]) * ks : 0.f;
          if (!SCALAR) y[e] = ok ? a[r].x[e] : 1.f;         // a token that is not there leaves S as it is
        }
        *(run_t*)&r_q[at][tt][chan(r)] = x;
        if (!SCALAR) *(run_t*)&r_a[at][SCALAR ? 0 : tt][chan(r)] = y;
      }
      if (SCALAR && ig == 0) r_a[at][0][tt] = on ? as : 1.f;
#pragma unroll
      for (int j = 0; j < VC; ++j) vf[j] = on && col0 + ig * VC + j < dv ? to_f32(v.x[j]) : 0.f;
    };
    float u[BONUS ? PC : 1];
    if (BONUS) {
#pragma unroll
      for (int j = 0; j < PC; ++j) {
        const int i = chan(j / RN) + j % RN;
        u[j] = i < dk ? p.bonus[h * dk + i] : 0.f;
      }
    }
    float n = 0.f;                                 // the normaliser's channel `tid`
    if (norm) {
      if (tid < dk) n = p.n_state[head * dk + tid];
      if (tid < DK) s_n[0][tid] = n;
    }
    // denominators of the chunk that the other waves work on
    auto normalise = [&](int c) {
      const int cur = c & 1, nxt = cur ^ 1;
      float d = 0.f;
#pragma unroll
      for (int r = 0; r < RUNS; ++r) {
        const run_t x = *(const run_t*)&s_q[cur][tt][ch_query(tt, chan(r))], y = *(const run_t*)&s_n[cur][chan(r)];
        float run = x[0] * y[0];
#pragma unroll
        for (int e = 1; e < RN; ++e) run = fmaf(x[e], y[e], run);
        d += run;
      }
      if (ig < 16) d += s_a[cur][tt][ig];          // (a row's sum: its pieces lie in another order)
      float none = 0.f;
      ta_sums2<32>(d, none);
      const int t = start + TA_CHUNK * c + tt;
      if (ig == 0 && t < end) p.den_out[(size_t)t * p.H + h] = d;
      if (tid < DK) {
        float keys[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4_t x = *(const f32x4_t*)&s_k[cur][tid][4 * g];
          keys[g] = (x[0] + x[1]) + (x[2] + x[3]);
        }
        n = fmaf(n, s_p[cur][0], (keys[0] + keys[1]) + (keys[2] + keys[3]));
        s_n[nxt][tid] = n;
      }
    };
    fetch(0);
    take(0);
    fetch(1);
    __syncthreads();
    // (no load in this loop is conditional: what it brings stays in its registers until it is used)
    for (int c = 0; c < chunks; ++c) {
      const int at = c & 1;
      bool odd = false;
#pragma unroll
      for (int j = 0; j < VC; ++j) {
        s_v[at][ig * VC + j][ch_place(ig * VC + j, tt % 4) + tt / 4] = vf[j];
        odd |= !(fabsf(vf[j]) < INFINITY);
      }
      const bool any = __any(odd);
      if (lane == 0) s_odd[at][wave] = any;
      // r + rl: the product of the decays up to token tt, from there on what the later tokens leave of the key
      float kl[SCALAR ? 1 : PC], r[PC], rl[PC], dq[PC], acc[16], fall[SCALAR ? 16 : 1], rs = 1.f, rsl = 0.f, ps = 1.f;
#pragma unroll
      for (int j = 0; j < PC; ++j) {
        if (!SCALAR) kl[SCALAR ? 0 : j] = ch_finite(kf[j]);
        r[j] = 1.f;
        rl[j] = 0.f;
      }
#pragma unroll
      for (int t = 0; t < 16; ++t) acc[t] = 0.f;
      f32x4_t da[SCALAR ? 4 : 1];
      if (SCALAR) {
#pragma unroll
        for (int e = 0; e < 4; ++e) da[SCALAR ? e : 0] = *(const f32x4_t*)&r_a[at][0][SCALAR ? 4 * e : 0];
      }
#pragma unroll
      for (int bq = 0; bq < 8; ++bq) {
        if (bq % 2 == 0) __builtin_amdgcn_sched_barrier(0);      // operands are not asked for far ahead: registers
        if (bq < wave) {                           // tokens in front of this wave's
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int t = 2 * bq + e;
            if (SCALAR) {
              ch_fall(rs, rsl, da[SCALAR ? t / 4 : 0][t % 4]);
              fall[SCALAR ? t : 0] = 0.f;
            } else {
#pragma unroll
              for (int x = 0; x < RUNS; ++x) {
                const run_t d = *(const run_t*)&r_a[at][SCALAR ? 0 : t][chan(x)];
#pragma unroll
                for (int i = 0; i < RN; ++i) ch_fall(r[RN * x + i], rl[RN * x + i], d[i]);
              }
            }
          }
        } else if (bq == wave) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int t = 2 * bq + e;
            const bool mine = own == e;
            if (SCALAR) {
              ch_fall(rs, rsl, da[SCALAR ? t / 4 : 0][t % 4]);
              ps = mine ? rs + rsl : ps;           // P_tt
              rs = mine ? 1.f : rs;
              rsl = mine ? 0.f : rsl;
              fall[SCALAR ? t : 0] = rs + rsl;
            }
#pragma unroll
            for (int x = 0; x < RUNS; ++x) {
              const run_t qv = *(const run_t*)&r_q[at][t][chan(x)];
              run_t d = 1.f;
              if (!SCALAR) d = *(const run_t*)&r_a[at][SCALAR ? 0 : t][chan(x)];
#pragma unroll
              for (int i = 0; i < RN; ++i) {
                const int j = RN * x + i;
                if (SCALAR) {
                  dq[j] = mine ? qv[i] : dq[j];
                  acc[t] = fmaf(qv[i], kf[j], acc[t]);
                } else {
                  if (BONUS) {
                    dq[j] = mine ? ch_times(qv[i], ch_finite(qv[i]), r[j], rl[j]) : dq[j];
                    acc[t] = fmaf(qv[i], mine ? u[BONUS ? j : 0] * kf[j] : ch_times(kf[j], kl[SCALAR ? 0 : j], r[j], rl[j]), acc[t]);
                  }
                  ch_fall(r[j], rl[j], d[i]);
                  if (!BONUS) {
                    dq[j] = mine ? ch_times(qv[i], ch_finite(qv[i]), r[j], rl[j]) : dq[j];
                    acc[t] = fmaf(qv[i], mine ? kf[j] : ch_times(kf[j], kl[SCALAR ? 0 : j], r[j], rl[j]), acc[t]);
                  }
                  if (t == 15 && mine) s_p[at][chan(x) + i] = r[j] + rl[j];
                  r[j] = mine ? 1.f : r[j];
                  rl[j] = mine ? 0.f : rl[j];
                }
              }
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int t = 2 * bq + e;
            if (SCALAR) {
              ch_fall(rs, rsl, da[SCALAR ? t / 4 : 0][t % 4]);
              fall[SCALAR ? t : 0] = rs + rsl;
            }
#pragma unroll
            for (int x = 0; x < RUNS; ++x) {
              const run_t qv = *(const run_t*)&r_q[at][t][chan(x)];
              run_t d = 1.f;
              if (!SCALAR) d = *(const run_t*)&r_a[at][SCALAR ? 0 : t][chan(x)];
#pragma unroll
              for (int i = 0; i < RN; ++i) {
                const int j = RN * x + i;
                if (SCALAR) {
                  acc[t] = fmaf(qv[i], kf[j], acc[t]);
                } else {
                  if (BONUS) acc[t] = fmaf(qv[i], ch_times(kf[j], kl[SCALAR ? 0 : j], r[j], rl[j]), acc[t]);
                  ch_fall(r[j], rl[j], d[i]);
                  if (!BONUS) acc[t] = fmaf(qv[i], ch_times(kf[j], kl[SCALAR ? 0 : j], r[j], rl[j]), acc[t]);
                }
              }
            }
          }
        }
      }
      float of = 0.f;                              // A[ig][tt]
#pragma unroll
      for (int t = 0; t < 16; t += 2) {
        ta_sums2<32>(acc[t], acc[t + 1]);
        of = ig == t ? (SCALAR ? acc[t] * fall[SCALAR ? t : 0] : acc[t]) : of;
        of = ig == t + 1 ? (SCALAR ? acc[t + 1] * fall[SCALAR ? t + 1 : 0] : acc[t + 1]) : of;
      }
      if (ig < 16) s_a[at][ig][ch_place(ig, tt % 4) + tt / 4] = ig >= tt ? of : 0.f;
      if (SCALAR && tid == CH_PRODUCERS - 1) s_p[at][0] = ps;
#pragma unroll
      for (int x = 0; x < RUNS; ++x) {
        run_t y;
#pragma unroll
        for (int i = 0; i < RN; ++i) {
          const int j = RN * x + i;
          y[i] = SCALAR ? dq[j] * ps : dq[j];
          s_k[at][chan(x) + i][ch_place(chan(x), tt % 4) + tt / 4] = SCALAR ? ch_times(kf[j], ch_finite(kf[j]), rs, rsl) : ch_times(kf[j], kl[SCALAR ? 0 : j], r[j], rl[j]);
        }
        *(run_t*)&s_q[at][tt][ch_query(tt, chan(x))] = y;
      }
      take(c + 1);                                 // (behind the last chunk: nothing)
      fetch(c + 2);
      if (norm && c > 0) normalise(c - 1);
      __syncthreads();
    }
    if (norm) normalise(chunks - 1);
    __syncthreads();
    if (norm && tid < dk) p.n_state[head * dk + tid] = n;
    return;
  }

  const int cw = (tid - CH_PRODUCERS) / TA_WAVE, ct = cw % CW, part = cw / CW, row0 = part * ROWS;
  const int m = lane % 16, g = lane / 16, col = col0 + 16 * ct + m, piece = ch_place(m, g);
  const bool mine = col < p.dv;
  float* st = p.state + head * p.dk * (size_t)p.dv + (mine ? col : 0);
  f32x4_t S[TILES];
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 16 * i + 4 * g + r;
      S[i][r] = mine && row < p.dk ? st[(size_t)row * p.dv] : 0.f;
    }
  auto store = [&](int c, f32x4_t o) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int t = start + TA_CHUNK * c + 4 * g + r;
      if (mine && t < end) {
        float* out = p.o_out + ((size_t)t * p.H + h) * p.dv + col;
        *out = o[r];
        for (int z = 1; z < p.planes; ++z) out[z * p.plane] = 0.f;
      }
    }
  };
  f32x4_t held = {0.f, 0.f, 0.f, 0.f};             // this half's readout of the chunk before
  auto join = [&](int c) {
#pragma unroll
    for (int r = 0; r < 4; ++r) held[r] += s_red[c & 1][RS > 1 ? ct : 0][4 * g + r][m];
    store(c, held);
  };
  __syncthreads();
  __syncthreads();
  for (int c = 0; c < chunks; ++c) {
    const int cur = c & 1;
    const f32x4_t v = *(const f32x4_t*)&s_v[cur][16 * ct + m][piece];
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t o = zero;
    // sixteen terms: four chains of four
    auto dot = [&](const f32x4_t& x, const f32x4_t& y) {
      f32x4_t c[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) c[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[j], y[j], zero, 0, 0, 0);
      return (c[0] + c[1]) + (c[2] + c[3]);
    };
    if (part == 0) {
      if (s_odd[cur][0] | s_odd[cur][1] | s_odd[cur][2] | s_odd[cur][3] | s_odd[cur][4] | s_odd[cur][5] | s_odd[cur][6] | s_odd[cur][7]) {
        // a later token's infinite or undefined value must not reach this token as 0 times it
#pragma unroll
        for (int r = 0; r < 4; ++r)
          for (int t = 0; t <= 4 * g + r; ++t)
            o[r] = fmaf(s_a[cur][4 * g + r][ch_place(4 * g, t % 4) + t / 4], s_v[cur][16 * ct + m][ch_place(m, t % 4) + t / 4], o[r]);
      } else {
        o = dot(*(const f32x4_t*)&s_a[cur][m][piece], v);
      }
    }
    // the tiles' sums in pairs, the pairs' in pairs: as short a chain as their number allows. The next tile's operands are on
    // their way, no others: registers.
    static_assert(TILES == 4 || TILES == 8, "fours of tiles");
    auto query = [&](int i) { return *(const f32x4_t*)&s_q[cur][m][ch_query(m, row0 + 16 * i + 4 * g)]; };
    f32x4_t x = query(0), pairs[2], fours = zero;
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      const f32x4_t mine = x;
      if (i + 1 < TILES) x = query(i + 1);
      __builtin_amdgcn_sched_barrier(0);
      f32x4_t sum = dot(mine, S[i]);
      ch_now(sum);
      if (i % 2 == 0) pairs[i / 2 % 2] = sum;
      else pairs[i / 2 % 2] += sum;
      if (i % 4 == 3) {
        const f32x4_t four = pairs[0] + pairs[1];
        if (i < 4) fours = four;
        else fours += four;
        ch_now(fours);
      }
    }
    o += fours;
    auto key = [&](int i) { return *(const f32x4_t*)&s_k[cur][row0 + 16 * i + m][piece]; };
    x = key(0);
    f32x4_t P = s_p[cur][0];
#pragma unroll
    for (int i = 0; i < TILES; ++i) {
      const f32x4_t mine = x;
      if (!SCALAR) P = *(const f32x4_t*)&s_p[cur][SCALAR ? 0 : row0 + 16 * i + 4 * g];
      if (i + 1 < TILES) x = key(i + 1);
      __builtin_amdgcn_sched_barrier(0);
      // the first eight tokens by themselves, then S, then the last eight: S that lasts is rounded nine times a chunk where
      // the walk rounds it sixteen times, S that fades as the walk would
      f32x4_t fresh = __builtin_amdgcn_mfma_f32_16x16x4f32(mine[0], v[0], zero, 0, 0, 0);
      fresh = __builtin_amdgcn_mfma_f32_16x16x4f32(mine[1], v[1], fresh, 0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) S[i][r] = fmaf(S[i][r], P[r], fresh[r]);
#pragma unroll
      for (int j = 2; j < 4; ++j) S[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(mine[j], v[j], S[i], 0, 0, 0);
    }
    if (RS == 1) {
      store(c, o);
    } else if (part > 0) {
#pragma unroll
      for (int r = 0; r < 4; ++r) s_red[cur][RS > 1 ? ct : 0][4 * g + r][m] = o[r];
    } else {
      if (c > 0) join(c - 1);
      held = o;
    }
    __syncthreads();
  }
  if (RS > 1 && part == 0) join(chunks - 1);
#pragma unroll
  for (int i = 0; i < TILES; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = row0 + 16 * i + 4 * g + r;
      if (mine && row < p.dk) st[(size_t)row * p.dv] = S[i][r];
    }
}

bool ta_chunked_takes(bool scalar_decay, bool bonus, int dk) {
  return dk <= 128 || (scalar_decay && !bonus && dk <= 256);
}

template <typename T, int DK, int CT, int MODE, bool VEC = true>
static void chunked_run(hipStream_t stream, const TaChunked& p, int batch) {
  const dim3 g(batch, p.H, (p.dv + CT - 1) / CT);
  chunked_kernel<T, DK, CT, MODE, VEC><<<g, CH_PRODUCERS + CT / 16 * (DK > 128 ? 2 : 1) * TA_WAVE, 0, stream>>>(p);
}

template <typename T, int DK, int MODE>
static void chunked_by_columns(hipStream_t stream, const TaChunked& p, int batch) {
  if (!p.vec) return chunked_run<T, DK, 32, MODE, false>(stream, p, batch);
  // as many columns a workgroup as leave three quarters of the CUs one: the preparation is then shared by more waves
  const long long heads = (long long)batch * p.H;
  constexpr int MOST = DK > 128 ? 64 : 128;
  if (MOST >= 128 && p.dv > 64 && heads * ((p.dv + 127) / 128) >= 192) chunked_run<T, DK, MOST, MODE>(stream, p, batch);
  else if (p.dv > 32 && heads * ((p.dv + 63) / 64) >= 192) chunked_run<T, DK, 64, MODE>(stream, p, batch);
  else chunked_run<T, DK, 32, MODE>(stream, p, batch);
}

template <typename T>
static void chunked_by_mode(hipStream_t stream, const TaChunked& p, int batch) {
  if (p.bonus) {
    if (p.dk <= 64) chunked_by_columns<T, 64, CH_BONUS>(stream, p, batch);
    else chunked_by_columns<T, 128, CH_BONUS>(stream, p, batch);
  } else if (p.alpha) {
    if (p.dk <= 64) chunked_by_columns<T, 64, CH_CHANNEL>(stream, p, batch);
    else chunked_by_columns<T, 128, CH_CHANNEL>(stream, p, batch);
  } else {
    if (p.dk <= 64) chunked_by_columns<T, 64, CH_SCALAR>(stream, p, batch);
    else if (p.dk <= 128) chunked_by_columns<T, 128, CH_SCALAR>(stream, p, batch);
    else chunked_by_columns<T, 256, CH_SCALAR>(stream, p, batch);
  }
}

int ta_chunked_launch(hipStream_t stream, int dtype, const TaChunked& in, int batch, const char* what) {
  TA_REQUIRE(ta_chunked_takes(in.alpha == nullptr, in.bonus != nullptr, in.dk), "%s: keys of %d do not go in chunks", what, in.dk);
  TA_REQUIRE((in.dv + 31) / 32 <= 65535, "%s: values of %d", what, in.dv);
  TaChunked p = in;
  const int item = dtype == TA_F32 ? 4 : 2;
  p.vec = p.stride % 4 == 0 && p.qoff % 4 == 0 && p.koff % 4 == 0 && p.voff % 4 == 0 && p.dk % 4 == 0 && p.dv % 4 == 0 &&
          (uintptr_t)p.proj % (4 * item) == 0 && (uintptr_t)p.alpha % 16 == 0;
  if (dtype == TA_F32) chunked_by_mode<float>(stream, p, batch);
  else if (dtype == TA_BF16) chunked_by_mode<bf16_t>(stream, p, batch);
  else return ta_fail("%s: unknown dtype %d", what, dtype);
  return ta_check_launch(what);
}
