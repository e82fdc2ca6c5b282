// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) in 32 bits for many rows, on the 16-bit matrix instructions (split.h, which also states the
// order of the sums: a row has the bits here that it has in the kernels for few rows).
#include <math.h>
#include <type_traits>
#include "split.h"
#include "gemm_split.h"

__device__ f32x4 split_zeros;      // where a piece past K is read from (never written: zero)

// A workgroup owns 32 WAVES x 16 NT of C. A wave owns 32 of the rows: it reads them from memory in operand layout and splits them,
// which no other wave needs; the columns' k are split once per workgroup, by all its waves, and go through LDS in operand layout,
// 32 k at a time in two buffers, one barrier a step. The next step's operands are split between this step's products and what comes after them is
// asked for right there. Bound by issue: 96 matrix instructions of 16 cycles, some 250 vector instructions and 30 of LDS a step of 32 k and wave. 1,021 x
// 16,384 x 2,048 301 to 330 us by card (208 to 228 TFLOP/s, up to 1.37 PFLOP/s of bfloat16; 535 to 610 in float32 tiles of 128 x 128 on the float32 matrix instructions), 1,021 x 3,072 x 2,048 78
// (122), x 2,048 x 2,048 56 (79), x 2,048 x 8,192 204 (292). A split once by a kernel in front: the same (386 us and 384). Four waves of 64 rows: 455 for 370. G groups of WAVES waves take the segments of k in turn and the first adds up what the others hand it through LDS,
// in ascending order.
//
// GLU: W holds gate rows, then up rows (N in all); every other 16 of the workgroup's columns are the ups of the 16 before, and C = silu(gate) * up. 1,021 rows x 8,192
// channels x 2,048 302 us, product and activation in turn 316; 2,000 rows 600 and 651; 3,000 x 14,336 x 4,096 3,400 and 3,477. Where the product goes by other
// tiles (513 rows) it is their difference that would be lost.
//
// FAR: rows further apart than offsets of 32 bits reach, in size_t.
template <int WAVES, int NT, int G, bool VEC, bool WHOLE, bool GLU = false, bool FAR = false>
__global__ __launch_bounds__(WAVES * G * 64, 2) void gemm_split_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W,
                                                                    int ldw, const float* __restrict__ bias, float* __restrict__ C,
                                                                    int ldc, int M, int N, int K, long long sa, long long sw,
                                                                    long long sc, int tiles_m, int tiles) {
  static_assert(NT >= 4 && NT % 2 == 0, "columns in pairs of tiles, the rows' splits between them");
  constexpr int MT = 2, COLS = GLU ? 8 * NT : 16 * NT, ROWS = 16 * MT * WAVES;       // COLS: of C
  constexpr int BRING = (NT + WAVES - 1) / WAVES;      // tiles of 16 columns that a wave brings
  __shared__ bf16x8 S[G][2][3][NT][TA_WAVE];
  __shared__ f32x4 handed[G > 1 ? G - 1 : 1][G > 1 ? WAVES : 1][G > 1 ? MT * NT : 1][G > 1 ? TA_WAVE : 1];
  const int lane = threadIdx.x % TA_WAVE, at = __builtin_amdgcn_readfirstlane(threadIdx.x / TA_WAVE), wave = at % WAVES, group = at / WAVES;
  const int r = lane % 16, kb = lane / 16;
  // an XCD's workgroups (every eighth) walk neighbouring tiles, rows first
  const int share = (tiles + 7) / 8, tile = blockIdx.x % 8 * share + blockIdx.x / 8;
  if (tile >= tiles) return;
  A += (size_t)blockIdx.y * sa;
  W += (size_t)blockIdx.y * sw;
  C += (size_t)blockIdx.y * sc;
  const int m0 = tile % tiles_m * ROWS, n0 = tile / tiles_m * COLS;
  const int n_out = GLU ? N / 2 : N;
  const int blocks = (K + 31) / 32, segs = (K + SEG - 1) / SEG, rounds = (segs + G - 1) / G;
  // steps of this group: 8 to a segment, and no further than the longest group's k
  const int last = segs - (rounds - 1) * G > 1 ? SEG / 32 : blocks - (segs - 1) * (SEG / 32);
  const int steps = (rounds - 1) * (SEG / 32) + last;
  const char* abase = reinterpret_cast<const char*>(A + (size_t)m0 * lda);
  const char* wbase = reinterpret_cast<const char*>(W + (size_t)n0 * ldw);
  typedef typename std::conditional<FAR, size_t, uint32_t>::type Offset;
  Offset aoff[MT], woff[BRING];                         // rows past M or N read another row and feed what is never stored
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = wave * 16 * MT + 16 * i + r;
    aoff[i] = ((Offset)(m0 + m < M ? m : M - 1 - m0) * lda + 4 * kb) * 4;
  }
#pragma unroll
  for (int i = 0; i < BRING; ++i) {
    const int f = wave + WAVES * i < NT ? wave + WAVES * i : NT - 1, n = 16 * (GLU ? f / 2 : f) + r;
    woff[i] = ((Offset)((n0 + n < n_out ? n : n_out - 1 - n0) + (GLU && f % 2 ? n_out : 0)) * ldw + 4 * kb) * 4;
  }
  auto piece = [&](const char* base, Offset off, int b, int h) {
    const char* p = base + (size_t)b * 128 + off + 64 * h;
    if (VEC) {
      if (!WHOLE) p = b * 32 + 16 * h + 4 * kb < K ? p : reinterpret_cast<const char*>(&split_zeros);
      return *reinterpret_cast<const f32x4*>(p);
    }
    f32x4 v;
    if (b * 32 + 32 <= K) {                            // 16 bytes from wherever they start (four loads of 4: 130 x 5,000 x 2,049 134 us)
      typedef float any4 __attribute__((ext_vector_type(4), aligned(4)));
      const any4 u = *reinterpret_cast<const any4*>(p);
      v = f32x4{u[0], u[1], u[2], u[3]};
      return v;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const char* q = b * 32 + 16 * h + 4 * kb + e < K ? p + 4 * e : reinterpret_cast<const char*>(&split_zeros);
      v[e] = *reinterpret_cast<const float*>(q);
    }
    return v;
  };
  f32x4 win[BRING][2], ain[MT][2];
  Split8 a[2][MT];
  // WHOLE (K of whole segments): behind the last block the same once more, unused; else zeros
  auto block_of = [&](int s) {
    const int b = (s / (SEG / 32) * G + group) * (SEG / 32) + s % (SEG / 32);
    return !WHOLE || b < blocks ? b : blocks - 1;
  };
  auto load_w = [&](int s) {
    const int b = block_of(s);
#pragma unroll
    for (int i = 0; i < BRING; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h) win[i][h] = piece(wbase, woff[i], b, h);
  };
  auto load_a = [&](int i, int s) {
    const int b = block_of(s);
#pragma unroll
    for (int h = 0; h < 2; ++h) ain[i][h] = piece(abase, aoff[i], b, h);
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < BRING; ++i) {
      const int f = wave + WAVES * i;
      if (NT % WAVES == 0 || f < NT) {
        const Split8 w = split8(win[i][0], win[i][1]);
        S[group][buf][0][f][lane] = w.h;
        S[group][buf][1][f][lane] = w.m;
        S[group][buf][2][f][lane] = w.l;
      }
    }
  };
  f32x4 acc[MT][NT], total[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  load_w(0);
#pragma unroll
  for (int i = 0; i < MT; ++i) load_a(i, 0);
  stash(0);
  load_w(1);
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    a[0][i] = split8(ain[i][0], ain[i][1]);
    load_a(i, 1);
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  auto step = [&](int s, int buf) {
#pragma unroll
    for (int j = 0; j < NT; j += 2) {
      Split8 w[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        w[x].h = S[group][buf][0][j + x][lane];
        w[x].m = S[group][buf][1][j + x][lane];
        w[x].l = S[group][buf][2][j + x][lane];
      }
      f32x4 t[MT][2];
#pragma unroll
      for (int i = 0; i < MT; ++i) t[i][0] = t[i][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int i = 0; i < MT; ++i) t[i][x] = split_mul(q, w[x], a[buf][i], t[i][x]);
      __builtin_amdgcn_s_setprio(0);
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int i = 0; i < MT; ++i) acc[i][j + x] += t[i][x];
      if (j == 0) {
        stash(buf ^ 1);
        load_w(s + 2);
      }
#pragma unroll
      for (int i = 0; i < MT; ++i)
        if (j == (NT > 4 ? 2 + 2 * i : 2 * i)) {
          a[buf ^ 1][i] = split8(ain[i][0], ain[i][1]);
          load_a(i, s + 2);
        }
      // two products, then up to six of the vector instructions between them
#pragma unroll
      for (int z = 0; z < 12; ++z) {
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 6, 0);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  for (int s0 = 0, round = 0; round < rounds; ++round) {
    const int end = s0 + SEG / 32 < steps ? s0 + SEG / 32 : steps;
    for (; s0 < end; s0 += 2) {
      step(s0, 0);
      if (s0 + 1 < end) step(s0 + 1, 1);
    }
    if (G > 1 && group > 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) handed[group - 1][wave][i * NT + j][lane] = acc[i][j];
    }
    if (G > 1) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    // (the next round's first barrier lies behind these reads and in front of its sums)
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        if (group == 0) {
          total[i][j] += acc[i][j];
#pragma unroll
          for (int g = 1; g < G; ++g)
            if (round * G + g < segs) total[i][j] += handed[g - 1][wave][i * NT + j][lane];
        }
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if (group > 0) return;
  // a lane's columns are four neighbours, stored at once where that is 16 bytes (1,021 x 16,384 x 2,048: 325 us one by one, 301 so)
  const bool wide = ldc % 4 == 0 && (uintptr_t)C % 16 == 0;
  auto store = [&](int m, int n, const f32x4& v) __attribute__((always_inline)) {
    float* c = C + (size_t)m * ldc + n;
    if (wide && n + 3 < n_out) {
      *reinterpret_cast<f32x4*>(c) = v;
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < n_out) c[e] = v[e];
  };
  // What is not finite: bit i PER + 4 j + e of the lane's, of gates and ups one set each. Rows with an undefined number are left as they are.
  constexpr int PER = GLU ? NT * 2 : NT * 4;           // results of one row tile
  uint64_t bad[GLU ? 2 : 1] = {};
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        bad[GLU ? j % 2 : 0] |= (uint64_t)(m0 + wave * 16 * MT + 16 * i + r < M && n0 + 16 * (GLU ? j / 2 : j) + 4 * kb + e < n_out &&
                                           split_bad(total[i][j][e])) << (i * PER + (GLU ? j / 2 : j) * 4 + e);
      total[i][j] *= SPLIT_DOWN;
    }
  auto of_row = [&](int m) { return [=](int k) { return A[(size_t)m * lda + k]; }; };
  uint64_t any = GLU ? bad[0] | bad[1 % (GLU ? 2 : 1)] : bad[0];
  if (__ballot(any != 0) != 0)
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const uint64_t own = (PER == 64 ? ~0ull : (1ull << PER) - 1) << (i * PER), lanes = __ballot((any & own) != 0);
#pragma unroll 1
      for (uint32_t rows = (lanes | lanes >> 16 | lanes >> 32 | lanes >> 48) & 0xffff; rows; rows &= rows - 1) {
        const int row = __builtin_ctz(rows);
        if (!split_undefined(of_row(m0 + wave * 16 * MT + 16 * i + row), K)) continue;
        if (r == row) any &= ~own, bad[0] &= ~own, bad[GLU ? 1 : 0] &= ~own;
      }
    }
  // The others, by the wave one after the other: form(bit, lane, row, column).
  auto again = [&](auto form) {
    if (__ballot(any != 0) == 0) return;
#pragma unroll 1
    for (int x = 0; x < MT * PER; ++x)
#pragma unroll 1
      for (uint64_t lanes = __ballot((any >> x & 1) != 0); lanes; lanes &= lanes - 1) {
        const int from = __builtin_ctzll(lanes);
        form(x, from, m0 + wave * 16 * MT + 16 * (x / PER) + from % 16, n0 + 16 * (x % PER / 4) + 4 * (from / 16) + x % 4);
      }
  };
  if constexpr (GLU) {
    // Of a gate and an up of which one is to be formed again C holds the other meanwhile.
    auto join = [&](float g, float u, int n) { return ta_glu(TaGlu{}, bias ? g + bias[n] : g, bias ? u + bias[n_out + n] : u); };
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + wave * 16 * MT + 16 * i + r;
      if (m >= M) continue;
#pragma unroll
      for (int j = 0; j < NT / 2; ++j) {
        const int n = n0 + 16 * j + 4 * kb;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = total[i][2 * j][e], u = total[i][2 * j + 1][e];
          const int x = i * PER + j * 4 + e;
          v[e] = bad[0] >> x & 1 ? u : bad[1] >> x & 1 ? g : n + e < n_out ? join(g, u, n + e) : 0.f;
        }
        store(m, n, v);
      }
    }
    again([&](int x, int from, int m, int n) {
      const bool gate = __builtin_amdgcn_readlane((int)(bad[0] >> x & 1), from), up = __builtin_amdgcn_readlane((int)(bad[1] >> x & 1), from);
      float g = 0.f, u = 0.f;
      if (gate) g = split_dot(of_row(m), W + (size_t)n * ldw, K);
      if (up) u = split_dot(of_row(m), W + (size_t)(n_out + n) * ldw, K);
      if (lane != from) return;
      float* c = C + (size_t)m * ldc + n;
      *c = join(gate ? g : *c, up ? u : *c, n);
    });
    return;
  }
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + wave * 16 * MT + 16 * i + r;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int n = n0 + 16 * j + 4 * kb;
      f32x4 v = total[i][j];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (bias && n + e < N) v[e] += bias[n + e];
      store(m, n, v);
    }
  }
  again([&](int, int from, int m, int n) {
    const float v = split_dot(of_row(m), W + (size_t)n * ldw, K);
    if (lane == from) C[(size_t)m * ldc + n] = bias ? v + bias[n] : v;
  });
}

// us a step of 32 k (of all groups) and us a round of workgroups beside its steps, when every CU has one: fitted to all forms at 7 to 3,000 rows of 2,048 to 28,672
// columns, k from 256 to 14,336, to 5 to 8 %. 256 x 128 reads and splits least per product but leaves CUs idle where there are few tiles: 16,384 x 2,048 at 1,021 rows
// 310 us there and 390 by 128 x 64, at 130 rows 132 and 105; 4,096 x 1,024 at 700 rows 70 and 51. Groups fill a CU that has a tile to itself: 2,048 x 8,192 at 1,021 rows 214 us by two,
// 6,144 x 8,192 at 64 rows 248 by one, 172 by two, 129 by four on 64 x 64. Two workgroups of 128 x 64 with one group share a CU.
// With split_few_cost they choose, of 633 sizes of 17 to 513 rows and k from 516, the fastest way to 0.5 % in the mean, 29 at the worst (16,384 x 516 at 17 rows: 20 us for 16).
struct SplitForm {
  int waves, nt, groups;
  float step, round;
};
constexpr SplitForm SPLIT_FORMS[] = {{0, 0, 0, 0.f, 0.f},      {8, 8, 1, 1.96f, 6.4f}, {4, 6, 2, 1.91f, 5.1f}, {4, 4, 2, 1.43f, 3.6f}, {2, 4, 4, 1.96f, 3.7f},
                                     {4, 4, 1, 1.47f, 3.1f}, {2, 4, 1, 1.02f, 3.6f}, {2, 4, 4, 1.96f, 3.7f}, {4, 4, 1, 1.47f, 3.1f}};
enum { SPLIT_GROUPS = 4, SPLIT_PAIRED = 5, SPLIT_SMALL = 6, SPLIT_FAR = 3, SPLIT_CUS = 256 };      // + SPLIT_FAR: the same, rows any distance apart
#define SPLIT_LAUNCH 2.0        // us of a launch
#define SPLIT_ALONE 0.94        // us a step of a SPLIT_PAIRED workgroup that has its CU to itself

static long long split_tiles(int form, int M, int N) {
  const SplitForm& f = SPLIT_FORMS[form];
  return (long long)((M + 32 * f.waves - 1) / (32 * f.waves)) * ((N + 16 * f.nt - 1) / (16 * f.nt));
}
static double split_cost(int form, int M, int N, int K, int batch) {
  const SplitForm& f = SPLIT_FORMS[form];
  const long long tiles = split_tiles(form, M, N) * batch;
  const int blocks = (K + 31) / 32, segs = (K + SEG - 1) / SEG, rounds = (segs + f.groups - 1) / f.groups;
  const int last = segs - (rounds - 1) * f.groups > 1 ? SEG / 32 : blocks - (segs - 1) * (SEG / 32);        // as in the kernel
  const int steps = f.groups == 1 ? blocks : (rounds - 1) * (SEG / 32) + last;
  const double round = (double)steps * f.step + f.round;
  if (form == SPLIT_SMALL) {                           // up to four share a CU
    const double share = (double)tiles / SPLIT_CUS, turns = share <= 4.0 ? (double)((tiles + SPLIT_CUS - 1) / SPLIT_CUS) : share;
    return SPLIT_LAUNCH + steps * f.step + f.round + (turns - 1.0) * (0.37 * steps + 1.2);
  }
  if (form != SPLIT_PAIRED) return SPLIT_LAUNCH + (double)((tiles + SPLIT_CUS - 1) / SPLIT_CUS) * round;
  const long long rest = tiles % (2 * SPLIT_CUS);
  return SPLIT_LAUNCH + (double)(tiles / (2 * SPLIT_CUS)) * round + (rest > SPLIT_CUS ? round : rest > 0 ? SPLIT_ALONE * steps + f.round : 0.0);
}

// what few rows take elsewhere. gemm_blocks: the blocks of a workgroup's waves one after the other, and all workgroups' work (10 % off in the mean).
// gemm_few_rows: a workgroup's rounds of segments or all workgroups' work, whichever is more (14 %).
static double split_few_cost(int M, int N, int K, int batch) {
  if (K <= SPLIT_BLOCKS_K) {
    const int form = M <= 8 ? 0 : M <= 16 ? 1 : M <= 32 ? 2 : 3, rows = M <= 16 ? 16 : M <= 32 ? 32 : 64, cols = M <= 8 ? 8 : 16;
    const double blocks = (K + 31) / 32 * (M <= 8 ? 0.5 : 1.0), share = (double)((N + cols - 1) / cols) * ((M + rows - 1) / rows) * batch / SPLIT_CUS;
    constexpr double chain[4] = {0.7, 0.7, 1.1, 1.8}, each[4] = {0.116, 0.134, 0.183, 0.247};
    return 2.3 + chain[form] * (int)((blocks + 7) / 8) + share * ((form == 3 ? 0.35 : 0.0) + each[form] * blocks);
  }
  const int segs = (K + SEG - 1) / SEG, rows = few_blocks_rows(M, N, K, batch), form = M <= 16 ? 0 : M <= 32 ? 1 : 2;
  if (rows) {
    const double share = (double)((N + 15) / 16) * ((M + rows - 1) / rows) * batch / SPLIT_CUS;
    return 0.4 + (rows == 16 ? 1.2 : 1.9) * (((K + 31) / 32 + 7) / 8) + share * segs * (rows == 16 ? 0.62 : 0.47);
  }
  const int waves = few_rows_waves(M, N, K, batch), tile = M <= 16 ? 16 : M <= 32 ? 32 : 64;
  const double share = (double)((N + 15) / 16) * ((M + tile - 1) / tile) * batch / SPLIT_CUS;
  constexpr double round4[3] = {3.8, 4.7, 8.5}, round8[3] = {7.5, 9.7, 14.7}, each[3] = {0.81, 1.42, 2.08};
  const double chain = (waves == 4 ? round4 : round8)[form] * (segs < waves ? (double)segs / waves : (segs + waves - 1) / waves), work = (segs > 8 ? ceil(share) : share) * segs * each[form];        // (over a long k a last, partly filled round counts whole)
  return 3.0 + cbrt(chain * chain * chain + work * work * work);
}

// Forms 1 to 4 only from k = 129 on, below which 5 and 6 start and end sooner; 6 only over a short k (12,300 x 48 at 300 rows 11.9 us, 15.3 by 5).
extern "C" int ta_gemm_split_form(int M, int N, int K, int lda, int ldw, int batch, bool vec) {
  const bool far = lda > 4194303 || ldw > 4194303;     // 256 rows by 32-bit offsets
  if (split_tiles(SPLIT_SMALL, M, N) * batch > 2147483640ll || (M <= 16 && K > SPLIT_BLOCKS_K)) return 0;
  int best = 0;
  double least = split_few_cost(M, N, K, batch);
  for (int f = !vec || K <= 128 ? SPLIT_PAIRED : far ? SPLIT_GROUPS : 1; f <= (K <= SPLIT_BLOCKS_K && !far ? SPLIT_SMALL : SPLIT_PAIRED); ++f) {
    const double cost = split_cost(f, M, N, K, batch);
    if (cost < least) best = f, least = cost;
  }
  return best && far ? best + SPLIT_FAR : best;
}

void ta_gemm_split(hipStream_t stream, int form, const float* A, int lda, long long sa, const float* W, int ldw, long long sw,
                   const float* bias, float* C, int ldc, long long sc, int M, int N, int K, int batch, bool vec) {
  const int tiles = (int)split_tiles(form, M, N), tiles_m = (M + 32 * SPLIT_FORMS[form].waves - 1) / (32 * SPLIT_FORMS[form].waves);
#define RUN_(WAVES, NT, G, VEC, ...)                                                                          \
  gemm_split_kernel<WAVES, NT, G, VEC, __VA_ARGS__><<<dim3((tiles + 7) / 8 * 8, batch), WAVES * G * 64, 0, stream>>>( \
      A, lda, W, ldw, bias, C, ldc, M, N, K, sa, sw, sc, tiles_m, tiles)
#define RUN(WAVES, NT, G)                              \
  if (K % SEG == 0) RUN_(WAVES, NT, G, true, true);    \
  else RUN_(WAVES, NT, G, true, false)
#define RUN_ANY(WAVES, NT, G)                          \
  if (!vec) RUN_(WAVES, NT, G, false, false);          \
  else RUN(WAVES, NT, G)
  switch (form) {
    case 1: RUN(8, 8, 1); break;
    case 2: RUN(4, 6, 2); break;
    case 3: RUN(4, 4, 2); break;
    case 4: RUN(2, 4, 4); break;
    case 5: RUN_ANY(4, 4, 1); break;
    case SPLIT_GROUPS + SPLIT_FAR: RUN_(2, 4, 4, true, false, false, true); break;
    case SPLIT_PAIRED + SPLIT_FAR:
      if (vec) RUN_(4, 4, 1, true, false, false, true);
      else RUN_(4, 4, 1, false, false, false, true);
      break;
    default: RUN_ANY(2, 4, 1); break;
  }
#undef RUN_ANY
#undef RUN
#undef RUN_
}

// Whether ta_gemm_split_glu takes the products of M rows with gates and ups (float32, rows on 16 bytes): where the product alone goes by
// tiles of 256 x 128.
extern "C" int ta_gemm_split_glu_takes(int M, int di, int K, int lda, int ldw) {
  return M > 16 && M <= 65535 * 64 && di > 0 && di <= 1073741823 && K % 4 == 0 && ((long long)di + 64) * ldw < 1 << 30 &&
         ta_gemm_split_form(M, 2 * di, K, lda, ldw, 1, true) == 1;
}

// C[M, di] = silu(A W[:di]^T + bias[:di]) * (A W[di:]^T + bias[di:]), W [2 di, K]: what the product and ta_swiglu give one after the other,
// bit for bit.
extern "C" int ta_gemm_split_glu(hipStream_t stream, const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc,
                                 int M, int di, int K) {
  TA_REQUIRE(ta_gemm_split_glu_takes(M, di, K, lda, ldw), "ta_gemm_split_glu: M=%d di=%d K=%d", M, di, K);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= di && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0,
             "ta_gemm_split_glu: rows of %d, %d, %d floats or their start", lda, ldw, ldc);
  const int tiles_m = (M + 255) / 256, tiles = tiles_m * ((di + 63) / 64);
#define RUN(WHOLE) \
  gemm_split_kernel<8, 8, 1, true, WHOLE, true><<<(tiles + 7) / 8 * 8, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, 2 * di, K, 0, 0, 0, tiles_m, tiles)
  if (K % SEG == 0) RUN(true);
  else RUN(false);
#undef RUN
  return ta_check_launch("ta_gemm_split_glu");
}
