// The gated feed-forward of many bfloat16 rows (prompts) in one kernel: C = act(A Wg^T) * (A Wu^T), W = [gate rows | up rows], float32 accumulate, on
// v_mfma_f32_16x16x32_bf16. The product with the activation behind it moves [M, 2 n] to memory and back; here gate and up of a channel meet in
// a lane's registers, in float32.
//
// The schedule is the published one of eight waves on this chip, two to a SIMD that take turns at reading and multiplying ("ping-pong").
// A workgroup of 8 waves, alone on its CU, owns 256 rows x 128 channels, wave (wm, wn) 128 rows and 32 channels of either kind in four quarters
// of 64 x 32. 64 k of the operands lie in LDS, row by row in 8 pieces of 16 bytes, permuted by the row so that the lanes that are
// served together meet no bank twice; they get there without passing through registers, in halves of 128 rows. A step of 64 k is four phases,
// each the 16 matrix instructions of a quarter behind the reads of 8 or 4 operands (never 12: a phase's reads by four waves then take longer
// than its products). The waves of a SIMD are half a phase apart, one reads and asks for memory while the other multiplies, with a
// barrier at every change; what a phase reads was asked for six phases earlier, into the place of what all waves have read two
// phases before. As a plain product 8,192 x 8,192 x 8,192 takes 713 us (1.54 PFLOP/s; 756 with 12 and 0 reads in turn; 765 and more with the barrier
// in front of a phase's last products), where the matrix pipelines are busy 80 % of the time and the clock is down to 1.8 GHz: power binds
// as much as issue. Four waves of 128 x 128, 32 k at a time in four buffers, 1,031 us.
//
// The last round of workgroups of up to half as many tiles as CUs is cut into tiles of 128 rows, as is what the matrix leaves of a tile with 128 rows or fewer: two phases
// a step, three buffers in LDS, the same order of sums, bound by LDS (0.8 of a whole tile's time). 2,011 x 28,672 x 4,096 (three and a half
// rounds) 370 us in whole tiles, 342 so; the library's product and the activation's kernel 379. 700 rows 152 and 164; 7,000 rows 1,167 and 1,255; 22,016 columns:
// 2,011 rows 273 and 426, 4,400 rows 589 and 684; 16,384 columns over k = 2,048: 512 rows 36 and 43, 5,632 rows 290 and 394.
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define HALF_TILE (128 * 64)     // bfloat16 of 128 rows and 64 k

struct GluArgs {
  const uint16_t *A, *W;
  const float* bias;             // [2 n] or null
  uint16_t* C;
  int lda, ldw, ldc, M, n, K;
  int tiles_m, whole, halves;    // rows of tiles; tiles of 256 rows; tiles of 128 rows behind them
  TaGlu glu;
  float* X;                      // PLAIN: the result [M][ldc], to which the product is added where `add`
  int add;
};

// 256 (SHORT: 128) rows from m0 on, 128 channels from n0 on. PLAIN: 256 columns, a product alone, in float32.
template <bool SHORT, bool PLAIN>
__device__ __forceinline__ void glu_tile(const GluArgs& p, uint16_t* S, int m0, int n0) {
  const int lane = threadIdx.x % TA_WAVE, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TA_WAVE), wm = wave / 4, wn = wave % 4;
  const int r = lane % 16, kb = lane / 16;
  constexpr int AH = SHORT ? 1 : 2;              // halves of the rows
  constexpr int STEP = (AH + 2) * HALF_TILE;     // of LDS
  // what this lane brings of a half: two pieces; rows past the end read the last one and feed what is never stored
  uint32_t aoff[AH][2], woff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = (wave * 2 + i) * 8 + lane / 8, piece = (lane % 8) ^ (row & 7);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (h < AH) {
        const int m = SHORT ? row : row / 64 * 128 + h * 64 + row % 64;
        aoff[h < AH ? h : 0][i] = ((uint32_t)(m0 + m < p.M ? m : p.M - 1 - m0) * p.lda + piece * 8) * 2;
      }
    }
    woff[i] = ((uint32_t)(PLAIN || n0 + row < p.n ? row : p.n - 1 - n0) * p.ldw + piece * 8) * 2;
  }
  const char* abase = reinterpret_cast<const char*>(p.A + (size_t)m0 * p.lda);
  const char* wbase[2] = {reinterpret_cast<const char*>(p.W + (size_t)n0 * p.ldw),      // gates, ups; PLAIN: 128 columns and the next 128
                          reinterpret_cast<const char*>(p.W + (size_t)((PLAIN ? 128 : p.n) + n0) * p.ldw)};
  const int steps = p.K / 64;
  const uint32_t lds = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)S) + wave * 2048;
  // half h of A (op 0), gates or ups (op 1) of step t into buffer `buf`; behind the last step that one once more, unused
  auto bring = [&](int op, int h, int t, int buf) {
    const char* base = (op ? wbase[h] : abase) + (size_t)(t < steps ? t : steps - 1) * 128;
#pragma unroll
    for (int i = 0; i < 2; ++i)      // (a scalar write of m0 wants one wait state; the base comes from the scalar unit)
      asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(op ? woff[i] : aoff[h < AH ? h : 0][i]), "s"(base),
                   "s"(lds + (buf * STEP + (op ? AH + h : h) * HALF_TILE + i * 512) * 2) : "m0", "memory");
  };
  bf16x8 a[4][2], w[4][2][2];      // [16 rows][32 k]; sets of [16 columns][32 k]
  f32x4 acc[AH][2][4][2];
#pragma unroll
  for (int x = 0; x < AH; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[x][y][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto read_a = [&](int buf, int h) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int row = wm * 64 + i * 16 + r;
        a[i][ks] = *reinterpret_cast<const bf16x8*>(S + buf * STEP + h * HALF_TILE + row * 64 + ((ks * 4 + kb) ^ (row & 7)) * 8);
      }
  };
  auto read_w = [&](int buf, int h, int set) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int row = wn * 32 + j * 16 + r;
        w[set][j][ks] = *reinterpret_cast<const bf16x8*>(S + buf * STEP + (AH + h) * HALF_TILE + row * 64 + ((ks * 4 + kb) ^ (row & 7)) * 8);
      }
  };
  auto meet = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  // a phase's products, between two barriers; behind the first all that this wave has read is there
  auto multiply = [&](int x, int y, int set) {
    meet();
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
          acc[x][y][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[set][j][ks], a[i][ks], acc[x][y][i][j], 0, 0, 0);
    __builtin_amdgcn_s_setprio(0);
    meet();
  };
  if constexpr (!SHORT) {
    bring(1, 0, 0, 0); bring(0, 0, 0, 0); bring(1, 1, 0, 0); bring(0, 1, 0, 0);
    bring(1, 0, 1, 1); bring(0, 0, 1, 1); bring(1, 1, 1, 1);
    ta_wait_loads<10>();
    meet();
    if (wm == 1) meet();                         // half a phase behind
    read_w(0, 0, 0);
    // Every phase asks for two pieces a lane, read six phases later; what the next phase reads is then all but the last ten.
    // The first half of W is read a phase ahead, into sets 0 and 2 in turn.
    auto step = [&](int t, int buf) {
      const int now = buf ? 2 : 0, next = buf ? 0 : 2;
      read_a(buf, 0);
      bring(0, 1, t + 1, buf ^ 1);
      ta_wait_loads<10>();
      multiply(0, 0, now);
      read_w(buf, 1, 1);
      bring(1, 0, t + 2, buf);
      ta_wait_loads<10>();
      multiply(0, 1, 1);
      read_a(buf, 1);
      bring(0, 0, t + 2, buf);
      ta_wait_loads<10>();
      multiply(AH - 1, 1, 1);
      read_w(buf ^ 1, 0, next);
      bring(1, 1, t + 2, buf);
      ta_wait_loads<10>();
      multiply(AH - 1, 0, now);
    };
    for (int t = 0; t < steps; t += 2) {
      step(t, 0);
      if (t + 1 < steps) step(t + 1, 1);
    }
  } else {
    bring(1, 0, 0, 0); bring(1, 1, 0, 0); bring(0, 0, 0, 0); bring(1, 0, 1, 1); bring(1, 1, 1, 1); bring(0, 0, 1, 1);
    bring(1, 0, 2, 2); bring(1, 1, 2, 2);
    ta_wait_loads<10>();
    meet();
    if (wm == 1) meet();
    read_w(0, 0, 0);
    read_w(0, 1, 1);
    int buf = 0;                                 // of step t; W is read a phase ahead, into sets 0, 1 and 2, 3 in turn
    auto step = [&](int t, int now) {
      const int after = buf == 2 ? 0 : buf + 1, third = buf == 0 ? 2 : buf - 1;
      read_a(buf, 0);
      bring(0, 0, t + 2, third);
      ta_wait_loads<8>();
      multiply(0, 0, now);
      read_w(after, 0, 2 - now);
      read_w(after, 1, 3 - now);
      bring(1, 0, t + 3, buf);
      bring(1, 1, t + 3, buf);
      ta_wait_loads<10>();
      multiply(0, 1, now + 1);
      buf = after;
    };
    for (int t = 0; t < steps; t += 2) {
      step(t, 0);
      if (t + 1 < steps) step(t + 1, 2);
    }
  }
  if (wm == 0) meet();
  ta_wait_loads<0>();                            // no wave ends with a load to LDS on its way
  if constexpr (PLAIN) {
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        float* to = p.X + n0 + y * 128 + wn * 32 + j * 16 + 4 * kb;
        f32x4 old[AH][4];
#pragma unroll
        for (int x = 0; x < AH; ++x)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = m0 + wm * 64 * AH + x * 64 + i * 16 + r;
            old[x][i] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (p.add) old[x][i] = *reinterpret_cast<const f32x4*>(to + (size_t)(m < p.M ? m : p.M - 1) * p.ldc);
          }
#pragma unroll
        for (int x = 0; x < AH; ++x)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int m = m0 + wm * 64 * AH + x * 64 + i * 16 + r;
            if (m < p.M) *reinterpret_cast<f32x4*>(to + (size_t)m * p.ldc) = old[x][i] + acc[x][y][i][j];
          }
      }
    return;
  }
  // a lane holds channels 4 kb .. + 3 of row r of each 16 x 16
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int n = n0 + wn * 32 + j * 16 + 4 * kb;
    if (n >= p.n) continue;
    f32x4 bg = {0.f, 0.f, 0.f, 0.f}, bu = bg;
    if (p.bias)
#pragma unroll
      for (int e = 0; e < 4; ++e) bg[e] = p.bias[n + e], bu[e] = p.bias[p.n + n + e];
#pragma unroll
    for (int x = 0; x < AH; ++x)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int m = m0 + wm * 64 * AH + x * 64 + i * 16 + r;
        if (m >= p.M) continue;
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = ta_glu(p.glu, acc[x][0][i][j][e] + bg[e], acc[x][1][i][j][e] + bu[e]);
        *reinterpret_cast<uint2*>(p.C + (size_t)m * p.ldc + n) = uint2{f32x2_to_bf16x2_bits(v[0], v[1]), f32x2_to_bf16x2_bits(v[2], v[3])};
      }
  }
}

// Tiles in groups of 8 rows of tiles, column by column, so that the 32 workgroups of an XCD (every eighth) share 8 + 4 operands.
template <bool PLAIN>
__global__ __launch_bounds__(512, 2) void gemm_glu_kernel(GluArgs p) {
  __shared__ __attribute__((aligned(16))) uint16_t S[3 * 3 * HALF_TILE];         // 2 x 4 or 3 x 3 halves
  constexpr int COLS = PLAIN ? 256 : 128;
  const int tiles_n = (p.n + COLS - 1) / COLS, grid_whole = (p.whole + 7) / 8 * 8;
  const bool rest = (int)blockIdx.x >= grid_whole;
  const int id = rest ? blockIdx.x - grid_whole : blockIdx.x, all = rest ? p.halves : p.whole, share = (all + 7) / 8;
  const int at = id % 8 * share + id / 8;
  if (at >= all) return;
  const int tile = rest ? p.whole + at / 2 : at;
  const int group = tile / (8 * tiles_n), in = tile % (8 * tiles_n), high = p.tiles_m - group * 8 < 8 ? p.tiles_m - group * 8 : 8;
  const int m0 = (group * 8 + in % high) * 256 + (rest ? at % 2 * 128 : 0), n0 = in / high * COLS;
  if (!rest && m0 + 128 < p.M) glu_tile<false, PLAIN>(p, S, m0, n0);
  else if (m0 < p.M) glu_tile<true, PLAIN>(p, S, m0, n0);
}

enum { GLU_CUS = 256 };

// Where it gains over the library's product (hipBLASLt of ROCm 7) and the activation's kernel: wide matrices, by how full the rounds of tiles are. Measured at 76 numbers of
// rows from 385 to 8,192 by 12 matrices (8,000 to 28,672 channels, k from 2,048 to 8,192), where it takes 1.11 times less in the mean. us there and here:
//   two rows of tiles of which the second is over half full, and three or more: 14,336 channels over 4,096: 512 rows 105 / 102, 700 161 / 156, 1,100 244 / 237, 2,060 399 / 384,
//   3,100 698 / 558, 7,500 1,361 / 1,271; 11,008 over 4,096: 700 154 / 143, 1,600 339 / 251; 8,000 over 4,096: 1,281 250 / 153; 22,016 over 4,096: 1,900 1.24 times.
//   513 to 640 rows, whose third row of tiles is the half form's, lose 2 to 12 % at most widths (but gain 26 to 36 % at 22,016, 5 at 11,008);
//   641 to 768 rows whose tiles leave a quarter of the CUs idle: 8,192 over 4,096 0.94 to 0.97 times, over 8,192 0.97 to 1.01 (8,000 over 4,096 would gain 2 to 8 %);
//   over k below 4,096 a second round of up to a quarter (8,192 over 2,048: 1,025 to 1,100 rows 0.94 to 0.98, 1,152 to 1,280 1.00 to 1.03), and whole rounds only,
//   four and more of them (16,384 over 2,048: 2,560 rows 0.98, 4,096 0.97, 5,632 0.96, 7,500 0.95, 8,192 0.90; 8,192 over 2,048 and 14,336 over 2,048: 8,192 rows 0.99, 1.00).
// The worst that is left of 837: 11,008 over 4,096 769 rows 0.94 (145 / 154; 780 0.99, 820 1.06), 8,192 over 4,096 1,100 rows 0.96, 14,336 over 4,096 1,040 rows 0.97;
// 400 rows, 28,672 over 8,192 at 2,060 and the like are ties. Fewer channels go either way: 5,632 over 2,048: 576 38 / 50, 830 55 / 47, 1,281 74 / 83, 2,011 98 / 94.
extern "C" int ta_gemm_glu_pays(int M, int n, int K) {
  if (M <= 384 || (M > 512 && M <= 640) || n < 8000 || n % 4 != 0 || K < 2048 || K % 64 != 0) return 0;
  const long long tiles = ((long long)M + 255) / 256 * ((n + 127) / 128), rest = tiles % GLU_CUS;
  if (M > 512 && M <= 768 && tiles <= 192) return 0;
  return K >= 4096 || !((tiles > GLU_CUS && tiles <= GLU_CUS + GLU_CUS / 4) || (rest == 0 && tiles >= 4 * GLU_CUS));
}

// C [M, n] = act(A W[:n]^T + bias[:n]) * (A W[n:]^T + bias[n:]); the activation as in ta_gemm_mid: a limit above 0 the limited form with its slope
// and shift, else gelu (tanh) or silu.
extern "C" int ta_gemm_glu(hipStream_t stream, const void* A, int lda, const void* W, int ldw, const float* bias, void* C, int ldc, int M,
                           int n, int K, int gelu, float limit, float slope, float shift) {
  TA_REQUIRE(M >= 0 && M <= 2147483392 && n > 0 && n <= 1073741823 && n % 4 == 0 && K > 0 && K % 64 == 0, "ta_gemm_glu: M=%d n=%d K=%d", M, n, K);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= n && lda % 8 == 0 && ldw % 8 == 0 && ldc % 4 == 0 && lda <= 4194304 && ldw <= 4194304 &&
                 ((uintptr_t)A | (uintptr_t)W) % 16 == 0 && (uintptr_t)C % 8 == 0,
             "ta_gemm_glu: rows of %d, %d, %d or their start", lda, ldw, ldc);
  const long long tm = (M + 255) / 256, tiles = tm * ((n + 127) / 128), rest = tiles % GLU_CUS;
  TA_REQUIRE(tiles <= 1073741823, "ta_gemm_glu: M=%d n=%d too large for one launch", M, n);
  if (M == 0) return 0;
  GluArgs p = {(const uint16_t*)A, (const uint16_t*)W, bias, (uint16_t*)C, lda, ldw, ldc, M, n, K, (int)tm, (int)tiles, 0, {limit, slope, shift, gelu}, nullptr, 0};
  if (rest <= GLU_CUS / 2) {
    p.whole = (int)(tiles - rest);
    p.halves = (int)(2 * rest);
  }
  gemm_glu_kernel<false><<<(p.whole + 7) / 8 * 8 + (p.halves + 7) / 8 * 8, 512, 0, stream>>>(p);
  return ta_check_launch("ta_gemm_glu");
}

// The same as a plain product with a float32 result. It is the library's equal while it multiplies (and sums in the same order except where that one cuts k);
// it gains where its rounds are full, and where the library cuts its last round along k and falls to half. us there and here (the product added to the stream):
// 4,096 columns over k = 14,336: 1,600 rows 333 / 182, 2,502 0.83 times the library's rate, 3,164 501 / 289, 3,400 309 / 295, 4,000 335 / 322, 4,500 424 / 473, 5,640 753 / 494; over
// 4,096 3,400 106 / 101, 4,000 112 / 110, but 8,159 216 / 224; 8,192 columns over 14,336: 1,573 328 / 303; 5,120 over 14,336: 1,166 321 / 171, 4,829 814 / 525; over 4,096 2,942 108 / 104.
// Measured anew at 23 matrices, k = 4,096, 5,120, 8,192, 11,008, 12,288, 12,352, 13,824, 14,336, 16,384, 20,480 and 28,672, at up to 54 numbers of rows each. Two rounds or less, over a long k:
//   full or from 208 tiles on: 0.98 to 1.75 times, mostly 1.03 (where the library keeps up) or 1.6 (where it falls); three rounds gain nowhere;
//   nearly half full, 100 to 128 tiles: 1.0 to 1.9; 96 to 128 as the second round: 1.0 to 1.84, but 8,192 columns over 28,672 0.95 to 0.98; 96 alone 0.77 to 0.98, whatever
//   the width; 128 over k above 12,288 0.98 (2,011 x 4,096 x 14,336 195 / 199).
// Over k below 8,192 one nearly full round: 1.00 to 1.06 added, 1.05 to 1.09 stored (16,384 columns over 4,096 0.97 and 0.98). Results in bfloat16 lose 3 to 5 % (5,000 rows x 6,144 over 4,096 182 / 194).
extern "C" int ta_gemm_plain_pays(int M, int n, int K) {
  if (M < 512 || n % 256 != 0 || K % 64 != 0 || K < 4096) return 0;
  const long long tiles = ((long long)M + 255) / 256 * (n / 256), rest = tiles % GLU_CUS;
  if (K < 8192) return n <= 8192 && tiles >= 208 && tiles <= GLU_CUS;
  if (tiles > 2 * GLU_CUS) return 0;
  if (rest == 0 || rest >= 208) return 1;
  return rest >= (tiles < GLU_CUS ? 100 : 96) && rest <= (K <= 12288 ? 128 : 120) && (n < 8192 || K <= 14336);
}

// C [M, n] = A W^T, or C += A W^T, float32.
extern "C" int ta_gemm_plain(hipStream_t stream, const void* A, int lda, const void* W, int ldw, float* C, int ldc, int M, int n, int K, int add) {
  TA_REQUIRE(M >= 0 && M <= 2147483392 && n > 0 && n % 256 == 0 && K > 0 && K % 64 == 0, "ta_gemm_plain: M=%d n=%d K=%d", M, n, K);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= n && lda % 8 == 0 && ldw % 8 == 0 && ldc % 4 == 0 && lda <= 4194304 && ldw <= 4194304 &&
                 ((uintptr_t)A | (uintptr_t)W | (uintptr_t)C) % 16 == 0,
             "ta_gemm_plain: rows of %d, %d, %d or their start", lda, ldw, ldc);
  const long long tm = ((long long)M + 255) / 256, tiles = tm * (n / 256), rest = tiles % GLU_CUS;
  TA_REQUIRE(tiles <= 1073741823, "ta_gemm_plain: M=%d n=%d too large for one launch", M, n);
  if (M == 0) return 0;
  GluArgs p = {(const uint16_t*)A, (const uint16_t*)W, nullptr, nullptr, lda, ldw, ldc, M, n, K, (int)tm, (int)tiles, 0, {}, C, add};
  if (rest <= GLU_CUS / 2) {
    p.whole = (int)(tiles - rest);
    p.halves = (int)(2 * rest);
  }
  gemm_glu_kernel<true><<<(p.whole + 7) / 8 * 8 + (p.halves + 7) / 8 * 8, 512, 0, stream>>>(p);
  return ta_check_launch("ta_gemm_plain");
}
