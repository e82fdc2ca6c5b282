// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) in 32 bits for up to 8 rows: the products of a float32 decode step, bound by
// reading W once. The sums are split.h's (a matrix instruction multiplies two segments side by side, 8 columns of W each), so a row
// has the same bits here and in the kernels for more rows.
//
// W goes from memory to LDS without passing through registers, whole lines at a time: 64 k of 8 columns of two segments are
// 16 runs of 256 bytes, 4 KB, and every wave has a ring of its own of such chunks, up to 128 KB a CU on their way, that is
// asked for across the ends of tiles. Operand layout straight from memory (gemm_walk, gemm_few_rows) touches half a line per row and
// instruction: at 4 rows 16,384 x 2,048 gated 28.2 us there and 24.9 here (5.4 TB/s), 28,672 x 4,096 gated 88 and 80, 2,048 x 8,192 19.2 and 15.4,
// 4,096 x 14,336 64 and 47, 8,192 x 8,192 70 and 55 (on the float32 matrix instructions). Splitting the operands costs a kernel up to 0.9 us more
// than those, in front of the first product and behind the last chunk: the four products of a layer of width 2,048 and 8,192 (3,072 and 2,048 x 2,048, 16,384 x 2,048 gated,
// 2,048 x 8,192) at 1 / 4 / 8 rows 54.0 / 55.6 / 58.5 us on the float32 instructions, 57.7 / 58.2 / 60.8 with A split by every lane and 55.1 / 56.5 / 61.1 with half of it (HALF); it is what
// keeps a row's bits the same as among many, which gain more.
//
// A product may take the RMS norm in front of it (its workgroups form the rows' factors once more each, which costs 1 to 3 us
// where the norm's own launch costs 4 to 5), and add its result to the residual stream where it stores it.
#include "gemm_stream.h"
#include "split.h"

__device__ float4 stream_zeros;    // where a piece past K is read from (never written: zero)

// 16 bytes per lane to LDS as ta_load_to_lds16; ONCE: past the caches
template <bool ONCE = true>
__device__ __forceinline__ void stream_to_lds16(const void* src, uint32_t to) {
  if (ONCE) asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off nt" ::"v"(src), "s"(to) : "m0", "memory");
  else asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(to) : "m0", "memory");
}

struct StreamNorm {
  const float* w;              // [K] weight of the norm in front, or null
  float eps;
};

// K up to 512 WAVES: a wave keeps its pair of segments of A in registers and the workgroup walks along the columns, two
// workgroups of 4 waves a CU or one of 8. A (and the norm's weight and rows) come behind the first two chunks of W and in front of the
// others: behind all of them they would be there only when those are, in front of all of them memory would wait for them (the norm's
// rows by waves of their own: 16,384 x 2,048 33 us instead of 27).
//
// HALF (up to 4 rows): rows 4 to 7 of the instruction hold the other half of rows 0 to 3, so that a lane reads, norms and splits half as much of A
// and gets the rest from its neighbour; what those rows then multiply is never stored.
template <int WAVES, int PF, bool GLU, bool NORM, bool TAIL, bool HALF>
__global__ __launch_bounds__(WAVES * 64, 2) void gemm_stream_kernel(const float* __restrict__ A, int lda,
                                                                 const float* __restrict__ W, int ldw,
                                                                 const float* __restrict__ bias, float* __restrict__ C, int ldc,
                                                                 int M, int N, int K, int tiles, int add, StreamNorm nm) {
  constexpr int TURN = 2 * WAVES;                // segments
  constexpr int CH = 4;                          // chunks of 64 k in a segment
  constexpr int SLOT = 1024;                     // floats of a chunk: 8 columns of two segments
  constexpr int EARLY = PF / 2;                 // chunks asked for in front of A
  __shared__ __attribute__((aligned(16))) float ring[WAVES][PF][SLOT];
  __shared__ __attribute__((aligned(16))) float part[2][TURN][64];
  __shared__ float sq[8][WAVES / 2];
  __shared__ int undefined[8];                   // of its rows, see split_undefined_once; one wave asks between two barriers
  if (threadIdx.x < 8) undefined[threadIdx.x] = 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TA_WAVE), lane = threadIdx.x % TA_WAVE;
  const int r = lane % 16, kb = lane / 16, lrow = lane / 16, lpiece = lane % 16;
  const int n_out = GLU ? N / 2 : N, segs = (K + SEG - 1) / SEG;
  const f32x4* zeros = reinterpret_cast<const f32x4*>(&stream_zeros);
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&ring[wave][0][0]);
  // instruction t of a chunk brings rows 4 t + lane / 16 of 16: columns 0 .. 7 of the wave's first segment, then of its second,
  // 16 lanes per 256 bytes, permuted by the row so that the operand reads meet no bank twice
  const float* src[4];
  int koff[4];
  auto aim = [&](int tile) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int row = 4 * t + lrow, col = row % 8;
      const int n = GLU ? 4 * tile + col % 4 : 8 * tile + col;
      koff[t] = (2 * wave + row / 8) * SEG + (lpiece ^ row) * 4;
      src[t] = W + (size_t)((n < n_out ? n : n_out - 1) + (GLU && col >= 4 ? n_out : 0)) * ldw + koff[t];
    }
  };
  int ask = blockIdx.x, chunk = 0, step = 64;    // what is asked for next
  aim(ask);
  auto request = [&](int slot) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const void* p = src[t] + step * chunk;
      if (TAIL) p = koff[t] + 64 * chunk < K ? p : (const void*)zeros;
      stream_to_lds16(p, base + (slot * SLOT + t * 256) * 4);
    }
    if (++chunk == CH) {
      chunk = 0;
      ask += gridDim.x;
      if (ask < tiles) {
        aim(ask);
      } else {                                   // behind the last tile: one address, not used
        step = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t) src[t] = reinterpret_cast<const float*>(zeros);
      }
    }
  };
#pragma unroll
  for (int s = 0; s < EARLY; ++s) request(s);

  // the lane's part of A, row r % 8, segment 2 wave + r / 8, PIECES of a chunk's four from piece half on
  constexpr int ROWS = HALF ? 4 : 8, PIECES = HALF ? 2 : 4;
  const int m_a = r % ROWS < M ? r % ROWS : 0, half = HALF ? r / 4 % 2 * 2 : 0;
  const float* arow = A + (size_t)m_a * lda;
  f32x4 a[CH * PIECES], g[NORM ? CH * PIECES : 1], v[NORM ? ROWS / 2 : 1][4];
  constexpr int T = WAVES * 32;                  // threads a row: add_rmsnorm's, 4 vectors of 4 each
  const int side = threadIdx.x / T, at = threadIdx.x % T;
  if (NORM) {
#pragma unroll
    for (int p = 0; p < ROWS / 2; ++p)
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int m = 2 * p + side, c = 4 * (at + u * T);
        v[p][u] = *(m < M && c < K ? reinterpret_cast<const f32x4*>(A + (size_t)m * lda + c) : zeros);
      }
  }
#pragma unroll
  for (int i = 0; i < CH * PIECES; ++i) {
    const int k = (2 * wave + r / 8) * SEG + (i / PIECES * 4 + half + i % PIECES) * BLK + 4 * kb;
    a[i] = *(k < K ? reinterpret_cast<const f32x4*>(arow + k) : zeros);
    if (NORM) g[i] = *(k < K ? reinterpret_cast<const f32x4*>(nm.w + k) : zeros);
  }
  // They have to be there before the rest is asked for: a wave's loads come back in order, and the compiler's waits for these
  // do not count those (a value that has been through an asm statement is waited for there).
  auto arrive = [](f32x4& x) { asm volatile("" : "+v"(x)); };
#pragma unroll
  for (int i = 0; i < CH * PIECES; ++i) {
    arrive(a[i]);
    if (NORM) arrive(g[i]);
    if (NORM) arrive(v[i / 4][i % 4]);
  }
#pragma unroll
  for (int s = EARLY; s < PF; ++s) request(s);
  if (NORM) {
#pragma unroll
    for (int p = 0; p < ROWS / 2; ++p) {
      float ss = 0.f;
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) ss += v[p][u][e] * v[p][u][e];
      ss = wave_sum(ss);
      if (lane == 0) sq[2 * p + side][wave % (WAVES / 2)] = ss;
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float tot = 0.f;
#pragma unroll
    for (int i = 0; i < WAVES / 2; ++i) tot += sq[m_a][i];
    const float rstd = 1.0f / sqrtf(tot / (float)K + nm.eps);
#pragma unroll
    for (int i = 0; i < CH * PIECES; ++i)
#pragma unroll
      for (int e = 0; e < 4; ++e) a[i][e] = a[i][e] * rstd * g[i][e];
  }
  Split8 as[CH * 2];                             // A, split in front of the first tile's chunks
  int slot = 0, turn = 0;
  auto multiply = [&](int tile, bool first) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      if (first) {                               // while the chunk is on its way
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < PIECES / 2; ++i) as[2 * c + i] = split8(a[PIECES * c + 2 * i], a[PIECES * c + 2 * i + 1]);
        if (HALF) as[2 * c + 1] = split_next4(as[2 * c]);
        __builtin_amdgcn_sched_barrier(0);
      }
      ta_wait_loads<(PF - 1) * 4>();
      f32x4 w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = *reinterpret_cast<const f32x4*>(&ring[wave][slot][r * 64 + ((4 * i + kb) ^ r) * 4]);
      // all of the slot is in registers before it is asked to hold another chunk
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
      request(slot);
      slot = slot + 1 == PF ? 0 : slot + 1;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        acc += split_block(split8(w[2 * i], w[2 * i + 1]), as[2 * c + i]);
      }
    }
    // a lane holds columns 4 kb .. + 3 of row r: of the products, the two squares on the diagonal are used
    auto* to = part[turn];
    if (kb / 2 == r / 8) *reinterpret_cast<f32x4*>(&to[2 * wave + r / 8][(r % 8) * 8 + 4 * (kb % 2)]) = acc;
    // one barrier a tile: who comes to this half again has passed the other half's, behind which all have read this one
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave == (tile / (int)gridDim.x) % WAVES) {                   // the waves take the tiles' sums in turn
      const int m = lane / 8, nn = lane % 8, n = GLU ? 4 * tile + nn % 4 : 8 * tile + nn;
      float total = 0.f;
      for (int s = 0; s < segs; ++s) total += to[s][lane];
      auto a_of = [&](int i, int k) {              // (of one row at a time: the factor is formed once)
        if (!NORM) return A[(size_t)i * lda + k];
        float all = 0.f;
#pragma unroll
        for (int q = 0; q < WAVES / 2; ++q) all += sq[i][q];
        return A[(size_t)i * lda + k] * (1.0f / sqrtf(all / (float)K + nm.eps)) * nm.w[k];
      };
      total = split_again(m < M && n < n_out && split_bad(total), total * SPLIT_DOWN, m, W + (size_t)(n + (GLU && nn >= 4 ? n_out : 0)) * ldw, K, a_of,
                          [&](int i) { return split_undefined_once(undefined, i, [&](int k) { return a_of(i, k); }, K); });
      if (bias && n < n_out) total += bias[n + (GLU && nn >= 4 ? n_out : 0)];
      if (GLU) {
        const float up = __shfl_xor(total, 4, TA_WAVE);
        if (m < M && nn < 4 && n < n_out) C[(size_t)m * ldc + n] = total / (1.0f + expf(-total)) * up;
      } else if (m < M && n < n_out) {
        float* c = C + (size_t)m * ldc + n;
        *c = add ? *c + total : total;
      }
    }
    turn ^= 1;
  };
  multiply(blockIdx.x, true);                    // (no more workgroups than tiles)
  for (int tile = blockIdx.x + gridDim.x; tile < tiles; tile += gridDim.x) multiply(tile, false);
  ta_wait_loads<0>();                            // no wave ends with a load to LDS on its way
}

// Longer K, a tile a workgroup, in rounds of 2 WAVES segments: pieces of A (up to 2 MR rows) go to LDS beside those of W. By 16 waves that keep A
// in registers, all of k = 8,192 in one round, 2,048 columns take 17.4 us at 4 rows instead of 15.4: all of W is then asked for in two bursts.
template <int WAVES, int PF, int MR, bool TAIL>
__global__ __launch_bounds__(WAVES * 64) void gemm_stream_long_kernel(const float* __restrict__ A, int lda,
                                                                      const float* __restrict__ W, int ldw,
                                                                      const float* __restrict__ bias, float* __restrict__ C, int ldc,
                                                                      int M, int N, int K, int add) {
  constexpr int TURN = 2 * WAVES;                // segments of a round
  constexpr int CH = 4;                          // chunks of 64 k in a segment
  constexpr int SLOT = 1024 + 256 * MR;          // floats of a chunk: 8 columns of W and 2 MR rows of A, of two segments
  __shared__ __attribute__((aligned(16))) float ring[WAVES][PF][SLOT];
  __shared__ __attribute__((aligned(16))) float part[2][TURN][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TA_WAVE), lane = threadIdx.x % TA_WAVE;
  const int r = lane % 16, kb = lane / 16, lrow = lane / 16, lpiece = lane % 16;
  const int segs = (K + SEG - 1) / SEG, rounds = (segs + TURN - 1) / TURN;
  const f32x4* zeros = reinterpret_cast<const f32x4*>(&stream_zeros);
  const uint32_t base = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)&ring[wave][0][0]);
  // instruction t of a chunk brings rows 4 t + lane / 16: columns 0 .. 7 of the wave's first segment, then of its second; rows
  // of A likewise; 16 lanes per 256 bytes, permuted by the row so that the operand reads meet no bank twice
  const float *src[4], *asrc[MR];
  int koff[4], aoff[MR];
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int row = 4 * t + lrow, n = 8 * blockIdx.x + row % 8;
    koff[t] = (2 * wave + row / 8) * SEG + (lpiece ^ row) * 4;
    src[t] = W + (size_t)(n < N ? n : N - 1) * ldw + koff[t];
  }
#pragma unroll
  for (int t = 0; t < MR; ++t) {
    const int row = 4 * t + lrow, m = row % (2 * MR);
    aoff[t] = (2 * wave + row / (2 * MR)) * SEG + (lpiece ^ row) * 4;
    asrc[t] = A + (size_t)(m < M ? m : 0) * lda + aoff[t];
  }
  int at = 0;                                    // k that the next request lies behind the wave's first
  const int end = rounds * TURN * SEG;
  auto request = [&](int slot) {
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const void* p = src[t] + at;
      if (TAIL || at >= end) p = koff[t] + at < K ? p : (const void*)zeros;
      stream_to_lds16(p, base + (slot * SLOT + t * 256) * 4);
    }
#pragma unroll
    for (int t = 0; t < MR; ++t) {
      const void* p = asrc[t] + at;
      if (TAIL || at >= end) p = aoff[t] + at < K ? p : (const void*)zeros;
      stream_to_lds16<false>(p, base + (slot * SLOT + 1024 + t * 256) * 4);
    }
    at += 64;
    if (at % SEG == 0) at += (TURN - 1) * SEG;   // on to the wave's segments of the next round
  };
#pragma unroll
  for (int s = 0; s < PF; ++s) request(s);
  const int arow = r / 8 * (2 * MR) + r % 8 % (2 * MR);
  constexpr bool HALF = MR <= 2;                 // as above
  const int half = HALF ? r / 4 % 2 * 2 : 0;
  const int m = lane / 8, n = 8 * blockIdx.x + lane % 8;
  float total = 0.f;
  int slot = 0;
  for (int round = 0; round < rounds; ++round) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      ta_wait_loads<(PF - 1) * (4 + MR)>();
      f32x4 w[4], a[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        w[i] = *reinterpret_cast<const f32x4*>(&ring[wave][slot][r * 64 + ((4 * i + kb) ^ r) * 4]);
        if (i < 2 || !HALF) a[i] = *reinterpret_cast<const f32x4*>(&ring[wave][slot][1024 + arow * 64 + ((4 * (half + i) + kb) ^ arow) * 4]);
        else a[i] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
      asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3])::"memory");
      request(slot);
      slot = slot + 1 == PF ? 0 : slot + 1;
      const Split8 first = split8(a[0], a[1]);
      acc += split_block(split8(w[0], w[1]), first);
      acc += split_block(split8(w[2], w[3]), HALF ? split_next4(first) : split8(a[2], a[3]));
    }
    auto* to = part[round & 1];
    if (kb / 2 == r / 8) *reinterpret_cast<f32x4*>(&to[2 * wave + r / 8][(r % 8) * 8 + 4 * (kb % 2)]) = acc;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (wave == 0) {
      const int live = segs - round * TURN < TURN ? segs - round * TURN : TURN;
      for (int s = 0; s < live; ++s) total += to[s][lane];
    }
  }
  if (wave == 0) {
    auto a_of = [&](int i, int k) { return A[(size_t)i * lda + k]; };
    total = split_again(m < M && n < N && split_bad(total), total * SPLIT_DOWN, m, W + (size_t)n * ldw, K, a_of,
                        [&](int i) { return split_undefined([&](int k) { return a_of(i, k); }, K); });
  }
  if (wave == 0 && m < M && n < N) {
    if (bias) total += bias[n];
    float* c = C + (size_t)m * ldc + n;
    *c = add ? *c + total : total;
  }
  ta_wait_loads<0>();                            // no wave ends with a load to LDS on its way
}

// Whether a plain product, or one with a gated activation, is better taken here than by gemm_simple's kernels (us there and here at 1 /
// 4 / 8 rows). From six of eight segments on: 2,048 x 1,540 6.3 / 6.5 / 7.3 and 6.1 / 5.9 / 6.6, but 2,048 x 1,100 4.8 / 5.1 / 5.7
// and 5.4 / 5.5 / 5.9. More than 4 rows of A weigh with a tile a workgroup and the CUs unevenly filled: 3,072 x 2,048 10.1 and 10.5 at
// 8. A gated activation with few tiles a workgroup: 2 x 2,049 columns x 1,996 10.4 / 10.7 / 11.8 and 11.0 / 11.2 / 12.3. Everything
// else measured gains, from 64 columns (x 8,192 12.6 / 14.7 / 17.6 and 9.4 / 10.4 / 11.4) to 32,000 (x 2,048 48 / 49 / 51 and 46 / 46 / 48).
static int stream_tiles(int N, int glu) { return glu ? (N / 2 + 3) / 4 : (N + 7) / 8; }
extern "C" int ta_gemm_stream_pays(int M, int N, int K, int glu) {
  if (M < 1 || M > 8 || K < 6 * SEG || K % 4 != 0) return 0;
  const int tiles = stream_tiles(N, glu), each = K <= 2048 ? 512 : 256;
  if (glu) return K <= 4096 && tiles >= 2 * each;
  return M <= 4 || K > 2048 || tiles <= 256 || tiles >= 512;
}
// The same with the norm in front, whose own kernel takes 4 to 5 us: 16,384 x 2,048 gated 30 / 32 / 33 and 26 / 27 / 28, 3,072 x 2,048 12.6 / 13.4
// / 14.3 and 12.0 / 12.9 / 14.3, 5,000 x 3,000 23.5 / 23.8 / 25.0 and 21.5 / 21.6 / 22.2; but 2,048 x 2,560, five of eight waves at
// work, 11.7 / 12.0 / 13.3 and 12.5 / 13.0 / 14.0.
extern "C" int ta_gemm_stream_normed_pays(int M, int N, int K) {
  return M >= 1 && M <= 8 && K % 4 == 0 && N > 0 && ((K >= 6 * SEG && K <= 8 * SEG) || (K > 11 * SEG && K <= 16 * SEG));
}

// C[M,N] = A W^T (+ bias), or with add C += A W^T (no bias). glu: W is [2 n, K] with gate rows first, N = 2 n and C [M, n] =
// silu(gate) * up. norm_w: A holds rows of the residual stream, which the RMS norm (weight norm_w [K], eps) goes over first, with the
// bits that ta_add_rmsnorm gives; K up to 4,096, as with glu.
extern "C" int ta_gemm_stream(hipStream_t stream, const float* A, int lda, const float* W, int ldw, const float* bias, float* C,
                              int ldc, int M, int N, int K, int glu, int add, const float* norm_w, float eps) {
  TA_REQUIRE(M >= 0 && M <= 8 && N > 0 && K > 0 && K % 4 == 0 && K <= 2147483647 - 32 * SEG, "ta_gemm_stream: M=%d N=%d K=%d", M, N, K);
  TA_REQUIRE(!glu || (N % 2 == 0 && !add), "ta_gemm_stream: %d rows of gates and ups", N);
  TA_REQUIRE(!add || !bias, "ta_gemm_stream: a product with a bias is not added");
  TA_REQUIRE(K <= 4096 || !(norm_w || glu), "ta_gemm_stream: a norm or gates over %d", K);
  TA_REQUIRE(!norm_w || (K > 1024 && eps >= 0.f), "ta_gemm_stream: a norm over %d, eps %g", K, (double)eps);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= (glu ? N / 2 : N) && lda % 4 == 0 && ldw % 4 == 0 &&
                 ((uintptr_t)A | (uintptr_t)W | (uintptr_t)norm_w) % 16 == 0,
             "ta_gemm_stream: rows of %d, %d, %d floats or their start", lda, ldw, ldc);
  if (M == 0) return 0;
  const int tiles = stream_tiles(N, glu);
  if (K > 4096) {
#define LONG(PF, MR)                                                                                                  \
  if (K % (16 * SEG) == 0)                                                                                            \
    gemm_stream_long_kernel<8, PF, MR, false><<<tiles, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, add); \
  else                                                                                                                \
    gemm_stream_long_kernel<8, PF, MR, true><<<tiles, 512, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, add)
    if (M <= 2) { LONG(3, 1); } else if (M <= 4) { LONG(3, 2); } else { LONG(2, 4); }
#undef LONG
    return ta_check_launch("ta_gemm_stream (long k)");
  }
  const int most = K <= 2048 ? 512 : 256, grid = tiles < most ? tiles : most;
  const StreamNorm nm = {norm_w, eps};
#define RUN_(WAVES, GLU, NORM, TAIL, HALF)                                                                        \
  gemm_stream_kernel<WAVES, 4, GLU, NORM, TAIL, HALF><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, tiles, add, nm)
#define RUN(WAVES, GLU, NORM)                                                                                     \
  if (K % (2 * WAVES * SEG) == 0) {                                                                               \
    if (M <= 4) RUN_(WAVES, GLU, NORM, false, true); else RUN_(WAVES, GLU, NORM, false, false);                   \
  } else {                                                                                                        \
    if (M <= 4) RUN_(WAVES, GLU, NORM, true, true); else RUN_(WAVES, GLU, NORM, true, false);                     \
  }
#define PICK(WAVES)                                                                                        \
  do {                                                                                                     \
    if (glu) { if (norm_w) { RUN(WAVES, true, true); } else { RUN(WAVES, true, false); } }                 \
    else { if (norm_w) { RUN(WAVES, false, true); } else { RUN(WAVES, false, false); } }                   \
  } while (0)
  if (K <= 2048) PICK(4); else PICK(8);
#undef PICK
#undef RUN
#undef RUN_
  return ta_check_launch("ta_gemm_stream");
}
