// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) in 32 bits on the matrix cores: the product of the true
// 32-bit path, and the fallback for storage types and shapes that no faster kernel takes.
//
// Every output element is summed in one order that depends on K and the types alone, whatever M, N, the kernel or the tile, so
// a row of A gives the same bits alone or inside any batch. float32 by float32: split.h's. With a bfloat16 operand, and over a k of up to 32, the products go to
// the float32 matrix instructions, which are chains of fused multiply-adds: v_mfma_f32_16x16x4_f32 and v_mfma_f32_32x32x2_f32 give the
// bits of fmaf over their 4 (2) k-slots in ascending order, denormals included. Then
//   k is cut into segments of 256 and these into blocks of 16; a segment's chain starts at zero and takes
//   its blocks in ascending order, and of a block k = 0 4 8 12, 1 5 9 13, 2 6 10 14, 3 7 11 15; the
//   segments' sums are added in ascending order.
// The order inside a block is the one in which a lane that has read 4 consecutive k holds them: no operand is turned round.
//
// gemm_few_rows: 16 columns a workgroup, whose waves take segments in turn; gemm_blocks: blocks of a short k. gemm_walk (float32): the same for
// wide matrices over a k of up to 4,096, where a workgroup keeps its rows of A and walks along the columns. gemm_tiles (a bfloat16
// operand, or a short k): a tile of 128 x 128 or 64 x 64 a workgroup, operands through LDS. Many rows of float32 are gemm_split.hip's, up to 8 of a long
// enough matrix gemm_stream.hip's, with the same bits.
#include "gemm_split.h"
#include "gemm_stream.h"
#include "split.h"

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

__device__ float4 gemm_zeros;      // where a piece past K is read from (never written: zero)

// 4 consecutive k of a row as floats. VEC: rows are 4-element aligned and K is a multiple of 4, so a piece
// lies wholly inside K or wholly outside. NT: read once, past the caches.
template <typename T, bool VEC, bool NT>
__device__ __forceinline__ f32x4 load_piece(const T* row, int k, int K) {
  if (VEC) {
    if (sizeof(T) == 4) {
      const f32x4* p = k < K ? reinterpret_cast<const f32x4*>(row + k) : reinterpret_cast<const f32x4*>(&gemm_zeros);
      return NT ? __builtin_nontemporal_load(p) : *p;
    }
    const u32x2* p = k < K ? reinterpret_cast<const u32x2*>(row + k) : reinterpret_cast<const u32x2*>(&gemm_zeros);
    const u32x2 v = NT ? __builtin_nontemporal_load(p) : *p;
    return f32x4{__uint_as_float(v[0] << 16), __uint_as_float(v[0] & 0xffff0000u), __uint_as_float(v[1] << 16),
                 __uint_as_float(v[1] & 0xffff0000u)};
  }
  f32x4 v;
#pragma unroll
  for (int j = 0; j < 4; ++j) v[j] = k + j < K ? to_f32(row[k + j]) : 0.f;
  return v;
}

// Few rows (up to 16 * RT of them a workgroup), bound by reading W. A lane reads 4 consecutive k of a row of W and
// of RT rows of A, which are operands as they are (a row's four lanes cover 64
// bytes); while one chunk of BC blocks is multiplied the next is on its way. The waves take the segments in
// turn and leave the partial tiles in LDS, where they are added in ascending order after every round.
// float32, 2,048 columns over k = 8,192 at 9 / 16 / 32 / 64 rows 32 / 38 / 55 / 85 us (31 / 36 / 52 / 86 on the float32 matrix instructions:
// from 32 rows on it is the splitting of A, once more for every 16 columns, that binds), 3,072 x 2,048 at 32 / 64 rows 15.6 / 24.0.
// PAIR (up to 8 rows): a matrix instruction multiplies two segments side by side, 8 columns of W each, of
// whose 16 x 16 products the two squares on the diagonal are used. A workgroup then owns 8 columns: a matrix of
// 2,048 rows keeps 256 CUs reading instead of 128.
// SHORT: k does not fill a round of segments, or leaves half of the last one empty. A wave then ends where k does instead of multiplying zeros to the end of
// its segment: 40 x 5,000 x 64 6.3 us (21 without), 1 x 5,000 x 768 6.9 (10.6). The test between the chunks costs
// long k 2 to 4 % (8 x 16,384 x 4,096 74.6 us without it, 77.3 with).
// CHAIN: float32 products over a short k (SHORT_K).
// Four waves a workgroup, or eight (few_rows_waves).
template <typename T, typename TW, typename TC, int WAVES, int RT, int BC, bool PAIR, bool SHORT, bool VEC, bool CHAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_few_rows_kernel(const T* __restrict__ A, int lda,
                                                                   const TW* __restrict__ W, int ldw,
                                                                   const float* __restrict__ bias,
                                                                   TC* __restrict__ C, int ldc, int M, int N, int K,
                                                                   long long sa, long long sw, long long sc) {
  static_assert(!PAIR || RT == 1, "two segments in one tile");
  static_assert(BC % 2 == 0, "blocks of split.h in pairs of 16 k");
  constexpr bool SPLIT = sizeof(T) == 4 && sizeof(TW) == 4 && !CHAIN;
  A += (size_t)blockIdx.z * sa;
  W += (size_t)blockIdx.z * sw;
  C += (size_t)blockIdx.z * sc;
  constexpr int COLS = PAIR ? 8 : 16, ROWS = PAIR ? 8 : 16 * RT;   // of the workgroup's tile
  constexpr int TURN = PAIR ? 2 * WAVES : WAVES;                   // segments per round
  constexpr int CPS = SEG / (BC * BLK);                            // chunks per segment
  constexpr int OUT = (ROWS * COLS + WAVES * 64 - 1) / (WAVES * 64);
  __shared__ __attribute__((aligned(16))) float part[2][TURN][ROWS * COLS];
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  const int r = lane % 16, kb = lane / 16;
  const int n0 = blockIdx.x * COLS, m0 = blockIdx.y * ROWS;
  const int first = PAIR ? 2 * wave + r / 8 : wave;                // this lane's segment of a round
  // rows past N or M read another row and feed outputs that are never stored
  const TW* wrow = W + (size_t)(n0 + r % COLS < N ? n0 + r % COLS : N - 1) * ldw;
  const T* arow[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + 16 * i + (PAIR ? r % 8 : r);
    arow[i] = A + (size_t)(m < M ? m : m0) * lda;
  }
  const int segs = (K + SEG - 1) / SEG, rounds = (segs + TURN - 1) / TURN;

  f32x4 wreg[2][BC], areg[2][RT][BC];
  // chunk c of this lane: chunk c % CPS of its segment of round c / CPS; past K: zeros from one address
  auto load = [&](int set, int c) {
    const int k0 = ((c / CPS) * TURN + first) * SEG + (c % CPS) * BC * BLK + 4 * kb;
#pragma unroll
    for (int i = 0; i < BC; ++i) {
      wreg[set][i] = load_piece<TW, VEC, (RT < 4)>(wrow, k0 + i * BLK, K);
#pragma unroll
      for (int t = 0; t < RT; ++t) areg[set][t][i] = load_piece<T, VEC, false>(arow[t], k0 + i * BLK, K);
    }
  };
  f32x4 acc[RT];
  auto multiply = [&](int set) {
    if constexpr (SPLIT) {
#pragma unroll
      for (int i = 0; i < BC; i += 2) {
        const Split8 w = split8(wreg[set][i], wreg[set][i + 1]);
#pragma unroll
        for (int t = 0; t < RT; ++t) acc[t] += split_block(w, split8(areg[set][t][i], areg[set][t][i + 1]));
      }
    } else {
#pragma unroll
      for (int i = 0; i < BC; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
          for (int t = 0; t < RT; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(wreg[set][i][j], areg[set][t][i][j], acc[t], 0, 0, 0);
    }
  };
  float total[OUT];
#pragma unroll
  for (int e = 0; e < OUT; ++e) total[e] = 0.f;

  load(0, 0);
  for (int round = 0; round < rounds; ++round) {
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    static_assert(CPS % 2 == 0, "chunks of a segment in pairs");
    const int seg0 = SHORT ? __builtin_amdgcn_readfirstlane((round * TURN + (PAIR ? 2 * wave : wave)) * SEG) : 0;
#pragma unroll
    for (int c = 0; c < CPS; c += 2) {
      if (SHORT && seg0 + c * BC * BLK >= K) break;       // the rest of this wave's segments lies past K
      load(1, round * CPS + c + 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      load(0, round * CPS + c + 2);
      __builtin_amdgcn_sched_barrier(0);
      multiply(1);
      __builtin_amdgcn_sched_barrier(0);
    }
    // a lane holds columns 4 kb .. + 3 of row r of each tile
    auto* to = part[round & 1];
    if (PAIR) {
      if (kb / 2 == r / 8) *reinterpret_cast<f32x4*>(&to[first][(r % 8) * 8 + 4 * (kb % 2)]) = acc[0];
    } else {
#pragma unroll
      for (int t = 0; t < RT; ++t) *reinterpret_cast<f32x4*>(&to[wave][t * 256 + r * 16 + 4 * kb]) = acc[t];
    }
    __syncthreads();
    const int live = segs - round * TURN < TURN ? segs - round * TURN : TURN;
#pragma unroll
    for (int e = 0; e < OUT; ++e) {
      const int at = (int)threadIdx.x + WAVES * 64 * e;
      if (at < ROWS * COLS)
        for (int w = 0; w < live; ++w) total[e] += to[w][at];
    }
  }
#pragma unroll
  for (int e = 0; e < OUT; ++e) {
    const int at = (int)threadIdx.x + WAVES * 64 * e;
    const int m = m0 + at / COLS, n = n0 + at % COLS;
    const bool own = at < ROWS * COLS && m < M && n < N;
    if constexpr (SPLIT) {
      auto row = [&](int i, int k) { return (float)A[(size_t)i * lda + k]; };
      total[e] = split_again(own && split_bad(total[e]), total[e] * SPLIT_DOWN, m, (const float*)(W + (size_t)n * ldw), K, row,
                             [&](int i) { return split_undefined([&](int k) { return row(i, k); }, K); });
    }
    if (!own) continue;
    C[(size_t)m * ldc + n] = from_f32<TC>(bias ? total[e] + bias[n] : total[e]);
  }
}

// Few rows over a k of up to 512 (up to 8 rows 1,280), float32: gemm_few_rows' tiles with the waves on blocks of 32 k instead of segments, so that a k of few segments
// has all of them at work (splitting doubles what a wave has to do for a block, which a wave alone on its SIMD cannot hide).
// Every block's tile goes to LDS (up to 64 KB), where a segment's blocks and the segments are added up in their order: the bits are the same. us of
// gemm_few_rows on the float32 instructions, on the split and here: 2,048 x 256 at 4 / 16 / 32 / 64 rows 4.8 / 4.9 / 6.0 / 8.4, 5.7 / 5.8 / 7.4 / 10.1 and 4.3 / 4.6 / 5.3 / 7.1; 16,384 x 128 at
// one row 7.0, 8.6, 5.3; 512 x 512 at 8 rows 4.9, 5.7, 4.7; 2,048 x 1,024 at one row 5.6, 6.4, 5.5.
template <int WAVES, int RT, bool PAIR, bool VEC>
__global__ __launch_bounds__(WAVES * 64) void gemm_blocks_kernel(const float* __restrict__ A, int lda, const float* __restrict__ W, int ldw,
                                                                 const float* __restrict__ bias, float* __restrict__ C, int ldc, int M, int N,
                                                                 int K, long long sa, long long sw, long long sc) {
  static_assert(!PAIR || RT == 1, "two blocks in one tile");
  A += (size_t)blockIdx.z * sa;
  W += (size_t)blockIdx.z * sw;
  C += (size_t)blockIdx.z * sc;
  constexpr int COLS = PAIR ? 8 : 16, ROWS = PAIR ? 8 : 16 * RT, OUT = (ROWS * COLS + WAVES * 64 - 1) / (WAVES * 64);
  constexpr int SIDE = PAIR ? 2 : 1;             // blocks that a matrix instruction multiplies side by side
  extern __shared__ __attribute__((aligned(16))) float part[];       // [blocks, rounded up to SIDE][ROWS * COLS]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TA_WAVE), lane = threadIdx.x % TA_WAVE;
  const int r = lane % 16, kb = lane / 16;
  const int n0 = blockIdx.x * COLS, m0 = blockIdx.y * ROWS;
  // rows past N or M read another row and feed outputs that are never stored
  const float* wrow = W + (size_t)(n0 + r % COLS < N ? n0 + r % COLS : N - 1) * ldw;
  const float* arow[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int m = m0 + 16 * i + r % (PAIR ? 8 : 16);
    arow[i] = A + (size_t)(m < M ? m : m0) * lda;
  }
  const int blocks = (K + 31) / 32, steps = (blocks + SIDE - 1) / SIDE;
  f32x4 w[2][2], a[2][RT][2];
  auto load = [&](int set, int step) {
    const int k0 = (step * SIDE + (PAIR ? r / 8 : 0)) * 32 + 4 * kb;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      w[set][h] = load_piece<float, VEC, (RT < 4)>(wrow, k0 + 16 * h, K);
#pragma unroll
      for (int t = 0; t < RT; ++t) a[set][t][h] = load_piece<float, VEC, false>(arow[t], k0 + 16 * h, K);
    }
  };
  auto multiply = [&](int set, int step) {
    const Split8 ws = split8(w[set][0], w[set][1]);
#pragma unroll
    for (int t = 0; t < RT; ++t) {
      // a lane holds columns 4 kb .. + 3 of row r; of two blocks side by side the two squares on the diagonal are used
      const f32x4 c = split_block(ws, split8(a[set][t][0], a[set][t][1]));
      if (!PAIR) *reinterpret_cast<f32x4*>(&part[(step * RT + t) * 256 + r * 16 + 4 * kb]) = c;
      else if (kb / 2 == r / 8) *reinterpret_cast<f32x4*>(&part[(step * 2 + r / 8) * 64 + r % 8 * 8 + 4 * (kb % 2)]) = c;
    }
  };
  load(0, wave);
  for (int s = wave; s < steps; s += 2 * WAVES) {
    load(1, s + WAVES);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0, s);
    if (s + WAVES >= steps) break;
    load(0, s + 2 * WAVES);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1, s + WAVES);
  }
  __syncthreads();
#pragma unroll
  for (int e = 0; e < OUT; ++e) {
    const int at = (int)threadIdx.x + WAVES * 64 * e;
    if (OUT * WAVES * 64 > ROWS * COLS && at / TA_WAVE * TA_WAVE >= ROWS * COLS) continue;       // whole waves
    float total = 0.f;
    for (int b0 = 0; b0 < blocks; b0 += SEG / 32) {
      float sum = 0.f;
      if (b0 + SEG / 32 <= blocks) {
#pragma unroll
        for (int b = 0; b < SEG / 32; ++b) sum += part[(b0 + b) * ROWS * COLS + at];
      } else {
        for (int b = b0; b < blocks; ++b) sum += part[b * ROWS * COLS + at];
      }
      total += sum;
    }
    const int m = m0 + at / COLS, n = n0 + at % COLS;
    const bool own = m < M && n < N;
    auto row = [&](int i, int k) { return A[(size_t)i * lda + k]; };
    total = split_again(own && split_bad(total), total * SPLIT_DOWN, m, W + (size_t)n * ldw, K, row,
                        [&](int i) { return split_undefined([&](int k) { return row(i, k); }, K); });
    if (own) C[(size_t)m * ldc + n] = bias ? total + bias[n] : total;
  }
}

// Up to 8 (PAIR) or 16 rows of A against a wide W over a k of at most one round of segments: every wave keeps its
// segments of A in registers, the workgroup walks over tiles of 8 (16) columns, and the next tile's k are on their way
// while the last ones of this are multiplied and added up. Bound by reading W. gemm_few_rows reads A again with every
// tile, as many bytes as W at 8 rows, and its workgroups, which live for four chunks, start and end all the time:
// 16,384 x 2,048 at 16 rows 39 us there, 29.9 here (29.3 on the float32 matrix instructions), 32,000 x 2,048 52, 8,192 x 4,096 at 9 rows 35.7
// (k above 2,048: eight waves with two segments each). One workgroup a CU with 8 KB of W a wave on their way is enough;
// two or three a CU are up to 4 % slower. W passes the caches like any other read here: past them 3 % slower.
// GLU: W holds gate rows, then up rows; a tile has half its columns of either and stores silu(gate) * up, with the bits
// that the product and the activation's kernel give one after the other (a launch and two passes over its rows less).
template <int WAVES, int OWN, bool PAIR, bool GLU>
__global__ __launch_bounds__(WAVES * 64) void gemm_walk_kernel(const float* __restrict__ A, int lda,
                                                               const float* __restrict__ W, int ldw,
                                                               const float* __restrict__ bias, float* __restrict__ C,
                                                               int ldc, int M, int N, int K, int tiles) {
  constexpr int SIDE = PAIR ? 8 : 16;            // rows and columns of a tile
  static_assert(!PAIR || OWN == 1, "a wave's segments side by side or one after the other");
  constexpr int TURN = PAIR ? 2 * WAVES : WAVES * OWN;   // segments
  constexpr int BC = OWN == 1 ? 8 : 4;           // pieces per chunk: more registers for A, fewer for W
  constexpr int CH = SEG / (BC * BLK);           // chunks per segment
  constexpr int HALF = SIDE / 2;
  static_assert(WAVES * 64 >= SIDE * SIDE, "a thread an output");
  __shared__ __attribute__((aligned(16))) float part[2][TURN][SIDE * SIDE];
  __shared__ int undefined[SIDE];                // of its rows, see split_undefined_once; a wave asks for its own only
  if (threadIdx.x < SIDE) undefined[threadIdx.x] = 0;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE;
  const int r = lane % 16, kb = lane / 16, col = r % SIDE;
  const int seg = PAIR ? 2 * wave + r / 8 : wave, segs = (K + SEG - 1) / SEG;
  const int k0 = seg * SEG + 4 * kb, n_out = GLU ? N / 2 : N;
  // columns past the last read another row and feed outputs that are never stored
  auto rows_of = [&](int tile) {
    const int n = GLU ? HALF * tile + col % HALF : SIDE * tile + col;
    return W + (size_t)((n < n_out ? n : n_out - 1) + (GLU && col >= HALF ? n_out : 0)) * ldw;
  };
  // the first k of a piece of chunk c: the wave's segments lie WAVES apart
  auto k_of = [&](int c, int i) { return k0 + c / CH * WAVES * SEG + (c % CH * BC + i) * BLK; };
  constexpr bool KEEP = OWN == 1;                // A split once; two segments of it take too many registers and are split every time
  f32x4 a[KEEP ? 1 : CH * OWN][BC], w[2][BC];
  Split8 as[KEEP ? CH : 1][BC / 2];
  auto load = [&](int c, const float* row) {
#pragma unroll
    for (int i = 0; i < BC; ++i) w[c % 2][i] = load_piece<float, true, false>(row, k_of(c, i), K);
  };
  int tile = blockIdx.x;
  const float* row = rows_of(tile);
  load(0, row);
  const float* arow = A + (size_t)(col < M ? col : 0) * lda;
#pragma unroll
  for (int c = 0; c < CH * OWN; ++c) {
    f32x4* to = a[KEEP ? 0 : c];
#pragma unroll
    for (int i = 0; i < BC; ++i) to[i] = load_piece<float, true, false>(arow, k_of(c, i), K);
    if (KEEP)
#pragma unroll
      for (int i = 0; i < BC; i += 2) as[KEEP ? c : 0][i / 2] = split8(to[i], to[i + 1]);
  }
  const int m = threadIdx.x / SIDE, nn = threadIdx.x % SIDE;
  for (int turn = 0; tile < tiles; tile += gridDim.x, turn ^= 1) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](int c) {
#pragma unroll
      for (int i = 0; i < BC; i += 2) {
        const Split8 wi = split8(w[c % 2][i], w[c % 2][i + 1]);
        if (KEEP) {
          acc += split_block(wi, as[KEEP ? c : 0][i / 2]);
        } else {
          f32x4 x = a[KEEP ? 0 : c][i], y = a[KEEP ? 0 : c][i + 1];
          asm volatile("" : "+v"(x), "+v"(y));   // or the compiler splits all of A in front of the loop and has no registers for it
          acc += split_block(wi, split8(x, y));
        }
      }
    };
    static_assert(CH % 2 == 0, "a segment's chunks in two sets of registers in turn");
    auto* to = part[turn];
#pragma unroll
    for (int c = 0; c < CH * OWN; ++c) {
      if (c + 1 < CH * OWN) {
        load(c + 1, row);
      } else {                                   // the next tile's first
        row = rows_of(tile + (int)gridDim.x < tiles ? tile + (int)gridDim.x : tile);
        load(0, row);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(c);
      __builtin_amdgcn_sched_barrier(0);
      if (c % CH != CH - 1) continue;
      // a segment's end: a lane holds columns 4 kb .. + 3 of row r
      if (PAIR) {
        if (kb / 2 == r / 8) *reinterpret_cast<f32x4*>(&to[seg][(r % 8) * 8 + 4 * (kb % 2)]) = acc;
      } else {
        *reinterpret_cast<f32x4*>(&to[seg + c / CH * WAVES][r * 16 + 4 * kb]) = acc;
      }
      acc = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // one barrier a tile: who comes to this half again has passed the other half's, behind which all have read this one
    __syncthreads();
    if (threadIdx.x < SIDE * SIDE) {
      float total = 0.f;
      for (int s = 0; s < segs; ++s) total += to[s][threadIdx.x];
      const int n = (GLU ? HALF * tile + nn % HALF : SIDE * tile + nn);
      auto a_of = [&](int i, int k) { return A[(size_t)i * lda + k]; };
      total = split_again(m < M && n < n_out && split_bad(total), total * SPLIT_DOWN, m, W + (size_t)(n + (GLU && nn >= HALF ? n_out : 0)) * ldw, K, a_of,
                          [&](int i) { return split_undefined_once(undefined, i, [&](int k) { return a_of(i, k); }, K); });
      if (bias && n < n_out) total += bias[n + (GLU && nn >= HALF ? n_out : 0)];
      if (GLU) {
        const float up = __shfl_xor(total, HALF, TA_WAVE);
        if (m < M && nn < HALF && n < n_out) C[(size_t)m * ldc + n] = total / (1.0f + expf(-total)) * up;
      } else if (m < M && n < n_out) {
        C[(size_t)m * ldc + n] = total;
      }
    }
  }
}

// Whether gemm_walk takes the product: as long a k as its waves' segments and a quarter more tiles than workgroups. With a tile a
// workgroup it is gemm_few_rows with A read first (2,048 x 2,048 6.3 us there, 6.7 here; 2,304 x 4,096, 288 tiles, at one row
// 14.8 and 15.2; 3,072 x 2,048, 384 tiles, at 4 rows 10.7 and 9.6). Up to k = 1,024 a workgroup of two waves has too little on its
// way for a CU, so there are two of them on each. Below k = 512 the waves would have no segment.
#define CUS 256
static int walk_groups(int M, int K) { return M <= 8 && K <= 1024 ? 2 * CUS : CUS; }
static bool walk_takes(int M, int N, int K) {
  const int side = M <= 8 ? 8 : 16;
  return M >= 1 && M <= 16 && K > 512 && K <= 4096 && (N + side - 1) / side >= walk_groups(M, K) * 5 / 4;
}
// Without an activation to save a launch: two tiles a workgroup where most of the last waves' k is past the end (6,000 x 520 at 1 /
// 8 rows 6.4 / 6.7 us by few rows, 7.0 / 7.2 here, but 16,384 x 520 15.5 and 12.9; 3,000 x 1,032 at one row 6 % more here). Up to 8
// rows of a k above 2,048 are gemm_stream's (28,672 x 4,096 at 4 rows, gated, 88 us here and 80 there).
static bool walk_pays(int M, int N, int K) {
  if (M <= 8 && K > 2048) return false;
  const bool thin = M <= 8 && (K <= 640 || (M == 1 && K > 1024 && K <= 1280));
  return walk_takes(M, N, K) && (!thin || (N + 7) / 8 >= 2 * walk_groups(M, K));
}
template <bool GLU>
static void walk(hipStream_t stream, const float* A, int lda, const float* W, int ldw, const float* bias, float* C, int ldc,
                 int M, int N, int K) {
  // Where the waves have many tiles and little of k each a second workgroup a CU, which splits while the first one waits (us with one, with two): 16,384 x 1,028 at 4 rows
  // 23.0 and 19.1, 32,000 x 1,280 at one row 45 and 36, 5,000 x 1,028 10.1 and 9.0; 32,000 x 516 at 16 rows 21.1 and 18.9. But 32,000 x 1,500 44 and 43, 8,192 x 1,500 15.2 and 15.4,
  // 3,000 x 1,280 (375 tiles) at 8 rows 8.8 and 9.8, 8,192 x 768 at 16 rows 9.6 and 10.9.
  const int side = M <= 8 ? 8 : 16, tiles = (N + side - 1) / side, twice = tiles >= 2 * CUS && (M <= 8 ? K > 1024 && K <= 1408 : K <= 640);
  const int most = walk_groups(M, K) * (twice ? 2 : 1), grid = tiles < most ? tiles : most;
#define WALK(WAVES, OWN, PAIR) \
  gemm_walk_kernel<WAVES, OWN, PAIR, GLU><<<grid, WAVES * 64, 0, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, tiles)
  if (M <= 8) {
    if (K <= 1024) WALK(2, 1, true);
    else if (K <= 2048) WALK(4, 1, true);
    else if constexpr (GLU) WALK(8, 1, true);
  } else {
    if (K <= 1024) WALK(4, 1, false);
    else if (K <= 2048) WALK(8, 1, false);
    else WALK(8, 2, false);
  }
#undef WALK
}

// Many rows with a bfloat16 operand, or any over a short k, bound by the matrix cores (a 32x32x2 instruction occupies its SIMD for 64 cycles and wants 512
// bytes of operands). 4 waves in 2 x 2 share a tile of 64 TT x 64 TT; each owns TT x TT tiles of 32 x 32. 32 k at a
// time go through registers, where they become float32, and LDS, double buffered: row by row in 8 pieces of 16 bytes, permuted by the row
// number so that the eight lanes that are served together meet no bank twice. Half h of a wave multiplies pieces h and h + 2 of a block's
// four, element by element: the order above.
template <typename T, typename TW, typename TC, int TT, bool VEC>
__global__ __launch_bounds__(256, 2) void gemm_tiles_kernel(const T* __restrict__ A, int lda,
                                                            const TW* __restrict__ W, int ldw,
                                                            const float* __restrict__ bias,
                                                            TC* __restrict__ C, int ldc, int M, int N, int K,
                                                            long long sa, long long sw, long long sc) {
  A += (size_t)blockIdx.z * sa;
  W += (size_t)blockIdx.z * sw;
  C += (size_t)blockIdx.z * sc;
  constexpr int BT = 64 * TT;                    // rows and columns of the tile
  constexpr int PER = BT * 8 / 256;              // pieces of an operand that a thread brings
  __shared__ f32x4 As[2][BT * 8], Ws[2][BT * 8];
  const int lane = threadIdx.x % TA_WAVE, wave = threadIdx.x / TA_WAVE;
  const int n0 = blockIdx.x * BT, m0 = blockIdx.y * BT;
  const int lrow = threadIdx.x / 8;              // 32 rows of 128 bytes at a time
  const int place = threadIdx.x % 8;             // piece of the row
  const T* asrc[PER];
  const TW* wsrc[PER];
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int row = lrow + 32 * i;
    asrc[i] = A + (size_t)(m0 + row < M ? m0 + row : M - 1) * lda;
    wsrc[i] = W + (size_t)(n0 + row < N ? n0 + row : N - 1) * ldw;
  }
  f32x4 ain[PER], win[PER];
  const int steps = (K + 31) / 32;               // of 32 k
  auto fetch = [&](int s) {
    const int k0 = (s < steps ? s : steps - 1) * 32;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      ain[i] = load_piece<T, VEC, false>(asrc[i], k0 + place * 4, K);
      win[i] = load_piece<TW, VEC, false>(wsrc[i], k0 + place * 4, K);
    }
  };
  auto stash = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int row = lrow + 32 * i, at = row * 8 + (place ^ (row & 7));
      As[buf][at] = ain[i];
      Ws[buf][at] = win[i];
    }
  };
  const int half = lane / 32, r = lane % 32;
  const int am = (wave % 2) * 32 * TT + r, wn = (wave / 2) * 32 * TT + r;    // this lane's rows in As and Ws
  f32x16 total[TT][TT], acc[TT][TT];
#pragma unroll
  for (int i = 0; i < TT; ++i)
#pragma unroll
    for (int j = 0; j < TT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) total[i][j][e] = acc[i][j][e] = 0.f;
  // a block's operands, one of a step's two while the other is multiplied
  f32x4 a[2][TT][2], w[2][TT][2];
  auto read = [&](int set, int buf) {
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int p = 0; p < 2; ++p) {
        const int at = (4 * set + 2 * p + half) ^ (r & 7);
        a[set][i][p] = As[buf][(am + 32 * i) * 8 + at];
        w[set][i][p] = Ws[buf][(wn + 32 * i) * 8 + at];
      }
  };
  auto multiply = [&](int set, int j) {          // a quarter of the block
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int x = 0; x < TT; ++x)
#pragma unroll
        for (int y = 0; y < TT; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[set][x][p][j], w[set][y][p][j], acc[x][y], 0, 0, 0);
  };

#pragma unroll
  for (int s = 0; s < 2; ++s) {
    fetch(s);
    stash(s);
  }
  __syncthreads();
  read(0, 0);
  // The barrier stands in the middle of a step: in front of it a step's second block is read, behind it the
  // step's buffer is free for the step after the next, and the next step's first block is read while the second
  // is multiplied, so that no wave waits for LDS right behind a barrier.
  for (int s = 0; s < steps; ++s) {
    const int buf = s % 2;
    fetch(s + 2);
    read(1, buf);
#pragma unroll
    for (int j = 0; j < 4; ++j) multiply(0, j);
    __syncthreads();
    stash(buf);
    read(0, (s + 1) % 2);
#pragma unroll
    for (int j = 0; j < 4; ++j) multiply(1, j);
    if ((s + 1) % (SEG / 32) == 0 || s + 1 == steps) {
#pragma unroll
      for (int x = 0; x < TT; ++x)
#pragma unroll
        for (int y = 0; y < TT; ++y)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            total[x][y][e] += acc[x][y][e];
            acc[x][y][e] = 0.f;
          }
    }
  }
  // accumulator: register e of a lane is row 8 (e / 4) + 4 half + e % 4 of the tile, column r
#pragma unroll
  for (int y = 0; y < TT; ++y) {
    const int n = n0 + wn + 32 * y;
    if (n >= N) continue;
    const float add = bias ? bias[n] : 0.f;
#pragma unroll
    for (int x = 0; x < TT; ++x)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const int m = m0 + (wave % 2) * 32 * TT + 32 * x + 8 * (e / 4) + 4 * half + e % 4;
        if (m < M) C[(size_t)m * ldc + n] = from_f32<TC>(bias ? total[x][y][e] + add : total[x][y][e]);
      }
  }
}

// float32 products over a k up to this stay on the float32 matrix instructions: a chain of so few fused multiply-adds rounds less than
// the split's left out products and last sums (k = 1 2.5e-8 and 3.8e-8, 2 3.1e-8 and 4.0e-8, 4 4.0e-8 and 3.7e-8; entries of very different size
// up to k = 16; 32 1.0e-7 and 4.2e-8).
#define SHORT_K 32

// Whether gemm_few_rows' waves look where k ends: less than a round of segments, or a last round of up to half of them behind at most three.
static bool few_short(int K, int turn) {
  const int segs = (K + SEG - 1) / SEG, rest = segs % turn;
  return segs < turn || (rest != 0 && rest <= turn / 2 && segs < 4 * turn);
}

template <typename T, typename TW, typename TC, bool VEC>
static void launch(hipStream_t stream, const void* A_, int lda, long long sa, const void* W_, int ldw, long long sw,
                   const float* bias, void* C_, int ldc, long long sc, int M, int N, int K, int batch) {
  const T* A = (const T*)A_;
  const TW* W = (const TW*)W_;
  TC* C = (TC*)C_;
  constexpr bool F32 = sizeof(T) == 4 && sizeof(TW) == 4;
  // A tile's time does not depend on how many there are, so few tiles are better cut along k (2,048 columns over
  // k = 8,192: 128 rows 85 us by few rows where 64 tiles take 187, 256 rows 170 against 187, 512 rows 187 by tiles
  // against 340). Tiles of 128 take two workgroups on every CU to fill. Over a short k it is the start and the end that
  // count: tiles for any rows (1 x 16,384 x 16 3.8 us, 7.2 by few rows; 32 products of 1 x 512 x 64 4.4 against 7.2).
  auto tiles = [&](int t) { return (long long)((M + t - 1) / t) * ((N + t - 1) / t) * batch; };
  if (tiles(64) >= 192 && (F32 ? K <= SHORT_K : M > 64 || K <= 128)) {
    if (tiles(128) >= 384)
      gemm_tiles_kernel<T, TW, TC, 2, VEC><<<dim3((N + 127) / 128, (M + 127) / 128, batch), 256, 0, stream>>>(
          A, lda, W, ldw, bias, C, ldc, M, N, K, sa, sw, sc);
    else
      gemm_tiles_kernel<T, TW, TC, 1, VEC><<<dim3((N + 63) / 64, (M + 63) / 64, batch), 256, 0, stream>>>(
          A, lda, W, ldw, bias, C, ldc, M, N, K, sa, sw, sc);
    return;
  }
#define FEW_(WAVES, RT, BC, PAIR, SHORT, CHAIN)                                                                \
  gemm_few_rows_kernel<T, TW, TC, WAVES, RT, BC, PAIR, SHORT, VEC, CHAIN>                                      \
      <<<dim3((N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), (M + 16 * RT - 1) / (16 * RT), batch), WAVES * 64, 0, stream>>>( \
          A, lda, W, ldw, bias, C, ldc, M, N, K, sa, sw, sc)
  if constexpr (F32) {
    if (K <= SHORT_K) {
      if (M <= 8) FEW_(4, 1, 4, true, true, true);
      else if (M <= 16) FEW_(4, 1, 4, false, true, true);
      else if (M <= 32) FEW_(4, 2, 2, false, true, true);
      else FEW_(4, 4, 2, false, true, true);
      return;
    }
    if (const int form = ta_gemm_split_form(M, N, K, lda, ldw, batch, VEC)) {
      ta_gemm_split(stream, form, A, lda, sa, W, ldw, sw, bias, C, ldc, sc, M, N, K, batch, VEC);
      return;
    }
  }
  if constexpr (VEC && F32)
    if (batch == 1 && walk_pays(M, N, K)) {
      walk<false>(stream, A, lda, W, ldw, bias, C, ldc, M, N, K);
      return;
    }
  // four waves a workgroup where there are many (4,096 x 48 at 130 rows, 768 workgroups, 7.3 us by eight and 6.3 by four; 8,192 x 384 at 16 rows, 512, 7.4 and 7.3)
#define BLOCKS_(WAVES, RT, PAIR)                                                                               \
  gemm_blocks_kernel<WAVES, RT, PAIR, VEC><<<grid, WAVES * 64, lds, stream>>>(A, lda, W, ldw, bias, C, ldc, M, N, K, sa, sw, sc)
#define BLOCKS(RT, PAIR)                                                                                       \
  do {                                                                                                         \
    const dim3 grid((N + (PAIR ? 7 : 15)) / (PAIR ? 8 : 16), (M + 16 * RT - 1) / (16 * RT), batch);            \
    const size_t lds = ((K + 31) / 32 + 1) / 2 * 2 * (PAIR ? 64 : 256 * RT) * sizeof(float);                   \
    if ((long long)grid.x * grid.y * grid.z <= 640) BLOCKS_(8, RT, PAIR);                                      \
    else BLOCKS_(4, RT, PAIR);                                                                                 \
  } while (0)
  if constexpr (F32)
    if (const int rows = few_blocks_rows(M, N, K, batch)) {
      if (rows == 8) BLOCKS(1, true);
      else if (rows == 16) BLOCKS(1, false);
      else if (rows == 32) BLOCKS(2, false);
      else BLOCKS(4, false);
      return;
    }
#undef BLOCKS
#undef BLOCKS_
#define FEW(WAVES, RT, BC, PAIR)                                                                               \
  do {                                                                                                         \
    if (few_short(K, WAVES * (PAIR ? 2 : 1))) FEW_(WAVES, RT, BC, PAIR, true, false);                          \
    else FEW_(WAVES, RT, BC, PAIR, false, false);                                                              \
  } while (0)
  // four waves a workgroup and 16 KB on their way in each: several workgroups share a CU and fill each other's
  // starts and ends (16,384 x 2,048 at 16 rows: 38 us; 44 with eight waves and twice the loads)
  const bool eight = F32 && few_rows_waves(M, N, K, batch) == 8;
  if (M <= 8) FEW(4, 1, 4, true);
  else if (M <= 16) { if (eight) FEW(8, 1, 4, false); else FEW(4, 1, 4, false); }
  else if (M <= 32) { if (eight) FEW(8, 2, 2, false); else FEW(4, 2, 2, false); }
  else if constexpr (F32) { if (eight) FEW(8, 4, 2, false); else FEW(4, 4, 2, false); }
  else FEW(4, 4, 2, false);
#undef FEW_
#undef FEW
}

// in_dtype: type of A; w_dtype: type of W (a bfloat16 engine keeps a matrix that its file
// stores in 32 bits as it is: bfloat16 A with float32 W); out_dtype: type of C. ``batch``
// products side by side: product i reads A + i*sa, W + i*sw and writes C + i*sc (elements).
extern "C" int ta_gemm_simple_batched(hipStream_t stream, int in_dtype, int w_dtype, int out_dtype,
                                      const void* A, int lda, long long sa, const void* W, int ldw,
                                      long long sw, const float* bias, void* C, int ldc, long long sc,
                                      int M, int N, int K, int batch) {
  TA_REQUIRE(M >= 0 && N > 0 && K > 0 && batch >= 1 && batch <= 65535,
             "ta_gemm_simple: bad sizes M=%d N=%d K=%d batch=%d", M, N, K, batch);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= N, "ta_gemm_simple: leading dimensions too small");
  if (M == 0) return 0;
  // the few-rows kernel counts up to two rounds of 8 segments past k
  TA_REQUIRE((M + 63) / 64 <= 65535 && K <= 2147483647 - 32 * SEG, "ta_gemm_simple: M=%d K=%d too large for one launch", M, K);
  // rows that start on 4 elements and hold whole pieces of 4
  auto aligned = [&](const void* p, int dtype, long long ld, long long stride) {
    return (uintptr_t)p % (dtype == TA_F32 ? 16 : 8) == 0 && ld % 4 == 0 && stride % 4 == 0;
  };
  const bool vec = K % 4 == 0 && aligned(A, in_dtype, lda, sa) && aligned(W, w_dtype, ldw, sw);
  if (vec && in_dtype == TA_F32 && w_dtype == TA_F32 && out_dtype == TA_F32 && batch == 1 && ta_gemm_stream_pays(M, N, K, 0))
    return ta_gemm_stream(stream, (const float*)A, lda, (const float*)W, ldw, bias, (float*)C, ldc, M, N, K, 0, 0, nullptr, 0.f);
#define LAUNCH(T, TW, TC)                                                                                   \
  do {                                                                                                      \
    if (vec) launch<T, TW, TC, true>(stream, A, lda, sa, W, ldw, sw, bias, C, ldc, sc, M, N, K, batch);     \
    else launch<T, TW, TC, false>(stream, A, lda, sa, W, ldw, sw, bias, C, ldc, sc, M, N, K, batch);        \
  } while (0)
  if (in_dtype == TA_F32 && w_dtype == TA_F32 && out_dtype == TA_F32) LAUNCH(float, float, float);
  else if (in_dtype == TA_BF16 && w_dtype == TA_BF16 && out_dtype == TA_BF16) LAUNCH(bf16_t, bf16_t, bf16_t);
  else if (in_dtype == TA_BF16 && w_dtype == TA_BF16 && out_dtype == TA_F32) LAUNCH(bf16_t, bf16_t, float);
  else if (in_dtype == TA_BF16 && w_dtype == TA_F32 && out_dtype == TA_BF16) LAUNCH(bf16_t, float, bf16_t);
  else if (in_dtype == TA_BF16 && w_dtype == TA_F32 && out_dtype == TA_F32) LAUNCH(bf16_t, float, float);
  else return ta_fail("ta_gemm_simple: unsupported dtypes a=%d w=%d out=%d", in_dtype, w_dtype, out_dtype);
#undef LAUNCH
  return ta_check_launch("ta_gemm_simple");
}

extern "C" int ta_gemm_simple(hipStream_t stream, int in_dtype, int w_dtype, int out_dtype,
                              const void* A, int lda, const void* W, int ldw, const float* bias,
                              void* C, int ldc, int M, int N, int K) {
  return ta_gemm_simple_batched(stream, in_dtype, w_dtype, out_dtype, A, lda, 0, W, ldw, 0, bias, C, ldc, 0,
                                M, N, K, 1);
}

// Whether ta_gemm_simple_glu takes such a product (float32, rows on 16 bytes).
extern "C" int ta_gemm_simple_glu_takes(int M, int di, int K) {
  return di > 0 && di <= 1073741823 && K % 4 == 0 && walk_takes(M, 2 * di, K);
}

// C[M, di] = silu(A W[:di]^T + bias[:di]) * (A W[di:]^T + bias[di:]), W [2 di, K]: what ta_gemm_simple and ta_swiglu give one
// after the other, bit for bit.
extern "C" int ta_gemm_simple_glu(hipStream_t stream, const float* A, int lda, const float* W, int ldw, const float* bias,
                                  float* C, int ldc, int M, int di, int K) {
  TA_REQUIRE(ta_gemm_simple_glu_takes(M, di, K), "ta_gemm_simple_glu: M=%d di=%d K=%d", M, di, K);
  TA_REQUIRE(lda >= K && ldw >= K && ldc >= di && lda % 4 == 0 && ldw % 4 == 0 && (uintptr_t)A % 16 == 0 && (uintptr_t)W % 16 == 0,
             "ta_gemm_simple_glu: rows of %d, %d, %d floats or their start", lda, ldw, ldc);
  if (ta_gemm_stream_pays(M, 2 * di, K, 1))
    return ta_gemm_stream(stream, A, lda, W, ldw, bias, C, ldc, M, 2 * di, K, 1, 0, nullptr, 0.f);
  walk<true>(stream, A, lda, W, ldw, bias, C, ldc, M, 2 * di, K);
  return ta_check_launch("ta_gemm_simple_glu");
}
