// Products of 32-bit numbers on the 16-bit matrix instructions, by the published way of taking a number apart into shorter ones whose products are
// exact (Ozaki's error-free transformation, Henry, Tang and Heinecke's three bfloat16 for a float32). A float32 x is the sum of three bfloat16,
// x = h + m + l, exactly (24 bits in three times 8; subnormal numbers too, see SPLIT_UP), and of the nine products of two such sums the six that matter are
// multiplied: h h, h m, m h, m m, h l, l h. What is left out is 2.9e-7 (2^-21.7) of a product at the most, of either sign. v_mfma_f32_16x16x32_bf16
// multiplies exactly and takes subnormal numbers: 32 k of all six occupy a SIMD for 96 cycles where the float32 instructions need 256.
//
// The order of the sums, the same in every kernel that uses this, whatever M, N, the kernel or the tile:
//   k is cut into segments of 256 and these into blocks of 32; a block's six products are a chain of instructions from zero, the
//   small ones first; the blocks' results are added in float32 in ascending order, and so are the segments'. Inside an
//   instruction lane (r, kb) holds k = 4 kb .. + 3 and 16 + 4 kb .. + 3 of the block: what a lane has that reads 16 bytes at a time.
// So a row of A gives the same bits alone or inside any batch. Segments let few rows be split over waves; they also round less.
// Against 64 bits (rms of the difference over rms of the result; normal entries, k = 2,048 / 8,192) 1.0e-7 / 1.6e-7, where chains of
// fused multiply-adds over segments of 256 give 2.9e-7 / 3.1e-7; positive entries 4.9e-8 / 7.8e-8 and 9.0e-8 / 8.7e-8; entries
// spread over e^(2 normal) 0.9e-7 / 1.2e-7 and 2.7e-7 / 2.8e-7; k = 64 5.0e-8 and 1.4e-7, 8 3.8e-8 and 5.4e-8. A product alone (k = 1, or a row with one entry
// that is not zero) 3.8e-8, some 3e-7 at the most, where one rounding is 2.5e-8 and 6e-8.
//
// An operand that is infinite, undefined or above some 2^112, and a sum above 2^96 on the way, give a result that
// is not finite here, never a wrong finite one; such a result is formed once more in fused multiply-adds, by a whole wave: lane i takes
// k = i, 64 + i, ..., and the lanes are added up by halves. What a row with an undefined number gives is undefined already, so that a row is
// looked through once and then left. 1,021 x 16,384 x 2,048: 350 us, with a NaN in one row 345, in every row 484, an infinity in one row 948 (8,400 for one
// row of either and 61,000 by one lane a result in series); 4 x 16,384 x 2,048: 25, 30, 31 and 150 (690).
#pragma once
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

#define SEG 256      // k per segment
#define BLK 16       // k that a row's four lanes read at once; two of them are a block

struct Split8 {
  bf16x8 h, m, l;
};
static_assert(sizeof(Split8) == 48, "twelve registers");

// What is split is x 2^16, exactly, so that l has a bfloat16 down to the smallest float32 there is (bfloat16 ends at 2^-133: without, numbers
// below 2^-110 would lose bits); a product is therefore 2^32 too large, and every kernel takes that out of its last sum.
#define SPLIT_UP 65536.0f
#define SPLIT_DOWN 0x1p-32f

// A lane's 8 numbers of a block: x its k = 4 kb .. + 3, y its 16 + 4 kb .. + 3. h is within 2^-7 of the number on either side of it (cut off after 8 bits
// behind a factor of 1 + 3 2^-10, which costs nothing beside the one above), m what is left cut off again, l the rest, which fits. Plain
// instructions, 6.5 a number: v_cvt_pk_bf16_f32 takes as long as three of them, and v_dot2_f32_bf16, which takes h away in one, holds up
// the matrix instructions (a tile of 256 x 128 over k = 8,192 590 us with it, 500 so).
__device__ __forceinline__ Split8 split8(const f32x4& x, const f32x4& y) {
#pragma clang fp contract(off)   // x and y may be products, which are rounded before they are split
  Split8 s;
  uint32_t *h = reinterpret_cast<uint32_t*>(&s.h), *m = reinterpret_cast<uint32_t*>(&s.m), *l = reinterpret_cast<uint32_t*>(&s.l);
  auto cut = [](uint32_t v) { return __uint_as_float(v & 0xffff0000u); };
  auto tops = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float a = i < 2 ? x[2 * i] : y[2 * i - 4], b = i < 2 ? x[2 * i + 1] : y[2 * i - 3];
    const uint32_t na = __float_as_uint(a * (SPLIT_UP * (1 + 0x3p-10f))), nb = __float_as_uint(b * (SPLIT_UP * (1 + 0x3p-10f)));
    const float ra = __builtin_fmaf(a, SPLIT_UP, -cut(na)), rb = __builtin_fmaf(b, SPLIT_UP, -cut(nb));
    const uint32_t ma = __float_as_uint(ra), mb = __float_as_uint(rb);
    h[i] = tops(na, nb);
    m[i] = tops(ma, mb);
    l[i] = tops(__float_as_uint(ra - cut(ma)), __float_as_uint(rb - cut(mb)));
  }
  return s;
}

// the numbers of the lane 4 further on in the row of 16
__device__ __forceinline__ Split8 split_next4(const Split8& x) {
  Split8 y;
  const int *from = reinterpret_cast<const int*>(&x);
  int* to = reinterpret_cast<int*>(&y);
#pragma unroll
  for (int i = 0; i < 12; ++i) to[i] = __builtin_amdgcn_update_dpp(0, from[i], 0x104, 0xf, 0xf, true);
  return y;
}

// step i (0 .. 5) of a block's chain
__device__ __forceinline__ f32x4 split_mul(int i, const Split8& w, const Split8& a, const f32x4& c) {
  const bf16x8& x = i == 0 ? w.l : i == 2 || i == 3 ? w.m : w.h;
  const bf16x8& y = i == 1 ? a.l : i == 2 || i == 4 ? a.m : a.h;
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
}

// a block's product: element e of lane (r, kb) is column 4 kb + e (w's row) of row r (a's)
__device__ __forceinline__ f32x4 split_block(const Split8& w, const Split8& a) {
  f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < 6; ++i) c = split_mul(i, w, a, c);
  return c;
}

__device__ __forceinline__ bool split_bad(float x) { return !(fabsf(x) <= 3.402823466e38f); }

// By whole waves, a(k) and w the same for all lanes: whether one of a's numbers is undefined; the sum over k of a(k) w[k].
template <typename A>
__device__ __forceinline__ bool split_undefined(A a, int K) {
  bool found = false;
#pragma unroll 4
  for (int k = threadIdx.x % TA_WAVE; k < K; k += TA_WAVE) {
    const float x = a(k);
    found |= x != x;
  }
  return __ballot(found) != 0;
}
template <typename A>
__device__ __forceinline__ float split_dot(A a, const float* w, int K) {
  float s = 0.f;
#pragma unroll 4
  for (int k = threadIdx.x % TA_WAVE; k < K; k += TA_WAVE) s = fmaf(a(k), w[k], s);
#pragma unroll
  for (int i = TA_WAVE / 2; i > 0; i /= 2) s += __shfl_xor(s, i, TA_WAVE);
  return s;
}
// Whether row m holds an undefined number, looked up once: state[m] in LDS is 0 before, 1 (no) or 2 behind it. No two waves ask for a row without a barrier between them.
template <typename A>
__device__ __forceinline__ bool split_undefined_once(int* state, int m, A a, int K) {
  int s = state[m];
  if (s == 0) {
    s = split_undefined(a, K) ? 2 : 1;
    if (threadIdx.x % TA_WAVE == 0) state[m] = s;
  }
  return s == 2;
}

// What a lane's result is, by a whole wave: `value` or, where that is `bad`, the sum over k of a(m, k) w[k]. undefined(m): whether row m
// holds an undefined number.
template <typename A, typename U>
__device__ __forceinline__ float split_again(bool bad, float value, int m, const float* w, int K, A a, U undefined) {
  uint64_t left = __ballot(bad);
  while (left) {
    const int from = __builtin_ctzll(left), row = __builtin_amdgcn_readlane(m, from);
    if (undefined(row)) {
      left &= ~__ballot(m == row);
      continue;
    }
    const uint64_t at = (uint64_t)(uintptr_t)w;
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)at, from), hi = __builtin_amdgcn_readlane((uint32_t)(at >> 32), from);
    const float v = split_dot([&](int k) { return a(row, k); }, (const float*)(uintptr_t)((uint64_t)hi << 32 | lo), K);
    if (threadIdx.x % TA_WAVE == from) value = v;
    left &= left - 1;
  }
  return value;
}
