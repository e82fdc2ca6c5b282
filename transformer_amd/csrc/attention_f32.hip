// Causal grouped-query attention over the paged cache in 32 bits on the matrix cores, for key and value
// widths that are multiples of 16 up to 128: what attention_generic.hip computes, options included, for the
// float32 engine's usual heads (other widths and storage types stay there).
//
// The float32 matrix instructions are chains of fused multiply-adds, so a row's result can be defined
// without them: pages of 64 keys are taken one by one, each with a maximum, a sum of exponentials and a sum
// of values of its own, and joined in ascending order:
//   M' = max(M, m), a = exp(M - M'), b = exp(m - M'); L = b l + a L; O = b o + a O.
// A page's numbers depend on the row's query and that page alone. So they may be formed anywhere: prompts walk
// a row's pages in one wave, single tokens hand every page to a wave of its own and join the pages in a second
// kernel, and both give the same bits, whatever the batch and the cut into steps.
//
// 16 rows (query token, query head of the kv head's group) a wave, v_mfma_f32_16x16x4_f32. Lane (r, kb), r < 16,
// kb < 4: scores K Q^T leave it row r's keys 16 t + 4 kb + i (t, i < 4), which is the layout in which the second
// product V^T P^T wants the weights; both operands of either product are runs of 4 consecutive numbers of a key
// or value row.
#include <type_traits>
#include "common.h"

typedef float f32x4 __attribute__((ext_vector_type(4)));

struct F32Attention {
  const float* q;
  float* out;
  const float *k, *v;          // one layer: [pages][nkv][64][dh], [pages][nkv][dv][64]
  const int *table, *cu_q, *pos0;
  const float *sink, *gate;
  // single tokens: [seqs][heads][max_blocks][dv] sums, then [seqs][heads][max_blocks][2] maxima and sums, of the sequences
  // from b0 on and the heads of the kv heads from kv0 on
  float* parts;
  int q_stride, out_stride, max_blocks, nh, nkv, dh, dv, window, sink_mode, gate_stride, gate_dv, keep, chunk;
  float scale, softcap;
  int b0, kv0, seqs, heads;
};

// what a row sees: keys start .. end - 1 and the first `keep`
struct Span {
  int start, end, keep;
  __device__ __forceinline__ bool key(int k) const { return (k >= start || k < keep) && k < end; }
  __device__ __forceinline__ bool page(int p) const { return p * 64 < end && (p * 64 + 64 > start || p * 64 < keep); }
};

// Both products read the next operands from LDS while the present ones are multiplied (left to itself the compiler reads them right in
// front of their use), where the widths are known (else the branches around the reads cost more registers than there are).
template <int NB, bool EXACT, int T, typename KF>
__device__ __forceinline__ void page_scores(const f32x4* qf, int nb, KF kfrag, f32x4* s) {
  f32x4 k[2][T];
  auto ask = [&](int d) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < T; ++t) k[d % 2][t] = kfrag(t, d);
  };
#pragma unroll
  for (int t = 0; t < T; ++t) s[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  if (EXACT) ask(0);
#pragma unroll
  for (int d = 0; d < NB; ++d)
    if (EXACT || d < nb) {
      if (!EXACT) ask(d);
      else if (d + 1 < NB) ask(d + 1);
      if (EXACT) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t) s[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[d % 2][t][j], qf[d][j], s[t], 0, 0, 0);
      if (EXACT) __builtin_amdgcn_sched_barrier(0);
    }
}

// scores -> weights relative to the page's maximum m, and their sum l. whole: every row of the wave sees the whole page.
__device__ __forceinline__ void page_softmax(const F32Attention& p, const Span& see, int key0, bool whole, f32x4* s, float& m, float& l) {
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) s[t][i] *= p.scale;
  if (p.softcap > 0.f)       // outside the loop above, or the compiler keeps a branch for every score
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[t][i] = p.softcap * tanhf(s[t][i] / p.softcap);
  if (!whole)
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[t][i] = see.key(key0 + 16 * t + i) ? s[t][i] : -INFINITY;
  m = -INFINITY;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) m = fmaxf(m, s[t][i]);
  const auto m16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(m), __float_as_uint(m), false, false);     // a lane's and its neighbour's
  m = fmaxf(__uint_as_float(m16[0]), __uint_as_float(m16[1]));
  const auto m32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(m), __float_as_uint(m), false, false);
  m = fmaxf(__uint_as_float(m32[0]), __uint_as_float(m32[1]));
  l = 0.f;
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      s[t][i] = s[t][i] == -INFINITY ? 0.f : expf(s[t][i] - m);
      l += s[t][i];
    }
  const auto l16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(l), __float_as_uint(l), false, false);
  l = __uint_as_float(l16[0]) + __uint_as_float(l16[1]);
  const auto l32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
  l = __uint_as_float(l32[0]) + __uint_as_float(l32[1]);
}

// o[d] = the page's sum of values, columns 16 d + 4 kb + i of row r. Keys from `live` on (of the page) were never
// written and count as zero.
template <int NB, bool EXACT, typename VF>
__device__ __forceinline__ void page_values(const f32x4* e, int nb, int live, int kb, VF vfrag, f32x4* o) {
  constexpr int G = !EXACT ? 1 : NB < 4 ? NB : 4, STEPS = 4 * NB / G;       // of G blocks of columns and 16 keys
  auto sum = [&](auto all) __attribute__((always_inline)) {
    f32x4 v[2][G];
    auto ask = [&](int step) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < G; ++i) v[step % 2][i] = vfrag(step / (NB / G), step % (NB / G) * G + i);
    };
#pragma unroll
    for (int d = 0; d < NB; ++d) o[d] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (EXACT) ask(0);
#pragma unroll
    for (int step = 0; step < STEPS; ++step) {
      const int t = step / (NB / G), d0 = step % (NB / G) * G;
      if (!EXACT && d0 >= nb) continue;
      if (!EXACT) ask(step);
      else if (step + 1 < STEPS) ask(step + 1);
      if (EXACT) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool there = decltype(all)::value || 16 * t + 4 * kb + j < live;
#pragma unroll
        for (int i = 0; i < G; ++i)
          o[d0 + i] = __builtin_amdgcn_mfma_f32_16x16x4f32(there ? v[step % 2][i][j] : 0.f, e[t][j], o[d0 + i], 0, 0, 0);
      }
      if (EXACT) __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (live >= 64) sum(std::true_type{});
  else sum(std::false_type{});
}

// factors with which what was joined so far and a page's numbers enter the sums
__device__ __forceinline__ void join(float& M, float m, float& a, float& b) {
  const float n = fmaxf(M, m);
  a = M == n ? 1.f : expf(M - n);
  b = m == n ? 1.f : expf(m - n);
  M = n;
}

// what stands between the sums and the result: the sink's term, the division, a gate per head
__device__ __forceinline__ float last_factor(const F32Attention& p, float M, float L, int head, size_t token, float& rescale) {
  rescale = 1.f;
  if (p.sink_mode != 0) {
    const float sv = p.sink_mode == 2 ? p.sink[head] : 0.f;
    const float n = fmaxf(M, sv);
    rescale = expf(M - n);               // M = -inf (no key seen) gives 0
    L = L * rescale + expf(sv - n);
  }
  float inv = L > 0.f ? 1.0f / L : 0.f;
  if (p.gate && p.gate_dv == 0) inv *= 1.0f / (1.0f + expf(-p.gate[token * p.gate_stride + head]));
  return inv;
}
__device__ __forceinline__ float gated(const F32Attention& p, float x, int head, size_t token, int col) {
  if (p.gate && col < p.gate_dv) x *= 1.0f / (1.0f + expf(-p.gate[token * p.gate_stride + (size_t)head * p.gate_dv + col]));
  return x;
}

// Prompts: 64 / SPLIT rows of one (sequence, kv head) a workgroup of four waves, SPLIT waves for 16 rows: each forms the scores of its share of a page's
// keys, takes the others' from LDS and sums its share of the columns, so every number comes about as with one wave. A page's keys and its
// values go through LDS once for the four. The next page's keys are on their way during the softmax and the second product, its values
// during the next scores; two workgroups share a CU. Bound by the chain of pages of the longest rows where they are few (a page is 256 matrix instructions of 32 cycles a
// wave, and with SPLIT 1 a prompt of 1,021 tokens has one wave a SIMD, whose longest walks twice the mean), by the matrix instructions where they are many. 16 heads of 128 over 4 kv heads, us
// before the split / with SPLIT 1, 2, 4: 256 tokens 30 / 28, 20, 16; 512 53 / 49, 35, 29; 1,021 102 / 95, 72, 88; 2,011 322 / 294, 231, 268; 3,000 535 / 487, 429, 548; 807 for 1,021 on the vector ALU.
template <int NB, bool EXACT, int SPLIT>
__global__ __launch_bounds__(256, EXACT ? 2 : 1) void attn_f32_rows_kernel(F32Attention p) {
  constexpr int ROWS = 64 / SPLIT, TILES = 4 / SPLIT, T = 4 / SPLIT, OWN = NB / SPLIT;
  __shared__ f32x4 Ks[64 * 4 * NB], Vs[16 * NB * 16], scores[SPLIT > 1 ? TILES : 1][SPLIT > 1 ? 4 : 1][TA_WAVE];
  const int group = p.nh / p.nkv, b = blockIdx.z, kvh = SPLIT > 1 ? blockIdx.x : blockIdx.y, nth = SPLIT > 1 ? blockIdx.y : blockIdx.x;
  const int q0 = p.cu_q[b], qlen = p.cu_q[b + 1] - q0, nrows = qlen * group;
  const int blocks = (nrows + ROWS - 1) / ROWS;
  if (nth >= blocks) return;
  // The longest first; with two workgroups a CU (SPLIT > 1) every other 256 the shortest first, so that a long and a short one meet
  // (1,300 tokens of the shape above 156 us without, 119 so).
  int row0 = (blocks - 1 - nth) * ROWS;
  if (SPLIT > 1) {
    const int turn = gridDim.x < 256 ? 256 / gridDim.x : 1, begin = b * gridDim.y;
    auto odd = [&](int n) { return n / (2 * turn) * turn + (n % (2 * turn) > turn ? n % (2 * turn) - turn : 0); };
    const int shorts = odd(begin + nth) - odd(begin);
    row0 = ((begin + nth) / turn % 2 ? shorts : blocks - 1 - (nth - shorts)) * ROWS;
  }
  const int pos0 = p.pos0[b];
  const int lane = threadIdx.x % TA_WAVE, wave = threadIdx.x / TA_WAVE, r = lane % 16, kb = lane / 16;
  const int tile = wave / SPLIT, part = wave % SPLIT;
  const int nkb = EXACT ? NB : p.dh / 16, nvb = EXACT ? NB : p.dv / 16;

  const int last = row0 + ROWS - 1 < nrows - 1 ? row0 + ROWS - 1 : nrows - 1;
  const Span all = {ta_first_key(pos0 + row0 / group + 1, p.window, p.chunk), pos0 + last / group + 1, p.keep};
  const int row = row0 + 16 * tile + r;
  const bool ok = row < nrows;
  const int qi = ok ? row / group : 0, head = kvh * group + (ok ? row % group : 0);
  Span see = {ta_first_key(pos0 + qi + 1, p.window, p.chunk), pos0 + qi + 1, p.keep};
  if (!ok) see = {0, 0, 0};
  // the wave's own rows
  const int wfirst = row0 + 16 * tile, wlast = wfirst + 15 < nrows - 1 ? wfirst + 15 : nrows - 1;
  const bool wlive = wfirst < nrows;
  const Span mine = {ta_first_key(pos0 + wfirst / group + 1, p.window, p.chunk), wlive ? pos0 + wlast / group + 1 : 0, p.keep};
  // pages that all 16 of them see whole
  const int whole0 = (ta_first_key(pos0 + wlast / group + 1, p.window, p.chunk) + 63) / 64;
  const int whole1 = wfirst + 15 < nrows ? (pos0 + wfirst / group + 1) / 64 : 0;

  f32x4 qf[NB], O[OWN];
  const float* qrow = p.q + (size_t)(q0 + qi) * p.q_stride + (size_t)head * p.dh;
#pragma unroll
  for (int d = 0; d < NB; ++d) {
    if (EXACT || d < nkb) qf[d] = *reinterpret_cast<const f32x4*>(qrow + 16 * d + 4 * kb);
    if (d < OWN) O[d] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float M = -INFINITY, L = 0.f;
  // here, or the compiler waits for them at their first use inside the loop, where that means all that is on its way
#pragma unroll
  for (int d = 0; d < NB; ++d)
    if (EXACT || d < nkb) asm volatile("" : "+v"(qf[d]));

  // pieces of 16 bytes, permuted inside a row by the row's number
  // by the scalar unit: a load of a wave's own would be waited for together with all that the wave has asked for before it
  const auto* table = (const __attribute__((address_space(4))) int*)(uintptr_t)(p.table + (size_t)b * p.max_blocks);
  auto entry = [&](int page) { return (size_t)table[__builtin_amdgcn_readfirstlane(page)]; };
  const int kper = 4 * nkb, kmask = nkb % 4 == 0 ? 15 : nkb % 2 == 0 ? 7 : 3;
  auto bring_keys = [&](int page) {
    const float* from = p.k + (entry(page) * p.nkv + kvh) * 64 * p.dh;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (EXACT || i < nkb) {
        const int at = i * 256 + (int)threadIdx.x, row_ = at / kper, piece = (at - row_ * kper) ^ (row_ & kmask);
        ta_load_to_lds16(from, (uint32_t)(row_ * p.dh + piece * 4) * 4, &Ks[i * 256 + wave * 64]);
      }
  };
  auto bring_values = [&](int page) {
    const float* from = p.v + (entry(page) * p.nkv + kvh) * 64 * p.dv;
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (EXACT || i < nvb) {
        const int at = i * 256 + (int)threadIdx.x, row_ = at / 16, piece = (at % 16) ^ (row_ & 15);
        ta_load_to_lds16(from, (uint32_t)(row_ * 64 + piece * 4) * 4, &Vs[i * 256 + wave * 64]);
      }
  };
  auto next_page = [&](int page) {
    do ++page; while (page * 64 < all.end && !all.page(page));
    return page;
  };

  int page = next_page(-1);
  bring_keys(page);
  bring_values(page);
  while (page * 64 < all.end) {
    const int next = next_page(page);
    const bool more = next * 64 < all.end;
    const bool use = mine.page(page);
    // the keys have come: they were asked for before the values
    if (EXACT) ta_wait_loads<NB>(); else ta_wait_loads<0>();
    __syncthreads();
    f32x4 s[4];
    if (use) {
      page_scores<NB, EXACT, T>(qf, nkb, [&](int t, int d) {
        return Ks[(16 * (part * T + t) + r) * kper + ((4 * d + kb) ^ (r & kmask))];
      }, s);
      if (SPLIT > 1)
#pragma unroll
        for (int t = 0; t < T; ++t) scores[tile][part * T + t][lane] = s[t];
    }
    __syncthreads();                               // everybody has done with the keys
    if (more) bring_keys(next);
    if (SPLIT > 1 && use)
#pragma unroll
      for (int t = 0; t < 4; ++t) s[t] = scores[tile][t][lane];
    float m = -INFINITY, l = 0.f;
    if (use) page_softmax(p, see, page * 64 + 4 * kb, page >= whole0 && page < whole1, s, m, l);
    if (EXACT && more) ta_wait_loads<NB>(); else ta_wait_loads<0>();          // the values
    __syncthreads();
    f32x4 o[OWN];
    if (use) {
      const int live = all.end - page * 64;
      page_values<OWN, EXACT>(s, (nvb - part + SPLIT - 1) / SPLIT, live, kb, [&](int t, int i) {
        return Vs[(16 * (part + SPLIT * i) + r) * 16 + ((4 * t + kb) ^ r)];
      }, o);
    }
    __syncthreads();                               // everybody has done with the values
    if (more) bring_values(next);
    if (use) {
      float a, c;
      join(M, m, a, c);
      L = fmaf(l, c, L * a);
#pragma unroll
      for (int d = 0; d < OWN; ++d)
        if (EXACT || part + SPLIT * d < nvb)
#pragma unroll
          for (int i = 0; i < 4; ++i) O[d][i] = fmaf(o[d][i], c, O[d][i] * a);
    }
    page = next;
  }
  if (!ok) return;
  const size_t token = (size_t)(q0 + qi);
  float rescale;
  const float inv = last_factor(p, M, L, head, token, rescale);
  float* orow = p.out + token * p.out_stride + (size_t)head * p.dv;
#pragma unroll
  for (int d = 0; d < OWN; ++d)
    if (EXACT || part + SPLIT * d < nvb) {
      const int col = 16 * (part + SPLIT * d) + 4 * kb;
      f32x4 x;
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] = gated(p, O[d][i] * rescale * inv, head, token, col + i);
      *reinterpret_cast<f32x4*>(orow + col) = x;
    }
}

// Single tokens: a workgroup takes pages of one (sequence, kv head, 16 of the group's heads), operands straight from
// memory, all of a page's 64 KB asked for at once. Wave t forms the scores of keys 16 t .. + 15, hands them round through
// LDS, and sums the values of columns 16 d .. + 15 for d = t, t + 4; weights, maximum and sum are formed by every wave, so
// that each number comes about as in the prompts' kernel. Bound by the trip to memory. The grid follows the page table's width, so
// that a recorded launch fits every length; the pages are its slowest index, since workgroups that find no page are then handed out
// last (with the pages fastest 4 x 200 keys, 16 heads over 4 kv heads, 14.0 us for both kernels where it now takes 9.1).
// Both kernels, those heads, 4 x 200 / 16 x 300 / 16 x 2,000 keys: 9.1 / 12.3 / 36 us; with a wave a page, which brings 64 KB by
// itself, 20.6 / 58 / 65; by one workgroup per sequence and kv head 279 (4 of 50 to 300). Heads of 64, whose pages are half as long: 8 x
// 1,000 keys, 16 heads over 4, 12.8 us where a wave a page took 15.2, but with every CU full the four waves' barrier shows (32 x
// 2,000 39.1 and 37.0; 64 x 1,000, 16 heads with keys of their own, 120 and 105); of 128, 64 x 1,000 214 and 278.
template <int NB, bool EXACT>
__global__ __launch_bounds__(256) void attn_f32_pages_kernel(F32Attention p) {
  __shared__ f32x4 scores[2][4][TA_WAVE];
  const int group = p.nh / p.nkv, tiles = (group + 15) / 16, b = p.b0 + blockIdx.y;
  const int kvh = p.kv0 + blockIdx.x / tiles, h0 = blockIdx.x % tiles * 16;
  const int wave = threadIdx.x / TA_WAVE, lane = threadIdx.x % TA_WAVE, r = lane % 16, kb = lane / 16;
  const int end = p.pos0[b] + 1;
  const Span see = {ta_first_key(end, p.window, p.chunk), end, p.keep};
  // no page behind the table's width, which the joining kernel goes by and which p.parts has room for
  const int pages = (end + 63) / 64 < p.max_blocks ? (end + 63) / 64 : p.max_blocks;
  if ((int)blockIdx.z >= pages) return;
  if (p.cu_q[b + 1] == p.cu_q[b]) return;          // a sequence that brings no token has no row
  constexpr int OWN = NB / 4;                      // blocks of value columns a wave owns
  const int nkb = EXACT ? NB : p.dh / 16, nvb = EXACT ? NB : p.dv / 16;
  const bool ok = h0 + r < group;
  const int head = kvh * group + (ok ? h0 + r : 0);
  const float* qrow = p.q + (size_t)p.cu_q[b] * p.q_stride + (size_t)head * p.dh;
  f32x4 qf[NB];
#pragma unroll
  for (int d = 0; d < NB; ++d)
    if (EXACT || d < nkb) qf[d] = *reinterpret_cast<const f32x4*>(qrow + 16 * d + 4 * kb);
  for (int page = blockIdx.z, turn = 0; page < pages; page += gridDim.z) {
    if (!see.page(page)) continue;
    const size_t at = ((size_t)p.table[(size_t)b * p.max_blocks + page] * p.nkv + kvh) * 64;
    const float *kp = p.k + (at + 16 * wave + r) * p.dh, *vp = p.v + at * p.dv;
    f32x4 kf[NB], vf[4][OWN];
#pragma unroll
    for (int d = 0; d < NB; ++d)
      if (EXACT || d < nkb) kf[d] = *reinterpret_cast<const f32x4*>(kp + 16 * d + 4 * kb);
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < OWN; ++i)
        if (EXACT || wave + 4 * i < nvb)
          vf[t][i] = *reinterpret_cast<const f32x4*>(vp + (size_t)(16 * (wave + 4 * i) + r) * 64 + 16 * t + 4 * kb);
    __builtin_amdgcn_sched_barrier(0);             // or the values are asked for behind the scores
    f32x4 own = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int d = 0; d < NB; ++d)
      if (EXACT || d < nkb)
#pragma unroll
        for (int j = 0; j < 4; ++j) own = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[d][j], qf[d][j], own, 0, 0, 0);
    // one barrier a page: who writes this half again has passed the other half's, behind which all have read this one
    scores[turn][wave][lane] = own;
    __syncthreads();
    f32x4 s[4], o[OWN];
#pragma unroll
    for (int t = 0; t < 4; ++t) s[t] = scores[turn][t][lane];
    turn ^= 1;
    float m, l;
    page_softmax(p, see, page * 64 + 4 * kb, false, s, m, l);
    page_values<OWN, EXACT>(s, (nvb - wave + 3) / 4, end - page * 64, kb, [&](int t, int i) { return vf[t][i]; }, o);
    if (!ok) continue;
    const size_t unit = ((size_t)blockIdx.y * p.heads + head - p.kv0 * group) * p.max_blocks + page;
    float* sums = p.parts + unit * p.dv;
#pragma unroll
    for (int i = 0; i < OWN; ++i)
      if (EXACT || wave + 4 * i < nvb) *reinterpret_cast<f32x4*>(sums + 16 * (wave + 4 * i) + 4 * kb) = o[i];
    if (wave == 0 && kb == 0) {
      float* ml = p.parts + (size_t)p.seqs * p.heads * p.max_blocks * p.dv + unit * 2;
      ml[0] = m;
      ml[1] = l;
    }
  }
}

// The pages of a single token's row joined in ascending order, eight asked for at a time; a thread a column.
__global__ __launch_bounds__(128) void attn_f32_join_kernel(F32Attention p) {
  const int head = p.kv0 * (p.nh / p.nkv) + blockIdx.x, b = p.b0 + blockIdx.y, d = threadIdx.x;
  if (p.cu_q[b + 1] == p.cu_q[b]) return;
  const int end = p.pos0[b] + 1;
  const Span see = {ta_first_key(end, p.window, p.chunk), end, p.keep};
  const size_t unit = ((size_t)blockIdx.y * p.heads + blockIdx.x) * p.max_blocks;
  const float* sums = p.parts + unit * p.dv;
  const float* ml = p.parts + (size_t)p.seqs * p.heads * p.max_blocks * p.dv + unit * 2;
  const int pages = (end + 63) / 64 < p.max_blocks ? (end + 63) / 64 : p.max_blocks;
  float M = -INFINITY, L = 0.f, O = 0.f;
  for (int p0 = 0; p0 < pages; p0 += 8) {
    float o[8], m[8], l[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const bool in = p0 + i < pages && see.page(p0 + i);
      const int at = in ? p0 + i : pages - 1;        // the last page is always seen
      o[i] = sums[(size_t)at * p.dv + (d < p.dv ? d : 0)];
      m[i] = ml[2 * at];
      l[i] = ml[2 * at + 1];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (p0 + i < pages && see.page(p0 + i)) {
        float a, c;
        join(M, m[i], a, c);
        L = fmaf(l[i], c, L * a);
        O = fmaf(o[i], c, O * a);
      }
  }
  if (d >= p.dv) return;
  const size_t token = (size_t)p.cu_q[b];
  float rescale;
  const float inv = last_factor(p, M, L, head, token, rescale);
  p.out[token * p.out_stride + (size_t)head * p.dv + d] = gated(p, O * rescale * inv, head, token, d);
}

// Single tokens go through in turns whose partial rows take 256 MB at most (or one kv head's, if that is more): whole
// sequences while one fits, else some kv heads of one sequence. (The prompts' kernel, which had such steps before, walks
// a row's pages one after the other: 8 sequences of 120,000 keys, 32 heads over 8, 11.0 ms, 2.9 in turns; 16 of 60,000
// 5.5 and 2.6.)
#define F32_PARTS (1ll << 26)
// Workgroups of single tokens: enough for every CU to hold a few, at least 8 a row, each with every so-manieth page (256 / 512 /
// 1,024 of them: 4 sequences of 4,000 keys, 16 heads of 64 with keys of their own, 47.6 / 46.9 / 42.5 us; 2 of 16,000 150 / 113 /
// 102; a workgroup per page of a table of 64 pages, most of them empty, 16 sequences of 300 keys over 4 kv heads 28.7, 12.3 here).
#define F32_PAGE_WGS 1024
static void f32_turn(int batch, int nh, int nkv, int max_blocks, int dv, int& seqs, int& kvs) {
  const long long unit = (long long)(nh / nkv) * max_blocks * (dv + 2), fit = F32_PARTS / unit > 1 ? F32_PARTS / unit : 1;
  kvs = fit < nkv ? (int)fit : nkv;
  seqs = fit / nkv < 1 ? 1 : fit / nkv < batch ? (int)(fit / nkv) : batch;
}

// Floats of scratch that ta_attention_f32 wants for a step of single tokens.
extern "C" long long ta_attention_f32_turn_scratch(int batch, int nh, int nkv, int max_blocks, int dv) {
  if (batch <= 0 || nkv <= 0 || nh < nkv || max_blocks <= 0 || dv <= 0) return 0;
  int seqs, kvs;
  f32_turn(batch, nh, nkv, max_blocks, dv, seqs, kvs);
  return (long long)seqs * kvs * (nh / nkv) * max_blocks * (dv + 2);
}
// The most that it wants, whatever the kv heads.
extern "C" long long ta_attention_f32_scratch(int batch, int nh, int max_blocks, int dv) {
  return (long long)batch * nh * max_blocks * (dv + 2);
}

// Which kernels take these widths: 128 and 128, 64 and 64, both up to 64, any. Up to 64 by half the registers and LDS: 16 heads of 32 over 4, a prompt of
// 1,021 76 us by the kernel for any and 55 by its own, 3,000 466 and 227.
static int f32_widths(int dh, int dv) { return dh == 128 && dv == 128 ? 0 : dh == 64 && dv == 64 ? 1 : dh <= 64 && dv <= 64 ? 2 : 3; }

// Waves for 16 rows by the blocks of 64 rows that the step has (half a block more a sequence), where SPLIT 4 keeps the CUs from idling and 2 the
// longest rows from walking alone. Many short sequences gain nothing: their pages are few and every workgroup brings them again. us of SPLIT 1, 2, 4, heads of 128
// over 4 kv heads: 2 + 34 blocks 22 / 16 / 14, 175 65 / 48 / 45, 4 x 50 to 300 tokens (190) 33 / 28 / 30, 4 x 400 (408) 63 / 58 / 67, 16 x 100 (432) 27 / 31 / 37, 8 x 300 (616) 63 / 67 / 78;
// 32 heads of 64 over 8: 200 29 / 23 / 26, 512 100 / 68 / 91, 1,005 265 / 242 / 300, 1,500 493 / 492 / 626.
// Heads of 16, whose pages cost little beside the barriers, not over several sequences (8 heads, 8 x 200 16 / 18, 8 x 300 21 / 24; 4 x 300 20 / 23; one of 1,021 53 / 44).
static int f32_split(int batch, int max_qlen, int tokens, int group, int nkv, int widest) {
  if (widest <= 16 && batch >= 4) return 1;
  const long long rows = (long long)max_qlen * group, blocks = ((long long)tokens * group + 63) / 64 * nkv + (long long)batch * nkv / 2;
  return rows > 65535 * 16 || blocks > (max_qlen >= 1000 ? 1024 : max_qlen >= 256 ? 512 : 256) ? 1 : blocks <= 180 ? 4 : 2;
}

// The prompts' kernel that ta_attention_f32 launches: f32_widths times 8 plus the waves for 16 rows; 0 for heads that it refuses.
extern "C" int ta_attention_f32_form(int batch, int max_qlen, int tokens, int nh, int nkv, int dh, int dv) {
  if (nh <= 0 || nkv <= 0 || nh % nkv != 0) return 0;
  return f32_widths(dh, dv) * 8 + f32_split(batch, max_qlen, tokens, nh / nkv, nkv, dh > dv ? dh : dv);
}

// As ta_attention_generic_sink, float32, dh and dv multiples of 16 up to 128, rows that start on 16 bytes. parts:
// scratch of ta_attention_f32_turn_scratch floats for steps in which every sequence brings one token or none (max_qlen 1), or
// null: the kernel for prompts then serves these too, with the same bits. tokens: of all sequences, by which the prompts' kernel is split.
extern "C" int ta_attention_f32(hipStream_t stream, const void* q, int q_stride, void* out, int out_stride,
                                const void* kcache, const void* vcache, const int* block_table, int max_blocks,
                                const int* cu_q, const int* pos0, int batch, int max_qlen, int nh, int nkv, int dh,
                                int dv, float scale, int window, float softcap, int sink_mode, const float* sink,
                                const void* gate, int gate_stride, int gate_dv, int keep, int chunk, float* parts,
                                int tokens) {
  TA_REQUIRE(batch >= 0 && max_qlen >= 0 && tokens >= 0, "ta_attention_f32: bad batch=%d max_qlen=%d tokens=%d", batch, max_qlen, tokens);
  TA_REQUIRE(sink_mode >= 0 && sink_mode <= 2 && (sink_mode != 2 || sink != nullptr) && softcap >= 0.f,
             "ta_attention_f32: sink mode %d, cap %f", sink_mode, softcap);
  TA_REQUIRE(gate == nullptr || (gate_dv >= 0 && gate_dv <= dv && gate_stride >= nh * (gate_dv > 0 ? gate_dv : 1)),
             "ta_attention_f32: gate rows of %d", gate_stride);
  TA_REQUIRE(keep >= 0 && (keep == 0 || window > 0), "ta_attention_f32: %d kept keys beside a window of %d", keep, window);
  TA_REQUIRE(chunk >= 0 && (chunk == 0 || window <= 0), "ta_attention_f32: chunks of %d beside a window of %d", chunk, window);
  TA_REQUIRE(nh > 0 && nkv > 0 && nh % nkv == 0, "ta_attention_f32: %d heads do not divide into %d kv heads", nh, nkv);
  TA_REQUIRE(dh % 16 == 0 && dh >= 16 && dh <= 128 && dv % 16 == 0 && dv >= 16 && dv <= 128,
             "ta_attention_f32: key width %d / value width %d", dh, dv);
  TA_REQUIRE(q_stride >= nh * dh && out_stride >= nh * dv && q_stride % 4 == 0 && out_stride % 4 == 0 &&
                 ((uintptr_t)q | (uintptr_t)out | (uintptr_t)kcache | (uintptr_t)vcache | (uintptr_t)parts) % 16 == 0,
             "ta_attention_f32: rows of %d and %d floats or their start", q_stride, out_stride);
  TA_REQUIRE(max_blocks > 0 && batch <= 65535 && (long long)nkv * ((nh / nkv + 15) / 16) <= 65535,
             "ta_attention_f32: grid of %d sequences, %d kv heads, %d pages", batch, nkv, max_blocks);
  if (batch == 0 || max_qlen == 0) return 0;
  F32Attention p = {(const float*)q, (float*)out, (const float*)kcache, (const float*)vcache, block_table, cu_q, pos0,
                          sink, (const float*)gate, parts, q_stride, out_stride, max_blocks, nh, nkv, dh, dv, window,
                          sink_mode, gate_stride, gate_dv, keep, chunk, scale, softcap, 0, 0, 0, 0};
  const int group = nh / nkv, widths = f32_widths(dh, dv);
#define PICK(kernel, grid, ...)                                                         \
  switch (widths) {                                                                     \
    case 0: kernel<8, true, ##__VA_ARGS__><<<grid, 256, 0, stream>>>(p); break;         \
    case 1: kernel<4, true, ##__VA_ARGS__><<<grid, 256, 0, stream>>>(p); break;         \
    case 2: kernel<4, false, ##__VA_ARGS__><<<grid, 256, 0, stream>>>(p); break;        \
    default: kernel<8, false, ##__VA_ARGS__><<<grid, 256, 0, stream>>>(p);              \
  }
  if (max_qlen == 1 && parts != nullptr) {
    int kvs;
    f32_turn(batch, nh, nkv, max_blocks, dv, p.seqs, kvs);
    p.heads = kvs * group;
    for (p.b0 = 0; p.b0 < batch; p.b0 += p.seqs)
      for (p.kv0 = 0; p.kv0 < nkv; p.kv0 += kvs) {
        const int bs = batch - p.b0 < p.seqs ? batch - p.b0 : p.seqs, ks = nkv - p.kv0 < kvs ? nkv - p.kv0 : kvs;
        const long long rows = (long long)ks * ((group + 15) / 16) * bs;
        const int each = (int)((F32_PAGE_WGS + rows - 1) / rows), turn = each < 8 ? 8 : each;
        PICK(attn_f32_pages_kernel, dim3(ks * ((group + 15) / 16), bs, max_blocks < turn ? max_blocks : turn))
        attn_f32_join_kernel<<<dim3(ks * group, bs), 128, 0, stream>>>(p);
      }
  } else {
    const long long rows = (long long)max_qlen * group;
    const int split = f32_split(batch, max_qlen, tokens, group, nkv, dh > dv ? dh : dv);
    if (split == 4) {
      PICK(attn_f32_rows_kernel, dim3(nkv, (unsigned)((rows + 15) / 16), batch), 4)
    } else if (split == 2) {
      PICK(attn_f32_rows_kernel, dim3(nkv, (unsigned)((rows + 31) / 32), batch), 2)
    } else {
      PICK(attn_f32_rows_kernel, dim3((unsigned)((rows + 63) / 64), nkv, batch), 1)
    }
  }
#undef PICK
  return ta_check_launch("ta_attention_f32");
}
