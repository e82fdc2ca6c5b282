// Matrix states of long steps, 16 tokens at a time (chunked.hip); called by the entry points of recurrent.hip and
// matrix_memory.hip, which have checked their arguments.
#pragma once
#include "common.h"

// S_t = diag(a_t) S_{t-1} + k_t v_t^T per head, o_t = S_t^T q_t. q, k, v lie at element offsets of rows ``stride``
// apart. The decay a_t comes from exactly one of alpha [nt, H, dk], tok_decay [nt, H] and head_decay [H].
struct TaChunked {
  const void* proj;
  int stride, qoff, koff, voff, qk_share;      // qk_share heads read the same q and k
  float qscale;
  const float *alpha, *tok_decay, *head_decay;
  const float* tok_kscale;                     // null, or [nt, H]: a factor on the key
  const float* bonus;                          // null, or [H, dk]: o_t = (S_{t-1} + diag(bonus) k_t v_t^T)^T q_t
  float* state;                                // [slots, H, dk, dv], moved on
  const int *cu_q, *slots;
  int H, dk, dv;
  size_t plane;
  int planes;                                  // planes of o_out; those behind the first are zeroed
  float* o_out;                                // [planes, nt, H, dv]
  float *n_state, *den_out;                    // null, or [slots, H, dk], moved on like a column of ones, and [nt, H] = n_t . q_t
  bool vec;                                    // q, k, v (and alpha) can be read four values at a time
};

#define TA_CHUNK 16
// Steps that may go in chunks: a chunk costs all of its 16 tokens.
static inline bool ta_chunked_long(int nt, int batch) { return nt > 48 && nt > 8 * batch; }

bool ta_chunked_takes(bool scalar_decay, bool bonus, int dk);
int ta_chunked_launch(hipStream_t stream, int dtype, const TaChunked& p, int batch, const char* what);
