// gdr_bwd_chunk.hip: the launch behind the reverse state scan of the gated delta rule backward, K and V in {64, 128}.
#pragma once
#include "fla_common.h"

// hT, dhT: the states and state gradients of every chunk, FLA_H_FRAGMENT_T; dv2 as the reverse scan leaves it; dg receives the
// gradient of the raw gate.  `chunks`, `ntfix`: chunk_grid() of the batch.
int gdr_bwd_chunk(const void* q, const void* k, const void* v, const void* v_new, const float* beta, const float* g_cumsum,
                  const void* Aw, const void* dout, const void* dv2, const void* hT, const void* dhT, void* dq, void* dk,
                  void* dv, float* dbeta, float* dg, const int64_t* offsets, const int64_t* indices, int64_t chunks,
                  int ntfix, int qkv_dtype, int64_t T, int64_t H, int64_t K, int64_t V, float scale, hipStream_t st);
