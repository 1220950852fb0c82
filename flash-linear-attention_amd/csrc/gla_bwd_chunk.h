// gla_bwd_chunk.hip: the launch behind the reverse state scan of the GLA backward, K and V in {64, 128}.
#pragma once
#include "fla_common.h"

// hT, dhT: the states and state gradients of every chunk, FLA_H_FRAGMENT_T.  head_gates: g and dg are fp32 [rows, H].  wide:
// chunks whose score terms are formed with pairwise exponents, or NULL.  `chunks`, `ntfix`: chunk_grid() of the batch.
int gla_bwd_chunk(const void* q, const void* k, const void* v, const void* g, const void* dout, const void* hT,
                  const void* dhT, const int* wide, void* dq, void* dk, void* dv, float* dg, const int64_t* offsets,
                  const int64_t* indices, int64_t chunks, int ntfix, int qkv_dtype, int gate_dtype, bool head_gates, int64_t T,
                  int64_t H, int64_t K, int64_t V, float scale, hipStream_t st);
