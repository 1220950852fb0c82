// gdr_bwd_scan.hip: the reverse state scan of the gated delta rule backward from the tiles the forward left, K in {64, 128}.
#pragma once
#include "fla_common.h"

// AT, Aqk: the packed tiles Tu and Aqk, [chunks, H, 10, 16, 16].  dv2 [rows, H, V] and dhtf (the gradient of the state leaving
// every chunk, FLA_H_FRAGMENT_T) are written; dh0 (fp32) unless NULL.  split: cut sequences (split->decays: the transposed
// transitions the forward left), or NULL.
int gdr_bwd_scan(const void* q, const void* k, const void* AT, const void* Aqk, const float* g_cumsum, const void* dout,
                 const float* dht, void* dv2, void* dhtf, float* dh0, const int64_t* offsets, const int64_t* chunk_offsets,
                 const fla_split* split, int qkv_dtype, int64_t T, int64_t H, int64_t K, int64_t V, int64_t N, float scale,
                 hipStream_t st);
