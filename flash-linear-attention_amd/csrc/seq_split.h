// Sequences cut into segments for the serial scans.
//
// A scan over chunks gives one workgroup to a (sequence, head, value slab), so a launch with few (sequence, head)
// pairs and long sequences leaves most CUs without one: a single prompt of 16 heads occupies 32 of 256.  The state
// recurrence is linear, so a sequence can be cut into segments that are scanned side by side once the state entering
// each is known:
//   1. a first pass forms, for every sub-block of `sub_chunks` chunks ahead of the last segment, what the sub-block adds
//      to a zero state and its transition (GLA: one decay per key channel; the delta rule: a K x K matrix);
//   2. a small launch folds them, sub-block after sub-block, into the state entering every segment;
//   3. the scan runs as before with (sequence, segment) in the place of a sequence.
// A segment is `ratio` sub-blocks: the first pass has no output to write and wants more, shorter pieces than the scan.
#pragma once
#include "chunk_common.h"

namespace {

struct SplitView {
  int sub_chunks = 0;               // chunks per sub-block
  int ratio = 0;                    // sub-blocks per segment; 0: sequences are not cut
  int nseg = 0;                     // equal-length sequences: segments of each
  int nsub = 0;                     //   ... and sub-blocks
  const int32_t* seg_table = nullptr;  // packed batch: rows (sequence, segment), those of the longest sequences first
  const int32_t* sub_table = nullptr;  //   rows (sequence, sub-block) of the first pass
  const int32_t* sub_base = nullptr;   //   [N+1] first sub-block of a sequence
  const float* states = nullptr;    // [sub-blocks, H, K, V]: the entering states sit in the slots segment_slot() names
};

inline SplitView split_view(const fla_split* s) {
  SplitView v;
  if (s) {
    v.sub_chunks = s->sub_chunks;
    v.ratio = s->ratio;
    v.nseg = s->nseg;
    v.nsub = s->nsub;
    v.seg_table = s->seg_table;
    v.sub_table = s->sub_table;
    v.sub_base = s->sub_base;
    v.states = s->states;
  }
  return v;
}

inline int check_split(const fla_split* s, const int64_t* offsets) {
  FLA_REQUIRE(s->sub_chunks > 0 && s->ratio > 0 && s->nseg > 0 && s->nsub > 0 && s->states, FLA_E_INVALID);
  if (offsets) FLA_REQUIRE(s->seg_table && s->sub_table && s->sub_base, FLA_E_INVALID);
  else FLA_REQUIRE(!s->seg_table && !s->sub_table && !s->sub_base, FLA_E_INVALID);
  FLA_REQUIRE((uintptr_t)s->states % 16 == 0 && (uintptr_t)s->decays % 16 == 0, FLA_E_ALIGNMENT);
  return FLA_OK;
}

// Sub-blocks of a sequence of `chunks` chunks (an empty sequence keeps one slot: its state passes through it).
FLA_DEVICE int64_t split_nsub(const SplitView& v, int64_t chunks) {
  const int64_t n = ((uint32_t)chunks + (uint32_t)v.sub_chunks - 1) / (uint32_t)v.sub_chunks;   // (below 2^31)
  return n > 0 ? n : 1;
}

// What one scan workgroup walks: a sequence, or one segment of it.
struct ScanSpan {
  int n;                // sequence
  SeqSpan sp;           // its token rows
  int64_t nchunks;
  int64_t chunk0;       // global index of its first chunk
  int64_t slot;         // sub-block slot that holds the state entering it (cut sequences)
  bool first, last;     // first / last piece of its sequence
};

// The slot of the state entering segment s: scanning forwards, that of the segment's first sub-block; backwards (the
// state gradient entering it from the right), that of its last one.
template <bool REVERSE>
FLA_DEVICE ScanSpan scan_span(const SplitView& v, int64_t i, const int64_t* seq_order, const int64_t* offsets,
                              const int64_t* chunk_offsets, int64_t T) {
  ScanSpan r;
  if (v.ratio == 0) {
    r.n = seq_order ? (int)seq_order[i] : (int)i;
    r.sp = seq_span(offsets, r.n, T);
    r.nchunks = (r.sp.len + BT - 1) / BT;
    r.chunk0 = chunk_offsets ? chunk_offsets[r.n] : (int64_t)r.n * ((T + BT - 1) / BT);
    r.slot = 0;
    r.first = r.last = true;
    return r;
  }
  int s;
  if (v.seg_table) {
    r.n = v.seg_table[2 * i];
    s = v.seg_table[2 * i + 1];
  } else {
    r.n = (int)((uint32_t)i / (uint32_t)v.nseg);
    s = (int)((uint32_t)i % (uint32_t)v.nseg);
  }
  const SeqSpan whole = seq_span(offsets, r.n, T);
  const int64_t all = (whole.len + BT - 1) / BT;
  const int64_t seg = (int64_t)v.sub_chunks * v.ratio, c0 = s * seg;
  r.first = s == 0;
  r.last = c0 + seg >= all;
  r.nchunks = r.last ? all - c0 : seg;
  if (r.nchunks < 0) r.nchunks = 0;
  r.sp.bos = whole.bos + c0 * BT;
  r.sp.len = r.last ? whole.len - c0 * BT : seg * BT;
  if (r.sp.len < 0) r.sp.len = 0;
  r.chunk0 = (chunk_offsets ? chunk_offsets[r.n] : (int64_t)r.n * ((T + BT - 1) / BT)) + c0;
  const int64_t nsub = split_nsub(v, all);
  const int64_t base = v.sub_base ? v.sub_base[r.n] : (int64_t)r.n * v.nsub;
  const int64_t end = (int64_t)(s + 1) * v.ratio;
  r.slot = base + (REVERSE ? (end < nsub ? end : nsub) - 1 : (int64_t)s * v.ratio);
  return r;
}

// Item i of a first pass from right to left over segments of one sub-block: every segment but a sequence's first.
FLA_DEVICE ScanSpan pass_span(const SplitView& v, int64_t i, int per_seq, const int64_t* offsets, const int64_t* chunk_offsets,
                              int64_t T) {
  ScanSpan r;
  int s;
  if (v.sub_table) {
    r.n = v.sub_table[2 * i];
    s = v.sub_table[2 * i + 1];
  } else {
    r.n = (int)((uint32_t)i / (uint32_t)per_seq);
    s = (int)((uint32_t)i % (uint32_t)per_seq) + 1;
  }
  const SeqSpan whole = seq_span(offsets, r.n, T);
  const int64_t all = (whole.len + BT - 1) / BT, c0 = (int64_t)s * v.sub_chunks;
  r.first = false;
  r.last = c0 + v.sub_chunks >= all;
  r.nchunks = r.last ? all - c0 : v.sub_chunks;
  r.sp.bos = whole.bos + c0 * BT;
  r.sp.len = r.last ? whole.len - c0 * BT : (int64_t)v.sub_chunks * BT;
  r.chunk0 = (chunk_offsets ? chunk_offsets[r.n] : (int64_t)r.n * ((T + BT - 1) / BT)) + c0;
  r.slot = (v.sub_base ? v.sub_base[r.n] : (int64_t)r.n * v.nsub) + s;
  return r;
}

}  // namespace

// gla_split.hip: the two launches ahead of a GLA scan over cut sequences.  Forward: a = k, b = v, g = the gates, init the
// initial states.  Reverse: a = the gated queries, b = do, g = the chunk decays, init the gradients of the final states.
int gla_split_states(const void* a, const void* b, const void* g, const float* init, const fla_split* split, bool head_gates,
                     bool reverse, bool logits, float gate_inv_norm, float gate_clamp_min, float scale,
                     const int64_t* offsets, const int64_t* chunk_offsets, int qkv_dtype, int gate_dtype, int64_t T,
                     int64_t H, int64_t K, int64_t V, int64_t N, hipStream_t st);

// gdr_split.hip: the two launches ahead of a delta-rule scan over cut sequences (segments of one sub-block).
int gdr_split_states(const void* k, const void* v, const void* AT, const float* g_cumsum, const float* k_rstd, const float* init,
                     const fla_split* split, const int64_t* offsets, const int64_t* chunk_offsets, int qkv_dtype, int64_t T,
                     int64_t H, int64_t K, int64_t V, int64_t N, hipStream_t st);
// ... and, backwards, the fold alone: `states` holds what every segment adds to a zero gradient, split->decays the transposed
// transitions the forward left, init the gradients of the final states.
int gdr_split_fold_reverse(const float* init, const fla_split* split, const int64_t* offsets, int64_t T, int64_t H, int64_t K,
                           int64_t V, int64_t N, hipStream_t st);
