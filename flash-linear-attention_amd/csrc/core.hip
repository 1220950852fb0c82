// ABI version, error strings and the host-side integer chunk bookkeeping.
#include "fla_common.h"

extern "C" int fla_abi_version(void) { return FLA_ABI_VERSION; }

extern "C" const char* fla_error_string(int code) {
  switch (code) {
    case FLA_OK: return "success";
    case FLA_E_INVALID: return "fla_hip: invalid argument (null pointer, negative size or inconsistent shapes)";
    case FLA_E_UNSUPPORTED: return "fla_hip: shape, dtype or chunk size not supported by the gfx950 kernels";
    case FLA_E_ALIGNMENT: return "fla_hip: pointer or row pitch not aligned for vector access";
    case FLA_E_SCRATCH: return "fla_hip: input larger than the static scratch buffer of the allocation-free entry point";
    default: break;
  }
  if (code > 0) return hipGetErrorString((hipError_t)code);
  return "fla_hip: unknown error code";
}

// One row (sequence, chunk-in-sequence) per chunk, sequences in order, and the
// exclusive prefix sum of per-sequence chunk counts.  Same result as the
// reference's host construction (fla/ops/gla/chunk.py:1323-1330;
// fla/ops/common/chunk_h.py:274-279), without a device round trip.
extern "C" int64_t fla_count_chunks(const int64_t* offsets, int64_t n_seqs, int64_t chunk_size) {
  if (!offsets || n_seqs < 0 || chunk_size <= 0) return FLA_E_INVALID;
  int64_t total = 0;
  for (int64_t n = 0; n < n_seqs; ++n) {
    int64_t len = offsets[n + 1] - offsets[n];
    if (len < 0) return FLA_E_INVALID;
    total += fla_cdiv(len, chunk_size);
  }
  return total;
}

extern "C" int fla_prepare_chunk_indices(const int64_t* offsets, int64_t n_seqs, int64_t chunk_size,
                                         int64_t* indices_out, int64_t* chunk_offsets_out) {
  if (!offsets || n_seqs < 0 || chunk_size <= 0) return FLA_E_INVALID;
  int64_t row = 0;
  for (int64_t n = 0; n < n_seqs; ++n) {
    int64_t len = offsets[n + 1] - offsets[n];
    if (len < 0) return FLA_E_INVALID;
    if (chunk_offsets_out) chunk_offsets_out[n] = row;
    int64_t nc = fla_cdiv(len, chunk_size);
    for (int64_t c = 0; c < nc; ++c, ++row) {
      if (indices_out) {
        indices_out[2 * row] = n;
        indices_out[2 * row + 1] = c;
      }
    }
  }
  if (chunk_offsets_out) chunk_offsets_out[n_seqs] = row;
  return FLA_OK;
}

// Where a sequence is cut.  A scan's time is its longest workgroup's chunks times the chunk period once every workgroup
// has a CU of its own, so the segments are as short as 256 CUs allow (GLA forward of 16 heads x 8192 tokens, K = V = 128:
// 4, 8, 16 and 32 segments 112, 81, 88 and 104 us, uncut 291).  The first pass gets about as many workgroups as there are
// CUs: 1, 2 and 4 sub-blocks per segment of that forward 97, 80 and 83 us, of one of 64 pairs in two segments 177, 141 and
// 126 us (uncut 156).  The delta rule's first pass costs as much as its scan (it walks K + V columns instead of V) and its
// fold 2.2 us per segment: segments of at least 0.7 sqrt(chunks) (forward of 128 chunks, 4 heads, in segments of 4, 8 and 16
// chunks 92, 71 and 77 us, uncut 174; training step of 64 chunks, 8 heads, in 4 and 8 187 and 165 us, uncut 251).
//
// Whether cutting pays is the longest sequence's chunk periods against those of a segment in the scan and in the first pass
// and the launches ahead of the scan, fitted to the times below (K = V = 128, uncut / cut in us, launches replayed from a
// graph; packed batches back to back).  The busier the CUs (triples of sequence, head and slab), the less a cut gains.
// (The training steps of GLA were read with a forward that also wrote k^ and the score tiles and with per-key gates: today's gain
// a little less from a cut than these figures say.)
//   GLA: one sequence of 16 heads, 12 and 16 chunks 37.7 / 36.1 and 46.0 / 37.2; four, 16, 20 and 24 chunks 50.4 / 53.5,
//     59.3 / 61.6 and 68.4 / 65.8, their training steps 145 / 162, 198 / 202 and 237 / 237.
//   Delta rule, forward: the uncut scan takes 1.1 us a chunk (64 key channels: 0.75), and a cut pays for: the chunks of a segment
//     in the scan, more where its segments no longer fit in slabs of 32 columns; the same in the first pass, whose workgroups of
//     128 of the K + V columns take as many rounds as 256 CUs need for them; the fold's steps; what the first pass loads and
//     stores; the launches.  K = V = 128: 4 heads, 24, 28 and 32 chunks 35.7 / 37.3, 40.1 / 40.4 and 44.5 / 42.1; 8 heads 35.8 /
//     38.6, 40.2 / 41.6 and 44.6 / 43.2; 12 heads, 36 and 40 chunks 51.0 / 53.5 and 55.7 / 53.8; 16 heads, 32, 36, 40 and 48
//     47.6 / 52.1, 52.3 / 56.1, 57.0 / 56.7 and 65.5 / 60.0; 24 heads, 44 and 52 63.8 / 64.6 and 73.1 / 70.9; 32 heads, 56, 60 and
//     68 80.3 / 83.6, 85.3 / 85.9 and 95.2 / 93.4; packed, 16 heads, 54, 94 and 77 chunks 132 / 146, 80 and 171 215 / 157.  128 keys,
//     64 values (the first pass as long as with 128, the scan with half the slabs): 16 heads, 24, 32 and 36 chunks 37.0 / 41.3,
//     46.8 / 47.0 and 52.0 / 50.1, 48 in two rounds 65.2 / 68.0; 32 heads, 32, 48 and 64 49.8 / 68.0, 69.3 / 80.2 and 89.0 / 91.7.
//     64 keys, 128 values: 16 heads, 28 and 36 32.4 / 34.5 and 39.5 / 38.5.  K = V = 64: 8 heads, 20 and 24 24.3 / 25.4 and 27.3 /
//     25.9; 16 heads, 24 28.7 / 28.3; 32 heads, 28, 36 and 40 35.3 / 37.2, 42.2 / 42.4 and 45.9 / 42.8; 64 heads, 64 73.1 / 76.3.
//   Delta rule, a forward that keeps its intermediates and its backward (training steps): the same terms over both directions; a
//     transition of every segment is formed.  K = V = 128: 4 heads, 23 and 24 chunks 87.0 / 89.0 and 89.3 / 88.5; 8 heads, 24 and
//     28 92.1 / 92.3 and 102.9 / 97.9; 12 heads, 36 and 40 132.8 / 141.6 and 143.5 / 142.8; 16 heads, 40, 44, 48 and 56 162 / 169,
//     172 / 178, 182 / 181 and 203 / 190; 24 heads, 72 and 80 311 / 323 and 350 / 340; 32 heads, 96 494 / 499; packed, 8 heads, 20, 63,
//     49 and 26 chunks 243 / 250.  K = V = 64: 8 heads, 20 and 24 63.1 / 61.3 and 70.9 / 63.1; 32 heads, 48 152 / 135.
//   The plain scan of chunk_simple_gla's forward takes half as long per chunk as the GLA kernel and fills the chip with half
//     the pairs (slabs of 32 columns).  K = V = 128: 4 heads, 12 and 16 chunks 16.5 / 18.1 and 20.6 / 18.8; 12 heads, 18 and 20 23.8
//     / 24.2 and 25.8 / 24.6; 16 heads, 20, 22 and 24 25.1 / 27.1, 27.1 / 27.5 and 29.2 / 27.8; 32 heads, 32, 36 and 40 38.4 / 39.6,
//     42.4 / 43.3 and 46.4 / 44.1; four sequences of 16, 64 and 128 76.8 / 87.9 and 159 / 164; packed, 16 heads, 54, 94 and 77
//     chunks 101 / 89.  64 keys, 128 values: 16 heads, 24 and 28 22.3 / 22.6 and 25.2 / 23.3.
//   The reverse scan of GLA's backward forms the state gradient alone, in half the time per chunk, and leaves every pass of the
//     backward behind it alone, so only what it saves itself counts (whole training steps; per-key gates, K = V = 128): 4
//     heads, 16, 24 and 32 chunks 63.5 / 67.3, 72.1 / 72.3 and 77.3 / 73.8; 8 heads, 24, 32 and 64 chunks 75.3 / 77.1, 84.0 /
//     83.1 and 118 / 106; 16 heads, 32, 48 and 64 chunks 99.2 / 101.6, 137.0 / 135.5 and 155.7 / 148.7; 24 heads, 64 and 96
//     chunks 225 / 229 and 340 / 336; two sequences of 16 heads, 32, 64 and 96 chunks 138 / 152, 286 / 291 and 400.0 / 398.5.
//     Per-head gates, K = V = 64: 8, 16, 32, 64, 96 and 128 heads, 24 chunks 52.9 / 51.5, 59.5 / 58.9, 65.9 / 66.9, 85.4 / 89.9,
//     107.8 / 115.1 and 120.8 / 131.5, 48 chunks 72.1 / 61.2, 79.5 / 68.9, 97.7 / 89.8, 137.4 / 138.9, 196.5 / 202.1 and 262 / 267.
extern "C" int fla_scan_split(const int64_t* offsets, int64_t N, int64_t T, int64_t H, int32_t slabs, int32_t reverse,
                              int32_t kind, fla_split* out, int32_t* seg_table, int32_t* sub_table, int32_t* sub_base) {
  constexpr int64_t kCUs = 256, kChunk = 64, kPassWorkgroups = 256;
  const bool keys64 = kind & FLA_SCAN_KEYS_64;
  kind &= ~FLA_SCAN_KEYS_64;
  const bool delta = kind == FLA_SCAN_DELTA || kind == FLA_SCAN_DELTA_KEPT;
  int64_t min_seg = 4;
  if (!out || kind < FLA_SCAN_GLA || kind > FLA_SCAN_GLA_GRADIENT || (keys64 && !delta)) return 0;
  if (N <= 0 || H <= 0 || slabs <= 0 || N > 65536) return 0;
  auto chunks_of = [&](int64_t n) { return offsets ? fla_cdiv(offsets[n + 1] - offsets[n], kChunk) : fla_cdiv(T, kChunk); };
  int64_t longest = 0, total = 0;
  for (int64_t n = 0; n < N; ++n) {
    const int64_t c = chunks_of(n);
    longest = c > longest ? c : longest;
    total += c;
  }
  if (delta)
    while (100 * min_seg * min_seg < 49 * longest) ++min_seg;
  const int64_t room = kCUs / (H * slabs);   // segments the chip holds at once
  if (longest == 0 || room < 2 || N > room || longest > 0x7fffffff / kChunk) return 0;
  // the shortest segment with which all of them fit
  auto segments = [&](int64_t len) {
    int64_t s = 0;
    for (int64_t n = 0; n < N; ++n) {
      const int64_t c = fla_cdiv(chunks_of(n), len);
      s += c > 0 ? c : 1;
    }
    return s;
  };
  int64_t seg = fla_cdiv(total, room);
  seg = seg < min_seg ? min_seg : seg;
  while (segments(seg) > room) ++seg;
  const int64_t triples = fla_cdiv(total, longest) * H * slabs;   // sequences of other lengths: as many of the longest
  const int64_t L = longest, segs = segments(seg), steps = fla_cdiv(L, seg) - 1;
  // the delta rule's first pass: workgroups of 128 of the K + V columns of a (segment, head); and the slabs its scan then has
  const int64_t pass = H * (segs - (kind == FLA_SCAN_DELTA_KEPT ? 0 : N)) * fla_cdiv(slabs + (keys64 ? 1 : 2), 2);
  const int64_t rounds = fla_cdiv(pass, kCUs), wide = 2 * segs * H * slabs > kCUs ? 1 : 0;
  bool pays;
  switch (kind) {   // the scan of whole sequences against that of the segments and what stands ahead of it, in twentieths of a chunk
                    // of the former (the last two in fifths and elevenths): see above
    case FLA_SCAN_DELTA:
      pays = keys64 ? 20 * L >= seg * (3 + 50 * rounds + 12 * wide) + 12 * steps + pass * 189 / 256 + 140
                    : 20 * L >= seg * (2 + 35 * rounds + 20 * wide) + 34 * steps + pass * 112 / 256 + 170;
      break;
    case FLA_SCAN_DELTA_KEPT:
      pays = keys64 ? 20 * L >= seg * (1 + 54 * rounds + 29 * wide) + 23 * steps + 57
                    : 20 * L >= seg * (6 * rounds + 55 * wide) + pass * 165 / 256 + 426;
      break;
    case FLA_SCAN_SIMPLE:
      pays = 5 * L >= 9 * seg + (triples < 8 ? 28 : triples < 32 ? 12 + 2 * triples : 52 + (triples < 64 ? triples : 64) * 3 / 4);
      break;
    case FLA_SCAN_GLA_GRADIENT: pays = 11 * (L - seg) >= 165 + 3 * triples; break;
    default: pays = 5 * L >= 7 * seg + 31;
  }
  if (steps == 0 || !pays) return 0;
  const int64_t formed = H * (segs - N);   // (segment, head) pairs the first pass works on
  int64_t ratio = formed > 0 ? kPassWorkgroups / formed : 1;
  ratio = ratio > seg / 2 ? seg / 2 : ratio;
  if (delta) ratio = 1;
  ratio = ratio < 1 ? 1 : ratio;
  const int64_t sub = fla_cdiv(seg, ratio);
  ratio = fla_cdiv(seg, sub);
  out->sub_chunks = (int32_t)sub;
  out->ratio = (int32_t)ratio;
  out->reserved = 0;
  out->seg_table = out->sub_table = out->sub_base = nullptr;
  auto subs_of = [&](int64_t n) {
    const int64_t s = fla_cdiv(chunks_of(n), sub);
    return s > 0 ? s : 1;
  };
  if (!offsets) {
    out->nsub = (int32_t)subs_of(0);
    out->nseg = (int32_t)fla_cdiv(out->nsub, ratio);
    out->slots = (int32_t)(out->nsub * N);
    return out->nseg > 1;
  }
  // packed batch: the tables list the segments in rounds, so that those of the longest sequences come first
  int64_t nseg = 0, nsub = 0, base = 0, most = 0;
  for (int64_t n = 0; n < N; ++n) {
    const int64_t s = subs_of(n), g = fla_cdiv(s, ratio);
    if (sub_base) sub_base[n] = (int32_t)base;
    base += s;
    nseg += g;
    most = g > most ? g : most;
    // (a forward that keeps its intermediates forms the last segment's transition too, for its backward)
    const int64_t lo = reverse ? ratio : 0, hi = reverse || kind == FLA_SCAN_DELTA_KEPT ? s : (g - 1) * ratio;
    for (int64_t j = lo; j < hi; ++j, ++nsub)
      if (sub_table) {
        sub_table[2 * nsub] = (int32_t)n;
        sub_table[2 * nsub + 1] = (int32_t)j;
      }
  }
  if (sub_base) sub_base[N] = (int32_t)base;
  if (seg_table) {
    int64_t row = 0;
    // whole segments before the shorter last pieces of the sequences
    for (int pass = 0; pass < 2; ++pass)
      for (int64_t n = 0; n < N; ++n) {
        const int64_t g = fla_cdiv(subs_of(n), ratio);
        for (int64_t s = pass ? g - 1 : 0; s < (pass ? g : g - 1); ++s, ++row) {
          seg_table[2 * row] = (int32_t)n;
          seg_table[2 * row + 1] = (int32_t)s;
        }
      }
  }
  out->nseg = (int32_t)nseg;
  out->nsub = (int32_t)nsub;
  out->slots = (int32_t)base;
  return most > 1;
}
