// The two launches ahead of a GLA scan over sequences cut into segments (seq_split.h): what every sub-block adds to a
// zero state, and the fold of these into the states entering the segments.
//
// Forward: with E_t the sum of the log-gates behind token t inside its chunk, a chunk takes the accumulators to
//   S <- e^{E of the whole chunk} S + sum_t (k_t e^{E_t}) v_t^T     (the decay per key row),
// and the sub-block multiplies the state entering it by the product of its chunks' decays.  The 16-bit k e^{E} is that of
// the scan itself, and decays further are applied in fp32: with E over the whole sub-block, early keys of an fp16 call
// would fall into the subnormal numbers (34 % of the state behind 512 tokens of -0.05 of which the last 280 have no key;
// it took 86.5 us instead of 88.6 for the forward of one sequence of 8192 tokens, 16 heads).
// Backward (the state gradient, right to left): S' = sum_c (prod_{earlier c'} e^{G_last,c'}) (q e^{G})_c^T do_c from the
// gated queries and chunk decays the forward kept, the accumulators scaled in the same way.
//
// One workgroup of four waves per (sub-block, head) holds the whole K x V tile (a wave a quarter of it), reads every
// operand once and runs two to a CU: 64 KB (GLA forward, fp32 gates) of loads per chunk against 64 matrix instructions, so
// it is bound by the loads: 28 us for 16 heads x 7168 tokens, K = V = 128 (117 MB in, 15 MB out: 4.7 TB/s, a large copy
// moves 5.1).  The fold behind it takes 6 us, the scan over 8 segments 50 us instead of 291 us over the whole sequences.
#include "gla_fused_staging.h"
#include "seq_split.h"

namespace {

struct SplitPassParams {
  const void* a;        // forward: k; backward: the gated queries q e^{G}; [rows, H, K]
  const void* b;        // forward: v; backward: do; [rows, H, V]
  const void* g;        // forward: log-gates (per key channel, or fp32 per head); backward: chunk decays fp32 [chunks, H, K]
  float* states;        // [sub-blocks, H, K, V]
  float* decays;        // [sub-blocks, H, K]
  const int64_t* offsets;
  const int64_t* chunk_offsets;
  SplitView split;
  int64_t T;
  int H, per_seq;       // equal-length sequences: sub-blocks of the pass per sequence
  float gate_inv_norm, gate_clamp_min;
};

enum { kPassKeyGates = 0, kPassHeadGates = 1, kPassGateLogits = 2, kPassReverse = 3 };

template <typename T, typename GT, int K, int V, int MODE>
__global__ __launch_bounds__(256, 2) void gla_split_pass_kernel(SplitPassParams p) {
  typedef typename Elem<T>::v8 v8;
  constexpr bool REV = MODE == kPassReverse;
  constexpr float LOG2E = 1.4426950408889634f;
  constexpr int LDA = K + 8, LDB = V + 8;
  constexpr int CPL = K / 16;                  // key channels per lane: 8 (K = 128) or 4 (K = 64)
  constexpr int NA = K / 64, NB = V / 64;      // 32 x 32 accumulator tiles per wave: NA x NB
  constexpr int BPR = V / 8;                   // 16-byte pieces of a row of b
  constexpr int NPB = BT * BPR / 256;          // ... per thread
  typedef T kvec __attribute__((ext_vector_type(CPL)));
  typedef GT gvec __attribute__((ext_vector_type(CPL)));
  __shared__ __attribute__((aligned(16))) T sA[2][BT * LDA];
  __shared__ __attribute__((aligned(16))) T sB[2][BT * LDB];
  __shared__ __attribute__((aligned(16))) float sD[2][K];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H;
  const int hh = (int)(blockIdx.x % (uint32_t)H);
  const int64_t i = blockIdx.x / (uint32_t)H;
  int n, j;
  if (p.split.sub_table) {
    n = p.split.sub_table[2 * i];
    j = p.split.sub_table[2 * i + 1];
  } else {
    n = (int)((uint32_t)i / (uint32_t)p.per_seq);
    j = (int)((uint32_t)i % (uint32_t)p.per_seq) + (REV ? p.split.ratio : 0);
  }
  const SeqSpan whole = seq_span(p.offsets, n, p.T);
  const int64_t all = (whole.len + BT - 1) / BT;
  const int64_t c0 = (int64_t)j * p.split.sub_chunks;
  const int64_t slot = (p.split.sub_base ? p.split.sub_base[n] : (int64_t)n * p.split.nsub) + j;
  const int nc = (int)(all - c0 < p.split.sub_chunks ? all - c0 : p.split.sub_chunks);
  const int64_t row0 = whole.bos + c0 * BT;
  const int64_t chunk0 = (p.chunk_offsets ? p.chunk_offsets[n] : (int64_t)n * ((p.T + BT - 1) / BT)) + c0;
  // rows of the sub-block: whole chunks except for the last one of a sequence, which only the reverse pass meets
  const int64_t rem = whole.len - c0 * BT;
  const int rows = (int)(rem < (int64_t)nc * BT ? rem : (int64_t)nc * BT);

  // A lane's operands of one chunk: four rows x CPL channels of a (16 row groups in the lanes of a DPP row, so that the
  // sums over time are DPP row scans), NPB 16-byte pieces of b.
  const int rg = lane & 15, kc = wave * (K / 4) + (lane >> 4) * CPL;
  const uint32_t apitch = (uint32_t)H * K * (uint32_t)sizeof(T), bpitch = (uint32_t)H * V * (uint32_t)sizeof(T);
  const char* pa = (const char*)p.a + ((row0 * H + hh) * (int64_t)K + kc) * (int64_t)sizeof(T);
  const char* pb = (const char*)p.b + ((row0 * H + hh) * (int64_t)V) * (int64_t)sizeof(T);
  const char* pg = REV ? (const char*)p.g + ((chunk0 * H + hh) * (int64_t)K) * 4
                       : MODE == kPassHeadGates ? (const char*)p.g + (row0 * H + hh) * 4
                                                : (const char*)p.g + ((row0 * H + hh) * (int64_t)K + kc) * (int64_t)sizeof(GT);
  const uint32_t gpitch = REV ? 0u : MODE == kPassHeadGates ? (uint32_t)H * 4u : (uint32_t)H * K * (uint32_t)sizeof(GT);
  uint32_t offb[NPB];
#pragma unroll
  for (int r = 0; r < NPB; ++r) offb[r] = (uint32_t)((tid + 256 * r) / BPR) * bpitch + (uint32_t)(tid % BPR) * 16u;
  struct Regs {
    kvec a[4];
    gvec g[MODE == kPassHeadGates || REV ? 1 : 4];
    float gh[MODE == kPassHeadGates ? 4 : 1];
    v8 b[NPB];
  } R;
  auto load = [&](int c) __attribute__((always_inline)) {
    const char* ca = pa + (int64_t)c * BT * apitch;
    const char* cb = pb + (int64_t)c * BT * bpitch;
    // reverse: rows past the end of the sequence are read from its last row and masked in b
    const int lastrow = rows - c * BT < BT ? rows - c * BT - 1 : BT - 1;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = REV ? min(rg * 4 + r, lastrow) : rg * 4 + r;
      R.a[r] = *(const kvec*)(ca + (uint32_t)row * apitch);
      if constexpr (MODE == kPassHeadGates) R.gh[r] = *(const float*)(pg + (int64_t)c * BT * gpitch + (uint32_t)row * gpitch);
      else if constexpr (!REV) R.g[r] = *(const gvec*)(pg + (int64_t)c * BT * gpitch + (uint32_t)row * gpitch);
    }
#pragma unroll
    for (int r = 0; r < NPB; ++r) {
      const uint32_t lim = (uint32_t)lastrow * bpitch + (uint32_t)(tid % BPR) * 16u;
      R.b[r] = *(const v8*)(cb + (REV ? min(offb[r], lim) : offb[r]));
    }
    if constexpr (REV) R.gh[0] = *(const float*)(pg + ((int64_t)c * H * K + (tid & (K - 1))) * 4);
  };
  float carry[CPL];   // forward: log2 decay of the chunks so far; backward: [0] the decay itself, of channel tid
#pragma unroll
  for (int jx = 0; jx < CPL; ++jx) carry[jx] = 0.f;
  [[maybe_unused]] const float clamp2 = p.gate_clamp_min * LOG2E;
  auto stage = [&](int c, int buf) __attribute__((always_inline)) {
    if constexpr (REV) {
#pragma unroll
      for (int r = 0; r < 4; ++r) *(kvec*)&sA[buf][(rg * 4 + r) * LDA + kc] = R.a[r];
      if (tid < K) sD[buf][tid] = R.gh[0];
    } else {
      // suffix sums over the rows of the chunk: in the lane from the last row up, then across the row groups
      float E[4][CPL];
      if constexpr (MODE == kPassHeadGates) {
        float run = 0.f, Es[4];
#pragma unroll
        for (int r = 3; r >= 0; --r) {
          Es[r] = run;
          run = fmaf(R.gh[r], LOG2E, run);
        }
        const float suf = row_suffix16(run), later = dpp_f32<0x101>(suf);   // row_shl:1, the later row groups
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int jx = 0; jx < CPL; ++jx) E[r][jx] = Es[r] + later;
        carry[0] += suf;                   // (lanes rg == 0, the sum over the whole chunk)
        if (rg == 0) {
          const float d = __builtin_amdgcn_exp2f(suf);
#pragma unroll
          for (int jx = 0; jx < CPL; ++jx) sD[buf][kc + jx] = d;
        }
      } else {
#pragma unroll
        for (int jx = 0; jx < CPL; ++jx) {
          float run = 0.f;
#pragma unroll
          for (int r = 3; r >= 0; --r) {
            E[r][jx] = run;
            if constexpr (MODE == kPassGateLogits) run += log2_sigmoid_gate((float)R.g[r][jx], p.gate_inv_norm, clamp2);
            else run = fmaf((float)R.g[r][jx], LOG2E, run);
          }
          // the later row groups' sum from the lane that has it: as a difference it would be lost behind a gate that
          // resets the state (-1e30), and NaN behind -inf
          const float suf = row_suffix16(run), later = dpp_f32<0x101>(suf);
#pragma unroll
          for (int r = 0; r < 4; ++r) E[r][jx] += later;
          carry[jx] += suf;   // (lanes rg == 0, the sum over the whole chunk)
          if (rg == 0) sD[buf][kc + jx] = __builtin_amdgcn_exp2f(suf);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        kvec x;
        if constexpr (MODE == kPassHeadGates) {
          const float e = __builtin_amdgcn_exp2f(E[r][0]);
#pragma unroll
          for (int jx = 0; jx < CPL; ++jx) x[jx] = (T)((float)R.a[r][jx] * e);
        } else {
#pragma unroll
          for (int jx = 0; jx < CPL; ++jx) x[jx] = (T)((float)R.a[r][jx] * __builtin_amdgcn_exp2f(E[r][jx]));
        }
        *(kvec*)&sA[buf][(rg * 4 + r) * LDA + kc] = x;
      }
    }
#pragma unroll
    for (int r = 0; r < NPB; ++r) {
      const int row = (tid + 256 * r) / BPR;
      v8 x = R.b[r];
      if (REV && c * BT + row >= rows) {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = (T)0.f;
      }
      *(v8*)&sB[buf][row * LDB + (tid % BPR) * 8] = x;
    }
  };

  const int rw = wave >> 1, cw = wave & 1;     // this wave's rows rw K/2 .., columns cw V/2 ..
  f32x16 acc[NA][NB];
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[a][b] = zero16();
  // Two tile buffers: the tiles of a chunk are written while slower waves still multiply those of the one before it,
  // and the barrier that publishes them says that everybody is done with the buffer the next chunk takes.
  load(REV ? nc - 1 : 0);
  for (int i = 0; i < nc; ++i) {
    const int c = REV ? nc - 1 - i : i, buf = i & 1;
    stage(c, buf);
    if (i + 1 < nc) load(REV ? c - 1 : c + 1);
    lds_barrier();
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int q4 = 0; q4 < 4; ++q4) {
        const f32x4 d = *(const f32x4*)&sD[buf][rw * (K / 2) + a * 32 + 8 * q4 + 4 * (lane >> 5)];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int b = 0; b < NB; ++b) acc[a][b][4 * q4 + e] *= d[e];
      }
    if (REV && tid < K) carry[0] = i == 0 ? sD[buf][tid] : carry[0] * sD[buf][tid];
#pragma unroll
    for (int ts = 0; ts < BT; ts += 16) {
      v8 fb[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) fb[b] = frag32_tr<T>(sB[buf], LDB, cw * (V / 2) + b * 32, ts, lane);
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        const v8 fa = frag32_tr<T>(sA[buf], LDA, rw * (K / 2) + a * 32, ts, lane);
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[a][b] = Elem<T>::mfma32(fa, fb[b], acc[a][b]);
      }
    }
  }
  float* out = p.states + (slot * H + hh) * (int64_t)(K * V);
#pragma unroll
  for (int a = 0; a < NA; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        out[(rw * (K / 2) + a * 32 + c32_row(r, lane)) * V + cw * (V / 2) + b * 32 + (lane & 31)] = acc[a][b][r];
  float* dec = p.decays + (slot * H + hh) * (int64_t)K;
  if constexpr (REV) {
    if (tid < K) dec[tid] = carry[0];
  } else if (rg == 0) {
#pragma unroll
    for (int jx = 0; jx < CPL; ++jx) dec[kc + jx] = __builtin_amdgcn_exp2f(carry[MODE == kPassHeadGates ? 0 : jx]);
  }
}

// The fold: a thread carries four adjacent value columns of one key row through the sub-blocks of its sequence,
//   h <- D_j h + S_j     (backwards: D_j h + scale S_j),
// and leaves h where a segment begins, over the sub-block's own S (read a moment before).  Loads of eight sub-blocks
// are in flight at a time; the slots of one (head, key row) are 64 KB apart, so the launch is a handful of dependent
// memory latencies whatever the length.
template <bool REVERSE>
__global__ __launch_bounds__(256) void gla_split_fold_kernel(float* __restrict__ states, const float* __restrict__ decays,
                                                             const float* __restrict__ init, float scale,
                                                             SplitView split,
                                                             const int64_t* offsets, int64_t T, int H, int K, int V) {
  const int nh = blockIdx.y;
  const int n = nh / H, hh = nh % H;
  const int e4 = (int)blockIdx.x * 256 + (int)threadIdx.x;
  const int KV4 = K * V / 4;
  if (e4 >= KV4) return;
  const int kk = e4 * 4 / V;
  const SeqSpan sp = seq_span(offsets, n, T);
  const int nsub = (int)split_nsub(split, (sp.len + BT - 1) / BT);
  const int nseg = (nsub + split.ratio - 1) / split.ratio;
  const int64_t base = split.sub_base ? split.sub_base[n] : (int64_t)n * split.nsub;
  f32x4* S = (f32x4*)states + (base * H + hh) * (int64_t)KV4 + e4;
  const float* D = decays + (base * H + hh) * (int64_t)K + kk;
  const int64_t sstr = (int64_t)H * KV4, dstr = (int64_t)H * K;
  f32x4 h = {0.f, 0.f, 0.f, 0.f};
  if (init) h = ((const f32x4_any*)init)[(int64_t)nh * KV4 + e4];   // the caller's: aligned to 4 bytes only
  constexpr int U = 8;
  const int todo = REVERSE ? nsub - split.ratio : (nseg - 1) * split.ratio;   // sub-blocks the first pass formed
  for (int d = 0; d < todo; d += U) {
    f32x4 s[U];
    float dc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int x = d + u < todo ? d + u : todo - 1;
      const int j = REVERSE ? nsub - 1 - x : x;
      s[u] = S[j * sstr];
      dc[u] = D[j * dstr];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (d + u < todo) {
        const int j = REVERSE ? nsub - 1 - (d + u) : d + u;
        if (REVERSE ? (j == nsub - 1 || (j + 1) % split.ratio == 0) : j % split.ratio == 0) S[j * sstr] = h;
        h = h * dc[u] + s[u] * scale;
      }
    }
  }
  // the segment no sub-block of which the first pass formed: the last one forwards, the first one backwards
  S[(REVERSE ? (split.ratio < nsub ? split.ratio : nsub) - 1 : (nseg - 1) * split.ratio) * sstr] = h;
}

template <typename T, typename GT, int MODE>
int launch_pass(const SplitPassParams& p, int K, int V, unsigned grid, hipStream_t st) {
#define FLA_CASE(KK, VV)                                                                              \
  if (K == KK && V == VV) {                                                                           \
    hipLaunchKernelGGL((gla_split_pass_kernel<T, GT, KK, VV, MODE>), dim3(grid), dim3(256), 0, st, p); \
    FLA_CHECK_LAUNCH();                                                                               \
    return FLA_OK;                                                                                    \
  }
  FLA_CASE(128, 128)
  FLA_CASE(64, 64)
  FLA_CASE(64, 128)
  FLA_CASE(128, 64)
#undef FLA_CASE
  return FLA_E_UNSUPPORTED;
}

template <typename T>
int dispatch_pass(const SplitPassParams& p, int mode, int gate_dtype, int K, int V, unsigned grid, hipStream_t st) {
  if (mode == kPassReverse) return launch_pass<T, float, kPassReverse>(p, K, V, grid, st);
  if (mode == kPassHeadGates) return launch_pass<T, float, kPassHeadGates>(p, K, V, grid, st);
  if (mode == kPassGateLogits)
    return gate_dtype == FLA_F32 ? launch_pass<T, float, kPassGateLogits>(p, K, V, grid, st)
                                 : launch_pass<T, T, kPassGateLogits>(p, K, V, grid, st);
  return gate_dtype == FLA_F32 ? launch_pass<T, float, kPassKeyGates>(p, K, V, grid, st)
                               : launch_pass<T, T, kPassKeyGates>(p, K, V, grid, st);
}

}  // namespace

// Both launches; `init` is the state entering the sequences (or, in reverse, the gradient leaving them), NULL for zero.
int gla_split_states(const void* a, const void* b, const void* g, const float* init, const fla_split* split, bool head_gates,
                     bool reverse, bool logits, float gate_inv_norm, float gate_clamp_min, float scale,
                     const int64_t* offsets, const int64_t* chunk_offsets, int qkv_dtype, int gate_dtype, int64_t T,
                     int64_t H, int64_t K, int64_t V, int64_t N, hipStream_t st) {
  int rc = check_split(split, offsets);
  if (rc) return rc;
  FLA_REQUIRE(split->decays, FLA_E_INVALID);
  FLA_REQUIRE(qkv_dtype == FLA_BF16 || qkv_dtype == FLA_F16, FLA_E_UNSUPPORTED);
  if (gate_dtype != FLA_F32) FLA_REQUIRE(gate_dtype == qkv_dtype, FLA_E_UNSUPPORTED);
  SplitPassParams p{a, b, g, split->states, split->decays, offsets, chunk_offsets, split_view(split), T, (int)H, 0,
                    gate_inv_norm, gate_clamp_min};
  int64_t subs;
  if (offsets) {
    subs = split->nsub;   // rows of sub_table
  } else {
    p.per_seq = reverse ? split->nsub - split->ratio : (split->nseg - 1) * split->ratio;
    FLA_REQUIRE(p.per_seq >= 0, FLA_E_INVALID);
    subs = (int64_t)p.per_seq * N;
  }
  FLA_REQUIRE(subs * H <= 0x7fffffffLL && N * H <= 65535, FLA_E_UNSUPPORTED);
  FLA_REQUIRE(BT * H * K * 4 <= 0x7fffffffLL && BT * H * V * 4 <= 0x7fffffffLL, FLA_E_UNSUPPORTED);   // 32-bit offsets inside a chunk
  const int mode = reverse ? kPassReverse : head_gates ? kPassHeadGates : logits ? kPassGateLogits : kPassKeyGates;
  if (subs > 0) {
    const unsigned grid = (unsigned)(subs * H);
    rc = qkv_dtype == FLA_BF16 ? dispatch_pass<bf16>(p, mode, gate_dtype, (int)K, (int)V, grid, st)
                               : dispatch_pass<f16>(p, mode, gate_dtype, (int)K, (int)V, grid, st);
    if (rc) return rc;
  }
  const dim3 fgrid((unsigned)((K * V / 4 + 255) / 256), (unsigned)(N * H));
  if (reverse)
    hipLaunchKernelGGL(gla_split_fold_kernel<true>, fgrid, dim3(256), 0, st, split->states, split->decays, init, scale,
                       p.split, offsets, T, (int)H, (int)K, (int)V);
  else
    hipLaunchKernelGGL(gla_split_fold_kernel<false>, fgrid, dim3(256), 0, st, split->states, split->decays, init, 1.f,
                       p.split, offsets, T, (int)H, (int)K, (int)V);
  FLA_CHECK_LAUNCH();
  return FLA_OK;
}
