// Chunked GLA backward for gfx950 (chunk size 64, 16-bit q/k/v/do, fp32 state).
//
// With G the chunk-local prefix sum of the log-gates, q~ = s q e^{G},
// k^ = k e^{G_last-G}, A = tril(q~ (k e^{-G})^T), dH_c the gradient w.r.t. the state
// LEAVING chunk c (fla/ops/gla/chunk.py:1217-1320, fla/ops/common/chunk_h.py:156-271):
//
//   gla_bwd_dh_kernel    reverse state scan:  store dH_c;  dH <- diag(e^{G_last}) dH + q~^T do.
//                        The tile is kept and stored transposed ([V,K], MFMA-fragment order), the
//                        orientation dk contracts it in; also emits dh0.
//   gla_bwd_dh_qg_kernel the same scan on the gated queries q e^{G} and the chunk decays e^{G_last} a
//                        states-keeping forward left: no prefix sums, no exponentials, 16-byte row pieces.
//   gla_bwd_chunk_kernel (gla_bwd_chunk.hip) per (chunk, head):  dq, dk, dv and dg from q, k, v, the gates, do, h_c and dH_c.
//                        As in the forward, one reference point per chunk replaces the 16x16 sub-block scheme.
//                        The score terms of chunks whose gates leave its range are added behind the last item.
#include <type_traits>

#include "chunk_common.h"
#include "gla_bwd_chunk.h"
#include "seq_split.h"

namespace {

// Gate operand of the chunk-parallel kernels: GT is the element type of per-key log-gates [rows, H, K], or
// HeadGate for one fp32 log-gate per (token, head), [rows, H], which a lane broadcasts over its key channels.
struct HeadGate {};
template <typename GT> struct GateOf { typedef GT elem; static constexpr bool per_head = false; };
template <> struct GateOf<HeadGate> { typedef float elem; static constexpr bool per_head = true; };

struct BDhParams {
  const void* q;
  const void* g;
  const void* dout;
  const float* dht;
  void* dhtf;         // out: dH, FLA_H_FRAGMENT_T
  float* dh0;         // out: fp32 [N,H,K,V] or null
  const int64_t* offsets;
  const int64_t* chunk_offsets;
  int64_t T;
  int64_t total_chunks;
  int H, K, V, N;
  float scale;
  const void* qg;      // optional: the gated queries q e^{G} the forward staged, [rows, H, K] in the q dtype
  const float* decay;  //   and e^{G_last} per chunk, [chunks, H, K]
  SplitView split;     // with qg: sequences cut into segments (ratio 0: not)
};

// The same scan from what a states-keeping forward left behind: dH_c = e^{G_last} dH_{c+1} + s (q e^{G})^T do with
// the gated queries and the decay factors read back instead of being formed from q and g again - no prefix sums,
// no exponentials, 16-byte loads (5 memory instructions per lane and chunk instead of 24) and half the bytes.  The
// tiles are plain row-major copies; both operands of the update contract over time, i.e. over the tiles' rows,
// and come out of LDS through the transposing load.  The scale is kept out of the operands: the accumulators
// carry dH / s (the incoming d ht is divided by s, every copy that leaves is multiplied by it).
template <typename T>
__global__ __launch_bounds__(256) void gla_bwd_dh_qg_kernel(BDhParams p) {
  typedef typename Elem<T>::v8 v8;
  __shared__ __attribute__((aligned(16))) T sQ[2][64 * LDT];  // [t][k] q e^{G}
  __shared__ __attribute__((aligned(16))) T sD[2][64 * LDT];  // [t][v] do
  __shared__ __attribute__((aligned(16))) float sDecay[2][64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = p.H, K = p.K, V = p.V;
  const int nkt = K / 64, nvt = V / 64, ntile = nkt * nvt;
  const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(id % (uint32_t)ntile);
  const int item = (int)(id / (uint32_t)ntile), hh = item % H;
  const int kbase = (tile % nkt) * 64, vbase = (tile / nkt) * 64;
  const ScanSpan span = scan_span<true>(p.split, item / H, nullptr, p.offsets, p.chunk_offsets, p.T);
  const int nh = span.n * H + hh;
  const SeqSpan sp = span.sp;
  const int64_t nchunks = span.nchunks, chunk0 = span.chunk0;
  // the gradient of the state leaving this workgroup's chunks
  const float* dht = p.split.ratio ? p.split.states + (span.slot * H + hh) * (int64_t)K * V
                     : p.dht       ? p.dht + (int64_t)nh * K * V
                                   : nullptr;

  // a lane owns two 16-byte pieces of each tile: rows prow and prow + 32, columns c8 ..
  const int prow = tid >> 3, c8 = (tid & 7) * 8;
  const char* qp = (const char*)((const T*)p.qg + (sp.bos * H + hh) * (int64_t)K + kbase + c8);
  const char* dp = (const char*)((const T*)p.dout + (sp.bos * H + hh) * (int64_t)V + vbase + c8);
  const float* cp = p.decay + (chunk0 * H + hh) * (int64_t)K + kbase + (tid & 63);
  const uint32_t pitchK = (uint32_t)H * K * (uint32_t)sizeof(T), pitchV = (uint32_t)H * V * (uint32_t)sizeof(T);
  const int64_t strideC = (int64_t)H * K;

  const int kq = wave & 1, vq = wave >> 1;
  const int kt32 = kbase / 32 + kq, vt32 = vbase / 32 + vq;
  const int kcol = kbase + kq * 32 + (lane & 31);
  // An empty sequence hands d ht through to d h0 bit for bit: no factor goes on and off it.
  const float scale = nchunks > 0 ? p.scale : 1.f, inv_scale = 1.f / scale;
  f32x16 acc2 = zero16();  // rows v, cols k: dH / s
  if (dht) {
#pragma unroll
    for (int r = 0; r < 16; ++r) acc2[r] = dht[(int64_t)kcol * V + vbase + vq * 32 + c32_row(r, lane)] * inv_scale;
  }
  struct Regs {
    v8 q[2], d[2];
    float dec;
  };
  auto chunk_len = [&](int64_t c) {
    int64_t rem = sp.len - c * BT;
    return (int)(rem < BT ? rem : BT);
  };
  // Every load is unconditional: rows past the end of a short (last) chunk are redirected to its last row and
  // their do rows zeroed where they are staged (the forward did not write gated queries there).
  auto load_chunk = [&](int64_t c, Regs& R) {
    const uint32_t last = (uint32_t)(chunk_len(c) - 1);
    const char* qb = qp + c * BT * (int64_t)pitchK;
    const char* db = dp + c * BT * (int64_t)pitchV;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t row = (uint32_t)(prow + 32 * i) < last ? (uint32_t)(prow + 32 * i) : last;
      R.q[i] = *(const v8*)(qb + row * pitchK);
      R.d[i] = *(const v8*)(db + row * pitchV);
    }
    R.dec = cp[c * strideC];
  };
  // One barrier per chunk, tiles double-buffered in LDS; two register sets, each refilled right after the
  // staging step that consumed it.
  auto step = [&](int64_t c, Regs& R, auto more) {
    const int buf = (int)(c & 1);
    const int L = chunk_len(c);
    // ---- gradient w.r.t. the state leaving chunk c, transposed fragment order
    {
      int64_t blk = ((chunk0 + c) * H + hh) * (int64_t)K * V;
      v8 lo, hi;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        lo[r] = (T)(acc2[r] * scale);
        hi[r] = (T)(acc2[r + 8] * scale);
      }
      // halves of 32 bytes exchanged between the halves of the wave: a store covers 1 KB on end instead of every other 16 bytes
      // of 2 KB (4 x 4096 tokens, 16 heads of 128: 66.1 -> 58.6 us)
      typedef uint32_t u4 __attribute__((ext_vector_type(4)));
      u4 x = __builtin_bit_cast(u4, lo), y = __builtin_bit_cast(u4, hi);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const auto sw = __builtin_amdgcn_permlane32_swap(x[r], y[r], false, false);
        x[r] = sw[0];
        y[r] = sw[1];
      }
      T* o2 = (T*)p.dhtf + blk + (((int64_t)vt32 * (K / 32) + kt32) * 64 + (lane & 31)) * 16 + 8 * (lane >> 5);
      *(u4*)o2 = x;
      *(u4*)(o2 + 32 * 16) = y;
    }
    const v8 z8 = {(T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int row = prow + 32 * i;
      *(v8*)&sQ[buf][row * LDT + c8] = R.q[i];
      *(v8*)&sD[buf][row * LDT + c8] = row < L ? R.d[i] : z8;
    }
    if (tid < 64) sDecay[buf][tid] = R.dec;
    if constexpr (decltype(more)::value) {
      load_chunk(c >= 2 ? c - 2 : 0, R);
      asm volatile("" ::: "memory");  // the loads stay here, ahead of the barrier
    }
    lds_barrier();
    {
      const float d = sDecay[buf][kq * 32 + (lane & 31)];
#pragma unroll
      for (int r = 0; r < 16; ++r) acc2[r] *= d;
    }
#pragma unroll
    for (int s = 0; s < BT; s += 16) {
      v8 fq = frag32_tr<T>(sQ[buf], LDT, kq * 32, s, lane);
      v8 fd = frag32_tr<T>(sD[buf], LDT, vq * 32, s, lane);
      acc2 = Elem<T>::mfma32(fd, fq, acc2);
    }
  };
  Regs R0, R1;
  if (nchunks > 0) {
    load_chunk(nchunks - 1, R0);
    asm volatile("" ::: "memory");
    load_chunk(nchunks > 1 ? nchunks - 2 : 0, R1);
    asm volatile("" ::: "memory");
    int64_t c = nchunks - 1;
    for (; c >= 3; c -= 2) {
      step(c, R0, std::true_type{});
      step(c - 1, R1, std::true_type{});
    }
    if (c == 2) {
      step(2, R0, std::true_type{});
      step(1, R1, std::false_type{});
      step(0, R0, std::false_type{});
    } else {
      step(c, R0, std::false_type{});
      if (c == 1) step(0, R1, std::false_type{});
    }
  }
  if (p.dh0 && span.first) {
    float* o = p.dh0 + (int64_t)nh * K * V;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *(f32x4*)&o[(int64_t)kcol * V + vbase + vq * 32 + 8 * r4 + 4 * (lane >> 5)] =
          f32x4{acc2[4 * r4] * scale, acc2[4 * r4 + 1] * scale, acc2[4 * r4 + 2] * scale, acc2[4 * r4 + 3] * scale};
  }
}

template <typename T, typename GT>
__global__ __launch_bounds__(256) void gla_bwd_dh_kernel(BDhParams p) {
  typedef typename Elem<T>::v8 v8;
  typedef T t2 __attribute__((ext_vector_type(2)));
  typedef GT g2 __attribute__((ext_vector_type(2)));
  __shared__ __attribute__((aligned(16))) T sQt[2][64 * LDT];  // [k][t] s q e^{G}
  __shared__ __attribute__((aligned(16))) T sDt[2][64 * LDT];  // [v][t] do
  __shared__ __attribute__((aligned(16))) float sDecay[2][64];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int H = p.H, K = p.K, V = p.V;
  const int nkt = K / 64, nvt = V / 64, ntile = nkt * nvt;
  const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
  const int tile = (int)(id % (uint32_t)ntile);
  const int nh = (int)(id / (uint32_t)ntile);
  const int n = nh / H, hh = nh % H;
  const int kbase = (tile % nkt) * 64, vbase = (tile / nkt) * 64;
  SeqSpan sp = seq_span(p.offsets, n, p.T);
  const int64_t nchunks = (sp.len + BT - 1) / BT;
  const int64_t chunk0 = p.chunk_offsets ? p.chunk_offsets[n] : (int64_t)n * ((p.T + BT - 1) / BT);

  const int rg = lane >> 3, c2 = wave * 16 + (lane & 7) * 2;
  const T* qp = (const T*)p.q + (sp.bos * H + hh) * (int64_t)K + kbase + c2;
  const GT* gp = (const GT*)p.g + (sp.bos * H + hh) * (int64_t)K + kbase + c2;
  const T* dp = (const T*)p.dout + (sp.bos * H + hh) * (int64_t)V + vbase + c2;
  const int64_t kstride = (int64_t)H * K, vstride = (int64_t)H * V;

  const int kq = wave & 1, vq = wave >> 1;
  const int kt32 = kbase / 32 + kq, vt32 = vbase / 32 + vq;
  const int vcol = vbase + vq * 32 + (lane & 31), kcol = kbase + kq * 32 + (lane & 31);
  f32x16 acc2 = zero16();  // rows v, cols k
  if (p.dht) {
    const float* dp0 = p.dht + (int64_t)nh * K * V;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc2[r] = dp0[(int64_t)kcol * V + vbase + vq * 32 + c32_row(r, lane)];
  }

  struct Regs {
    g2 g[8];
    t2 q[8];
    t2 d[8];
  };
  auto chunk_len = [&](int64_t c) {
    int64_t rem = sp.len - c * BT;
    return (int)(rem < BT ? rem : BT);
  };
  // Every load is unconditional: rows past the end of a short (last) chunk are redirected to its
  // last row (one unsigned minimum on a byte offset) and masked where they are used.
  const uint32_t pitchK = (uint32_t)kstride * sizeof(T), pitchG = (uint32_t)kstride * sizeof(GT);
  const uint32_t pitchV = (uint32_t)vstride * sizeof(T);
  auto load_chunk = [&](int64_t c, Regs& R) {
    const uint32_t last = (uint32_t)(chunk_len(c) - 1);
    const uint32_t limk = last * pitchK, limg = last * pitchG, limv = last * pitchV;
    const char* qb = (const char*)(qp + c * BT * kstride);
    const char* gb = (const char*)(gp + c * BT * kstride);
    const char* db = (const char*)(dp + c * BT * vstride);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const uint32_t row = (uint32_t)(rg * 8 + i);
      uint32_t ok = row * pitchK, og = row * pitchG, ov = row * pitchV;
      R.g[i] = *(const g2*)(gb + (og < limg ? og : limg));
      R.q[i] = *(const t2*)(qb + (ok < limk ? ok : limk));
      R.d[i] = *(const t2*)(db + (ov < limv ? ov : limv));
    }
  };

  // One barrier per chunk, operand tiles double-buffered in LDS.  Two register sets, each
  // refilled right after the staging step that consumed it: a chunk is in flight for almost two
  // iterations and no register copy sits between a load and its use.
  auto step = [&](int64_t c, Regs& R, auto more) {
    const int buf = (int)(c & 1);
    const int L = chunk_len(c);
    // ---- gradient w.r.t. the state leaving chunk c, transposed fragment order
    {
      int64_t blk = ((chunk0 + c) * H + hh) * (int64_t)K * V;
      v8 lo, hi;
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        lo[r] = (T)acc2[r];
        hi[r] = (T)acc2[r + 8];
      }
      T* o2 = (T*)p.dhtf + blk + (((int64_t)vt32 * (K / 32) + kt32) * 64 + lane) * 16;
      *(v8*)o2 = lo;
      *(v8*)(o2 + 8) = hi;
    }
    // ---- chunk-local prefix sums of the gates
    float G[8][2], glast0, glast1;
    {
      float r0 = 0.f, r1 = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        bool valid = (rg * 8 + i) < L;
        r0 += valid ? finite_gate((float)R.g[i][0]) : 0.f;
        r1 += valid ? finite_gate((float)R.g[i][1]) : 0.f;
        G[i][0] = r0;
        G[i][1] = r1;
      }
      float s0 = r0, s1 = r1;
#pragma unroll
      for (int d = 8; d < 64; d <<= 1) {
        float u0 = __shfl_up(s0, d, 64), u1 = __shfl_up(s1, d, 64);
        if (lane >= d) {
          s0 += u0;
          s1 += u1;
        }
      }
      float off0 = s0 - r0, off1 = s1 - r1;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        G[i][0] += off0;
        G[i][1] += off1;
      }
      glast0 = __shfl(s0, 56 + (lane & 7), 64);
      glast1 = __shfl(s1, 56 + (lane & 7), 64);
    }
    {
      v8 qa, qb, da, db;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        bool valid = (rg * 8 + i) < L;
        qa[i] = (T)(valid ? (float)R.q[i][0] * p.scale * __expf(G[i][0]) : 0.f);
        qb[i] = (T)(valid ? (float)R.q[i][1] * p.scale * __expf(G[i][1]) : 0.f);
        da[i] = R.d[i][0];
        db[i] = R.d[i][1];
      }
      *(v8*)&sQt[buf][(c2 + 0) * LDT + rg * 8] = qa;
      *(v8*)&sQt[buf][(c2 + 1) * LDT + rg * 8] = qb;
      *(v8*)&sDt[buf][(c2 + 0) * LDT + rg * 8] = da;
      *(v8*)&sDt[buf][(c2 + 1) * LDT + rg * 8] = db;
      if (rg == 0) *(f32x2*)&sDecay[buf][c2] = f32x2{__expf(glast0), __expf(glast1)};
    }
    if constexpr (decltype(more)::value) {
      load_chunk(c >= 2 ? c - 2 : 0, R);
      asm volatile("" ::: "memory");  // the loads stay here, ahead of the barrier
    }
    lds_barrier();
    {
      const float d = sDecay[buf][kq * 32 + (lane & 31)];
#pragma unroll
      for (int r = 0; r < 16; ++r) acc2[r] *= d;
    }
#pragma unroll
    for (int s = 0; s < BT; s += 16) {
      v8 fq = lds_frag32<T>(sQt[buf], LDT, kq * 32, s, lane);
      v8 fd = lds_frag32<T>(sDt[buf], LDT, vq * 32, s, lane);
      acc2 = Elem<T>::mfma32(fd, fq, acc2);
    }
  };
  Regs R0, R1;
  if (nchunks > 0) {
    load_chunk(nchunks - 1, R0);
    asm volatile("" ::: "memory");  // the two sets are issued one after the other, as in the loop:
    load_chunk(nchunks > 1 ? nchunks - 2 : 0, R1);  // interleaved, the loop's first wait would cover both
    asm volatile("" ::: "memory");
    int64_t c = nchunks - 1;
    for (; c >= 3; c -= 2) {
      step(c, R0, std::true_type{});
      step(c - 1, R1, std::true_type{});
    }
    // the last one to three chunks: nothing is left to prefetch for the final two
    if (c == 2) {
      step(2, R0, std::true_type{});
      step(1, R1, std::false_type{});
      step(0, R0, std::false_type{});
    } else {
      step(c, R0, std::false_type{});
      if (c == 1) step(0, R1, std::false_type{});
    }
  }
  if (p.dh0) {
    float* o = p.dh0 + (int64_t)nh * K * V;
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4)
      *(f32x4*)&o[(int64_t)kcol * V + vbase + vq * 32 + 8 * r4 + 4 * (lane >> 5)] =
          f32x4{acc2[4 * r4], acc2[4 * r4 + 1], acc2[4 * r4 + 2], acc2[4 * r4 + 3]};
  }
}

template <typename T, typename GT>
int launch_bwd(const void* q, const void* k, const void* v, const void* g, const void* dout, const float* dht,
               const void* hT, const void* qg, const float* decay, void* dhtf, void* dq, void* dk, void* dv, float* dg,
               float* dg_head, float* dh0, const int* wide,
               const int64_t* offsets, const int64_t* indices, const int64_t* chunk_offsets, int64_t NT, int64_t B,
               int64_t T_, int64_t H, int64_t K, int64_t V, int64_t N, float scale, hipStream_t st,
               const fla_split* split = nullptr) {
  constexpr int kDtype = std::is_same<T, bf16>::value ? FLA_BF16 : FLA_F16;
  constexpr int kGates = std::is_same<GT, bf16>::value ? FLA_BF16 : std::is_same<GT, f16>::value ? FLA_F16 : FLA_F32;
  dim3 grid;
  int ntfix;
  int rc = chunk_grid(offsets, indices, B, T_, H, NT, &grid, &ntfix);
  if (rc) return rc;
  if (grid.x == 0) return copy_or_zero(dht, dh0, N * H * K * V, st);   // no chunk at all: d h0 = d ht
  const int64_t total_chunks = grid.x;
  {
    BDhParams p{q, g, dout, dht, dhtf, dh0, offsets, chunk_offsets, T_, total_chunks,
                (int)H, (int)K, (int)V, (int)N, scale, qg, decay, split_view(split)};
    int64_t seqs = N;
    if (split) {
      // the gradient leaving every segment: dH <- decay dH + scale (q e^{G})^T do over the sub-blocks
      rc = gla_split_states(qg, dout, decay, dht, split, false, true, false, 1.f, 0.f, scale, offsets, chunk_offsets, kDtype,
                            FLA_F32, T_, H, K, V, N, st);
      if (rc) return rc;
      seqs = offsets ? split->nseg : split->nseg * N;
    }
    const int64_t total = (K / 64) * (V / 64) * seqs * H;
    FLA_REQUIRE(total <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
    if (qg) hipLaunchKernelGGL((gla_bwd_dh_qg_kernel<T>), dim3((unsigned)total), dim3(256), 0, st, p);
    else if constexpr (GateOf<GT>::per_head) return FLA_E_INVALID;   // per-head gates come with kept gated queries
    else hipLaunchKernelGGL((gla_bwd_dh_kernel<T, GT>), dim3((unsigned)total), dim3(256), 0, st, p);
    FLA_CHECK_LAUNCH();
  }
  rc = gla_bwd_chunk(q, k, v, g, dout, hT, dhtf, wide, dq, dk, dv, GateOf<GT>::per_head ? dg_head : dg, offsets, indices,
                     grid.x, ntfix, kDtype, kGates, GateOf<GT>::per_head, T_, H, K, V, scale, st);
  return rc;
}

}  // namespace

static int gla_bwd_impl(const void* q, const void* k, const void* v, const void* gates, const void* dout,
                        const float* dht, const void* hT, const void* q_gated, const float* chunk_decay,
                        void* dh_frag_t, void* dq, void* dk, void* dv, float* dg, float* dg_head, float* dh0,
                        const int* wide,
                        const int64_t* offsets, const int64_t* indices, const int64_t* chunk_offsets, int64_t NT,
                        int qkv_dtype, int gate_dtype, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V,
                        int64_t N, float scale, fla_stream_t stream, bool head_gates = false,
                        const void* kh_t = nullptr, const void* scores = nullptr, const fla_split* split = nullptr) {
  if (split) FLA_REQUIRE(q_gated, FLA_E_INVALID);
  FLA_REQUIRE(q && k && v && gates && dout && hT && dh_frag_t && dq && dk && dv && (dg || dg_head),
              FLA_E_INVALID);
  if (head_gates) FLA_REQUIRE(q_gated && dg_head, FLA_E_INVALID);
  FLA_REQUIRE((kh_t == nullptr) == (scores == nullptr) && (kh_t == nullptr || q_gated != nullptr), FLA_E_INVALID);
  FLA_REQUIRE(((uintptr_t)kh_t | (uintptr_t)scores) % 16 == 0, FLA_E_ALIGNMENT);
  FLA_REQUIRE(B >= 0 && T >= 0 && H > 0 && K > 0 && V > 0 && N >= 0 && NT >= 0, FLA_E_INVALID);
  FLA_REQUIRE(K % 64 == 0 && V % 64 == 0 && K <= 128 && V <= 128, FLA_E_UNSUPPORTED);
  if (offsets) FLA_REQUIRE(indices && chunk_offsets && B == 1, FLA_E_INVALID);
  else FLA_REQUIRE(N == B, FLA_E_INVALID);
  FLA_REQUIRE((q_gated == nullptr) == (chunk_decay == nullptr), FLA_E_INVALID);
  if (q_gated) FLA_REQUIRE(scale != 0.f, FLA_E_INVALID);
  FLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (head_gates ? 0 : (uintptr_t)gates) | (uintptr_t)dout |
               (uintptr_t)hT | (uintptr_t)dh_frag_t | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv |
               (uintptr_t)dg | (uintptr_t)q_gated) % 16 == 0,
              FLA_E_ALIGNMENT);
  hipStream_t st = (hipStream_t)stream;
#define FLA_BWD(TT, GG)                                                                                           \
  return launch_bwd<TT, GG>(q, k, v, gates, dout, dht, hT, q_gated, chunk_decay, dh_frag_t, dq, dk, dv, dg, dg_head, dh0, wide,   \
                            offsets, indices, chunk_offsets, NT, B, T, H, K, V, N, scale, st, split)
  if (head_gates && qkv_dtype == FLA_BF16) FLA_BWD(bf16, HeadGate);
  if (head_gates && qkv_dtype == FLA_F16) FLA_BWD(f16, HeadGate);
  if (head_gates) return FLA_E_UNSUPPORTED;
  if (qkv_dtype == FLA_BF16 && gate_dtype == FLA_F32) FLA_BWD(bf16, float);
  if (qkv_dtype == FLA_BF16 && gate_dtype == FLA_BF16) FLA_BWD(bf16, bf16);
  if (qkv_dtype == FLA_F16 && gate_dtype == FLA_F32) FLA_BWD(f16, float);
  if (qkv_dtype == FLA_F16 && gate_dtype == FLA_F16) FLA_BWD(f16, f16);
#undef FLA_BWD
  return FLA_E_UNSUPPORTED;
}

extern "C" int fla_chunk_gla_bwd(const void* q, const void* k, const void* v, const void* gates, const void* dout,
                                 const float* dht, const void* hT, void* dh_frag_t,
                                 void* dq, void* dk, void* dv, float* dg, float* dh0, const int* wide,
                                 const int64_t* offsets, const int64_t* indices, const int64_t* chunk_offsets,
                                 int64_t NT, int qkv_dtype,
                                 int gate_dtype, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t N,
                                 float scale, fla_stream_t stream) {
  return gla_bwd_impl(q, k, v, gates, dout, dht, hT, nullptr, nullptr, dh_frag_t, dq, dk, dv, dg, nullptr, dh0, wide, offsets,
                      indices, chunk_offsets, NT, qkv_dtype, gate_dtype, B, T, H, K, V, N, scale, stream);
}

extern "C" int fla_chunk_gla_bwd_kept(const void* q, const void* k, const void* v, const void* gates,
                                      const void* dout, const float* dht, const void* hT, const void* q_gated,
                                      const float* chunk_decay, const void* khat_t, const void* scores,
                                      void* dh_frag_t, void* dq, void* dk, void* dv,
                                      float* dg, float* dh0, const int* wide, const int64_t* offsets,
                                      const int64_t* indices, const int64_t* chunk_offsets, int64_t NT,
                                      int qkv_dtype, int gate_dtype, int64_t B, int64_t T, int64_t H, int64_t K,
                                      int64_t V, int64_t N, float scale, fla_stream_t stream) {
  FLA_REQUIRE(q_gated && chunk_decay, FLA_E_INVALID);
  return gla_bwd_impl(q, k, v, gates, dout, dht, hT, q_gated, chunk_decay, dh_frag_t, dq, dk, dv, dg, nullptr, dh0, wide,
                      offsets, indices, chunk_offsets, NT, qkv_dtype, gate_dtype, B, T, H, K, V, N, scale, stream, false,
                      khat_t, scores);
}

extern "C" int fla_chunk_simple_gla_bwd(const void* q, const void* k, const void* v, const float* g, const void* dout,
                                        const float* dht, const void* hT, const void* q_gated,
                                        const float* chunk_decay, const void* khat_t, const void* scores,
                                        void* dh_frag_t, void* dq, void* dk, void* dv, float* dg, float* dh0, const int* wide, const int64_t* offsets,
                                        const int64_t* indices, const int64_t* chunk_offsets, int64_t NT,
                                        int qkv_dtype, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V,
                                        int64_t N, float scale, fla_stream_t stream) {
  FLA_REQUIRE(q_gated && chunk_decay && dg, FLA_E_INVALID);
  return gla_bwd_impl(q, k, v, g, dout, dht, hT, q_gated, chunk_decay, dh_frag_t, dq, dk, dv, nullptr, dg, dh0, wide,
                      offsets, indices, chunk_offsets, NT, qkv_dtype, FLA_F32, B, T, H, K, V, N, scale, stream, true,
                      khat_t, scores);
}

extern "C" int fla_chunk_gla_bwd_split(const void* q, const void* k, const void* v, const void* gates, const void* dout,
                                       const float* dht, const void* hT, const void* q_gated, const float* chunk_decay,
                                       const void* khat_t, const void* scores, void* dh_frag_t, void* dq, void* dk,
                                       void* dv, float* dg, float* dh0, const int* wide, const int64_t* offsets,
                                       const int64_t* indices, const int64_t* chunk_offsets, const fla_split* split,
                                       int64_t NT, int qkv_dtype, int gate_dtype, int64_t B, int64_t T, int64_t H,
                                       int64_t K, int64_t V, int64_t N, float scale, int head_gates,
                                       fla_stream_t stream) {
  FLA_REQUIRE(q_gated && chunk_decay && split && dg, FLA_E_INVALID);
  return gla_bwd_impl(q, k, v, gates, dout, dht, hT, q_gated, chunk_decay, dh_frag_t, dq, dk, dv, head_gates ? nullptr : dg,
                      head_gates ? dg : nullptr, dh0, wide, offsets, indices, chunk_offsets, NT, qkv_dtype,
                      head_gates ? FLA_F32 : gate_dtype, B, T, H, K, V, N, scale, stream, head_gates != 0, khat_t, scores,
                      split);
}
