// The chunk-parallel half of the chunked GLA backward in one launch: dq, dk, dv and the gate gradient of a (chunk, head)
// from q, k, v, the log-gates, do, the state entering the chunk and the gradient of the state leaving it
// (fla/ops/gla/chunk.py:409-837, :982-1061).  With G the chunk-local prefix sums of the gates, q~ = q e^G, k~ = k e^{-G},
// k^ = k e^{G_last - G}:
//   P = tril(q~ k~^T)   dA = tril(do v^T)
//   dq = s e^G (dA k~ + do h^T)     dk = s e^{-G} (dA^T q~) + e^{G_last - G} (v dH^T)     dv = s P^T do + k^ dH
//   dg_t = sum_{t' >= t} s (q~ (dA k~ + do h^T) - k~ (dA^T q~))_t' + sum_{t' < t} (k^ (v dH^T))_t' + e^{G_last} sum_v h dH
// (the pairs of the first sum are formed with the rounded operands of the products, so that they cancel exactly unless they
// straddle t; see gla_bwd.hip).
//
// What bounds it: bytes, 1.0 GB for 4 x 4096 tokens, 16 heads, K = V = 128, in 202 us: 5.0 TB/s, the rate of a large copy
// (208 behind the gradient scan, 216 inside a training step).
// Before, dv was formed inside the reverse state scan from three tiles the forward kept for it (P, k^ and the gated
// queries: 128 us, and 20 us more in the forward) and the rest in a launch per 64 key channels (206 us); the scan alone is
// 70 us.  Sums over time cost VALU cycles here, not LDS or barriers: 3600 vector instructions per wave and item are 214 us,
// 2950 are 202.
#include <type_traits>

#include "chunk_rows.h"
#include "gla_bwd_chunk.h"

namespace {

struct GlaChunkParams {
  const void* q;
  const void* k;
  const void* v;
  const void* g;       // log-gates [rows, H, K], or per head fp32 [rows, H]
  const void* dout;
  const void* hT;      // forward states, FLA_H_FRAGMENT_T
  const void* dhtf;    // dH, FLA_H_FRAGMENT_T
  const int* wide;     // [chunks, H] or NULL: chunks whose score terms (P, dA) are left to exact_scores()
  void* dq;
  void* dk;
  void* dv;
  float* dg;           // fp32 [rows, H, K], or per head [rows, H]
  const int64_t* offsets;
  const int64_t* indices;
  int64_t T;
  int H, NTfix;
  float scale;
};

// A copy the compiler takes for another value
template <typename X>
FLA_DEVICE X opaque(X x) {
  typedef uint32_t u2 __attribute__((ext_vector_type(2)));
  u2 u = __builtin_bit_cast(u2, x);
  asm volatile("" : "+v"(u));
  return __builtin_bit_cast(X, u);
}

// One fp32 log-gate per (token, head) instead of per-key log-gates of type GT
struct PerHead {};

// Element (i, j), j <= i, of a 64 x 64 lower triangle of floats
FLA_DEVICE int tri_at(int i, int j) { return i * (i + 1) / 2 + j; }
constexpr int kTriFloats = BT * (BT + 1) / 2;

// The score terms of a chunk whose gates leave the range of one reference point, added to what gla_bwd_chunk_kernel left for
// it: pairwise exponents G_i - G_j <= 0, the arithmetic of the reference's diagonal sub-blocks (fla/ops/gla/chunk.py:409-567):
//   A_ij  = s sum_k q_ik k_jk e^{G_ik-G_jk},  dA_ij = do_i . v_j            (j <= i)
//   dv_j += sum_{i>=j} A_ij do_i
//   dq_ik += s sum_{j<=i} dA_ij k_jk e^{G_ik-G_jk},  dk_jk += s sum_{i>=j} dA_ij q_ik e^{G_ik-G_jk}
//   dg_ik += sum_{t>=i} (q_tk dq'_tk - k_tk dk'_tk)          (dq', dk': the terms added here)
// Plain fp32 arithmetic on the vector ALU, by the workgroup that formed the chunk, behind its last item and in the LDS of the
// items.  ab, c, d, tri: room for 64 rows of gates and sums over channels (or v and do), for q (or do), for k (or A), for dA.
//
// What bounds it: with per-key gates 3 x 2080 K exponentials an item and what stands around them, as long as the operands come
// wide enough and far enough ahead.  Pairs: a thread takes rows a + 16 m and columns b + 16 n, the ten blocks m >= n, so that
// four channels of eight rows feed forty products and all threads have the same work.  dq and dk: a thread takes four channels
// of a row, four steps of the sum per trip, the ends of the triangle by selection.
// Backward with every chunk flagged, us, as a launch of its own with 136 KB of LDS / here, one channel a trip and a single sum /
// so: fp16, 2 x 2000 tokens, 32 heads of 64, per-key gates 819 / 687 / 412, per head 672 / 535 / 232; bf16, 4 x 4096 tokens, 16
// heads of 128, per-key 3176 / 3260 / 1568, per head 2728 / 2577 / 928, a chunk in twenty flagged 987 / 1316 / 666; 2 x 256 tokens,
// 4 heads of 64, one item a workgroup, 120 / 194 / 76.  Where nothing is flagged the launch took 4 us to find that out.
template <typename T, typename GT, int K, int V>
FLA_DEVICE void exact_scores(const GlaChunkParams& p, const ChunkLoc& cl, int hh, char* ab, T* c, T* d, float* tri, float* sGam) {
  typedef typename Elem<T>::v4 v4;
  constexpr bool PH = std::is_same<GT, PerHead>::value;
  typedef typename std::conditional<PH, float, GT>::type GE;
  constexpr int LDG = K + 4, LDQ = K + 8, LDW = V + 8;
  constexpr int RP = 1024 / K, NR = BT / RP;   // rows of K / 4 threads each that stand side by side, and how often
  float *sG = (float*)ab, *sX = sG;
  T *sQ = c, *sK = d, *sV = (T*)ab, *sDo = sV + BT * LDW, *sDo2 = c;
  float *sA = (float*)d, *sdA = tri;
  // (fresh_tid: nothing formed here may live in registers over the items)
  const int tid0 = threadIdx.x, tid = fresh_tid(tid0), H = p.H, L = cl.L;
  const int64_t strideK = (int64_t)H * K, strideV = (int64_t)H * V;
  const int64_t baseK = (cl.row0 * H + hh) * (int64_t)K, baseV = (cl.row0 * H + hh) * (int64_t)V;
  const v4 z4 = {(T)0.f, (T)0.f, (T)0.f, (T)0.f};
  auto f4 = [](v4 x) __attribute__((always_inline)) { return f32x4{(float)x[0], (float)x[1], (float)x[2], (float)x[3]}; };
  const int pa = tid >> 4, pb = tid & 15;
  // f(block number, m, n) over the ten blocks of pairs (pa + 16 m, pb + 16 n)
  auto blocks = [](auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
      for (int n = 0; n <= m; ++n) f(m * (m + 1) / 2 + n, m, n);
  };

#pragma unroll 4
  for (int e = tid; e < BT * (V / 4); e += 256) {
    const int row = e / (V / 4), c4 = (e % (V / 4)) * 4;
    const int64_t off = baseV + row * strideV + c4;
    *(v4*)&sV[row * LDW + c4] = row < L ? *(const v4*)((const T*)p.v + off) : z4;
    *(v4*)&sDo[row * LDW + c4] = row < L ? *(const v4*)((const T*)p.dout + off) : z4;
  }
#pragma unroll 4
  for (int e = tid; e < BT * (K / 4); e += 256) {
    const int row = e / (K / 4), c4 = (e % (K / 4)) * 4;
    const int64_t off = baseK + row * strideK + c4;
    *(v4*)&sQ[row * LDQ + c4] = row < L ? *(const v4*)((const T*)p.q + off) : z4;
    *(v4*)&sK[row * LDQ + c4] = row < L ? *(const v4*)((const T*)p.k + off) : z4;
  }
  if (PH && tid < BT) sGam[tid] = tid < L ? finite_gate(((const float*)p.g)[(cl.row0 + tid) * H + hh]) : 0.f;
  __syncthreads();
  if (PH && tid == 0) {
    float run = 0.f;
#pragma unroll 16
    for (int t = 0; t < BT; ++t) {
      run += sGam[t];
      sGam[t] = run;
    }
  }
  float da[10];
  blocks([&](int x, int, int) { da[x] = 0.f; });
#pragma unroll 2
  for (int ch = 0; ch < V; ch += 4) {
    f32x4 di[4], vj[4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      di[m] = f4(*(const v4*)&sDo[(pa + 16 * m) * LDW + ch]);
      vj[m] = f4(*(const v4*)&sV[(pb + 16 * m) * LDW + ch]);
    }
    blocks([&](int x, int m, int n) {
#pragma unroll
      for (int z = 0; z < 4; ++z) da[x] = fmaf(di[m][z], vj[n][z], da[x]);
    });
  }
  __syncthreads();   // v and do make room for the gates
  if constexpr (!PH) {
#pragma unroll 4
    for (int e = tid; e < BT * (K / 4); e += 256) {
      const int row = e / (K / 4), c4 = (e % (K / 4)) * 4;
      float gv[4] = {0.f, 0.f, 0.f, 0.f};
      if (row < L) Load<GE>::x4((const GE*)p.g + baseK + row * strideK + c4, gv);
      *(f32x4*)&sG[row * LDG + c4] = f32x4{finite_gate(gv[0]), finite_gate(gv[1]), finite_gate(gv[2]), finite_gate(gv[3])};
    }
    __syncthreads();
    if (tid < K) {
      float run = 0.f;
#pragma unroll 1
      for (int t0 = 0; t0 < BT; t0 += 16) {
        float y[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) y[t] = sG[(t0 + t) * LDG + tid];
#pragma unroll
        for (int t = 0; t < 16; ++t) sG[(t0 + t) * LDG + tid] = run += y[t];
      }
    }
    __syncthreads();
  }
  float a[10];   // A
  blocks([&](int x, int, int) { a[x] = 0.f; });
#pragma unroll 2
  for (int ch = 0; ch < K; ch += 4) {
    f32x4 qi[4], kj[4], gi[PH ? 1 : 4], gj[PH ? 1 : 4];
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      qi[m] = f4(*(const v4*)&sQ[(pa + 16 * m) * LDQ + ch]);
      kj[m] = f4(*(const v4*)&sK[(pb + 16 * m) * LDQ + ch]);
      if constexpr (!PH) {
        gi[m] = *(const f32x4*)&sG[(pa + 16 * m) * LDG + ch];
        gj[m] = *(const f32x4*)&sG[(pb + 16 * m) * LDG + ch];
      }
    }
    blocks([&](int x, int m, int n) {
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        if constexpr (PH) a[x] = fmaf(qi[m][z], kj[n][z], a[x]);
        else a[x] = fmaf(qi[m][z] * kj[n][z], __expf(gi[m][z] - gj[n][z]), a[x]);
      }
    });
  }
  // (per head the exponential is the pair's and goes onto dA as well)
  blocks([&](int x, int m, int n) {
    const int i = pa + 16 * m, j = pb + 16 * n;
    const float e = PH ? __expf(sGam[i] - sGam[j]) : 1.f;
    a[x] *= p.scale * e;
    if (j <= i) sdA[tri_at(i, j)] = da[x] * p.scale * e;
  });
  __syncthreads();
  float x[NR][4];    // q dq' - k dk', rows and channels as below
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const int t = fresh_tid(tid0), r = t / (K / 4) + RP * n, c4 = (t % (K / 4)) * 4;
    const int w0 = __builtin_amdgcn_readfirstlane(t >> 6) * (RP / 4) + RP * n;   // the wave's first row
    const f32x4 gr = PH ? zero4() : *(const f32x4*)&sG[r * LDG + c4];
    f32x4 dq = zero4(), dk = zero4();
#pragma unroll 1
    for (int j0 = 0; j0 < w0 + RP / 4; j0 += 4) {   // row r as the query row i
      f32x4 kj[4], gj[4];
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        kj[u] = f4(*(const v4*)&sK[(j0 + u) * LDQ + c4]);
        if constexpr (!PH) gj[u] = *(const f32x4*)&sG[(j0 + u) * LDG + c4];
        w[u] = sdA[tri_at(r, j0 + u)];   // (past the diagonal: another element of the triangle, not used)
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int z = 0; z < 4; ++z) {
          const float y = PH ? w[u] * kj[u][z] : w[u] * kj[u][z] * __expf(gr[z] - gj[u][z]);
          dq[z] += j0 + u <= r ? y : 0.f;
        }
    }
#pragma unroll 1
    for (int i0 = w0 & ~3; i0 < L; i0 += 4) {       // row r as the key row j
      f32x4 qi[4], gi[4];
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        qi[u] = f4(*(const v4*)&sQ[(i0 + u) * LDQ + c4]);
        if constexpr (!PH) gi[u] = *(const f32x4*)&sG[(i0 + u) * LDG + c4];
        w[u] = sdA[tri_at(i0 + u, r)];   // (r > i0 + u: another element)
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int z = 0; z < 4; ++z) {
          const float y = PH ? w[u] * qi[u][z] : w[u] * qi[u][z] * __expf(gi[u][z] - gr[z]);
          dk[z] += i0 + u >= r && i0 + u < L ? y : 0.f;
        }
    }
#pragma unroll
    for (int z = 0; z < 4; ++z) x[n][z] = 0.f;
    if (r < L) {
      const v4 qr = *(const v4*)&sQ[r * LDQ + c4], kr = *(const v4*)&sK[r * LDQ + c4];
      T *dqp = (T*)p.dq + baseK + r * strideK + c4, *dkp = (T*)p.dk + baseK + r * strideK + c4;
      const v4 oq = *(const v4*)dqp, ok = *(const v4*)dkp;
      v4 nq, nk;
#pragma unroll
      for (int z = 0; z < 4; ++z) {
        nq[z] = (T)((float)oq[z] + dq[z]);
        nk[z] = (T)((float)ok[z] + dk[z]);
        x[n][z] = (float)qr[z] * dq[z] - (float)kr[z] * dk[z];
      }
      *(v4*)dqp = nq;
      *(v4*)dkp = nk;
    }
  }
  __syncthreads();   // the gates make room for x, q for do, k for A
#pragma unroll
  for (int n = 0; n < NR; ++n) {
    const int r = tid / (K / 4) + RP * n, c4 = (tid % (K / 4)) * 4;
    if constexpr (PH) {   // the channels of a row are added up in the K / 4 lanes that hold it
      float sum = (x[n][0] + x[n][1]) + (x[n][2] + x[n][3]);
#pragma unroll
      for (int m = K / 8; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, 64);
      if (c4 == 0) sGam[r] = sum;
    } else {
      *(f32x4*)&sX[r * LDG + c4] = f32x4{x[n][0], x[n][1], x[n][2], x[n][3]};
    }
  }
  blocks([&](int y, int m, int n) {
    const int i = pa + 16 * m, j = pb + 16 * n;
    if (j <= i) sA[tri_at(i, j)] = a[y];
  });
#pragma unroll 4
  for (int e = tid; e < BT * (V / 4); e += 256) {
    const int row = e / (V / 4), c4 = (e % (V / 4)) * 4;
    *(v4*)&sDo2[row * LDW + c4] = row < L ? *(const v4*)((const T*)p.dout + baseV + row * strideV + c4) : z4;
  }
  __syncthreads();
  // dg: sums over the rows from the last one up
  if constexpr (PH) {
    if (tid < L) {
      float run = 0.f;
#pragma unroll 16
      for (int t = BT - 1; t >= 0; --t) run += t >= tid ? sGam[t] : 0.f;
      p.dg[(cl.row0 + tid) * H + hh] += run;
    }
  } else if (tid < K) {
    float run = 0.f;
    float* dg = p.dg + baseK + tid;
#pragma unroll 1
    for (int t0 = BT - 8; t0 >= 0; t0 -= 8) {
      float old[8], y[8];
#pragma unroll
      for (int t = 7; t >= 0; --t) {
        y[t] = sX[(t0 + t) * LDG + tid];
        if (t0 + t < L) old[t] = dg[(t0 + t) * strideK];
      }
#pragma unroll
      for (int t = 7; t >= 0; --t) {
        run += y[t];
        if (t0 + t < L) dg[(t0 + t) * strideK] = old[t] + run;
      }
    }
  }
  // dv_j += sum_{i>=j} A_ij do_i
  constexpr int VP = 1024 / V;
#pragma unroll 1
  for (int n = 0; n < BT / VP; ++n) {
    const int r = tid / (V / 4) + VP * n, c4 = (tid % (V / 4)) * 4;
    const int w0 = __builtin_amdgcn_readfirstlane(tid >> 6) * (VP / 4) + VP * n;
    f32x4 acc = zero4();
#pragma unroll 1
    for (int i0 = w0 & ~3; i0 < L; i0 += 4) {
      f32x4 y[4];
      float w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        y[u] = f4(*(const v4*)&sDo2[(i0 + u) * LDW + c4]);
        w[u] = sA[tri_at(i0 + u, r)];   // (r > i0 + u: another element)
      }
#pragma unroll
      for (int u = 0; u < 4; ++u)
#pragma unroll
        for (int z = 0; z < 4; ++z) acc[z] += i0 + u >= r && i0 + u < L ? w[u] * y[u][z] : 0.f;
    }
    if (r < L) {
      T* dst = (T*)p.dv + baseV + r * strideV + c4;
      const v4 old = *(const v4*)dst;
      v4 nw;
#pragma unroll
      for (int z = 0; z < 4; ++z) nw[z] = (T)((float)old[z] + acc[z]);
      *(v4*)dst = nw;
    }
  }
  __syncthreads();
}

// Four waves.  In products with K (V) result columns a wave owns 32 of them and, with 128 columns, all 64 rows, with 64
// columns one half of the rows; such products are formed transposed, so that a lane owns one time row and, per register
// quad, four adjacent columns, and everything elementwise - the gates and their prefix sums over time, which run along the
// lanes, the epilogue, the gate gradient - happens in that one layout.  In the 64 x 64 products waves 0, 2 and 3 own the
// 32 x 32 blocks on and below the diagonal.  LDS (80 KB, two workgroups per CU):
//   AB: gates -> do | v -> dH [k][v]     C: k -> k~ -> k^ -> dv     D: q -> q~ -> dq -> dk     S: dA -> P
template <typename T, typename GT, int K, int V>
__global__ __launch_bounds__(256, 2) void gla_bwd_chunk_kernel(GlaChunkParams p, uint32_t nitems) {
  typedef typename Elem<T>::v8 v8;
  typedef typename Elem<T>::v4 v4;
  typedef RowTile<T, K> TK;
  typedef RowTile<T, V> TV;
  constexpr bool PH = std::is_same<GT, PerHead>::value;
  typedef typename std::conditional<PH, float, GT>::type GE;
  constexpr int GP = 16 / sizeof(GE), NG = PH ? 1 : BT * K / GP / 256;   // gates: elements per 16-byte piece, pieces per lane
  typedef GE gvec __attribute__((ext_vector_type(GP)));
  constexpr int LDK = K + 8, LDV = V + 8, LDG = K + 4;
  // the gates and their sums are carried times log2 e
  constexpr float kLog2e = 1.4426950408889634f, kInvLimit = InvDecayLimit<T>::value * kLog2e;
  constexpr int VT32 = V / 32, KT32 = K / 32;
  constexpr int RK = K / 64, RV = V / 64;   // row tiles of a wave in products with K (V) result columns
  constexpr int AB_DOV = 2 * BT * LDV * 2, AB_G = PH ? 0 : BT * LDG * 4, AB_DH = K * LDV * 2;
  constexpr int AB0 = AB_DOV > AB_G ? AB_DOV : AB_G, AB = AB0 > AB_DH ? AB0 : AB_DH;
  __shared__ __attribute__((aligned(16))) char sAB[AB];
  __shared__ __attribute__((aligned(16))) T sC[BT * (LDK > LDV ? LDK : LDV)];
  __shared__ __attribute__((aligned(16))) T sD[BT * LDK];
  __shared__ __attribute__((aligned(16))) T sS[BT * LDT];
  __shared__ __attribute__((aligned(16))) float sHd[4][32];    // per wave: <h, dH> of its key channels
  __shared__ __attribute__((aligned(16))) float sGl[4][32];    // per wave: G_last of its key channels
  // K = 64: totals of the gate gradient's terms over a wave's half of the rows.  Per head: [0] prefix sums of the gate
  __shared__ __attribute__((aligned(16))) float sX[PH ? 1 : 4][PH ? BT : 32], sKd[PH ? 1 : 4][PH ? 4 : 32];
  float* sG = (float*)sAB;
  T* sDo = (T*)sAB;
  T* sV = sDo + BT * LDV;
  T* sDH = (T*)sAB;
  float* sGam = &sX[0][0];
  // Per head: row sums of the gate gradient's terms, one slot per wave, in the padding behind every row of a tile
  auto slotC = [&](int s_, int r) -> float& { return ((float*)&sC[r * LDK + K])[s_]; };
  auto slotD = [&](int s_, int r) -> float& { return ((float*)&sD[r * LDK + K])[s_]; };

  const int tid0 = threadIdx.x;
  const int H = p.H;
  struct Item {
    ChunkLoc cl;
    int hh;
  };
  auto locate = [&](uint32_t it) {
    Item r;
    r.cl = locate_chunk_at32(it, p.offsets, p.indices, p.T, p.NTfix, H, &r.hh);
    return r;
  };
  // The rows an item starts with; requested in the last third of the item before it.
  struct Raw {
    v8 k[TK::N], q[TK::N];
    gvec g[NG];
    float gh;
  };
  auto request = [&](const Item& im, int tid, Raw& R) __attribute__((always_inline)) {
    const int64_t r0h = im.cl.row0 * H + im.hh;
    const int L = im.cl.L;
    if constexpr (PH) {
      const int row = tid >= BT ? 0 : tid < L ? tid : L - 1;   // (one wave's; the others read one word, not 64 lines)
      R.gh = ((const float*)p.g)[r0h + (int64_t)row * H];
    } else {
      constexpr int CG = K / GP;
      const char* base = (const char*)p.g + r0h * K * (int64_t)sizeof(GE);
      const uint32_t pitch = (uint32_t)H * K * (uint32_t)sizeof(GE), col = (uint32_t)(tid % CG) * 16u;
      const uint32_t lim = (uint32_t)(L - 1) * pitch + col;
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const uint32_t o = (uint32_t)((tid + 256 * i) / CG) * pitch + col;
        R.g[i] = *(const gvec*)(base + (o < lim ? o : lim));
      }
    }
    TK::load(p.k, r0h, L, H, tid, R.k);
    TK::load(p.q, r0h, L, H, tid, R.q);
  };
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6) & 3;   // (the mask tells the compiler its range)
  const int ib = wave >> 1, jb = wave & 1;
  const int ctk = RK == 2 ? wave : wave & 1, rk0 = RK == 2 ? 0 : wave >> 1;
  const int ctv = RV == 2 ? wave : wave & 1, rv0 = RV == 2 ? 0 : wave >> 1;
  // An item's first tiles to LDS (rows past the end of a short chunk zero, i.e. a gate of 1)
  auto stage = [&](const Item& im, const Raw& R) __attribute__((always_inline)) {
    FLA_PHASE(tid0);
    const int L = im.cl.L;
    if constexpr (PH) {
      if (wave == 0) {
        float x = half_prefix(lane < L ? finite_gate(R.gh) * kLog2e : 0.f);
        x += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x143, 0xC, 0xF, true));   // row_bcast:31
        sGam[lane] = x;
      }
    } else {
      constexpr int CG = K / GP;
#pragma unroll
      for (int i = 0; i < NG; ++i) {
        const int e = tid + 256 * i, row = e / CG, c = (e % CG) * GP;
        const float unit = row < L ? kLog2e : 0.f;
#pragma unroll
        for (int j = 0; j < GP; j += 4) {
          f32x4 x;
#pragma unroll
          for (int b = 0; b < 4; ++b) x[b] = finite_gate((float)R.g[i][j + b]) * unit;
          *(f32x4*)&sG[row * LDG + c + j] = x;
        }
      }
    }
    TK::put(sC, LDK, L, tid, R.k);
    TK::put(sD, LDK, L, tid, R.q);
  };

  // room for exact_scores()
  static_assert(2 * BT * LDV * 2 <= AB && (PH || BT * LDG * 4 <= AB) && kTriFloats * 4 <= BT * LDK * 2 &&
                    kTriFloats * 4 <= BT * LDT * 2,
                "tiles of the pairwise score terms");
  bool any_flagged = false;
  const uint32_t it0 = xcd_remap(blockIdx.x, gridDim.x);
  uint32_t it = it0;   // adjacent heads of a chunk at the same time on one XCD
  if (it >= nitems) return;
  Item im = locate(it);
  Raw R;
  request(im, tid0, R);
  stage(im, R);
  for (;;) {
    const ChunkLoc cl = im.cl;
    const int L = cl.L;
    const int64_t r0h = cl.row0 * H + im.hh;
    const bool flagged = p.wide && p.wide[cl.cglob * H + im.hh];
    any_flagged |= flagged;
    // what the item needs next: do and v, and the state tiles of this wave's key columns
    v8 rd[TV::N], rv[TV::N], hf[VT32][2], dhf[VT32][2];
    {
      FLA_PHASE(tid0);
      TV::load(p.dout, r0h, L, H, tid, rd);
      TV::load(p.v, r0h, L, H, tid, rv);
      const int64_t blk = (cl.cglob * H + im.hh) * (int64_t)K * V * (int64_t)sizeof(T);
      const char* hb = (const char*)p.hT + blk;
      const char* dhb = (const char*)p.dhtf + blk;
#pragma unroll
      for (int vt = 0; vt < VT32; ++vt) {
        const uint32_t o = (uint32_t)(((vt * KT32 + ctk) * 64 + lane) * 16) * (uint32_t)sizeof(T);
        hf[vt][0] = *(const v8*)(hb + o);
        hf[vt][1] = *(const v8*)(hb + o + 16);
        dhf[vt][0] = *(const v8*)(dhb + o);
        dhf[vt][1] = *(const v8*)(dhb + o + 16);
      }
    }
    lds_barrier();
    // ---- prefix sums of the gates along the lanes; q~ and k~ take the place of q and k
    float G[RK][PH ? 1 : 16];
    float glh = 0.f;   // per head: G_last
    v4 kk[RK][4];      // k in storage precision, for the epilogue
    {
      FLA_PHASE(tid0);
      if constexpr (PH) {
        glh = sGam[BT - 1];
#pragma unroll
        for (int r = 0; r < RK; ++r) G[r][0] = sGam[(rk0 + r) * 32 + l32];
      } else {
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 g[2];
#pragma unroll
          for (int r = 0; r < 2; ++r) g[r] = *(const f32x4*)&sG[(r * 32 + l32) * LDG + ctk * 32 + 8 * a + hi4];
          f32x4 gl;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const float x0 = half_prefix(g[0][b]), t0 = of_half<31>(x0);
            const float x1 = half_prefix(g[1][b]) + t0;
            if constexpr (RK == 2) {
              G[0][4 * a + b] = x0;
              G[1][4 * a + b] = x1;
            } else {
              G[0][4 * a + b] = rk0 ? x1 : x0;
            }
            gl[b] = x1;
          }
          if (l32 == 31) *(f32x4*)&sGl[wave][8 * a + hi4] = gl;
          __builtin_amdgcn_sched_barrier(0);
        }
      }
#pragma unroll
      for (int r = 0; r < RK; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int o = ((rk0 + r) * 32 + l32) * LDK + ctk * 32 + 8 * a + hi4;
          const v4 k4 = *(const v4*)&sC[o], q4 = *(const v4*)&sD[o];
          kk[r][a] = opaque(k4);   // (packed; not the fp32 copies below)
          v4 kt, qt;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            const float gg = G[r][PH ? 0 : 4 * a + b];
            kt[b] = (T)((float)k4[b] * __builtin_amdgcn_exp2f(fminf(-gg, kInvLimit)));   // e^{-G}, clamped
            qt[b] = (T)((float)q4[b] * __builtin_amdgcn_exp2f(gg));
          }
          *(v4*)&sC[o] = kt;
          *(v4*)&sD[o] = qt;
          __builtin_amdgcn_sched_barrier(0);
        }
    }
    lds_barrier();
    // ---- do, v; this wave's block of P = tril(q~ k~^T), kept until S is free
    v4 pq[4] = {};
    {
      FLA_PHASE(tid0);
      TV::put(sDo, LDV, L, tid, rd);
      TV::put(sV, LDV, L, tid, rv);
    }
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 s = zero16();
#pragma unroll
      for (int ks = 0; ks < K; ks += 16)
        s = Elem<T>::mfma32(lds_frag32<T>(sC, LDK, jb * 32, ks, lane), lds_frag32<T>(sD, LDK, ib * 32, ks, lane), s);
#pragma unroll
      for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b)
          pq[a][b] = (T)(jb * 32 + 8 * a + hi4 + b <= ib * 32 + l32 && !flagged ? s[4 * a + b] : 0.f);
    }
    lds_barrier();
    // ---- dA = tril(do v^T)
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 s = zero16();
#pragma unroll
      for (int vs = 0; vs < V; vs += 16)
        s = Elem<T>::mfma32(lds_frag32<T>(sV, LDV, jb * 32, vs, lane), lds_frag32<T>(sDo, LDV, ib * 32, vs, lane), s);
      const int i = ib * 32 + l32;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int j0 = jb * 32 + 8 * a + hi4;
        v4 x;
#pragma unroll
        for (int b = 0; b < 4; ++b) x[b] = (T)(j0 + b <= i && !flagged ? s[4 * a + b] : 0.f);
        *(v4*)&sS[i * LDT + j0] = x;
      }
    }
    lds_barrier();
    // ---- aq = dA k~ + do h^T, ak1 = dA^T q~, ak2 = v dH^T and the epilogue: dq (in place of q~), dk, the gate gradient.  One
    // row tile after the other, the first rows first (the products of the second need q~ of its own rows only): both at once
    // do not fit the registers.
    __builtin_amdgcn_sched_barrier(0);   // (nothing here waits for the states ahead of the barrier)
    v4 dkx[RK][4];
    float xs[PH ? RK : 1][PH ? 1 : 16], ks[PH ? RK : 1][PH ? 1 : 16];   // sums of the gate gradient's terms
    {
      const int lane = fresh_tid(tid0) & 63;
      float hd = 0.f;   // sum over the value columns of h dH: one key channel per lane
#pragma unroll
      for (int vt = 0; vt < VT32; ++vt)
#pragma unroll
        for (int half = 0; half < 2; ++half) hd = Elem<T>::dot8(hf[vt][half], dhf[vt][half], hd);
      hd += __shfl_xor(hd, 32, 64);
      if (lane < 32) sHd[wave][lane] = hd;
    }
#pragma unroll
    for (int r = 0; r < RK; ++r) {
      FLA_PHASE(tid0);
      const int row0 = (rk0 + r) * 32, row = row0 + l32;
      f32x16 aq = zero16(), ak1 = zero16(), ak2 = zero16();
#pragma unroll
      for (int s = 0; s < BT; s += 16) {
        if (s < row0 + 32) aq = Elem<T>::mfma32(frag32_tr<T>(sC, LDK, ctk * 32, s, lane), lds_frag32<T>(sS, LDT, row0, s, lane), aq);
        if (s >= row0) ak1 = Elem<T>::mfma32(frag32_tr<T>(sD, LDK, ctk * 32, s, lane), frag32_tr<T>(sS, LDT, row0, s, lane), ak1);
      }
#pragma unroll
      for (int vt = 0; vt < VT32; ++vt)
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          aq = Elem<T>::mfma32(hf[vt][half], lds_frag32_perm<T>(sDo, LDV, row0, vt * 32 + half * 16, lane), aq);
          ak2 = Elem<T>::mfma32(dhf[vt][half], lds_frag32_perm<T>(sV, LDV, row0, vt * 32 + half * 16, lane), ak2);
        }
      if constexpr (RK == 1) lds_barrier();   // the other wave of these columns has read q~
      if constexpr (PH) xs[r][0] = ks[r][0] = 0.f;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        f32x4 gl, hd;
        if constexpr (PH) {
          gl = f32x4{glh, glh, glh, glh};
        } else {
          gl = *(const f32x4*)&sGl[wave][8 * a + hi4];
          hd = *(const f32x4*)&sHd[wave][8 * a + hi4];
        }
        const int o = row * LDK + ctk * 32 + 8 * a + hi4;
        const v4 qt = *(const v4*)&sD[o], kt = *(const v4*)&sC[o];
        v4 dq, dk, kh;
        f32x4 dg;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          float gg = G[r][PH ? 0 : 4 * a + b];
          asm volatile("" : "+v"(gg));   // (the factors are formed again instead of being kept since q~ and k~)
          const float eg = __builtin_amdgcn_exp2f(gg), ei = __builtin_amdgcn_exp2f(fminf(-gg, kInvLimit)),
                      el = __builtin_amdgcn_exp2f(gl[b] - gg);
          const float q_ = p.scale * aq[4 * a + b], k1 = p.scale * ak1[4 * a + b], k2 = el * ak2[4 * a + b];
          const float x = (float)qt[b] * q_ - (float)kt[b] * k1, kd = (float)kk[r][a][b] * k2;
          dq[b] = (T)(eg * q_);
          dk[b] = (T)(ei * k1 + k2);
          kh[b] = (T)((float)kk[r][a][b] * el);
          if constexpr (PH) {
            xs[r][0] += x;
            ks[r][0] += kd;
          } else {
            const float su = half_suffix(x, lane), pr = half_prefix(kd);
            const float own = su + (pr - kd);
            if constexpr (RK == 1) {
              // the totals of these rows go to the wave of the other rows
              xs[0][4 * a + b] = own + __builtin_amdgcn_exp2f(gl[b]) * hd[b];
              if (l32 == 0) sX[wave][8 * a + hi4 + b] = su;
              if (l32 == 31) sKd[wave][8 * a + hi4 + b] = pr;
            } else if (r == 0) {
              xs[0][4 * a + b] = own + __builtin_amdgcn_exp2f(gl[b]) * hd[b];
              ks[0][4 * a + b] = of_half<31>(pr);
              asm volatile("" : "+v"(xs[0][4 * a + b]), "+v"(ks[0][4 * a + b]));   // (formed here, not where they are used)
            } else {
              xs[0][4 * a + b] += of_half<0>(su);
              dg[b] = own + __builtin_amdgcn_exp2f(gl[b]) * hd[b] + ks[0][4 * a + b];
            }
          }
        }
        *(v4*)&sD[o] = dq;
        dkx[r][a] = opaque(dk);   // (rounded here, not where they are stored)
        kk[r][a] = opaque(kh);
        if constexpr (!PH && RK == 2) {
          if (r == 1) {
            float* og = p.dg + (r0h + (int64_t)l32 * H) * K + ctk * 32 + 8 * a + hi4;
            if (l32 < L) *(f32x4*)og = f32x4{xs[0][4 * a], xs[0][4 * a + 1], xs[0][4 * a + 2], xs[0][4 * a + 3]};
            if (32 + l32 < L) *(f32x4*)(og + (int64_t)32 * H * K) = dg;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (PH) {
        const float x = xs[r][0] + __shfl_xor(xs[r][0], 32, 64), y = ks[r][0] + __shfl_xor(ks[r][0], 32, 64);
        if (lane < 32) {
          slotC(ctk, row) = x;
          slotD(ctk, row) = y;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();   // k~, dA and v are spent
    {
      FLA_PHASE(tid0);
      if (jb <= ib)
#pragma unroll
        for (int a = 0; a < 4; ++a) *(v4*)&sS[(ib * 32 + l32) * LDT + jb * 32 + 8 * a + hi4] = pq[a];
#pragma unroll
      for (int r = 0; r < RK; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) *(v4*)&sC[((rk0 + r) * 32 + l32) * LDK + ctk * 32 + 8 * a + hi4] = kk[r][a];
      if constexpr (PH) {
        if (wave == 0) {   // one row per lane
          float x = 0.f, y = 0.f, h = 0.f;
#pragma unroll
          for (int s = 0; s < KT32; ++s) {
            x += slotC(s, lane);
            y += slotD(s, lane);
            h += sHd[s][l32];
          }
          h = of_half<31>(half_prefix(h));
          x = half_suffix(x, lane);
          x += lane < 32 ? __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 32)) : 0.f;
          float q_ = half_prefix(y);
          q_ += lane < 32 ? 0.f : __int_as_float(__builtin_amdgcn_readlane(__float_as_int(q_), 31));
          if (lane < L) p.dg[r0h + (int64_t)lane * H] = x + (q_ - y) + __builtin_amdgcn_exp2f(glh) * h;
        }
      } else if constexpr (RK == 1) {
        const int row = rk0 * 32 + l32;
        const float* tot = rk0 ? &sKd[ctk][0] : &sX[2 + ctk][0];   // what the other rows add
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          f32x4 o = *(const f32x4*)&tot[8 * a + hi4];
#pragma unroll
          for (int b = 0; b < 4; ++b) o[b] += xs[0][4 * a + b];
          if (row < L) *(f32x4*)(p.dg + (r0h + (int64_t)row * H) * K + ctk * 32 + 8 * a + hi4) = o;
        }
      }
    }
    lds_barrier();
    {
      FLA_PHASE(tid0);
      v8 x[TK::N];
      TK::get(sD, LDK, tid, x);
      TK::store(p.dq, r0h, L, H, tid, x);
    }
    const uint32_t nit = it + gridDim.x;
    const bool more = nit < nitems;             // workgroup-uniform
    const Item nim = locate(more ? nit : it);   // (past the last item the request repeats it: no load under a branch)
    request(nim, fresh_tid(tid0), R);
    // ---- dv = s P^T do + k^ dH
    f32x16 dv[RV];
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int r = 0; r < RV; ++r) dv[r] = zero16();
#pragma unroll
      for (int s = 0; s < BT; s += 16) {
        const v8 f = frag32_tr<T>(sDo, LDV, ctv * 32, s, lane);
#pragma unroll
        for (int r = 0; r < RV; ++r)
          if (s >= (rv0 + r) * 32) dv[r] = Elem<T>::mfma32(f, frag32_tr<T>(sS, LDT, (rv0 + r) * 32, s, lane), dv[r]);
      }
#pragma unroll
      for (int r = 0; r < RV; ++r)
#pragma unroll
        for (int e = 0; e < 16; ++e) dv[r][e] *= p.scale;
    }
    lds_barrier();   // do and P are spent, dq is on its way
    {
      FLA_PHASE(tid0);
      if (RK == 2 || rk0 == 0) {   // (with 64 key columns waves 2 and 3 hold the tiles of waves 0 and 1)
#pragma unroll
        for (int vt = 0; vt < VT32; ++vt)
#pragma unroll
          for (int half = 0; half < 2; ++half) {
            T* o = &sDH[(ctk * 32 + l32) * LDV + vt * 32 + half * 16 + hi4];
            const v8 x = dhf[vt][half];
            *(v4*)o = __builtin_shufflevector(x, x, 0, 1, 2, 3);
            *(v4*)(o + 8) = __builtin_shufflevector(x, x, 4, 5, 6, 7);
          }
      }
#pragma unroll
      for (int r = 0; r < RK; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) *(v4*)&sD[((rk0 + r) * 32 + l32) * LDK + ctk * 32 + 8 * a + hi4] = dkx[r][a];
    }
    lds_barrier();
    {
      FLA_PHASE(tid0);
      v8 x[TK::N];
      TK::get(sD, LDK, tid, x);
      TK::store(p.dk, r0h, L, H, tid, x);
    }
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int s = 0; s < K; s += 16) {
        const v8 f = frag32_tr<T>(sDH, LDV, ctv * 32, s, lane);
#pragma unroll
        for (int r = 0; r < RV; ++r) dv[r] = Elem<T>::mfma32(f, lds_frag32<T>(sC, LDK, (rv0 + r) * 32, s, lane), dv[r]);
      }
    }
    lds_barrier();   // k^ is spent: its tile takes dv
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int r = 0; r < RV; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          v4 x;
#pragma unroll
          for (int b = 0; b < 4; ++b) x[b] = (T)dv[r][4 * a + b];
          *(v4*)&sC[((rv0 + r) * 32 + l32) * LDV + ctv * 32 + 8 * a + hi4] = x;
        }
    }
    lds_barrier();
    v8 dvx[TV::N];
    TV::get(sC, LDV, fresh_tid(tid0), dvx);
    // (the next item's tiles are written ahead of this item's last stores: the wait for their loads would otherwise be a wait
    // for the stores in front of them as well)
    if (more) {
      lds_barrier();
      stage(nim, R);
    }
    TV::store(p.dv, r0h, L, H, fresh_tid(tid0), dvx);
    if (!more) break;
    it = nit;
    im = nim;
  }
  if (!any_flagged) return;   // workgroup-uniform
  for (it = it0; it < nitems; it += gridDim.x) {
    im = locate(it);
    if (!p.wide[im.cl.cglob * H + im.hh]) continue;
    __syncthreads();   // (what this workgroup stored is what it reads back)
    exact_scores<T, GT, K, V>(p, im.cl, im.hh, sAB, sC, sD, (float*)sS, sGam);
  }
}

template <typename T, typename GT>
int launch_gla_chunk(const GlaChunkParams& p, int64_t K, int64_t V, int64_t total, hipStream_t st) {
#define LAUNCH(KK, VV)                                                                                                   \
  {                                                                                                                      \
    const int64_t res = resident_workgroups(gla_bwd_chunk_kernel<T, GT, KK, VV>);                                        \
    hipLaunchKernelGGL((gla_bwd_chunk_kernel<T, GT, KK, VV>), dim3((unsigned)(total < res ? total : res)), dim3(256), 0, \
                       st, p, (uint32_t)total);                                                                          \
  }
  if (K == 128 && V == 128) LAUNCH(128, 128)
  else if (K == 64 && V == 64) LAUNCH(64, 64)
  else if (K == 128 && V == 64) LAUNCH(128, 64)
  else if (K == 64 && V == 128) LAUNCH(64, 128)
  else return FLA_E_UNSUPPORTED;
#undef LAUNCH
  FLA_CHECK_LAUNCH();
  return FLA_OK;
}

}  // namespace

int gla_bwd_chunk(const void* q, const void* k, const void* v, const void* g, const void* dout, const void* hT,
                  const void* dhT, const int* wide, void* dq, void* dk, void* dv, float* dg, const int64_t* offsets,
                  const int64_t* indices, int64_t chunks, int ntfix, int qkv_dtype, int gate_dtype, bool head_gates, int64_t T,
                  int64_t H, int64_t K, int64_t V, float scale, hipStream_t st) {
  const int64_t total = chunks * H;
  FLA_REQUIRE(total <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
  GlaChunkParams p{q, k, v, g, dout, hT, dhT, wide, dq, dk, dv, dg, offsets, indices, T, (int)H, ntfix, scale};
#define GLA_CHUNK(TT, GG) return launch_gla_chunk<TT, GG>(p, K, V, total, st)
  if (head_gates && qkv_dtype == FLA_BF16) GLA_CHUNK(bf16, PerHead);
  if (head_gates && qkv_dtype == FLA_F16) GLA_CHUNK(f16, PerHead);
  if (head_gates) return FLA_E_UNSUPPORTED;
  if (qkv_dtype == FLA_BF16 && gate_dtype == FLA_F32) GLA_CHUNK(bf16, float);
  if (qkv_dtype == FLA_BF16 && gate_dtype == FLA_BF16) GLA_CHUNK(bf16, bf16);
  if (qkv_dtype == FLA_F16 && gate_dtype == FLA_F32) GLA_CHUNK(f16, float);
  if (qkv_dtype == FLA_F16 && gate_dtype == FLA_F16) GLA_CHUNK(f16, f16);
#undef GLA_CHUNK
  return FLA_E_UNSUPPORTED;
}
