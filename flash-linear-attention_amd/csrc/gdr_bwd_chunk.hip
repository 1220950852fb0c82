// The chunk-parallel half of the gated delta rule backward in one launch: what follows the reverse state scan
// (gdr_bwd.hip) - dq, dk, dw and their gate terms (fla/ops/common/chunk_o.py:602-...) and the gradient through the WY
// representation (fla/ops/gated_delta_rule/wy_fast.py:429-560) - formed by one workgroup per (chunk, head).
//
// What bounds it: bytes.  q, k, v, v_new, do, dv2, Aw and the two states enter once, dq, dk and dv leave once (0.91 GB for
// 4 x 4096 tokens, 16 heads, K = V = 128); dw, the part of dk that does not go through the inverse and the partial gate
// gradients stay on the chip, and w is not needed: its gate term is the row sum of w . dw = Aw ((dw k^T) diag beta), whose
// second factor the WY gradient forms anyway.  191 us there, 4.75 TB/s (a large copy: 5.0; 195 behind the reverse scan, 202
// inside a training step), where the two launches it replaces took 200 + 146 us for 1.3 GB; 2 x 2048 tokens 50 us instead of
// 50 + 39.
#include "chunk_rows.h"
#include "gdr_bwd_chunk.h"

namespace {

struct ChunkBwdParams {
  const void* q;
  const void* k;
  const void* v;
  const void* vnew;
  const void* dout;
  const void* dv2;
  const float* beta;
  const float* gam;    // chunk-local prefix sums of the gate, or NULL
  const void* Aw;
  const void* hT;      // forward states, FLA_H_FRAGMENT_T
  const void* dhtf;    // dH, FLA_H_FRAGMENT_T
  void* dq;
  void* dk;
  void* dv;
  float* dbeta;
  float* dg;           // gradient of the raw gate
  const int64_t* offsets;
  const int64_t* indices;
  int64_t T;
  int H, NTfix;
  float scale;
};

// Four waves.  In products with K (V) result columns a wave owns 32 of them and, with 128 columns, all 64 rows, with 64
// columns one half of the rows: what a wave later needs of such a result (gate terms, in-place replacement of q by dq, k
// by dk, v by dv) it finds in its own columns.  In the 64 x 64 products waves 0, 2 and 3 own the three 32 x 32 blocks on and
// below the diagonal.  All products with a wide result are formed transposed (the state or the transposed tile as the first
// operand): a lane then owns one time row and, per register quad, four adjacent columns.
// Five tiles fit 80 KB, i.e. two workgroups per CU, because each is reused as its contents are spent:
//   A: do -> dv2 -> dw -> dM diag(beta)    B: v_new -> v -> dv    C: k -> dk
//   D: q -> dq -> Au | - -> dA, later dM | X1    S: ds -> Aw
template <typename T, int K, int V>
__global__ __launch_bounds__(256, 2) void gdr_bwd_chunk_kernel(ChunkBwdParams p, uint32_t nitems) {
  typedef typename Elem<T>::v8 v8;
  typedef typename Elem<T>::v4 v4;
  typedef RowTile<T, K> TK;
  typedef RowTile<T, V> TV;
  typedef RowTile<T, BT> TA;
  constexpr int LDK = K + 8, LDV = V + 8, LDA = LDK > LDV ? LDK : LDV;
  constexpr int VT32 = V / 32, KT32 = K / 32;
  constexpr int RK = K / 64, RV = V / 64;   // row tiles of a wave in products with K (V) result columns
  constexpr int SD = BT * LDK > 2 * BT * LDT ? BT * LDK : 2 * BT * LDT;
  __shared__ __attribute__((aligned(16))) T sA[BT * LDA];
  __shared__ __attribute__((aligned(16))) T sB[BT * LDV];
  __shared__ __attribute__((aligned(16))) T sC[BT * LDK];
  __shared__ __attribute__((aligned(16))) T sD[SD];
  __shared__ __attribute__((aligned(16))) T sS[BT * LDT];
  __shared__ __attribute__((aligned(16))) float sGam[BT], sBeta[BT];
  // Row sums of dgamma from the two column blocks and column sums from the two row blocks of the score products
  __shared__ float sRow[2][BT], sCol[2][BT];
  __shared__ float sKin[4], sHd[4];
  T* sD1 = sD;
  T* sD2 = sD + BT * LDT;
  // Partial row sums, one slot per contributing wave, added in a fixed order (no atomics: the gradients are
  // bit-reproducible).  They live in the 16 bytes of padding behind every tile row, which no tile access touches.
  auto slotB = [&](int s_, int r) -> float& { return ((float*)&sB[r * LDV + V])[s_]; };      // dbeta, value side
  auto slotC = [&](int s_, int r) -> float& { return ((float*)&sC[r * LDK + K])[s_]; };      // dgamma: q dq - k dk
  auto slotS = [&](int s_, int r) -> float& { return ((float*)&sS[r * LDT + BT])[s_]; };     // dbeta, key side

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
  // The rows an item starts with; requested while the item before it is in its last third.
  struct Raw {
    v8 d[TV::N], vn[TV::N], k[TK::N], q[TK::N];
    float gam, beta;
  };
  auto request = [&](const Item& im, int tid, Raw& R) __attribute__((always_inline)) {
    const int64_t r0h = im.cl.row0 * H + im.hh;
    TV::load(p.dout, r0h, im.cl.L, H, tid, R.d);
    TV::load(p.vnew, r0h, im.cl.L, H, tid, R.vn);
    TK::load(p.k, r0h, im.cl.L, H, tid, R.k);
    TK::load(p.q, r0h, im.cl.L, H, tid, R.q);
    // a column of 64 gates is 64 requests to the L2: the waves that do not use it read one word
    const int row = tid >= BT ? 0 : tid < im.cl.L ? tid : im.cl.L - 1;
    R.beta = p.beta[r0h + (int64_t)row * H];
    R.gam = *(p.gam ? p.gam + r0h + (int64_t)row * H : &kZeroWord);   // (without gates one zero word: no branch)
  };
  const int wave = __builtin_amdgcn_readfirstlane(tid0 >> 6) & 3;   // (the mask tells the compiler its range)
  const int ib = wave >> 1, jb = wave & 1;
  const int ctk = RK == 2 ? wave : wave & 1, rk0 = RK == 2 ? 0 : wave >> 1;
  const int ctv = RV == 2 ? wave : wave & 1, rv0 = RV == 2 ? 0 : wave >> 1;
  // An item's first tiles to LDS
  auto stage = [&](const Item& im, const Raw& R) __attribute__((always_inline)) {
    FLA_PHASE(tid0);
    const int L = im.cl.L;
    TV::put(sA, LDV, L, tid, R.d);
    TV::put(sB, LDV, L, tid, R.vn);
    TK::put(sC, LDK, L, tid, R.k);
    TK::put(sD, LDK, L, tid, R.q);
    if (tid < BT) {
      sGam[tid] = R.gam;
      sBeta[tid] = tid < L ? R.beta : 0.f;
      if (tid < 32) sRow[1][tid] = 0.f;   // the block above the diagonal contributes nothing
      else sCol[0][tid] = 0.f;
    }
  };
  // adjacent items, i.e. adjacent heads of a chunk, run on one XCD at the same time (198 -> 191 us)
  uint32_t it = xcd_remap(blockIdx.x, gridDim.x);
  if (it >= nitems) return;
  Item im = locate(it);
  Raw R;
  request(im, tid0, R);
  stage(im, R);
  for (;;) {
    const ChunkLoc cl = im.cl;
    const int L = cl.L;
    const int64_t r0h = cl.row0 * H + im.hh;
    // what the item needs behind ds: the state tiles of this wave's key columns and the value side of the WY gradient
    v8 hf[VT32][2], dhf[VT32][2];
    v8 rd2[TV::N], rv[TV::N], ra[TA::N];
    {
      FLA_PHASE(tid0);
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
      TV::load(p.dv2, r0h, L, H, tid, rd2);
      TV::load(p.v, r0h, L, H, tid, rv);
      TA::load(p.Aw, r0h, L, H, tid, ra);
    }
    lds_barrier();
    // ---- ds = s tril((do v_new^T) * Gamma), row-major
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 s = zero16();
#pragma unroll
      for (int vs = 0; vs < V; vs += 16)
        s = Elem<T>::mfma32(lds_frag32<T>(sB, LDV, jb * 32, vs, lane), lds_frag32<T>(sA, LDV, ib * 32, vs, lane), s);
      const int i = ib * 32 + l32;
      const float gi = sGam[i];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int j0 = jb * 32 + 8 * a + hi4;
        const f32x4 gj = *(const f32x4*)&sGam[j0];
        v4 x;
#pragma unroll
        for (int b = 0; b < 4; ++b) x[b] = (T)(j0 + b <= i ? s[4 * a + b] * p.scale * __expf(gi - gj[b]) : 0.f);
        *(v4*)&sS[i * LDT + j0] = x;
      }
    }
    lds_barrier();
    // ---- dq = s e^gamma (do h^T) + ds k ;  dk so far = e^{gamma_last - gamma} (v_new dH^T) + ds^T q
    f32x16 aq[RK], ak[RK];
#pragma unroll
    for (int r = 0; r < RK; ++r) aq[r] = ak[r] = zero16();
    const float glast = sGam[L - 1];
    {
    FLA_PHASE(tid0);
    float hd = 0.f;   // <h, dH> over this wave's tiles (the same fragment order on both sides)
#pragma unroll
    for (int vt = 0; vt < VT32; ++vt)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        hd = Elem<T>::dot8(hf[vt][half], dhf[vt][half], hd);
#pragma unroll
        for (int r = 0; r < RK; ++r) {
          const int row0 = (rk0 + r) * 32, c0 = vt * 32 + half * 16;
          aq[r] = Elem<T>::mfma32(hf[vt][half], lds_frag32_perm<T>(sA, LDV, row0, c0, lane), aq[r]);
          ak[r] = Elem<T>::mfma32(dhf[vt][half], lds_frag32_perm<T>(sB, LDV, row0, c0, lane), ak[r]);
        }
      }
    float kin = 0.f;   // sum of k * the inter-chunk part of dk
#pragma unroll
    for (int r = 0; r < RK; ++r) {
      const int row = (rk0 + r) * 32 + l32;
      const float gm = sGam[row], eq = p.scale * __expf(gm), ek = __expf(glast - gm);
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const v4 kk = *(const v4*)&sC[row * LDK + ctk * 32 + 8 * a + hi4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          aq[r][4 * a + b] *= eq;
          ak[r][4 * a + b] *= ek;
          kin += (float)kk[b] * ak[r][4 * a + b];
        }
      }
    }
#pragma unroll
    for (int s = 0; s < BT; s += 16) {
      const v8 fk = frag32_tr<T>(sC, LDK, ctk * 32, s, lane), fq = frag32_tr<T>(sD, LDK, ctk * 32, s, lane);
#pragma unroll
      for (int r = 0; r < RK; ++r) {
        const int row0 = (rk0 + r) * 32;
        if (s < row0 + 32) aq[r] = Elem<T>::mfma32(fk, lds_frag32<T>(sS, LDT, row0, s, lane), aq[r]);
        if (s >= row0) ak[r] = Elem<T>::mfma32(fq, frag32_tr<T>(sS, LDT, row0, s, lane), ak[r]);
      }
    }
    if constexpr (RK == 1) lds_barrier();   // the other wave of these columns has read q
#pragma unroll
    for (int r = 0; r < RK; ++r) {
      const int row = (rk0 + r) * 32 + l32;
      float part = 0.f;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int o = row * LDK + ctk * 32 + 8 * a + hi4;
        const v4 kk = *(const v4*)&sC[o], qq = *(const v4*)&sD[o];
        v4 x;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          part += (float)qq[b] * aq[r][4 * a + b] - (float)kk[b] * ak[r][4 * a + b];
          x[b] = (T)aq[r][4 * a + b];
        }
        *(v4*)&sD[o] = x;   // dq takes the place of the q elements this lane has just read
      }
      part += __shfl_xor(part, 32, 64);
      if (lane < 32) slotC(ctk, row) = part;
    }
    kin = wave_sum_lane63(kin);
    hd = wave_sum_lane63(hd);
    if (lane == 63) {
      sKin[wave] = kin;
      sHd[wave] = hd;
    }
    }
    lds_barrier();   // do, v_new and ds are spent
    {
      FLA_PHASE(tid0);
      TV::put(sA, LDV, L, tid, rd2);
      TV::put(sB, LDV, L, tid, rv);
#pragma unroll
      for (int i = 0; i < TA::N; ++i) {
        const int e = tid + 256 * i, row = e / 8, c8 = (e % 8) * 8;
        if (row >= L)   // rows past the end: identity
#pragma unroll
          for (int j = 0; j < 8; ++j) ra[i][j] = (T)(c8 + j == row ? 1.f : 0.f);
        *(v8*)&sS[row * LDT + c8] = ra[i];
      }
    }
    lds_barrier();
    {
      FLA_PHASE(tid0);
      v8 x[TK::N];
      TK::get(sD, LDK, tid, x);
      TK::store(p.dq, r0h, L, H, tid, x);
    }
    // ---- dw = -e^gamma (dv2 h^T) ; dAu = (dv2 v^T) diag(beta)
    f32x16 aw[RK], dAu = zero16();
#pragma unroll
    for (int r = 0; r < RK; ++r) aw[r] = zero16();
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int vt = 0; vt < VT32; ++vt)
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int r = 0; r < RK; ++r)
            aw[r] = Elem<T>::mfma32(hf[vt][half], lds_frag32_perm<T>(sA, LDV, (rk0 + r) * 32, vt * 32 + half * 16, lane), aw[r]);
    }
    if (jb <= ib) {
      FLA_PHASE(tid0);
#pragma unroll
      for (int vs = 0; vs < V; vs += 16)
        dAu = Elem<T>::mfma32(lds_frag32<T>(sB, LDV, jb * 32, vs, lane), lds_frag32<T>(sA, LDV, ib * 32, vs, lane), dAu);
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const f32x4 bj = *(const f32x4*)&sBeta[jb * 32 + 8 * a + hi4];
#pragma unroll
        for (int b = 0; b < 4; ++b) dAu[4 * a + b] *= bj[b];
      }
    }
    lds_barrier();   // dq is on its way: its tile takes Au_ij = Aw_ij e^{gamma_i - gamma_j}, i >= j
    {
      FLA_PHASE(tid0);
      const int c8 = (tid % 8) * 8;
      const f32x4 g0 = *(const f32x4*)&sGam[c8], g1 = *(const f32x4*)&sGam[c8 + 4];
#pragma unroll
      for (int i = 0; i < TA::N; ++i) {
        const int row = (tid + 256 * i) / 8;
        const float gi = sGam[row];
        v8 x;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          x[j] = (T)(c8 + j <= row ? (float)ra[i][j] * __expf(gi - (j < 4 ? g0[j & 3] : g1[j & 3])) : 0.f);
        *(v8*)&sD1[row * LDT + c8] = x;
      }
    }
    lds_barrier();
    // ---- value side: d(vb) = Au^T dv2 ; dv = beta d(vb) ; dbeta += sum_v d(vb) v
    v4 dvst[RV][4];
    {
      FLA_PHASE(tid0);
      f32x16 dvb[RV];
#pragma unroll
      for (int r = 0; r < RV; ++r) dvb[r] = zero16();
#pragma unroll
      for (int s = 0; s < BT; s += 16) {
        const v8 f = frag32_tr<T>(sA, LDV, ctv * 32, s, lane);
#pragma unroll
        for (int r = 0; r < RV; ++r)
          if (s >= (rv0 + r) * 32) dvb[r] = Elem<T>::mfma32(f, frag32_tr<T>(sD1, LDT, (rv0 + r) * 32, s, lane), dvb[r]);
      }
#pragma unroll
      for (int r = 0; r < RV; ++r) {
        const int row = (rv0 + r) * 32 + l32;
        const float bj = sBeta[row];
        float part = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const v4 vv = *(const v4*)&sB[row * LDV + ctv * 32 + 8 * a + hi4];
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            part += dvb[r][4 * a + b] * (float)vv[b];
            dvst[r][a][b] = (T)(dvb[r][4 * a + b] * bj);
          }
        }
        part += __shfl_xor(part, 32, 64);
        if (lane < 32) slotB(ctv, row) = part;
      }
    }
    lds_barrier();   // dv2, v and Au are spent
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int r = 0; r < RV; ++r)
#pragma unroll
        for (int a = 0; a < 4; ++a) *(v4*)&sB[((rv0 + r) * 32 + l32) * LDV + ctv * 32 + 8 * a + hi4] = dvst[r][a];
#pragma unroll
      for (int r = 0; r < RK; ++r) {
        const int row = (rk0 + r) * 32 + l32;
        const float ew = -__expf(sGam[row]);
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          v4 x;
#pragma unroll
          for (int b = 0; b < 4; ++b) x[b] = (T)(aw[r][4 * a + b] * ew);
          *(v4*)&sA[row * LDK + ctk * 32 + 8 * a + hi4] = x;
        }
      }
    }
    lds_barrier();
    {
      FLA_PHASE(tid0);
      v8 x[TV::N];
      TV::get(sB, LDV, tid, x);
      TV::store(p.dv, r0h, L, H, tid, x);
    }
    const uint32_t nit = it + gridDim.x;
    const bool more = nit < nitems;             // workgroup-uniform
    const Item nim = locate(more ? nit : it);   // (past the last item the request repeats it: no load under a branch)
    request(nim, fresh_tid(tid0), R);
    // ---- key side: d(kb) = Aw^T dw ; dAw = (dw k^T) diag(beta) ; dA = strict_lower(dAw + dAu * Gamma)
    f32x16 dkb[RK];
#pragma unroll
    for (int r = 0; r < RK; ++r) dkb[r] = zero16();
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int s = 0; s < BT; s += 16) {
        const v8 f = frag32_tr<T>(sA, LDK, ctk * 32, s, lane);
#pragma unroll
        for (int r = 0; r < RK; ++r)
          if (s >= (rk0 + r) * 32) dkb[r] = Elem<T>::mfma32(f, frag32_tr<T>(sS, LDT, (rk0 + r) * 32, s, lane), dkb[r]);
      }
    }
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 dA = zero16();
#pragma unroll
      for (int ks = 0; ks < K; ks += 16)
        dA = Elem<T>::mfma32(lds_frag32<T>(sC, LDK, jb * 32, ks, lane), lds_frag32<T>(sA, LDK, ib * 32, ks, lane), dA);
      const int i = ib * 32 + l32;
      const float gi = sGam[i];
      float rs = 0.f;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int j0 = jb * 32 + 8 * a + hi4;
        const f32x4 gj = *(const f32x4*)&sGam[j0], bj = *(const f32x4*)&sBeta[j0];
        const v4 aw4 = *(const v4*)&sS[i * LDT + j0];
        v4 tot;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const int j = j0 + b;
          const float d1 = dA[4 * a + b] * bj[b], w = (float)aw4[b];
          const float dg = dAu[4 * a + b] * (j < i ? __expf(gi - gj[b]) : 0.f);
          const float x = j < i ? dg * w : 0.f;   // dAu * Au below the diagonal: + at row i, - at row j
          rs += x + (j <= i ? w * d1 : 0.f);                     // (w d1: the row sums of w dw)
          tot[b] = (T)(j < i ? d1 + dg : 0.f);
          const float cs = half_wave_sum_hi(x);
          if (l32 == 16) sCol[ib][j] = -cs;
        }
        *(v4*)&sD1[i * LDT + j0] = tot;
      }
      rs += __shfl_xor(rs, 32, 64);
      if (lane < 32) sRow[jb][i] = rs;
    }
    lds_barrier();
    // ---- X1 = dA Aw^T, stored transposed; dM = -strict_lower(Aw^T X1) and, for the transposed product, its rows times beta
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 x1 = zero16();
      for (int s = 0; s < (jb + 1) * 32; s += 16)   // Aw_jb is zero for b > j
        x1 = Elem<T>::mfma32(lds_frag32<T>(sD1, LDT, ib * 32, s, lane), lds_frag32<T>(sS, LDT, jb * 32, s, lane), x1);
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        v4 x;
#pragma unroll
        for (int b = 0; b < 4; ++b) x[b] = (T)x1[4 * a + b];
        *(v4*)&sD2[(jb * 32 + l32) * LDT + ib * 32 + 8 * a + hi4] = x;   // X1^T[j][a]
      }
    }
    lds_barrier();
    if (jb <= ib) {
      FLA_PHASE(tid0);
      f32x16 m = zero16();
      for (int s = ib * 32; s < BT; s += 16)   // Aw_ai is zero for a < i
        m = Elem<T>::mfma32(lds_frag32<T>(sD2, LDT, jb * 32, s, lane), frag32_tr<T>(sS, LDT, ib * 32, s, lane), m);
      const int i = ib * 32 + l32;
      const float bi = sBeta[i];
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int j0 = jb * 32 + 8 * a + hi4;
        v4 x, y;
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          const float z = j0 + b < i ? -m[4 * a + b] : 0.f;
          x[b] = (T)z;
          y[b] = (T)(z * bi);
        }
        *(v4*)&sD1[i * LDT + j0] = x;
        *(v4*)&sA[i * LDT + j0] = y;
      }
    }
    lds_barrier();
    // ---- d(kb) += dM k ; dk += (dM^T diag(beta)) k + beta d(kb) ; dbeta += sum_k d(kb) k
    {
      FLA_PHASE(tid0);
#pragma unroll
      for (int s = 0; s < BT; s += 16) {
        const v8 f = frag32_tr<T>(sC, LDK, ctk * 32, s, lane);
#pragma unroll
        for (int r = 0; r < RK; ++r) {
          const int row0 = (rk0 + r) * 32;
          if (s < row0 + 32) dkb[r] = Elem<T>::mfma32(f, lds_frag32<T>(sD1, LDT, row0, s, lane), dkb[r]);
          if (s >= row0) ak[r] = Elem<T>::mfma32(f, frag32_tr<T>(sA, LDT, row0, s, lane), ak[r]);
        }
      }
      if constexpr (RK == 1) lds_barrier();   // the other wave of these columns has read k
#pragma unroll
      for (int r = 0; r < RK; ++r) {
        const int row = (rk0 + r) * 32 + l32;
        const float bj = sBeta[row];
        float part = 0.f;
#pragma unroll
        for (int a = 0; a < 4; ++a) {
          const int o = row * LDK + ctk * 32 + 8 * a + hi4;
          const v4 kk = *(const v4*)&sC[o];
          v4 x;
#pragma unroll
          for (int b = 0; b < 4; ++b) {
            part += dkb[r][4 * a + b] * (float)kk[b];
            x[b] = (T)(ak[r][4 * a + b] + dkb[r][4 * a + b] * bj);
          }
          *(v4*)&sC[o] = x;   // dk takes the place of the k elements this lane has just read
        }
        part += __shfl_xor(part, 32, 64);
        if (lane < 32) slotS(ctk, row) = part;
      }
    }
    lds_barrier();
    v8 dkx[TK::N];
    TK::get(sC, LDK, fresh_tid(tid0), dkx);
    float db = 0.f, dgm = 0.f;
    if (wave == 0) {   // one row per lane
      const int lane = fresh_tid(tid0) & 63;
#pragma unroll
      for (int s = 0; s < VT32; ++s) db += slotB(s, lane);
#pragma unroll
      for (int s = 0; s < KT32; ++s) {
        db += slotS(s, lane);
        dgm += slotC(s, lane);
      }
      dgm += (sRow[0][lane] + sRow[1][lane]) + (sCol[0][lane] + sCol[1][lane]);
      if (lane == L - 1) {
        // (with 64 key columns waves 2 and 3 hold the tiles of waves 0 and 1)
        const float hd_all = RK == 2 ? (sHd[0] + sHd[1]) + (sHd[2] + sHd[3]) : sHd[0] + sHd[1];
        dgm += (sKin[0] + sKin[1]) + (sKin[2] + sKin[3]) + __expf(glast) * hd_all;
      }
      // inclusive suffix sum over the 64 rows (the gate's reverse chunk-local cumulative sum): DPP row scans plus the
      // totals of the later rows of 16
      dgm = row_suffix16(lane < L ? dgm : 0.f);
      const float t1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dgm), 16));
      const float t2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dgm), 32));
      const float t3 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dgm), 48));
      const int r = lane >> 4;
      dgm += (r < 1 ? t1 : 0.f) + (r < 2 ? t2 : 0.f) + (r < 3 ? t3 : 0.f);
    }
    // The next item's tiles are written ahead of this item's last stores: a wait for
    // a load would otherwise be a wait for the stores in front of it as well.
    if (more) {
      lds_barrier();   // dk and the row sums are read
      stage(nim, R);
    }
    {
      FLA_PHASE(tid0);
      TK::store(p.dk, r0h, L, H, tid, dkx);
      if (tid < BT && tid < L) {
        p.dbeta[r0h + (int64_t)tid * H] = db;
        p.dg[r0h + (int64_t)tid * H] = dgm;
      }
    }
    if (!more) break;
    it = nit;
    im = nim;
  }
}

template <typename T>
int launch_chunk_bwd(const ChunkBwdParams& p, int64_t K, int64_t V, int64_t total, hipStream_t st) {
#define LAUNCH(KK, VV)                                                                                                     \
  {                                                                                                                        \
    const int64_t res = resident_workgroups(gdr_bwd_chunk_kernel<T, KK, VV>);                                              \
    hipLaunchKernelGGL((gdr_bwd_chunk_kernel<T, KK, VV>), dim3((unsigned)(total < res ? total : res)), dim3(256), 0, st, p, \
                       (uint32_t)total);                                                                                   \
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

int gdr_bwd_chunk(const void* q, const void* k, const void* v, const void* v_new, const float* beta, const float* g_cumsum,
                  const void* Aw, const void* dout, const void* dv2, const void* hT, const void* dhT, void* dq, void* dk,
                  void* dv, float* dbeta, float* dg, const int64_t* offsets, const int64_t* indices, int64_t chunks,
                  int ntfix, int qkv_dtype, int64_t T, int64_t H, int64_t K, int64_t V, float scale, hipStream_t st) {
  const int64_t total = chunks * H;
  FLA_REQUIRE(total <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
  ChunkBwdParams p{q, k, v, v_new, dout, dv2, beta, g_cumsum, Aw, hT, dhT, dq, dk, dv, dbeta, dg, offsets, indices,
                   T, (int)H, ntfix, scale};
  if (qkv_dtype == FLA_BF16) return launch_chunk_bwd<bf16>(p, K, V, total, st);
  if (qkv_dtype == FLA_F16) return launch_chunk_bwd<f16>(p, K, V, total, st);
  return FLA_E_UNSUPPORTED;
}
