// The two launches ahead of a delta-rule scan over sequences cut into segments (seq_split.h): what every segment adds to a
// zero state and its K x K transition, and the fold of these into the states entering the segments.
//
// Over one chunk the state is an affine function of the state entering it,
//   h <- e^{gamma_last} h + k^T (e^{gamma_last - gamma} * Tu (v - e^{gamma} * (k h)))
// so a segment takes h to M h + S: S is the recurrence from a zero state, M the same recurrence on the identity with
// v = 0.  The recurrence is independent per column, and the V columns of S and the K columns of M are walked side by
// side with the arithmetic of the scan (gdr_fwd_fused.hip: state in fp32 accumulators, 16-bit operands).
//
// gdr_split_pass_kernel: a workgroup of four waves takes 128 of the V + K columns of one (segment, head), 32 per wave as two
// 16-column blocks, so that an operand read from LDS serves two matrix instructions (16 columns per wave: twice the LDS
// reads), beside four waves that stage the tiles.  Neither q nor an output is touched: a chunk costs 21 KB of k and Tu, and
// 16 KB of v for the columns of S, and its load latency is longer than its arithmetic: the staging waves hold three chunks
// in registers: 2.0 us per chunk (23 us for 7 segments of 10 chunks of 16 heads, K = V = 128).  Tiles staged by the waves
// that multiply, one chunk ahead: 3.9 - 4.5 us.
// gdr_split_fold_kernel: h <- M h + S; a workgroup carries 16 value columns of one head through the segments, 16 key rows
// per wave.  The state is fp32 in the scan and stays so between the segments: M and h are multiplied as sums of three bf16
// numbers (exactly their 24 bits; eight products, the ninth is below 2^-30 of the result), a transition that is the
// identity hands on every bit.  M is stored in fp32, in operand order, and requested two segments ahead: a step is 64 KB of
// M into every CU, 15.4 us for 7 steps.  Two bf16 numbers apiece and three products lost the last 8 bits for 11.5 us (forward
// of one sequence of 5003 tokens, 16 heads: 80.4 against 84.0); M split a step ahead out of three register sets: 15.6 us;
// fp32 M in rows, 16x16x4 fp32 instructions, one segment ahead: 2.1 us per segment.
#include "seq_split.h"

namespace {

struct GdrPassParams {
  const void* k;
  const void* v;
  const void* AT;       // [chunks, H, 10, 16, 16]: Tu
  const float* gam;     // chunk-local prefix sums of the gate, or NULL
  const float* rk;      // L2N: 1 / |k|, [rows, H]
  float* states;        // out: S, [slots, H, K, V]
  float* trans;         // out: M, [slots, H, K/32 slices, K/16 row tiles, 2, 64 lanes, 4]
  float* trans_t;       // out, or NULL: M^T in the same order
  const int64_t* offsets;
  const int64_t* chunk_offsets;
  SplitView split;
  int64_t T;
  int H, per_seq, col_wgs;
};

// Eight fp32 numbers as sums of three bf16 numbers each, exactly: 8 significant bits apiece, cut off, never rounded up (a
// finite number stays finite).
FLA_DEVICE void split3(f32x4 a, f32x4 b, bf16x8* out) {
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  u4 w[3];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float x0 = i < 2 ? a[2 * i] : b[2 * i - 4], x1 = i < 2 ? a[2 * i + 1] : b[2 * i - 3];
#pragma unroll
    for (int part = 0; part < 3; ++part) {
      const uint32_t u0 = __float_as_uint(x0), u1 = __float_as_uint(x1);
      w[part][i] = __builtin_amdgcn_perm(u1, u0, 0x07060302);   // the upper halves, x0's in the low one
      x0 -= __uint_as_float(u0 & 0xffff0000u);
      x1 -= __uint_as_float(u1 & 0xffff0000u);
    }
  }
#pragma unroll
  for (int part = 0; part < 3; ++part) out[part] = __builtin_bit_cast(bf16x8, w[part]);
}

template <typename T, int K, int V, bool L2N>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdr_split_pass_kernel(GdrPassParams p) {
  typedef typename Elem<T>::v8 v8;
  typedef typename Elem<T>::v4 v4;
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4 lds_s4;
  constexpr int LDR = K + 8, LDV = V + 8;
  constexpr int KS = K / 32, KT = K / 16;
  constexpr int CK = K / 8, NPK = BT * CK / 256, CV = V / 8, NPV = BT * CV / 256;
  __shared__ __attribute__((aligned(16))) T sK[2][BT * LDR];
  __shared__ __attribute__((aligned(16))) T sV[2][BT * LDV];
  __shared__ __attribute__((aligned(16))) T sTu[2][kTriElems];
  __shared__ __attribute__((aligned(16))) float sEg[2][BT];    // e^{gamma} (L2N: / |k|)
  __shared__ __attribute__((aligned(16))) float sEd[2][BT];    // e^{gamma_last - gamma} (L2N: / |k|)
  __shared__ float sDec[2];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H;
  const int cw = (int)(blockIdx.x % (uint32_t)p.col_wgs);     // which 128 of the V + K columns
  const uint32_t item = blockIdx.x / (uint32_t)p.col_wgs;
  const int hh = (int)(item % (uint32_t)H);
  const int64_t i = item / (uint32_t)H;
  int n, j;
  if (p.split.sub_table) {
    n = p.split.sub_table[2 * i];
    j = p.split.sub_table[2 * i + 1];
  } else {
    n = (int)((uint32_t)i / (uint32_t)p.per_seq);
    j = (int)((uint32_t)i % (uint32_t)p.per_seq);
  }
  const SeqSpan whole = seq_span(p.offsets, n, p.T);
  const int64_t all = (whole.len + BT - 1) / BT;
  const int64_t c0 = (int64_t)j * p.split.sub_chunks;
  const int64_t slot = (p.split.sub_base ? p.split.sub_base[n] : (int64_t)n * p.split.nsub) + j;
  const int nc = (int)(all - c0 < p.split.sub_chunks ? all - c0 : p.split.sub_chunks);
  const int64_t row0 = (whole.bos + c0 * BT) * H + hh;
  const int64_t chunk0 = (p.chunk_offsets ? p.chunk_offsets[n] : (int64_t)n * ((p.T + BT - 1) / BT)) + c0;
  const int64_t rem = whole.len - c0 * BT;
  const int rows = (int)(rem < (int64_t)nc * BT ? rem : (int64_t)nc * BT);   // < nc * BT in the last segment of a sequence only

  if (nc <= 0) return;
  if (wave >= 4) {
    // =========================== staging waves ===========================
    const int st = tid - 256;
    struct Regs {
      v8 k[NPK], v[NPV], tu0, tu1;
      float gam, rk;
    };
    const uint32_t pitchk = 2u * (uint32_t)H * K, pitchv = 2u * (uint32_t)H * V, colk = (uint32_t)(st % CK) * 16u,
                   colv = (uint32_t)(st % CV) * 16u;
    uint32_t offk[NPK], offv[NPV];
#pragma unroll
    for (int x = 0; x < NPK; ++x) offk[x] = (uint32_t)((st + 256 * x) / CK) * pitchk + colk;
#pragma unroll
    for (int x = 0; x < NPV; ++x) offv[x] = (uint32_t)((st + 256 * x) / CV) * pitchv + colv;
    const int Llast = rows - (nc - 1) * BT;   // < BT at the end of a sequence only
    const uint32_t tail = wave == 4 ? (uint32_t)lane : 0u, grow = wave == 7 ? (uint32_t)lane : 0u;
    // One barrier per chunk: it publishes the next chunk's tiles and says that the matrix waves are done with the other
    // buffer.  Every memory operation is unconditional (rows and chunks past the end are read from the last one), so
    // that the compiler's wait counts leave the other register sets in flight.
    auto run = [&](auto with_v) __attribute__((always_inline)) {
      constexpr bool NEED_V = decltype(with_v)::value;
      int lc = 0;   // next chunk to load
      auto load = [&](Regs& R) __attribute__((always_inline)) {
        const int cc = lc < nc - 1 ? lc : nc - 1;
        const uint32_t last = (uint32_t)((cc == nc - 1 ? Llast : BT) - 1);
        const int64_t r0 = row0 + (int64_t)cc * BT * H;
        const char* kb = (const char*)p.k + r0 * K * 2;
        const uint32_t limk = last * pitchk + colk;
#pragma unroll
        for (int x = 0; x < NPK; ++x) R.k[x] = *(const v8*)(kb + (offk[x] < limk ? offk[x] : limk));
        if constexpr (NEED_V) {
          const char* vb = (const char*)p.v + r0 * V * 2;
          const uint32_t limv = last * pitchv + colv;
#pragma unroll
          for (int x = 0; x < NPV; ++x) R.v[x] = *(const v8*)(vb + (offv[x] < limv ? offv[x] : limv));
        }
        const char* tb = (const char*)p.AT + ((chunk0 + cc) * H + hh) * (int64_t)kTriElems * 2;
        R.tu0 = *(const v8*)(tb + st * 16);
        // the last 64 pieces of Tu and the gates: one wave's each; the others load one word, without a branch (a column of
        // 64 gates is 64 requests to the L2)
        R.tu1 = *(const v8*)(tb + (256 + tail) * 16);
        const uint32_t gr = (grow < last ? grow : last) * (uint32_t)H;
        R.gam = *(p.gam ? p.gam + r0 + gr : &kZeroWord);
        if constexpr (L2N) R.rk = p.rk[r0 + gr];
        ++lc;
      };
      int wc = 0;   // next chunk to write
      auto write = [&](Regs& R) __attribute__((always_inline)) {
        const int b = wc & 1;
        if (wc >= nc - 1 && Llast < BT) {
#pragma unroll
          for (int x = 0; x < NPK; ++x)
            if ((st + 256 * x) / CK >= Llast)
#pragma unroll
              for (int z = 0; z < 8; ++z) R.k[x][z] = (T)0.f;
          if constexpr (NEED_V) {
#pragma unroll
            for (int x = 0; x < NPV; ++x)
              if ((st + 256 * x) / CV >= Llast)
#pragma unroll
                for (int z = 0; z < 8; ++z) R.v[x][z] = (T)0.f;
          }
        }
#pragma unroll
        for (int x = 0; x < NPK; ++x) *(v8*)&sK[b][(st + 256 * x) / CK * LDR + st % CK * 8] = R.k[x];
        if constexpr (NEED_V) {
#pragma unroll
          for (int x = 0; x < NPV; ++x) *(v8*)&sV[b][(st + 256 * x) / CV * LDV + st % CV * 8] = R.v[x];
        }
        *(v8*)&sTu[b][st * 8] = R.tu0;
        if (wave == 4) *(v8*)&sTu[b][2048 + lane * 8] = R.tu1;
        if (wave == 7) {
          const float glast = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(R.gam), 63));
          float eg = __expf(R.gam), ed = __expf(glast - R.gam);
          if constexpr (L2N) {
            eg *= R.rk;
            ed *= R.rk;
          }
          sEg[b][lane] = eg;
          sEd[b][lane] = ed;
          if (lane == 0) sDec[b] = __expf(glast);
        }
        ++wc;
      };
      Regs R0, R1, R2;
      load(R0);
      asm volatile("" ::: "memory");   // the sets are issued one after the other
      load(R1);
      asm volatile("" ::: "memory");
      load(R2);
      write(R0);
      load(R0);
      lds_barrier();
      auto iter = [&](Regs& R) __attribute__((always_inline)) {
        write(R);
        load(R);
        lds_barrier();
      };
      for (int ci = 0;;) {
        iter(R1);
        if (++ci == nc) break;
        iter(R2);
        if (++ci == nc) break;
        iter(R0);
        if (++ci == nc) break;
      }
    };
    if (cw * 128 < V) run(std::true_type{});
    else run(std::false_type{});
    return;
  }
  // =========================== matrix waves ===========================
  // this wave's 32 columns: of S (value columns) or of M, or none
  const int col = (cw * 4 + wave) * 32;
  const bool is_s = col < V, is_m = !is_s && col < V + K;
  const int c = lane & 15, g = lane >> 4;
  f32x4 acc[2][KT];   // acc[j][kt][r] = column (col + 16 j + c) at key row 16 kt + 4 g + r
#pragma unroll
  for (int jb = 0; jb < 2; ++jb)
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[jb][kt][r] = is_m && 16 * kt + 4 * g + r == col - V + 16 * jb + c ? 1.f : 0.f;
  lds_barrier();
  for (int ci = 0; ci < nc; ++ci) {
    const int b = ci & 1;
    if (!is_s && !is_m) {   // wave-uniform
      lds_barrier();
      continue;
    }
    const T *Kr = sK[b], *Tu = sTu[b];
    // LDS reads are issued a group ahead of the matrix instructions that consume them (the fences keep them there)
    v8 fa[KS], fb[KS];
    auto read_k = [&](int tt, v8* f) __attribute__((always_inline)) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) f[ks] = frag16<T>(Kr, LDR, 16 * tt, 32 * ks, lane);
    };
    read_k(0, fa);
    read_k(1, fb);
    __builtin_amdgcn_sched_barrier(0);
    v8 hb[2][KS];
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          hb[jb][ks][e] = (T)acc[jb][2 * ks][e];
          hb[jb][ks][4 + e] = (T)acc[jb][2 * ks + 1][e];
        }
    f32x4 d[2][4];
    auto mul_k = [&](int tt, const v8* f) __attribute__((always_inline)) {
      d[0][tt] = d[1][tt] = zero4();
#pragma unroll
      for (int ks = 0; ks < KS; ++ks)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) d[jb][tt] = Elem<T>::mfma16(f[ks], hb[jb][ks], d[jb][tt]);
    };
    mul_k(0, fa);
    __builtin_amdgcn_sched_barrier(0);
    read_k(2, fa);
    __builtin_amdgcn_sched_barrier(0);
    mul_k(1, fb);
    __builtin_amdgcn_sched_barrier(0);
    read_k(3, fb);
    __builtin_amdgcn_sched_barrier(0);
    mul_k(2, fa);
    __builtin_amdgcn_sched_barrier(0);
    v8 ft[6];
    ft[0] = frag_tri<T>(Tu, 0, 0, lane);
    ft[1] = frag_tri<T>(Tu, 1, 0, lane);
    ft[2] = frag_tri<T>(Tu, 2, 0, lane);
    ft[3] = frag_tri<T>(Tu, 2, 1, lane);
    ft[4] = frag_tri<T>(Tu, 3, 0, lane);
    ft[5] = frag_tri<T>(Tu, 3, 1, lane);
    f32x4 eg[4], ed[4];
    v4 vv[2][4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
      eg[tt] = *(const f32x4*)&sEg[b][16 * tt + 4 * g];
      ed[tt] = *(const f32x4*)&sEd[b][16 * tt + 4 * g];
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        vv[jb][tt] = v4{(T)0.f, (T)0.f, (T)0.f, (T)0.f};
        if (is_s) {   // four rows of one value column: the transposing load
          const T* pv = &sV[b][(16 * tt + 4 * g + (c >> 2)) * LDV + col + 16 * jb + 4 * (c & 3)];
          vv[jb][tt] = __builtin_bit_cast(v4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)pv));
        }
      }
    }
    const float dec = sDec[b];
    __builtin_amdgcn_sched_barrier(0);
    mul_k(3, fb);
    __builtin_amdgcn_sched_barrier(0);
    v8 fk[4];
    auto read_kt = [&](int kt2) __attribute__((always_inline)) {   // two 16-row tiles of k^T
#pragma unroll
      for (int x = 0; x < 4; ++x) fk[x] = frag16_tr<T>(Kr, LDR, 16 * (2 * kt2 + (x >> 1)), 32 * (x & 1), lane);
    };
    read_kt(0);
    __builtin_amdgcn_sched_barrier(0);
    v8 vs[2][2];
#pragma unroll
    for (int jb = 0; jb < 2; ++jb) {
      // r = v - e^{gamma} (k h) as the operand contracting over time, v_new = Tu r, and its decayed copy as an operand
      v8 rb[2];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) rb[tt >> 1][(tt & 1) * 4 + r] = (T)((float)vv[jb][tt][r] - d[jb][tt][r] * eg[tt][r]);
      f32x4 vn[4];
      vn[0] = Elem<T>::mfma16(ft[0], rb[0], zero4());
      vn[1] = Elem<T>::mfma16(ft[1], rb[0], zero4());
      vn[2] = Elem<T>::mfma16(ft[2], rb[0], zero4());
      vn[3] = Elem<T>::mfma16(ft[4], rb[0], zero4());
      vn[2] = Elem<T>::mfma16(ft[3], rb[1], vn[2]);
      vn[3] = Elem<T>::mfma16(ft[5], rb[1], vn[3]);
#pragma unroll
      for (int tt = 0; tt < 4; ++tt)
#pragma unroll
        for (int r = 0; r < 4; ++r) vs[jb][tt >> 1][(tt & 1) * 4 + r] = (T)(vn[tt][r] * ed[tt][r]);
    }
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[jb][kt][r] *= dec;
#pragma unroll
    for (int kt2 = 0; kt2 < KT / 2; ++kt2) {
      v8 f[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) f[x] = fk[x];
      if (kt2 + 1 < KT / 2) read_kt(kt2 + 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
          acc[jb][2 * kt2 + (x >> 1)] = Elem<T>::mfma16(f[x], vs[jb][x & 1], acc[jb][2 * kt2 + (x >> 1)]);
    }
    lds_barrier();
  }
  if (is_s) {
    float* out = p.states + (slot * H + hh) * (int64_t)(K * V) + col + c;
#pragma unroll
    for (int jb = 0; jb < 2; ++jb)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int r = 0; r < 4; ++r) out[(16 * kt + 4 * g + r) * V + 16 * jb] = acc[jb][kt][r];
  } else if (is_m) {
    // This wave's columns are one slice of 32 of the contraction index.  An accumulator pair multiplied by the identity in
    // accumulator-row order, part by part, comes out with lanes and registers exchanged and every bit in place: a lane then
    // holds four columns of one row, and both column blocks of the wave together are its eight slots of the fold's operand.
    typedef bf16x8 b8;
    b8 eye[2];
#pragma unroll
    for (int half = 0; half < 2; ++half)
#pragma unroll
      for (int e = 0; e < 8; ++e) eye[half][e] = (bf16)(((e >> 2) == half && 4 * g + (e & 3) == c) ? 1.f : 0.f);
    float* out = p.trans + (slot * H + hh) * (int64_t)(K * K) + ((col - V) / 32 * KT * 128 + lane) * 4;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
      for (int jb = 0; jb < 2; ++jb) {
        b8 x[3];
        split3(acc[jb][2 * ks], acc[jb][2 * ks + 1], x);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
          f32x4 t = Elem<bf16>::mfma16(x[0], eye[half], zero4());
          t = Elem<bf16>::mfma16(x[1], eye[half], t);
          *(f32x4*)(out + ((2 * ks + half) * 2 + jb) * 256) = Elem<bf16>::mfma16(x[2], eye[half], t);
        }
      }
      if (p.trans_t) {   // a column of M is a row of M^T: the accumulators are the operand as they are
        float* ot = p.trans_t + (slot * H + hh) * (int64_t)(K * K) + ((ks * KT + (col - V) / 16) * 128 + lane) * 4;
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
          for (int half = 0; half < 2; ++half) *(f32x4*)(ot + (jb * 2 + half) * 256) = acc[jb][2 * ks + half];
      }
    }
  }
}

template <int K, bool REVERSE>
__global__ __launch_bounds__(64 * (K / 16)) void gdr_split_fold_kernel(float* states, const float* trans, const float* init,
                                                                       SplitView split, const int64_t* offsets, int64_t T,
                                                                       int H, int V) {
  constexpr int KS = K / 32, KT = K / 16;
  typedef bf16x4 b4;
  typedef bf16x8 b8;
  __shared__ __attribute__((aligned(16))) bf16 sH[2][3][KT * 64 * 4];   // the parts of the slab, [row tile][lane][4]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // heads fastest: the column slabs of a head, which read the same M, land on one XCD and its L2
  const int nh = blockIdx.x, n = nh / H, hh = nh % H, cb = (int)blockIdx.y * 16;
  const int c = lane & 15, g = lane >> 4;
  const SeqSpan sp = seq_span(offsets, n, T);
  const int nseg = (int)split_nsub(split, (sp.len + BT - 1) / BT);   // a segment is one sub-block
  const int64_t base = split.sub_base ? split.sub_base[n] : (int64_t)n * split.nsub;
  float* S = states + (base * H + hh) * (int64_t)K * V + (int64_t)(16 * wave + 4 * g) * V + cb + c;
  const float* M = trans + (base * H + hh) * (int64_t)(K * K) + (wave * 128 + lane) * 4;
  const int64_t sstr = (int64_t)H * K * V, mstr = (int64_t)H * K * K;
  f32x4 h;   // rows 16 wave + 4 g .. + 3 of column cb + c
#pragma unroll
  for (int r = 0; r < 4; ++r) h[r] = init ? init[(int64_t)nh * K * V + (int64_t)(16 * wave + 4 * g + r) * V + cb + c] : 0.f;
  struct Regs {
    f32x4 m[KS][2];
    f32x4 s;
  } A, B;
  auto load = [&](Regs& R, int seg) __attribute__((always_inline)) {
    // `seg` counts in the order of the walk: backwards the segments come from the last to the second
    const int y = seg < nseg - 1 ? seg : nseg - 2, x = REVERSE ? nseg - 1 - y : y;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks)
#pragma unroll
      for (int half = 0; half < 2; ++half) R.m[ks][half] = *(const f32x4*)(M + x * mstr + ks * KT * 512 + half * 256);
#pragma unroll
    for (int r = 0; r < 4; ++r) R.s[r] = S[x * sstr + (int64_t)r * V];
  };
  auto step = [&](Regs& R, int seg) __attribute__((always_inline)) {
    b8 hp[3];
    split3(h, h, hp);
#pragma unroll
    for (int part = 0; part < 3; ++part)
      *(b4*)&sH[seg & 1][part][(wave * 64 + lane) * 4] = __builtin_shufflevector(hp[part], hp[part], 0, 1, 2, 3);
    // the state entering this segment takes the place of its S, which this lane has read
    f32x4 a[6] = {R.s, zero4(), zero4(), zero4(), zero4(), zero4()};   // by the order of the products
#pragma unroll
    for (int r = 0; r < 4; ++r) S[(REVERSE ? nseg - 1 - seg : seg) * sstr + (int64_t)r * V] = h[r];
    lds_barrier();
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      b8 m[3], x[3];
      split3(R.m[ks][0], R.m[ks][1], m);
#pragma unroll
      for (int part = 0; part < 3; ++part) {
        const b4 t0 = *(const b4*)&sH[seg & 1][part][(2 * ks * 64 + lane) * 4];
        const b4 t1 = *(const b4*)&sH[seg & 1][part][((2 * ks + 1) * 64 + lane) * 4];
        x[part] = __builtin_shufflevector(t0, t1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
      a[0] = Elem<bf16>::mfma16(m[0], x[0], a[0]);
      a[1] = Elem<bf16>::mfma16(m[0], x[1], a[1]);
      a[2] = Elem<bf16>::mfma16(m[1], x[0], a[2]);
      a[3] = Elem<bf16>::mfma16(m[0], x[2], a[3]);
      a[4] = Elem<bf16>::mfma16(m[1], x[1], a[4]);
      a[5] = Elem<bf16>::mfma16(m[2], x[0], a[5]);
      a[3] = Elem<bf16>::mfma16(m[1], x[2], a[3]);
      a[5] = Elem<bf16>::mfma16(m[2], x[1], a[5]);
    }
    load(R, seg + 2);
    h = a[0] + ((a[1] + a[2]) + (a[3] + (a[4] + a[5])));
  };
  if (nseg > 1) {
    load(A, 0);
    asm volatile("" ::: "memory");   // the sets are issued one after the other
    load(B, 1);
    for (int seg = 0;;) {
      step(A, seg);
      if (++seg == nseg - 1) break;
      step(B, seg);
      if (++seg == nseg - 1) break;
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) S[(REVERSE ? 0 : nseg - 1) * sstr + (int64_t)r * V] = h[r];
}

template <typename T, bool L2N>
int launch_gdr_pass(const GdrPassParams& p, int K, int V, unsigned grid, hipStream_t st) {
#define FLA_CASE(KK, VV)                                                                               \
  if (K == KK && V == VV) {                                                                            \
    hipLaunchKernelGGL((gdr_split_pass_kernel<T, KK, VV, L2N>), dim3(grid), dim3(512), 0, st, p);      \
    FLA_CHECK_LAUNCH();                                                                                \
    return FLA_OK;                                                                                     \
  }
  FLA_CASE(128, 128)
  FLA_CASE(64, 64)
  FLA_CASE(64, 128)
  FLA_CASE(128, 64)
#undef FLA_CASE
  return FLA_E_UNSUPPORTED;
}

template <bool REVERSE>
int launch_gdr_fold(const float* init, const fla_split* split, const int64_t* offsets, int64_t T, int64_t H, int64_t K, int64_t V,
                    int64_t N, hipStream_t st) {
  const dim3 grid((unsigned)(N * H), (unsigned)(V / 16));
  if (K == 128)
    hipLaunchKernelGGL((gdr_split_fold_kernel<128, REVERSE>), grid, dim3(512), 0, st, split->states, split->decays,
                       init, split_view(split), offsets, T, (int)H, (int)V);
  else
    hipLaunchKernelGGL((gdr_split_fold_kernel<64, REVERSE>), grid, dim3(256), 0, st, split->states, split->decays,
                       init, split_view(split), offsets, T, (int)H, (int)V);
  FLA_CHECK_LAUNCH();
  return FLA_OK;
}

}  // namespace

int gdr_split_states(const void* k, const void* v, const void* AT, const float* g_cumsum, const float* k_rstd, const float* init,
                     const fla_split* split, const int64_t* offsets, const int64_t* chunk_offsets, int qkv_dtype, int64_t T,
                     int64_t H, int64_t K, int64_t V, int64_t N, hipStream_t st) {
  int rc = check_split(split, offsets);
  if (rc) return rc;
  FLA_REQUIRE(split->decays && split->ratio == 1, FLA_E_INVALID);
  FLA_REQUIRE(BT * H * K * 2 <= 0x7fffffffLL && BT * H * V * 2 <= 0x7fffffffLL, FLA_E_UNSUPPORTED);   // 32-bit offsets in a chunk
  GdrPassParams p{k, v, AT, g_cumsum, k_rstd, split->states, split->decays, split->transitions_t, offsets,
                  chunk_offsets, split_view(split), T, (int)H, split->nseg - (split->transitions_t ? 0 : 1),
                  (int)((V + K + 127) / 128)};
  const int64_t subs = offsets ? split->nsub : (int64_t)p.per_seq * N;
  FLA_REQUIRE(subs * H * p.col_wgs <= 0x7fffffffLL && N * H <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
  if (subs > 0) {
    const unsigned grid = (unsigned)(subs * H * p.col_wgs);
    if (qkv_dtype == FLA_BF16)
      rc = k_rstd ? launch_gdr_pass<bf16, true>(p, (int)K, (int)V, grid, st) : launch_gdr_pass<bf16, false>(p, (int)K, (int)V, grid, st);
    else if (qkv_dtype == FLA_F16)
      rc = k_rstd ? launch_gdr_pass<f16, true>(p, (int)K, (int)V, grid, st) : launch_gdr_pass<f16, false>(p, (int)K, (int)V, grid, st);
    else
      rc = FLA_E_UNSUPPORTED;
    if (rc) return rc;
  }
  return launch_gdr_fold<false>(init, split, offsets, T, H, K, V, N, st);
}

int gdr_split_fold_reverse(const float* init, const fla_split* split, const int64_t* offsets, int64_t T, int64_t H, int64_t K,
                           int64_t V, int64_t N, hipStream_t st) {
  return launch_gdr_fold<true>(init, split, offsets, T, H, K, V, N, st);
}
