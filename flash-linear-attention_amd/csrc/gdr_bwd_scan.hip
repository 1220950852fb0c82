// The reverse state scan of the gated delta rule backward (fla/ops/common/chunk_delta_h.py:136-237), from what the two-launch
// forward leaves: per (chunk, head) the packed lower-triangular tiles Tu = (Aw * Gamma) diag(beta) and Aqk.  With dH the
// gradient of the state leaving a chunk,
//   dv2 = Aqk^T do + e^{gamma_last-gamma} * (k dH)          the gradient of v_new = Tu (v - e^gamma (k h))
//   dr  = Tu^T dv2
//   dH <- e^{gamma_last} dH + q^T (s e^gamma * do) - k^T (e^gamma * dr)
// so neither dv_loc = Aqk^T do nor w = Aw (beta k) is read, or kept by the forward: k, which the scan reads anyway, takes
// w's place at the price of one small triangular product in the chain.
//
// What bounds it: the serial chain where the chip is half empty (2 x 2048 tokens, 16 heads, K = V = 128: 128 workgroups,
// 1.4 us a chunk), and what 256 CUs take in through their row loads where it is full (4 x 4096 tokens: 2.2 us a chunk, 58 KB
// in and out per CU).  There it takes 46.5 and 141 us; the scan that reads w, with two barriers and both orientations of dH
// in the matrix waves, 61 and 162 us (gdr_bwd_dhu_kernel).  Requesting rows two chunks ahead instead of one: 48 and 144 us.
#include <type_traits>

#include "gdr_bwd_scan.h"
#include "seq_split.h"

namespace {

// LDS tiles and the transposing loads: a load of 32 operand rows reads, per half wave, four tile rows x 64 bytes, so with the
// pitch of K + 8 elements that suits row fragments (16 rows x 16 bytes) its four rows share banks - measured, half of the LDS
// cycles of the scan.  A tile read only through them takes a pitch of 16 words more than a multiple of 32 (q), 16 words
// (s e^gamma do) or, for 16 operand rows, 24 (do).  k and dH^T are read both ways: no padding, and the 16-byte slot of a row
// is XORed with bits of the row such that both 16 rows of one slot and 4 rows of 4 slots cover all banks.
template <int K>
FLA_DEVICE int swz_slot(int row) {
  return K == 128 ? ((row & 3) << 2) | ((row >> 2) & 3) : (((row >> 1) & 1) << 2) | ((row >> 2) & 3);
}
// element offset of (row, col) in such a tile, col a multiple of 4
template <int K>
FLA_DEVICE int swz(int row, int col) {
  return row * K + ((((col >> 3) ^ swz_slot<K>(row)) << 3) | (col & 4));
}

struct BwdScanParams {
  const void* q;
  const void* k;
  const void* AT;
  const void* Aqk;
  const float* gam;    // chunk-local prefix sums of the gate, or NULL
  const void* dout;
  const float* dht;
  void* dv2;
  void* dhtf;          // dH, FLA_H_FRAGMENT_T
  float* dh0;
  const int64_t* offsets;
  const int64_t* chunk_offsets;
  int64_t T;
  int H, V, N;
  float scale;
  SplitView split;     // sequences cut into segments (ratio 0: not)
  float* local;        // PASS: what the segments add to a zero gradient, [slots, H, K, V]
  int per_seq;         // PASS, equal-length sequences: segments of the pass per sequence
};

// One workgroup of eight waves: all K rows x 32 value columns of one (sequence, head).  Waves 0-3 ("matrix") carry the state
// gradient and form the products; waves 4-7 ("staging") bring in the rows, write the operand tiles and store the results.
// Per chunk c, walking backwards, the groups meet three times:
//   B1(c)  matrix:  dv2 = dl + e^{gamma_last-gamma} * (k dH) -> LDS (dl = Aqk^T do and the rows of k are in registers)
//          staging: k of chunk c-1 -> LDS; dH of chunk c -> memory
//   B2(c)  matrix:  dH <- e^{gamma_last} dH + q^T (s e^gamma * do) while the operands of dr arrive; -e^gamma * dr -> LDS
//          staging: do, Aqk and gates of chunk c-1 -> LDS; dv2 of chunk c -> memory
//   B3(c)  matrix:  dH += k^T (-e^gamma * dr); k rows and dl of chunk c-1; publishes dH in 16 bit
//          staging: Tu, s e^gamma * do and q of chunk c-1 -> LDS
// The work is dealt out so that neither group waits long in any of the three.  A staging wave requests the rows of chunk c-2
// as soon as those of c-1 have left its registers, a period ahead.  Only one orientation of dH is carried: the copy in
// fragment order is turned round by the staging waves out of the 16-bit tile (with both in the matrix waves half of their
// products, and their stores, stood in the chain: 57 -> 61 us at 32 chunks).
// PASS: the first pass over sequences cut into segments (seq_split.h): every segment but a sequence's first, from a zero
// gradient, without outputs but the gradient it ends with.
template <typename T, int K, bool PASS>
__global__ __launch_bounds__(512, K == 64 ? 4 : 2) void gdr_bwd_scan_kernel(BwdScanParams p) {
  typedef typename Elem<T>::v8 v8;
  typedef typename Elem<T>::v4 v4;
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4 lds_s4;
  constexpr int BV = 32;
  constexpr int LDQ = K + 32, LDO = BV + 16, LDD = BV;   // pitches of q, do, s e^{gamma} * do
  constexpr int C8 = K / 8, NP = BT * C8 / 256, NH = NP / 2;   // q, k: 16-byte pieces per row / per staging lane, half of them
  constexpr int PR = 256 / C8;                                 // rows between two pieces of a lane
  constexpr int KT32 = K / 32;
  __shared__ __attribute__((aligned(16))) T sK[2][BT * K];     // k of chunk c at [c & 1], swz
  __shared__ __attribute__((aligned(16))) T sQ[BT * LDQ];      // q, row-major
  __shared__ __attribute__((aligned(16))) T sDo[BT * LDO];     // do, row-major [t][v]
  __shared__ __attribute__((aligned(16))) T sDs[BT * LDD];    // s e^{gamma} * do
  __shared__ __attribute__((aligned(16))) T sP[kTriElems];     // Aqk, packed
  __shared__ __attribute__((aligned(16))) T sU[kTriElems];     // Tu, packed
  __shared__ __attribute__((aligned(16))) T sDHt[BV * K];      // dH^T in 16-bit, swz
  __shared__ __attribute__((aligned(16))) T sDv2T[BV * LDT];   // dv2^T
  __shared__ __attribute__((aligned(16))) T sDrT[BV * LDT];    // (-e^{gamma} * dr)^T
  // of chunk c at [c & 1]: e^{gamma_t}, e^{gamma_last - gamma_t} (both 0 past the end of a short chunk); the other rows are
  // where the lanes with nothing to say write
  __shared__ __attribute__((aligned(16))) float sG[2][4][BT];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H, V = p.V;
  const int nvt = V / BV;
  const uint32_t id = xcd_remap(blockIdx.x, gridDim.x);
  const int vt = (int)(id % (uint32_t)nvt);
  const int item = (int)(id / (uint32_t)nvt);
  const int hh = item % H;
  const int vbase = vt * BV;
  const ScanSpan span = PASS ? pass_span(p.split, item / H, p.per_seq, p.offsets, p.chunk_offsets, p.T)
                             : scan_span<true>(p.split, item / H, nullptr, p.offsets, p.chunk_offsets, p.T);
  const int nh = span.n * H + hh;
  const SeqSpan sp = span.sp;
  const int64_t nchunks = span.nchunks, chunk0 = span.chunk0;
  // the gradient of the state leaving this workgroup's chunks
  const float* dht = PASS            ? nullptr
                     : p.split.ratio ? p.split.states + (span.slot * H + hh) * (int64_t)K * V
                     : p.dht         ? p.dht + (int64_t)nh * K * V
                                     : nullptr;
  auto chunk_len = [&](int64_t c) {
    int64_t rem = sp.len - c * BT;
    return (int)(rem < BT ? rem : BT);
  };

  if (wave >= 4) {
    // =========================== staging waves ===========================
    if (nchunks == 0) return;
    const int st = tid - 256;
    const int prow = st / C8, c8 = (st % C8) * 8;   // piece i of a lane: row prow + PR i, columns c8 ..
    const int vrow = st >> 2, vc8 = (st & 3) * 8;   // do, dv2: one row, 8 of the 32 columns
    // Loads are unconditional (a load under a branch makes the wave drain its whole load queue at the join) and take few
    // instructions: a wave-uniform base per operand that steps back chunk by chunk, and byte offsets of this lane's rows
    // from the first row of a chunk.  Only the last chunk of a sequence can be short: in the prologue rows past its end are
    // redirected to its last row.  What a redirected row holds never counts: its gate factors are zero.
    const int64_t c0 = nchunks - 1;
    const int L0 = chunk_len(c0);
    const uint32_t pitchK = (uint32_t)H * K * (uint32_t)sizeof(T), pitchV = (uint32_t)H * V * (uint32_t)sizeof(T);
    const uint32_t pitchG = p.gam ? (uint32_t)H * 4u : 0u;   // without gates every gate load reads one zero word
    constexpr int64_t TB = (int64_t)kTriElems * (int64_t)sizeof(T);
    uint32_t offk[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) offk[i] = (uint32_t)(prow + PR * i) * pitchK + (uint32_t)c8 * (uint32_t)sizeof(T);
    const uint32_t offv = (uint32_t)vrow * pitchV + (uint32_t)vc8 * (uint32_t)sizeof(T);
    const uint32_t offg = (uint32_t)vrow * pitchG;
    const uint32_t off0 = 16 * (uint32_t)st, off1 = 4096 + 4 * (uint32_t)st;   // a tile: 16 bytes per lane, then 4
    auto lim = [](uint32_t o, uint32_t m) { return o < m ? o : m; };
    const uint32_t row0 = (uint32_t)(L0 - 1);
    struct Base {
      const char* p;
      int64_t step;
    };
    auto base = [&](const void* x, int64_t first, int64_t step) { return Base{(const char*)x + first + c0 * step, step}; };
    // a byte offset the compiler does not widen ahead of the loop: the load then takes base and offset as they are
    auto at = [](const Base& b, uint32_t o) __attribute__((always_inline)) {
      asm volatile("" : "+v"(o));
      return b.p + o;
    };
    const int64_t firstk = (sp.bos * H + hh) * (int64_t)K * (int64_t)sizeof(T);
    Base bq = base(p.q, firstk, BT * (int64_t)pitchK), bk = base(p.k, firstk, BT * (int64_t)pitchK);
    Base bd = base(p.dout, ((sp.bos * H + hh) * (int64_t)V + vbase) * (int64_t)sizeof(T), BT * (int64_t)pitchV);
    Base ba = base(p.Aqk, (chunk0 * H + hh) * TB, H * TB), bu = base(p.AT, (chunk0 * H + hh) * TB, H * TB);
    Base bg = base(p.gam ? (const void*)p.gam : (const void*)&kZeroWord, p.gam ? (sp.bos * H + hh) * 4 : 0, BT * (int64_t)pitchG);

    v8 kr[NP], qr[NP], dr, a0, u0;
    uint32_t a1, u1;
    float gam, glast;
    // tail: the chunk may be the short one
    auto load_rows = [&](Base& b, v8* R, auto tail) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NP; ++i)
        R[i] = *(const v8*)at(b, decltype(tail)::value ? lim(offk[i], row0 * pitchK + (uint32_t)c8 * 2u) : offk[i]);
      b.p -= b.step;
    };
    auto load_do = [&](auto tail) __attribute__((always_inline)) {   // do, Aqk and gates
      constexpr bool TAIL = decltype(tail)::value;
      dr = *(const v8*)at(bd, TAIL ? lim(offv, row0 * pitchV + (uint32_t)vc8 * 2u) : offv);
      a0 = *(const v8*)at(ba, off0);
      a1 = *(const uint32_t*)at(ba, off1);
      gam = *(const float*)at(bg, TAIL ? lim(offg, row0 * pitchG) : offg);
      glast = *(const float*)at(bg, (TAIL ? row0 : (uint32_t)(BT - 1)) * pitchG);
      bd.p -= bd.step;
      ba.p -= ba.step;
      bg.p -= bg.step;
    };
    auto load_u = [&]() __attribute__((always_inline)) {
      u0 = *(const v8*)at(bu, off0);
      u1 = *(const uint32_t*)at(bu, off1);
      bu.p -= bu.step;
    };
    auto stage_q = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NP; ++i) *(v8*)&sQ[(prow + PR * i) * LDQ + c8] = qr[i];
    };
    const int ksw = swz<K>(prow, c8);   // PR is a multiple of 16: the same slot in every piece
    auto stage_k = [&](T* tile) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NP; ++i) *(v8*)&tile[ksw + PR * i * K] = kr[i];
    };
    // the raw do row, and s e^{gamma} times it (zero past the end of its chunk), which waits in registers for its tile
    v8 ds;
    float* gdst = &sG[0][st & 3][vrow];
    auto stage_do = [&](int64_t c, auto tail) __attribute__((always_inline)) {
      asm volatile("" : "+v"(gam), "+v"(glast));   // not ahead of the barrier: it would wait for loads of the last phase
      const bool in = !decltype(tail)::value || vrow < L0;
      *(v8*)&sDo[vrow * LDO + vc8] = dr;
      *(v8*)&sP[st * 8] = a0;
      *(uint32_t*)&sP[2048 + st * 2] = a1;
      const float eg = in ? __expf(gam) : 0.f, ed = in ? __expf(glast - gam) : 0.f;
      gdst[(c & 1) * (4 * BT)] = (st & 3) == 1 ? ed : eg;
      const float x = p.scale * eg;
#pragma unroll
      for (int j = 0; j < 8; ++j) ds[j] = (T)((float)dr[j] * x);
    };
    auto stage_u = [&]() __attribute__((always_inline)) {
      *(v8*)&sU[st * 8] = u0;
      *(uint32_t*)&sU[2048 + st * 2] = u1;
    };
    // dH of chunk c in fragment order: transposing loads turn the 16-bit tile round.  The K / 32 tiles have 32 bytes per lane of
    // a wave; four adjacent lanes of a 16-lane group take the 4 key channels of an 8-byte piece, the group both halves of 8
    // such 32 bytes, 256 bytes on end (16 bytes of every lane's 32 per store: 127.6 us for 4 x 4096 tokens, 16 heads of 128; so:
    // 123.1)
    const T *hlo[KT32 / 2], *hhi[KT32 / 2];
    char* hdst[KT32 / 2];
#pragma unroll
    for (int i = 0; i < KT32 / 2; ++i) {
      const int pc = (wave - 4) * (KT32 / 2) + i, kt = pc >> 1, x = pc & 1;
      const int g = lane >> 4, j = lane & 15;
      const int hrow = 16 * (j & 1) + 4 * x + (j >> 2), hcol = kt * 32 + 8 * g + 2 * (j & 2);
      hlo[i] = &sDHt[swz<K>(hrow, hcol)];
      hhi[i] = &sDHt[swz<K>(hrow + 8, hcol)];
      hdst[i] = (char*)((T*)p.dhtf + ((chunk0 + c0) * H + hh) * (int64_t)K * V +
                        (((int64_t)vt * KT32 + kt) * 64 + 32 * x + 8 * g + 4 * (j >> 3) + (j & 3)) * 16 + 8 * ((j >> 2) & 1));
    }
    const int64_t hstep = (int64_t)H * K * V * (int64_t)sizeof(T);
    auto store_dh = [&]() __attribute__((always_inline)) {
      if constexpr (PASS) return;
#pragma unroll
      for (int i = 0; i < KT32 / 2; ++i) {
        s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)hlo[i]);
        s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)hhi[i]);
        *(v8*)hdst[i] =
            __builtin_shufflevector(__builtin_bit_cast(v4, lo), __builtin_bit_cast(v4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
        hdst[i] -= hstep;
      }
    };
    // dv2 leaves as whole rows, 16 bytes per lane: a 16-lane group turns a block of 8 value columns x 16 time rows of the
    // transposed tile round with two transposing LDS loads (lane j ends up with time row 16 tb + j, columns 8 vb ..)
    const int dgrp = st >> 4, dtb = dgrp >> 2, dvb = dgrp & 3, dj = st & 15, drow = 16 * dtb + dj;
    const int dsrc = (8 * dvb + (dj >> 2)) * LDT + 16 * dtb + 4 * (dj & 3);
    char* vdst = (char*)((T*)p.dv2 + ((sp.bos + c0 * BT + drow) * H + hh) * (int64_t)V + vbase + 8 * dvb);
    auto store_dv2 = [&](auto tail) __attribute__((always_inline)) {
      if constexpr (PASS) return;
      s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&sDv2T[dsrc]);
      s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&sDv2T[dsrc + 4 * LDT]);
      const v8 x = __builtin_shufflevector(__builtin_bit_cast(v4, lo), __builtin_bit_cast(v4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
      if (!decltype(tail)::value || drow < L0) *(v8*)vdst = x;
      vdst -= BT * (int64_t)pitchV;
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    load_rows(bk, kr, yes);
    load_do(yes);
    load_u();
    load_rows(bq, qr, yes);
    stage_k(sK[c0 & 1]);
    stage_do(c0, yes);
    stage_u();
    *(v8*)&sDs[vrow * LDD + vc8] = ds;
    stage_q();
    if (nchunks > 1) {
      load_rows(bk, kr, no);
      load_do(no);
      load_u();
      load_rows(bq, qr, no);
    }
    lds_barrier();  // B0
    // more: chunk c - 1 exists; ahead: chunk c - 2 exists
    auto period = [&](int64_t c, auto tail, auto more, auto ahead) __attribute__((always_inline)) {
      constexpr bool MORE = decltype(more)::value, AHEAD = decltype(ahead)::value;
      lds_barrier();  // B1(c)
      if constexpr (MORE) stage_k(sK[(c - 1) & 1]);
      if constexpr (AHEAD) load_rows(bk, kr, no);
      store_dh();
      lds_barrier();  // B2(c)
      if constexpr (MORE) stage_do(c - 1, no);
      if constexpr (AHEAD) load_do(no);
      store_dv2(tail);
      lds_barrier();  // B3(c)
      if constexpr (MORE) stage_u();
      if constexpr (AHEAD) load_u();
      if constexpr (MORE) {
        *(v8*)&sDs[vrow * LDD + vc8] = ds;
        stage_q();
      }
      if constexpr (AHEAD) load_rows(bq, qr, no);
    };
    // The last chunk (processed first) and the first two are peeled off: the steady-state loop has no memory operation under
    // a branch.
    if (nchunks > 2) {
      period(c0, yes, yes, yes);
      for (int64_t c = c0 - 1; c >= 2; --c) period(c, no, yes, yes);
      period(1, no, yes, no);
      period(0, no, no, no);
    } else {
      if (nchunks > 1) {
        period(1, yes, yes, no);
        period(0, no, no, no);
      } else {
        period(0, yes, no, no);
      }
    }
  } else {
    // =========================== matrix waves ===========================
    // wave w: rows 32 w .. of dH; rows 16 w .. of dv2 and dr (16 x 16 tiles: a lane holds four time rows of one column)
    const bool own = KT32 >= 4 || wave < KT32;
    const int tr = wave * 16 + 4 * (lane >> 4), l16 = lane & 15;
    // operands of q^T and k^T read a phase ahead of their products: not with 64 key channels, where two workgroups share a CU
    // (128 registers) and hide each other's latency (one sequence of 16384 tokens, 8 heads: step 211 -> 195 us)
    constexpr bool EARLY = K == 128;
    f32x16 acc = zero16();
    if (dht && own) {
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[r] = dht[(int64_t)(wave * 32 + c32_row(r, lane)) * V + vbase + (lane & 31)];
    }
    // swizzled tiles: a lane's piece of row fragment i (16 rows), and of the 32 key channels of this wave as operand rows
    int roff[K / 32];
#pragma unroll
    for (int i = 0; i < K / 32; ++i) roff[i] = swz<K>(l16, 32 * i + 8 * (lane >> 4));
    const int krow = 8 * (lane >> 5) + (l16 >> 2), kcol = wave * 32 + (lane & 16) + 4 * (lane & 3);
    const int klo = swz<K>(krow, kcol), khi = swz<K>(krow + 4, kcol);
    // dH^T in 16 bit, the operand of k dH
    auto publish = [&]() __attribute__((always_inline)) {
      if (own) {
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
          v4 x;
#pragma unroll
          for (int b = 0; b < 4; ++b) x[b] = (T)acc[4 * q4 + b];
          *(v4*)&sDHt[swz<K>(lane & 31, wave * 32 + 8 * q4 + 4 * (lane >> 5))] = x;
        }
      }
    };
    // Rows 32 s .. 32 s + 31 of column block `wave` of a packed lower-triangular tile, transposed: a 16-lane group holds
    // four rows of row block 2 s, then four of 2 s + 1.  Blocks above the diagonal are not stored: the address is that of
    // another block and what it holds is dropped (a branch round the load would make the wave wait for each by itself).
    const int toff = (4 * (lane >> 4) + (l16 >> 2)) * 16 + 4 * (lane & 3);
    auto tri_frag = [&](const T* tile, int s) __attribute__((always_inline)) {
      const int t0 = 2 * s, t1 = 2 * s + 1;
      s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&tile[(t0 * (t0 + 1) / 2 + wave) * 256 + toff]);
      s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&tile[(t1 * (t1 + 1) / 2 + wave) * 256 + toff]);
      const s4 z = {0, 0, 0, 0};
      lo = t0 >= wave ? lo : z;
      hi = t1 >= wave ? hi : z;
      return __builtin_shufflevector(__builtin_bit_cast(v4, lo), __builtin_bit_cast(v4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
    };
    // The first 32 rows lie above the diagonal for waves 2 and 3: their product is left out and not formed with zeros, which
    // would make every later row NaN where an earlier one of do holds an infinity or NaN.
    auto tri_product = [&](const v8* a, v8 b0, v8 b1) __attribute__((always_inline)) {
      f32x4 x = zero4();
      if (wave < 2) x = Elem<T>::mfma16(a[0], b0, x);   // wave-uniform
      return Elem<T>::mfma16(a[1], b1, x);
    };
    // what dv2 of chunk c takes that does not depend on dH: this wave's rows of k, dl = Aqk^T do, the gate factors
    v8 ka[K / 32];
    f32x4 dl[2], ed;
    auto front = [&](int64_t c) __attribute__((always_inline)) {
      const T* kc = sK[c & 1];
      v8 pa[2], db[2][2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        pa[s] = tri_frag(sP, s);
#pragma unroll
        for (int j = 0; j < 2; ++j) db[s][j] = frag16_tr<T>(sDo, LDO, 16 * j, 32 * s, lane);
      }
#pragma unroll
      for (int i = 0; i < K / 32; ++i) ka[i] = *(const v8*)&kc[wave * 16 * K + roff[i]];
      ed = *(const f32x4*)&sG[c & 1][1][tr];
#pragma unroll
      for (int j = 0; j < 2; ++j) dl[j] = tri_product(pa, db[0][j], db[1][j]);
    };
    if (nchunks > 0) {
      publish();
      lds_barrier();  // B0
      front(nchunks - 1);
    }
    for (int64_t c = nchunks - 1; c >= 0; --c) {
      const int L = chunk_len(c);
      v8 fq[BT / 16], fd[BT / 16];   // q^T and s e^gamma do, half of the reads in each of two phases
      auto load_qd = [&](int s0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = s0; s < s0 + BT / 32; ++s) {
          fq[s] = frag32_tr<T>(sQ, LDQ, wave * 32, 16 * s, lane);
          fd[s] = frag32_tr<T>(sDs, LDD, 0, 16 * s, lane);
        }
      };
      lds_barrier();  // B1(c)
      {
        v8 b[2][K / 32];
#pragma unroll
        for (int i = 0; i < K / 32; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) b[j][i] = *(const v8*)&sDHt[j * 16 * K + roff[i]];
        if (EARLY && own) load_qd(0);
        __builtin_amdgcn_sched_barrier(0);   // all reads in flight before the first product waits
        f32x4 d[2] = {zero4(), zero4()};
#pragma unroll
        for (int i = 0; i < K / 32; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) d[j] = Elem<T>::mfma16(ka[i], b[j][i], d[j]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          v4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (T)(tr + r < L ? dl[j][r] + ed[r] * d[j][r] : 0.f);
          *(v4*)&sDv2T[(16 * j + l16) * LDT + tr] = o;
        }
      }
      lds_barrier();  // B2(c)
      const T* kc = sK[c & 1];
      v8 fk[BT / 16];
      auto load_k = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < BT / 16; ++s) {
          s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&kc[klo + 16 * s * K]);
          s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)&kc[khi + 16 * s * K]);
          fk[s] = __builtin_shufflevector(__builtin_bit_cast(v4, lo), __builtin_bit_cast(v4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
        }
      };
      {
        v8 ua[2], db[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          ua[s] = tri_frag(sU, s);
#pragma unroll
          for (int j = 0; j < 2; ++j) {
            // the same order of the 32 summed rows as in `ua`: four of each row block per lane group
            const T* d2 = &sDv2T[(16 * j + l16) * LDT + 32 * s + 4 * (lane >> 4)];
            db[s][j] = __builtin_shufflevector(*(const v4*)d2, *(const v4*)(d2 + 16), 0, 1, 2, 3, 4, 5, 6, 7);
          }
        }
        if (EARLY && own) load_qd(2);
        const f32x4 eg = *(const f32x4*)&sG[c & 1][0][tr];
        const float dec = sG[c & 1][0][L - 1];
        __builtin_amdgcn_sched_barrier(0);
        if (EARLY && own) {   // in the shade of those reads
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] *= dec;
#pragma unroll
          for (int s = 0; s < BT / 16; ++s) acc = Elem<T>::mfma32(fq[s], fd[s], acc);
        }
        f32x4 dr[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) dr[j] = tri_product(ua, db[0][j], db[1][j]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          v4 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) o[r] = (T)(-eg[r] * dr[j][r]);
          *(v4*)&sDrT[(16 * j + l16) * LDT + tr] = o;
        }
        if (EARLY && own) load_k();
        if (!EARLY && own) {
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[r] *= dec;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            load_qd(2 * h);
#pragma unroll
            for (int s = 2 * h; s < 2 * h + 2; ++s) acc = Elem<T>::mfma32(fq[s], fd[s], acc);
          }
        }
      }
      lds_barrier();  // B3(c)
      if (own) {
        if (!EARLY) load_k();
        v8 f2[BT / 16];
#pragma unroll
        for (int s = 0; s < BT / 16; ++s) f2[s] = lds_frag32<T>(sDrT, LDT, 0, 16 * s, lane);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < BT / 16; ++s) acc = Elem<T>::mfma32(fk[s], f2[s], acc);
      }
      if (c > 0) {
        front(c - 1);
        publish();
      }
    }
    if (own && (PASS || (p.dh0 && span.first))) {
      float* o = PASS ? p.local + (span.slot * H + hh) * (int64_t)K * V : p.dh0 + (int64_t)nh * K * V;
#pragma unroll
      for (int r = 0; r < 16; ++r) o[(int64_t)(wave * 32 + c32_row(r, lane)) * V + vbase + (lane & 31)] = acc[r];
    }
  }
}

template <typename T>
int launch_scan(BwdScanParams p, const fla_split* split, int64_t K, hipStream_t st) {
#define LS(KK, PASS) hipLaunchKernelGGL((gdr_bwd_scan_kernel<T, KK, PASS>), dim3((unsigned)total), dim3(512), 0, st, p)
  const int64_t slabs = (int64_t)(p.V / 32) * p.H;
  if (split) {
    // the gradient leaving every segment: the first pass, then the fold with the transitions the forward left
    p.local = split->states;
    p.per_seq = split->nseg - 1;
    const int64_t total = slabs * (p.offsets ? (int64_t)split->nsub : (int64_t)p.per_seq * p.N);
    FLA_REQUIRE(total <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
    if (total > 0) {
      if (K == 64) LS(64, true);
      else LS(128, true);
      FLA_CHECK_LAUNCH();
    }
    const int rc = gdr_split_fold_reverse(p.dht, split, p.offsets, p.T, p.H, K, p.V, p.N, st);
    if (rc) return rc;
  }
  const int64_t total = slabs * (!split ? (int64_t)p.N : p.offsets ? (int64_t)split->nseg : (int64_t)split->nseg * p.N);
  FLA_REQUIRE(total <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
  if (total > 0) {
    if (K == 64) LS(64, false);
    else LS(128, false);
    FLA_CHECK_LAUNCH();
  }
#undef LS
  return FLA_OK;
}

}  // namespace

int gdr_bwd_scan(const void* q, const void* k, const void* AT, const void* Aqk, const float* g_cumsum, const void* dout,
                 const float* dht, void* dv2, void* dhtf, float* dh0, const int64_t* offsets, const int64_t* chunk_offsets,
                 const fla_split* split, int qkv_dtype, int64_t T, int64_t H, int64_t K, int64_t V, int64_t N, float scale,
                 hipStream_t st) {
  FLA_REQUIRE((K == 64 || K == 128) && V % 32 == 0, FLA_E_UNSUPPORTED);
  const BwdScanParams p{q, k, AT, Aqk, g_cumsum, dout, dht, dv2, dhtf, dh0, offsets, chunk_offsets, T, (int)H, (int)V, (int)N,
                        scale, split_view(split), nullptr, 0};
  if (qkv_dtype == FLA_BF16) return launch_scan<bf16>(p, split, K, st);
  if (qkv_dtype == FLA_F16) return launch_scan<f16>(p, split, K, st);
  return FLA_E_UNSUPPORTED;
}
