// One-pass gated-delta-rule forward for gfx950: state scan and output in one launch.  Inputs are q, k, v, the chunk-local
// gate prefix sums gamma and the packed triangular 64x64 tile Tu = (Aw * Gamma) diag(beta) that fla_gdr_fwd_prep leaves per
// (chunk, head).  Per chunk
//   v_new = Tu (v - e^{gamma} * (k h))
//   h    <- e^{gamma_last} h + k^T (e^{gamma_last - gamma} * v_new)            the chain
//   o     = s e^{gamma} * (q h) + s tril(q k^T * Gamma) v_new                   behind it
// (fla/ops/common/chunk_delta_h.py:71-119, chunk_o.py:68-101; v_new equals the reference's u - e^{gamma} (w h), see
// gdr_fwd.hip).  A workgroup of eight waves walks the chunks of a (sequence, head, 32 or 64 value columns):
//   waves 4-7 ("staging")  bring k, v, Tu and the gates of chunk c+1 and q of chunk c into LDS and, in a forward that will be
//                          differentiated, write v_new and the entering state of chunk c-1 to memory;
//   waves 0-1 ("chain")    hold the fp32 state, 16 columns of every 32 each and all K rows, and do nothing but the chain; they
//                          leave the entering state and v_new of the chunk in LDS as the 16-bit operands they use themselves;
//   waves 2-3 ("output")   form the scores and the output of chunk c-1 from those, two row tiles each (0 and 3, 1 and 2: five
//                          blocks of the scores), and store it.
// One barrier per chunk.  State, k h, the residual and v_new go from accumulators straight back into MFMA operands (the
// contraction index of the LDS-side operand is permuted to the accumulator row order instead), and so do the scores: they and
// the output are computed transposed.
//
// What bounds it: with a CU to every workgroup the two groups of matrix waves, 2500 cycles a chunk each, whichever is left out
// (2 x 2048 tokens, 16 heads, K = V = 128: 40 us; without the output waves' work 37, without the chain's 37); on a full chip the
// bytes (8 x 4096 tokens: 579 MB in 130 us, 4.5 TB/s), and where everything is kept the stores (4 x 4096 tokens: 149 us, 89
// without them).  With four waves that each form their 16 columns' share of all products, scores of the next chunk included,
// and store v_new and the states themselves, the same shapes took 46, 152 and 149 us, a packed batch of 12 sequences 179
// (now 155) and the mixing layer's 2 x 2048 tokens, everything kept, 54.7 (now 45).
#include <type_traits>

#include "seq_split.h"

namespace {

struct GdrScanParams {
  const void* q;
  const void* k;
  const void* v;
  const void* AT;   // [chunks, H, 10, 16, 16]: Tu
  const float* gam;
  const float* h0;
  void* o;
  float* ht;
  void* v_new;      // KEEP: [rows, H, V]
  void* h_frag_t;   // KEEP: [chunks, H, K*V], FLA_H_FRAGMENT_T
  void* Aqk_out;    // KEEP: [chunks, H, 10, 16, 16], the gated scores (or NULL)
  const int64_t* offsets;
  const int64_t* chunk_offsets;
  const int64_t* seq_order;  // sequence ids, longest first (or NULL)
  int64_t T;
  int H, V, N;
  float scale;
  float l2_eps;     // L2N: q and k are un-normalised; the launch works with x / sqrt(sum x^2 + l2_eps) ...
  const float* rk;  //      ... the factors of k, fp32 [rows, H], come from fla_gdr_fwd_prep_l2norm
  SplitView split;  // sequences cut into segments (ratio 0: not)
};

// Tiles of W columns (128 or 64) without padding.  The 16-byte slot of a row is XORed with bits of the row such that row
// fragments (8-byte pieces of 16 rows) as well as transposing reads (4 or 8 rows x 32 or 64 bytes) cover all banks.
template <int W>
FLA_DEVICE int tile_slot(int row) {
  return (W == 128 ? (row & 3) << 2 : (row & 2) << 1) | ((row & 4) >> 1) | ((row >> 3) & 1);
}
// element offset of (row, col), col a multiple of 4
template <int W>
FLA_DEVICE int tile_at(int row, int col) {
  return row * W + ((((col >> 3) ^ tile_slot<W>(row)) << 3) | (col & 4));
}

// The value columns of a slab are held in an order of their own: column 32 n + 8 a + 4 x + r (a, r < 4; x < 2) is row
// 32 n + 16 x + 4 a + r of the transposed tiles of h and v_new, and lane 4 a + r of chain wave x.  Two accumulators of an
// output wave (x = 0, 1) then are eight adjacent columns of a row of o, and sixteen adjacent rows of the state tile are what
// a lane holds of FLA_H_FRAGMENT_T.
template <typename T, int K, bool KEEP, int NC, bool L2N, bool DELTA>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdr_fwd_scan_kernel(GdrScanParams p) {
  static_assert(!(KEEP && L2N), "a forward that keeps its intermediates takes normalised q and k");
  static_assert(DELTA || (!KEEP && !L2N), "the plain scan: forward only, no l2 norm");
  typedef typename Elem<T>::v8 v8;
  typedef typename Elem<T>::v4 v4;
  typedef short s4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) s4 lds_s4;
  typedef __attribute__((address_space(3))) const volatile v4 lds_v4;   // (volatile: not fused into paired reads)
  constexpr int BV = 32 * NC, KS = K / 32, KT = K / 16;
  __shared__ __attribute__((aligned(16))) T sK[3][BT * K];       // k of chunk c at [c % 3], [t][k]
  __shared__ __attribute__((aligned(16))) T sQ[2][BT * K];       // q of chunk c at [c & 1], [t][k]
  __shared__ __attribute__((aligned(16))) T sV[2][BT * BV];      // v, [t][v]
  __shared__ __attribute__((aligned(16))) T sTu[DELTA ? 2 : 1][DELTA ? kTriElems : 8];   // Tu, packed
  __shared__ __attribute__((aligned(16))) T sH[2][BV * K];       // the state entering the chunk, transposed
  __shared__ __attribute__((aligned(16))) T sVn[2][BV * BT];     // v_new, transposed
  __shared__ __attribute__((aligned(16))) float sGam[3][BT];     // gamma_t
  __shared__ __attribute__((aligned(16))) float sEg[3][BT];      // e^{gamma_t}
  __shared__ __attribute__((aligned(16))) float sEd[3][BT];      // e^{gamma_last - gamma_t} (L2N: / |k_t|)
  __shared__ float sDec[3];                                      // e^{gamma_last}
  __shared__ __attribute__((aligned(16))) float sRq[L2N ? 2 : 1][L2N ? BT : 4];    // L2N: 1 / |q_t|
  __shared__ __attribute__((aligned(16))) float sRk[L2N ? 3 : 1][L2N ? BT : 4];    // L2N: 1 / |k_t|
  __shared__ __attribute__((aligned(16))) float sEgk[L2N ? 3 : 1][L2N ? BT : 4];   // L2N: e^{gamma_t} / |k_t|

  const int tid = threadIdx.x, lane = tid & 63;
  // wave-uniform by construction: keeps the role split and the barriers on scalar branches
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int H = p.H, V = p.V;
  const ScanItem wi = scan_item(V / BV);
  const int vb = wi.slab, vbase = vb * BV;
  const int hh = (int)(wi.item % (uint32_t)H);
  const ScanSpan span = scan_span<false>(p.split, wi.item / (uint32_t)H, p.seq_order, p.offsets, p.chunk_offsets, p.T);
  const int nh = span.n * H + hh;
  const SeqSpan sp = span.sp;
  const int nchunks = (int)span.nchunks;
  const int64_t chunk0 = span.chunk0;
  const int Llast = (int)(sp.len - (int64_t)(nchunks - 1) * BT);
  const int c = lane & 15, g = lane >> 4;

  if (wave >= 4) {
    // =========================== staging waves ===========================
    if (nchunks == 0) return;
    const int st = tid - 256;
    constexpr int C8 = K / 8, NPW = BT * C8 / 256, CV8 = BV / 8, NPV = BT * CV8 / 256;   // 16-byte pieces: row, lane
    static_assert(kTriElems == 8 * (256 + 64), "Tu: a 16-byte piece per staging lane and 64 more");
    const uint32_t pitchk = 2u * (uint32_t)H * K, pitchv = 2u * (uint32_t)H * V;
    struct Regs {
      v8 q[NPW], k[NPW], v[NPV], a0, a1;
      uint32_t gam, rk;   // fp32 bits
    };
    // The steady state carries no address arithmetic: byte offsets of this lane's pieces from a chunk's first row are formed
    // once and the bases advance by constant strides.  Every memory operation of the loop is unconditional (under a branch the
    // wave would wait for everything it has in flight at the join): rows past the end of a sequence's last chunk are
    // redirected to its last row and cleared on the way to LDS, past the last chunk the bases stay on it.
    const uint32_t colk = 16u * (uint32_t)(st % C8), colv = 16u * (uint32_t)(st % CV8);
    uint32_t offk[NPW], offv[NPV];
#pragma unroll
    for (int i = 0; i < NPW; ++i) offk[i] = (uint32_t)((st + 256 * i) / C8) * pitchk + colk;
#pragma unroll
    for (int i = 0; i < NPV; ++i) offv[i] = (uint32_t)((st + 256 * i) / CV8) * pitchv + colv;
    const int64_t row00 = sp.bos * H + hh;
    const char* lq = (const char*)p.q + row00 * K * 2;
    const char* lk = (const char*)p.k + row00 * K * 2;
    const char* lv = (const char*)p.v + (row00 * V + vbase) * 2;
    const char* la = (const char*)p.AT + (chunk0 * H + hh) * (int64_t)kTriElems * 2;
    const uint32_t gmask = p.gam ? 0xffffffffu : 0u;   // without gates: a dummy address, bits masked to zero
    const char* lg = p.gam ? (const char*)p.gam + row00 * 4 : lq;
    const char* lr = L2N ? (const char*)p.rk + row00 * 4 : lq;
    const int64_t strk = (int64_t)BT * pitchk, strv = (int64_t)BT * pitchv, strr = (int64_t)BT * H * 4;
    const int64_t stra = (int64_t)H * kTriElems * 2, strg = p.gam ? strr : 0;
    // Only the first staging wave uses the gate rows and only the second the last 64 pieces of Tu; the others' loads are all of
    // one word: a column of 64 gates, H apart, is 64 requests to the L2.
    const uint32_t offg = wave == 4 ? 4 * (uint32_t)lane * H : 0u;
    const uint32_t offa0 = 16 * (uint32_t)st, offa1 = 16 * (uint32_t)(256 + (wave == 5 ? lane : 0));
    const uint32_t limk_full = (BT - 1) * pitchk + colk, limk_last = (uint32_t)(Llast - 1) * pitchk + colk;
    const uint32_t limv_full = (BT - 1) * pitchv + colv, limv_last = (uint32_t)(Llast - 1) * pitchv + colv;
    // register set j: k, v, Tu and gates of chunk j, q of chunk j - 1
    int lc = 0;
    auto load = [&](Regs& R) __attribute__((always_inline)) {
      const bool last = lc >= nchunks - 1, qlast = (lc > 0 ? lc - 1 : 0) >= nchunks - 1;
      const uint32_t limk = last ? limk_last : limk_full, limq = qlast ? limk_last : limk_full;
      const uint32_t limv = last ? limv_last : limv_full, limg = 4 * (uint32_t)((last ? Llast : BT) - 1) * H;
#pragma unroll
      for (int i = 0; i < NPW; ++i) R.k[i] = *(const v8*)(lk + (offk[i] < limk ? offk[i] : limk));
      if constexpr (DELTA) {
        R.a0 = *(const v8*)(la + offa0);   // a full tile whatever the chunk length
        R.a1 = *(const v8*)(la + offa1);
      }
#pragma unroll
      for (int i = 0; i < NPV; ++i) R.v[i] = *(const v8*)(lv + (offv[i] < limv ? offv[i] : limv));
      R.gam = *(const uint32_t*)(lg + (offg < limg ? offg : limg));
      if constexpr (L2N) R.rk = *(const uint32_t*)(lr + (offg < limg ? offg : limg));
#pragma unroll
      for (int i = 0; i < NPW; ++i) R.q[i] = *(const v8*)(lq + (offk[i] < limq ? offk[i] : limq));
      if (lc + 1 < nchunks) {
        lk += strk;
        lv += strv;
        la += stra;
        lg += strg;
        if constexpr (L2N) lr += strr;
      }
      if (lc > 0 && lc < nchunks) lq += strk;
      ++lc;
    };
    int dk[NPW];
#pragma unroll
    for (int i = 0; i < NPW; ++i) dk[i] = tile_at<K>((st + 256 * i) / C8, st % C8 * 8);
    int wc = 0, w3 = 0;   // next set to write, and its buffer of three
    auto write = [&](Regs& R) __attribute__((always_inline)) {
      const int b = wc & 1;
      if (wc == nchunks - 1 && Llast < BT) {
#pragma unroll
        for (int i = 0; i < NPW; ++i)
          if ((st + 256 * i) / C8 >= Llast)
#pragma unroll
            for (int j = 0; j < 8; ++j) R.k[i][j] = (T)0.f;
#pragma unroll
        for (int i = 0; i < NPV; ++i)
          if ((st + 256 * i) / CV8 >= Llast)
#pragma unroll
            for (int j = 0; j < 8; ++j) R.v[i][j] = (T)0.f;
      }
#pragma unroll
      for (int i = 0; i < NPW; ++i) *(v8*)&sK[w3][dk[i]] = R.k[i];
      if constexpr (DELTA) {
        *(v8*)&sTu[b][st * 8] = R.a0;
        if (wave == 5) *(v8*)&sTu[b][2048 + lane * 8] = R.a1;
      }
#pragma unroll
      for (int i = 0; i < NPV; ++i) *(v8*)&sV[b][(st + 256 * i) * 8] = R.v[i];
      if (wave == 4) {
        // lanes past the end of a short chunk carry the last row's gate
        float gam = __uint_as_float(R.gam & gmask);
        if constexpr (!DELTA) {
          // raw gates: inclusive prefix sum over the 64 rows (rows past the end add zero)
          const float x = row_prefix16(lane < (wc == nchunks - 1 ? Llast : BT) ? gam : 0.f);
          const float x0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 15));
          const float x1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 31));
          const float x2 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), 47));
          gam = x + (g >= 1 ? x0 : 0.f) + (g >= 2 ? x1 : 0.f) + (g >= 3 ? x2 : 0.f);
        }
        const float glast = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gam), 63));
        sGam[w3][lane] = gam;
        sEg[w3][lane] = __expf(gam);
        if constexpr (L2N) {
          const float rk = __uint_as_float(R.rk);
          sRk[w3][lane] = rk;
          sEgk[w3][lane] = __expf(gam) * rk;
          sEd[w3][lane] = __expf(glast - gam) * rk;
        } else {
          sEd[w3][lane] = __expf(glast - gam);
        }
        if (lane == 0) sDec[w3] = __expf(glast);
      }
      if (wc == nchunks && Llast < BT) {
#pragma unroll
        for (int i = 0; i < NPW; ++i)
          if ((st + 256 * i) / C8 >= Llast)
#pragma unroll
            for (int j = 0; j < 8; ++j) R.q[i][j] = (T)0.f;
      }
#pragma unroll
      for (int i = 0; i < NPW; ++i) *(v8*)&sQ[b ^ 1][dk[i]] = R.q[i];
      if constexpr (L2N) {
#pragma unroll
        for (int i = 0; i < NPW; ++i) {
          const float rq = l2norm_rstd<T, K / 8>(R.q[i], p.l2_eps);
          if (st % C8 == 0) sRq[b ^ 1][(st + 256 * i) / C8] = rq;
        }
      }
      ++wc;
      w3 = w3 == 2 ? 0 : w3 + 1;
    };
    // KEEP: what the chain left of a chunk, turned round by transposing loads, four adjacent lanes of a 16-lane group taking
    // the 4 columns of an 8-byte piece in four tile rows.  State: the tile of 32 columns x 32 key rows of FLA_H_FRAGMENT_T has
    // 32 bytes per lane of a wave, sixteen adjacent rows of sH at one key row; a 16-lane group takes both halves of 8 of these,
    // 256 bytes on end.  v_new: 4 time rows x 32 columns (four rows of sVn and the four 16 further down are 8 columns).
    constexpr int HP = NC * KS / 2;   // pieces of the state per lane
    const int vrow = 16 * (wave - 4) + 4 * g + (c & 3);
    int hsrc = 0, vsrc = 0;
    uint32_t hlane = 0;
    char *hbase = nullptr, *vdst = nullptr;
    int kc = 0;   // next chunk to keep
    if constexpr (KEEP) {
      hsrc = tile_at<K>(8 * (c & 1) + (c >> 2), 8 * g + 2 * (c & 2));
      hlane = (uint32_t)((8 * g + 4 * (c >> 3) + (c & 3)) * 32 + 16 * ((c >> 2) & 1));
      hbase = (char*)p.h_frag_t + ((chunk0 * H + hh) * (int64_t)K * V + (int64_t)(vbase / 32) * KS * 1024) * 2;
      vsrc = tile_at<BT>(4 * (c & 3) + (c >> 2), 16 * (wave - 4) + 4 * g);
      vdst = (char*)p.v_new + (((sp.bos + vrow) * H + hh) * (int64_t)V + vbase + 8 * (c >> 2)) * 2;
    }
    auto tr2 = [&](const T* lo, const T* hi) __attribute__((always_inline)) {
      const s4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)lo), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)hi);
      return __builtin_shufflevector(__builtin_bit_cast(v4, a), __builtin_bit_cast(v4, b), 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto keep = [&](auto maybe_last) __attribute__((always_inline)) {
      if constexpr (KEEP) {
        const int b = kc & 1;
#pragma unroll
        for (int i = 0; i < HP; ++i) {
          const int pc = (wave - 4) * HP + i, x = pc & 1, kt = (pc >> 1) % KS, n = (pc >> 1) / KS;   // uniform
          const T* src = &sH[b][(32 * n + 16 * x) * K];
          // (rows 4 further: another value of row bit 2, which moves the slot by 2)
          const v8 h = tr2(src + (hsrc ^ 32 * kt), src + ((hsrc ^ 32 * kt ^ 16) + 4 * K));
          // (non-temporal: the backward pass reads it much later.  4 x 4096 tokens, training step 518.6 -> 511.1 us; v_new as well
          // 514.9, and 67 -> 72 us for the scan of 32 heads of 64.  Steps whose states the last-level cache would hold, plain / so:
          // 0.3 to 34 MB within 0.9 % of each other, but 32 heads of 64 of 2 x 2000 tokens, 17 MB, 136.6 / 138.6; 16 x 512 tokens, 32
          // heads of 64, 34 MB, 238 / 233, 16 heads of 128, 67 MB, 247 / 241)
          __builtin_nontemporal_store(h, (v8*)(hbase + (n * KS + kt) * 2048 + x * 1024 + hlane));
        }
        hbase += (int64_t)H * K * V * 2;
        const bool in = !decltype(maybe_last)::value || vrow < Llast;
#pragma unroll
        for (int n = 0; n < NC; ++n) {
          const T* s = &sVn[b][vsrc + 32 * n * BT];
          const v8 x = tr2(s, s + 16 * BT);
          if (in) *(v8*)(vdst + 64 * n) = x;
        }
        vdst += strv;
        ++kc;
      }
    };
    constexpr std::true_type any_chunk{};
    constexpr std::false_type inner_chunk{};
    Regs R0, R1, R2;
    load(R0);
    asm volatile("" ::: "memory");   // the sets are issued one after the other
    load(R1);
    asm volatile("" ::: "memory");
    // Iteration c (the chain works on chunk c) writes set c + 1 and loads set c + 4 into the registers just emptied.  Where
    // there is one chunk nothing behind set 1 is wanted (16 sequences of 64 tokens, 32 heads of 128: 39.5 -> 36.6 us).
    if (nchunks > 1) {
      load(R2);
      write(R0);
      load(R0);
      lds_barrier();
      write(R1);
      load(R1);
    } else {
      write(R0);
      lds_barrier();
      write(R1);
    }
    lds_barrier();
    auto iter = [&](Regs& R) __attribute__((always_inline)) {
      write(R);
      load(R);
      keep(inner_chunk);
      lds_barrier();
    };
    const int inner = nchunks - 1;
    for (int trips = inner / 3; trips > 0; --trips) {
      iter(R2);
      iter(R0);
      iter(R1);
    }
    const int rem = inner % 3;
    if (rem >= 1) iter(R2);
    if (rem >= 2) iter(R0);
    keep(any_chunk);
  } else if (wave >= 2) {
    // =========================== output waves ===========================
    if (nchunks == 0) return;
    // Row fragments (16 rows x 32 columns, 8-byte pieces 4 g .. and 16 + 4 g ..): slot of this lane's row, XORed per piece
    const int xk = tile_slot<K>(c) << 3, xt = tile_slot<BT>(c) << 3, g4 = 4 * g;
    auto row_frag = [&](const T* tile, int row0, int k0) __attribute__((always_inline)) {   // tiles of K columns
      const T* r = tile + (row0 + c) * K + (g4 & 4);
      const v4 lo = *(lds_v4*)(r + (((g4 & 8) + k0) ^ xk)), hi = *(lds_v4*)(r + (((g4 & 8) + k0 + 16) ^ xk));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto vn_frag = [&](const T* tile, int row0, int t0) __attribute__((always_inline)) {
      const T* r = tile + (row0 + c) * BT + (g4 & 4);
      const v4 lo = *(lds_v4*)(r + (((g4 & 8) + t0) ^ xt)), hi = *(lds_v4*)(r + (((g4 & 8) + t0 + 16) ^ xt));
      return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    char* ob = (char*)p.o + ((sp.bos * H + hh) * (int64_t)V + vbase) * 2;
    // 32 columns: a lane stores what it holds, 16 bytes of row c.  64 columns: o goes through LDS and leaves as whole rows of
    // 128 bytes, eight lanes each (8 x 4096 tokens, 16 heads of 128: 134.8 -> 130.0 us, 32 heads of 64: 149.3 -> 141.9; with
    // 32 columns the detour costs more than it gives, 2 x 2048 tokens 40.0 -> 41.0).
    const int orow = NC == 1 ? c : lane >> 3;
    const uint32_t opitch = (uint32_t)H * (uint32_t)V * 2u;
    const uint32_t olane = (uint32_t)orow * opitch + 16u * (uint32_t)(NC == 1 ? g : lane & 7);
    T* Pg = nullptr;   // KEEP: the first value slab of a head also leaves the scores in memory for the backward pass
    if constexpr (KEEP) {
      if (vb == 0 && p.Aqk_out) Pg = (T*)p.Aqk_out + (chunk0 * H + hh) * (int64_t)kTriElems;
    }
    int b3 = 0;   // oc modulo 3
    auto output = [&](int oc, auto t0, auto t1) __attribute__((always_inline)) {
      constexpr int TI[2] = {decltype(t0)::value, decltype(t1)::value};   // TI[0] < TI[1]
      const int b = oc & 1;
      const T *Kr = sK[b3], *Q = sQ[b];
      [[maybe_unused]] T* own = sQ[b];   // the rows of q of this wave's row tiles, read by nobody else: o takes their place
      // LDS reads are issued a group ahead of the matrix instructions that consume them, and the products of a column of blocks
      // ahead of the elementwise work on the one before it (the fences keep both there)
      v8 fq[2][KS], fh[2][KS], fka[KS], fkb[KS];
      auto read_k = [&](int tj, v8* f) __attribute__((always_inline)) {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) f[ks] = row_frag(Kr, 16 * tj, 32 * ks);
      };
      auto read_h = [&](int n) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) fh[x][ks] = row_frag(sH[b], 32 * n + 16 * x, 32 * ks);
      };
      f32x4 gj[4], rj[4];
      float gi[2], eg[2], ri[2];
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        gi[a] = sGam[b3][16 * TI[a] + c];
        eg[a] = sEg[b3][16 * TI[a] + c];
        if constexpr (L2N) ri[a] = sRq[b][16 * TI[a] + c];
      }
#pragma unroll
      for (int tj = 0; tj <= TI[1]; ++tj) {
        gj[tj] = *(const f32x4*)&sGam[b3][16 * tj + 4 * g];
        if constexpr (L2N) rj[tj] = *(const f32x4*)&sRk[b3][16 * tj + 4 * g];
      }
      __builtin_amdgcn_sched_barrier(0);
      read_k(0, fka);
#pragma unroll
      for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) fq[a][ks] = row_frag(Q, 16 * TI[a], 32 * ks);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 ex[2][4];   // e^{gamma_i - gamma_j}
#pragma unroll
      for (int tj = 0; tj <= TI[1]; ++tj)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          if (tj > TI[a]) continue;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            ex[a][tj][r] = __expf(gi[a] - gj[tj][r]);
            if constexpr (L2N) ex[a][tj][r] *= ri[a] * rj[tj][r];
          }
        }
      if constexpr (L2N) {
#pragma unroll
        for (int a = 0; a < 2; ++a) eg[a] *= ri[a];
      }
      __builtin_amdgcn_sched_barrier(0);
      // the scores, block by block transposed: this lane has row 16 ti + c, columns 16 tj + 4 g ..
      v4 P[2][4];
      f32x4 sc[2][4];
      auto products = [&](int tj, const v8* f) __attribute__((always_inline)) {
        sc[0][tj] = sc[1][tj] = zero4();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int a = 0; a < 2; ++a)
            if (tj <= TI[a]) sc[a][tj] = Elem<T>::mfma16(f[ks], fq[a][ks], sc[a][tj]);
      };
      auto scores = [&](int tj) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          if (tj > TI[a]) continue;
#pragma unroll
          for (int r = 0; r < 4; ++r)
            P[a][tj][r] = (T)((TI[a] > tj || 4 * g + r <= c) ? p.scale * sc[a][tj][r] * ex[a][tj][r] : 0.f);
          if constexpr (KEEP) {
            if (Pg) *(v4*)&Pg[(TI[a] * (TI[a] + 1) / 2 + tj) * 256 + c * 16 + 4 * g] = P[a][tj];
          }
        }
      };
      f32x4 acc[NC][2][2];   // [n][row tile][x]: row 16 ti + c, columns 32 n + 8 g + 4 x ..
      auto mul_h = [&](int n) __attribute__((always_inline)) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int x = 0; x < 2; ++x) acc[n][a][x] = zero4();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int x = 0; x < 2; ++x) acc[n][a][x] = Elem<T>::mfma16(fh[x][ks], fq[a][ks], acc[n][a][x]);
      };
      v8 fv[2][2];   // [x][32 time rows]
      auto read_v = [&](int n) __attribute__((always_inline)) {
#pragma unroll
        for (int x = 0; x < 2; ++x)
#pragma unroll
          for (int s = 0; s < 2; ++s)
            if (2 * s <= TI[1]) fv[x][s] = vn_frag(sVn[b], 32 * n + 16 * x, 32 * s);
      };
      read_k(1, fkb);
      __builtin_amdgcn_sched_barrier(0);
      products(0, fka);
      __builtin_amdgcn_sched_barrier(0);
      read_k(2, fka);
      __builtin_amdgcn_sched_barrier(0);
      products(1, fkb);
      scores(0);
      __builtin_amdgcn_sched_barrier(0);
      if (TI[1] == 3) read_k(3, fkb);
      read_h(0);
      __builtin_amdgcn_sched_barrier(0);
      products(2, fka);
      scores(1);
      __builtin_amdgcn_sched_barrier(0);
      if (TI[1] == 3) products(3, fkb);
      scores(2);
      __builtin_amdgcn_sched_barrier(0);
      read_v(0);
      __builtin_amdgcn_sched_barrier(0);
      mul_h(0);
      if (TI[1] == 3) scores(3);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (NC > 1) {
        read_h(1);
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (KEEP) {
        if (Pg) Pg += (int64_t)H * kTriElems;
      }
      const int L = oc == nchunks - 1 ? Llast : BT;
#pragma unroll
      for (int n = 0; n < NC; ++n) {
        if (n > 0) {
          read_v(n);
          mul_h(n);
        }
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int x = 0; x < 2; ++x)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[n][a][x][r] *= p.scale * eg[a];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
          for (int a = 0; a < 2; ++a) {
            if (2 * s > TI[a]) continue;
            v4 hi = {(T)0.f, (T)0.f, (T)0.f, (T)0.f};   // above the diagonal
            if (2 * s + 1 <= TI[a]) hi = P[a][2 * s + 1];
            const v8 fp = __builtin_shufflevector(P[a][2 * s], hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
            for (int x = 0; x < 2; ++x) acc[n][a][x] = Elem<T>::mfma16(fv[x][s], fp, acc[n][a][x]);
          }
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          v8 o;
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            o[r] = (T)acc[n][a][0][r];
            o[4 + r] = (T)acc[n][a][1][r];
          }
          if constexpr (NC == 1) {
            if (16 * TI[a] + c < L) *(v8*)(ob + (olane + (uint32_t)(16 * TI[a]) * opitch)) = o;
          } else {
            *(v8*)&own[16 * TI[a] * K + c * BV + (((4 * n + g) ^ (c & 7)) << 3)] = o;
          }
        }
      }
      if constexpr (NC == 2) {
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            const int row = 8 * i + orow;
            const v8 o = *(const v8*)&own[16 * TI[a] * K + row * BV + (((lane & 7) ^ (row & 7)) << 3)];
            if (16 * TI[a] + row < L) *(v8*)(ob + (olane + (uint32_t)(16 * TI[a] + 8 * i) * opitch)) = o;
          }
      }
      ob += (int64_t)BT * H * V * 2;
      b3 = b3 == 2 ? 0 : b3 + 1;
    };
    auto run = [&](auto t0, auto t1) __attribute__((always_inline)) {
      lds_barrier();
      lds_barrier();
      for (int ci = 1; ci < nchunks; ++ci) {
        output(ci - 1, t0, t1);
        lds_barrier();
      }
      output(nchunks - 1, t0, t1);
    };
    if (wave == 2) run(std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
    else run(std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
  } else {
    // =========================== chain waves ===========================
    const float* hin = p.split.ratio ? p.split.states + (span.slot * H + hh) * (int64_t)K * V
                       : p.h0        ? p.h0 + (int64_t)nh * K * V
                                     : nullptr;
    const int vcol = 8 * (c >> 2) + 4 * wave + (c & 3);   // of every 32 columns
    f32x4 acc[NC][KT];   // acc[n][kt][r] = h[16 kt + 4 g + r][32 n + vcol]
#pragma unroll
    for (int n = 0; n < NC; ++n)
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) {
        acc[n][kt] = zero4();
        if (hin) {
          const float* h0p = hin + vbase + 32 * n + vcol;
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[n][kt][r] = h0p[(int64_t)(16 * kt + 4 * g + r) * V];
        }
      }
    if (nchunks > 0) {
      // this lane's places in the tiles: row fragments of k and of the two tiles it writes, transposed fragments of k
      int roff[2 * KS], coff[KT];
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) roff[i] = tile_at<K>(c, 16 * i + 4 * g);
#pragma unroll
      for (int kt = 0; kt < KT; ++kt) coff[kt] = tile_at<K>(4 * g + (c >> 2), 16 * kt + 4 * (c & 3));
      int toff[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) toff[tt] = tile_at<BT>(16 * wave + c, 16 * tt + 4 * g);
      const int voff = (4 * g + (c >> 2)) * BV + 8 * (c & 3) + 4 * wave;
      lds_barrier();
      int b3 = 0;   // ci modulo 3
      for (int ci = 0; ci < nchunks; ++ci) {
        const int b = ci & 1;
        const T *Kr = sK[b3], *Tu = sTu[b];
        // LDS reads are issued a group ahead of the matrix instructions that consume them (the fences keep that order; with 128
        // key channels a group of k is sixteen reads, and two are on their way before the first is used)
        v8 fa[2][KS], fb[2][KS];
        auto read_k = [&](int t0, v8 (*f)[KS]) __attribute__((always_inline)) {   // two row tiles
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
              const T* r = Kr + 16 * (t0 + i) * K;
              const v4 lo = *(lds_v4*)(r + roff[2 * ks]), hi = *(lds_v4*)(r + roff[2 * ks + 1]);
              f[i][ks] = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
            }
        };
        if constexpr (DELTA) read_k(0, fa);
        __builtin_amdgcn_sched_barrier(0);
        // the state as an operand: two stacked accumulators per 32-slice; its two halves are what the tile takes
        v8 hb[NC][KS];
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              hb[n][ks][e] = (T)acc[n][2 * ks][e];
              hb[n][ks][4 + e] = (T)acc[n][2 * ks + 1][e];
            }
          }
        if constexpr (DELTA) read_k(2, fb);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 d[NC][4];
        auto mul_k = [&](int t0, const v8 (*f)[KS]) __attribute__((always_inline)) {
#pragma unroll
          for (int n = 0; n < NC; ++n) d[n][t0] = d[n][t0 + 1] = zero4();
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
              for (int n = 0; n < NC; ++n) d[n][t0 + i] = Elem<T>::mfma16(f[i][ks], hb[n][ks], d[n][t0 + i]);
        };
        if constexpr (DELTA) mul_k(0, fa);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 eg[4], ed[4];
        v4 vv[NC][4];
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          if constexpr (L2N) eg[tt] = *(const f32x4*)&sEgk[b3][16 * tt + 4 * g];
          else eg[tt] = *(const f32x4*)&sEg[b3][16 * tt + 4 * g];
#pragma unroll
          for (int n = 0; n < NC; ++n)   // four rows of one value column: the transposing load
            vv[n][tt] = __builtin_bit_cast(v4, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                                   (lds_s4*)&sV[b][voff + 16 * tt * BV + 32 * n]));
        }
        v8 ft[6];
        if constexpr (DELTA) {
          ft[0] = frag_tri<T>(Tu, 0, 0, lane);
          ft[1] = frag_tri<T>(Tu, 1, 0, lane);
          ft[2] = frag_tri<T>(Tu, 2, 0, lane);
          ft[4] = frag_tri<T>(Tu, 3, 0, lane);
          __builtin_amdgcn_sched_barrier(0);
          mul_k(2, fb);
          __builtin_amdgcn_sched_barrier(0);
          ft[3] = frag_tri<T>(Tu, 2, 1, lane);
          ft[5] = frag_tri<T>(Tu, 3, 1, lane);
        }
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) ed[tt] = *(const f32x4*)&sEd[b3][16 * tt + 4 * g];
        const float dec = sDec[b3];
        v8 fk[2][KT];   // [half of the row tiles][tile, 32 time rows]
        auto read_kt = [&](int half) __attribute__((always_inline)) {
#pragma unroll
          for (int x = 0; x < KT; ++x) {
            const T* r = Kr + coff[half * (KT / 2) + (x >> 1)] + 32 * (x & 1) * K;
            const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)r);
            const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(r + 16 * K));
            fk[half][x] =
                __builtin_shufflevector(__builtin_bit_cast(v4, lo), __builtin_bit_cast(v4, hi), 0, 1, 2, 3, 4, 5, 6, 7);
          }
        };
        __builtin_amdgcn_sched_barrier(0);
        v8 vs[NC][2];
        f32x4 vn[NC][4];
        if constexpr (DELTA) {
          v8 rb[NC][2];
          // r = v - e^{gamma} (k h), as the operand contracting over time
#pragma unroll
          for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
              for (int r = 0; r < 4; ++r) rb[n][tt >> 1][(tt & 1) * 4 + r] = (T)((float)vv[n][tt][r] - d[n][tt][r] * eg[tt][r]);
          // v_new = Tu r; Tu is lower triangular: row tiles 0 and 1 only meet the first 32 rows of r
#pragma unroll
          for (int n = 0; n < NC; ++n) {
            vn[n][2] = Elem<T>::mfma16(ft[2], rb[n][0], zero4());
            vn[n][3] = Elem<T>::mfma16(ft[4], rb[n][0], zero4());
            vn[n][0] = Elem<T>::mfma16(ft[0], rb[n][0], zero4());
            vn[n][1] = Elem<T>::mfma16(ft[1], rb[n][0], zero4());
            vn[n][2] = Elem<T>::mfma16(ft[3], rb[n][1], vn[n][2]);
            vn[n][3] = Elem<T>::mfma16(ft[5], rb[n][1], vn[n][3]);
          }
        } else {
#pragma unroll
          for (int n = 0; n < NC; ++n)
#pragma unroll
            for (int tt = 0; tt < 4; ++tt)
#pragma unroll
              for (int r = 0; r < 4; ++r) vn[n][tt][r] = (float)vv[n][tt][r];
        }
        __builtin_amdgcn_sched_barrier(0);
        read_kt(0);
        __builtin_amdgcn_sched_barrier(0);
        // in the shade of those: the entering state for the output waves, the decay of the accumulators
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int ks = 0; ks < KS; ++ks) {
            T* h = &sH[b][(32 * n + 16 * wave) * K];
            *(v4*)(h + roff[2 * ks]) = __builtin_shufflevector(hb[n][ks], hb[n][ks], 0, 1, 2, 3);
            *(v4*)(h + roff[2 * ks + 1]) = __builtin_shufflevector(hb[n][ks], hb[n][ks], 4, 5, 6, 7);
          }
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int kt = 0; kt < KT; ++kt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[n][kt][r] *= dec;
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt)
#pragma unroll
            for (int r = 0; r < 4; ++r) vs[n][tt >> 1][(tt & 1) * 4 + r] = (T)(vn[n][tt][r] * ed[tt][r]);
        __builtin_amdgcn_sched_barrier(0);
        auto mul_kt = [&](int half) __attribute__((always_inline)) {
#pragma unroll
          for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < KT / 2; ++i)
#pragma unroll
              for (int n = 0; n < NC; ++n)
                acc[n][half * (KT / 2) + i] = Elem<T>::mfma16(fk[half][2 * i + s], vs[n][s], acc[n][half * (KT / 2) + i]);
        };
        read_kt(1);
        __builtin_amdgcn_sched_barrier(0);
        mul_kt(0);
#pragma unroll
        for (int n = 0; n < NC; ++n)
#pragma unroll
          for (int tt = 0; tt < 4; ++tt) {
            v4 x;
#pragma unroll
            for (int r = 0; r < 4; ++r) x[r] = (T)vn[n][tt][r];
            *(v4*)&sVn[b][32 * n * BT + toff[tt]] = x;
          }
        __builtin_amdgcn_sched_barrier(0);
        mul_kt(1);
        lds_barrier();
        b3 = b3 == 2 ? 0 : b3 + 1;
      }
    }
    if (p.ht && span.last) {
      float* htp = p.ht + (int64_t)nh * K * V + vbase + vcol;
#pragma unroll
      for (int n = 0; n < NC; ++n)
#pragma unroll
        for (int kt = 0; kt < KT; ++kt)
#pragma unroll
          for (int r = 0; r < 4; ++r) htp[(int64_t)(16 * kt + 4 * g + r) * V + 32 * n] = acc[n][kt][r];
    }
  }
}

template <typename T>
int launch_scan(const GdrScanParams& p, int K, hipStream_t st) {
  // (sequence, head) pairs, or (segment, head) pairs of sequences cut into segments
  const int64_t seqs = !p.split.ratio ? p.N : p.split.seg_table ? p.split.nseg : (int64_t)p.split.nseg * p.N;
  const int64_t nblk = seqs * p.H * (p.V / 32);
  FLA_REQUIRE(nblk <= 0x7fffffffLL, FLA_E_UNSUPPORTED);
  if (nblk == 0) return FLA_OK;
  const bool keep = p.v_new != nullptr, l2n = p.l2_eps >= 0.f, delta = p.AT != nullptr;
  if ((keep && l2n) || (!delta && (keep || l2n))) return FLA_E_UNSUPPORTED;
  const dim3 block(512);
#define FLA_SCAN(KK, NC)                                                                                             \
  {                                                                                                                   \
    const dim3 grid((unsigned)(nblk / NC));                                                                           \
    if (!delta) hipLaunchKernelGGL((gdr_fwd_scan_kernel<T, KK, false, NC, false, false>), grid, block, 0, st, p);    \
    else if (keep) hipLaunchKernelGGL((gdr_fwd_scan_kernel<T, KK, true, NC, false, true>), grid, block, 0, st, p);   \
    else if (l2n) hipLaunchKernelGGL((gdr_fwd_scan_kernel<T, KK, false, NC, true, true>), grid, block, 0, st, p);    \
    else hipLaunchKernelGGL((gdr_fwd_scan_kernel<T, KK, false, NC, false, true>), grid, block, 0, st, p);            \
  }
  // 32-column slabs while they still give every workgroup a CU of its own
  const bool narrow = nblk <= kNumCUs;
  if (K == 64 && narrow) FLA_SCAN(64, 1)
  else if (K == 64) FLA_SCAN(64, 2)
  else if (K == 128 && narrow) FLA_SCAN(128, 1)
  else if (K == 128) FLA_SCAN(128, 2)
  else return FLA_E_UNSUPPORTED;
#undef FLA_SCAN
  FLA_CHECK_LAUNCH();
  return FLA_OK;
}

}  // namespace

static int gdr_fwd_scan_impl(const void* q, const void* k, const void* v, const void* AT, const float* g_cumsum,
                             const float* h0, void* o, float* ht, void* v_new, void* h_frag_t, void* Aqk_out,
                             const int64_t* offsets, const int64_t* chunk_offsets, const int64_t* seq_order,
                             int qkv_dtype, int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t N,
                             float scale, float l2_eps, fla_stream_t stream, const float* k_rstd = nullptr,
                             const fla_split* split = nullptr) {
  FLA_REQUIRE(q && k && v && o, FLA_E_INVALID);   // AT == NULL: the plain scan (fla_chunk_simple_gla_fwd_scan)
  FLA_REQUIRE((l2_eps >= 0.f) == (k_rstd != nullptr), FLA_E_INVALID);
  FLA_REQUIRE(B >= 0 && T >= 0 && H > 0 && K > 0 && V > 0 && N >= 0, FLA_E_INVALID);
  FLA_REQUIRE(offsets ? (B == 1 && chunk_offsets != nullptr) : N == B, FLA_E_INVALID);
  FLA_REQUIRE(V % 64 == 0 && H <= 0x7fffff, FLA_E_UNSUPPORTED);
  FLA_REQUIRE((v_new == nullptr) == (h_frag_t == nullptr), FLA_E_INVALID);
  FLA_REQUIRE(Aqk_out == nullptr || v_new != nullptr, FLA_E_INVALID);
  FLA_REQUIRE(((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)AT | (uintptr_t)o | (uintptr_t)v_new |
               (uintptr_t)h_frag_t | (uintptr_t)Aqk_out) % 16 == 0, FLA_E_ALIGNMENT);
  GdrScanParams p{q, k, v, AT, g_cumsum, h0, o, ht, v_new, h_frag_t, Aqk_out, offsets, chunk_offsets, seq_order, T,
                  (int)H, (int)V, (int)N, scale, l2_eps, k_rstd, split_view(split)};
  if (split) {
    const int rc = AT ? gdr_split_states(k, v, AT, g_cumsum, k_rstd, h0, split, offsets, chunk_offsets, qkv_dtype, T, H, K, V, N,
                                         (hipStream_t)stream)
                      : gla_split_states(k, v, g_cumsum, h0, split, true, false, false, 1.f, 0.f, 1.f, offsets, chunk_offsets,
                                         qkv_dtype, FLA_F32, T, H, K, V, N, (hipStream_t)stream);
    if (rc) return rc;
  }
  if (qkv_dtype == FLA_BF16) return launch_scan<bf16>(p, (int)K, (hipStream_t)stream);
  if (qkv_dtype == FLA_F16) return launch_scan<f16>(p, (int)K, (hipStream_t)stream);
  return FLA_E_UNSUPPORTED;
}

extern "C" int fla_chunk_gated_delta_rule_fwd_scan(const void* q, const void* k, const void* v, const void* AT,
                                                   const float* g_cumsum, const float* h0, void* o, float* ht,
                                                   void* v_new, void* h_frag_t, void* Aqk_out, const int64_t* offsets, const int64_t* chunk_offsets,
                                                   const int64_t* seq_order, int qkv_dtype, int64_t B, int64_t T,
                                                   int64_t H, int64_t K, int64_t V, int64_t N, float scale,
                                                   fla_stream_t stream) {
  FLA_REQUIRE(AT, FLA_E_INVALID);
  return gdr_fwd_scan_impl(q, k, v, AT, g_cumsum, h0, o, ht, v_new, h_frag_t, Aqk_out, offsets, chunk_offsets,
                           seq_order, qkv_dtype, B, T, H, K, V, N, scale, -1.f, stream);
}

extern "C" int fla_chunk_gated_delta_rule_fwd_scan_l2norm(const void* q, const void* k, const void* v, const void* AT,
                                                          const float* g_cumsum, const float* k_rstd, const float* h0,
                                                          void* o, float* ht,
                                                          const int64_t* offsets, const int64_t* chunk_offsets,
                                                          const int64_t* seq_order, int qkv_dtype, int64_t B,
                                                          int64_t T, int64_t H, int64_t K, int64_t V, int64_t N,
                                                          float scale, float eps, fla_stream_t stream) {
  FLA_REQUIRE(eps >= 0.f && k_rstd, FLA_E_INVALID);
  return gdr_fwd_scan_impl(q, k, v, AT, g_cumsum, h0, o, ht, nullptr, nullptr, nullptr, offsets, chunk_offsets,
                           seq_order, qkv_dtype, B, T, H, K, V, N, scale, eps, stream, k_rstd);
}

extern "C" int fla_chunk_simple_gla_fwd_scan(const void* q, const void* k, const void* v, const float* g,
                                             const float* h0, void* o, float* ht, const int64_t* offsets,
                                             const int64_t* chunk_offsets, const int64_t* seq_order, int qkv_dtype,
                                             int64_t B, int64_t T, int64_t H, int64_t K, int64_t V, int64_t N,
                                             float scale, fla_stream_t stream) {
  return gdr_fwd_scan_impl(q, k, v, nullptr, g, h0, o, ht, nullptr, nullptr, nullptr, offsets, chunk_offsets,
                           seq_order, qkv_dtype, B, T, H, K, V, N, scale, -1.f, stream);
}

extern "C" int fla_chunk_gated_delta_rule_fwd_scan_split(const void* q, const void* k, const void* v, const void* AT,
                                                         const float* gates, const float* k_rstd, const float* h0, void* o,
                                                         float* ht, void* v_new, void* h_frag_t, void* Aqk_out,
                                                         const int64_t* offsets, const int64_t* chunk_offsets,
                                                         const fla_split* split, int qkv_dtype, int64_t B, int64_t T,
                                                         int64_t H, int64_t K, int64_t V, int64_t N, float scale, float eps,
                                                         fla_stream_t stream) {
  FLA_REQUIRE(split && (AT || gates), FLA_E_INVALID);
  FLA_REQUIRE(K <= 128 && V <= 128, FLA_E_UNSUPPORTED);
  return gdr_fwd_scan_impl(q, k, v, AT, gates, h0, o, ht, v_new, h_frag_t, Aqk_out, offsets, chunk_offsets, nullptr, qkv_dtype, B,
                           T, H, K, V, N, scale, k_rstd ? eps : -1.f, stream, k_rstd, split);
}
