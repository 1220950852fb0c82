// Pieces shared by the kernels that form all gradients of a (chunk, head) in one workgroup of four waves
// (gdr_bwd_chunk.hip, gla_bwd_chunk.hip).
#pragma once
#include "chunk_common.h"

namespace {

// A [64][D] tile moved in 16-byte pieces, whole rows per group of D / 8 lanes.  Rows past the end of a short chunk
// re-read its last row (no load sits under a branch) and are cleared on the way to LDS.
template <typename T, int D>
struct RowTile {
  typedef typename Elem<T>::v8 v8;
  static constexpr int C8 = D / 8, N = BT * C8 / 256;
  static FLA_DEVICE void load(const void* src, int64_t r0h, int L, int H, int tid, v8* reg) {
    const char* base = (const char*)src + r0h * D * (int64_t)sizeof(T);
    const uint32_t pitch = (uint32_t)H * D * (uint32_t)sizeof(T), col = (uint32_t)(tid % C8) * 16u;
    const uint32_t lim = (uint32_t)(L - 1) * pitch + col;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const uint32_t o = (uint32_t)((tid + 256 * i) / C8) * pitch + col;
      reg[i] = *(const v8*)(base + (o < lim ? o : lim));
    }
  }
  static FLA_DEVICE void put(T* dst, int ld, int L, int tid, const v8* reg) {
    const v8 z = {(T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f};
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = tid + 256 * i, row = e / C8, c8 = (e % C8) * 8;
      *(v8*)&dst[row * ld + c8] = row < L ? reg[i] : z;
    }
  }
  static FLA_DEVICE void get(const T* tile, int ld, int tid, v8* reg) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int e = tid + 256 * i;
      reg[i] = *(const v8*)&tile[e / C8 * ld + (e % C8) * 8];
    }
  }
  static FLA_DEVICE void store(void* dst, int64_t r0h, int L, int H, int tid, const v8* reg) {
    char* base = (char*)dst + r0h * D * (int64_t)sizeof(T);
    const uint32_t pitch = (uint32_t)H * D * (uint32_t)sizeof(T), col = (uint32_t)(tid % C8) * 16u;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int row = (tid + 256 * i) / C8;
      // This launch does not read the gradients again: they need not push the operands of other workgroups out of the L2.
      // Whole steps with plain stores / with these: gla_bwd_chunk, 4 x 4096 tokens, 16 heads of 128, 474 / 465 us, 2 x 2000
      // tokens, 32 heads of 64, 117 / 102; gdr_bwd_chunk, the first shape, 527 / 525; a mixing layer of 2 x 2048 tokens, whose
      // norms and convolutions read them in the next launches, 319.9 / 320.7 (the runs of one side differ by 0.6).
      if (row < L) __builtin_nontemporal_store(reg[i], (v8*)(base + ((uint32_t)row * pitch + col)));
    }
  }
};

// The lane id through an opaque copy: addresses formed from it are formed where they are used.  Left to itself the compiler
// forms the LDS and row addresses of all phases once per item and keeps them, a hundred registers it then spills - and every
// reload of a spilled register waits for all loads and stores in flight (gdr_bwd_chunk_kernel: 245 us instead of 204).
FLA_DEVICE int fresh_tid(int tid) {
  asm volatile("" : "+v"(tid));
  return tid;
}
#define FLA_PHASE(t0)                                    \
  const int tid = fresh_tid(t0), lane = tid & 63;        \
  const int l32 = lane & 31, hi4 = 4 * (lane >> 5);      \
  (void)l32, (void)hi4

// Lane SRC of each half wave, in all its lanes (through the LDS crossbar: no VALU cycles)
template <int SRC>
FLA_DEVICE float of_half(float x) {
  return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(x), SRC << 5));
}
// Inclusive prefix / suffix sums over the 32 lanes of each half wave: its total is in lanes 31 and 63 of the prefix sums, in
// lanes 0 and 32 of the suffix sums.
FLA_DEVICE float half_prefix(float x) {
  x = row_prefix16(x);
  // lane 15 (47) on top of lanes 16-31 (48-63); the other rows keep their sums.  (As a builtin this is three instructions.)
  asm("s_nop 1\n\tv_add_f32_dpp %0, %0, %0 row_bcast:15 row_mask:0xa bank_mask:0xf" : "+v"(x));
  return x;
}
FLA_DEVICE float half_suffix(float x, int lane) {
  x = row_suffix16(x);
  const float t = of_half<16>(x);
  return x + ((lane & 16) ? 0.f : t);
}

}  // namespace
