// Depthwise causal short convolution over time in the layers' own [B,T,D] layout (channels
// last), with optional bias and SiLU:  y[b,t,d] = act(bias[d] + sum_i w[d,i] x[b,t-(W-1)+i,d]).
// Replaces the external causal_conv1d package the reference's ShortConvolution needs
// (fla/modules/convolution.py:79-211; forward :171-186, single-token step :188-211).
//
// HBM-streaming kernels: a lane owns 4 or 2 adjacent channels of one tile of consecutive time steps, all rows of the tile
// (and the W-1 rows of halo that the neighbouring tile reads too) in flight at once, the last W inputs (and, in backward,
// the last W pre-activation gradients) in registers.  The weight/bias gradients are accumulated in registers over all
// tiles a lane visits, summed over the workgroup's waves in LDS and written once per workgroup (the host adds the
// per-workgroup partial sums: deterministic, no atomics).
#include "fla_common.h"

namespace {

// A lane's slice of one row: N adjacent channels, kept in storage precision until use so that
// a whole tile of rows can be in flight at once.
template <typename T, int N>
struct Chan {
  typedef T raw __attribute__((ext_vector_type(N)));
  static FLA_DEVICE void to_f32(raw r, float* o) {
#pragma unroll
    for (int i = 0; i < N; ++i) o[i] = (float)r[i];
  }
  static FLA_DEVICE raw from_f32(const float* v) {
    raw r;
#pragma unroll
    for (int i = 0; i < N; ++i) r[i] = (T)v[i];
    return r;
  }
};

struct ConvParams {
  const void* x;       // [B,T,D]
  const float* w;      // [D,W] fp32
  const float* bias;   // [D] fp32 or NULL
  void* y;             // [B,T,D]
  const void* dy;      // backward
  void* dx;
  float* dw;           // [conv_bwd_parts(B, T), D, W] fp32 partial sums
  float* dbias;        // [conv_bwd_parts(B, T), D] fp32 partial sums or NULL
  int64_t B, T;
  int D;
  unsigned cblocks, tiles_per_seq, tiles;   // channel blocks of a row, tiles of a sequence and of all
  unsigned tile0;                           // forward: the launch's first tile
};

FLA_DEVICE float silu_f(float z) { return z * __builtin_amdgcn_rcpf(1.f + __expf(-z)); }
FLA_DEVICE float silu_grad(float z) {
  const float s = __builtin_amdgcn_rcpf(1.f + __expf(-z));  // hardware reciprocal (1 ulp), not an IEEE division
  return s * (1.f + z * (1.f - s));
}

// The taps w[i][j] and bias of CV adjacent channels: W CV consecutive floats, four at a time
template <int W, int CV>
FLA_DEVICE void load_weights(const ConvParams& p, int d0, float (*w)[CV], float* bias) {
  const float* src = p.w + (int64_t)d0 * W;
  if constexpr (W * CV % 4 == 0) {
#pragma unroll
    for (int e = 0; e < W * CV; e += 4) {
      const f32x4 x = *(const f32x4_any*)(src + e);
#pragma unroll
      for (int z = 0; z < 4; ++z) w[(e + z) % W][(e + z) / W] = x[z];
    }
  } else {
#pragma unroll
    for (int e = 0; e < W * CV; ++e) w[e % W][e / W] = src[e];
  }
#pragma unroll
  for (int j = 0; j < CV; ++j) bias[j] = p.bias ? p.bias[d0 + j] : 0.f;
}

// A row's address in scalar registers: the lane's part of it is then one 32-bit offset for all rows.  The compiler on its
// own folds the lane's part into every row's address, two vector registers and a 64-bit multiply and add for each.
typedef const char __attribute__((address_space(1)))* RowIn;
typedef char __attribute__((address_space(1)))* RowOut;
FLA_DEVICE RowIn row_in(const char* base, int64_t byte) {
  RowIn r = (RowIn)(base + byte);
  asm("" : "+s"(r));
  return r;
}
FLA_DEVICE RowOut row_out(char* base, int64_t byte) {
  RowOut r = (RowOut)(base + byte);
  asm("" : "+s"(r));
  return r;
}
template <typename RAW>
FLA_DEVICE RAW load_at(RowIn row, unsigned byte) { return *(const RAW __attribute__((address_space(1)))*)(row + byte); }
template <typename RAW>
FLA_DEVICE void store_at(RowOut row, unsigned byte, RAW x) { *(RAW __attribute__((address_space(1)))*)(row + byte) = x; }

// One tile of TT steps from t0.  FULL: all of them lie inside the sequence, so that every load and store is
// unconditional.  Loads and stores share one counter of what is outstanding: behind a store under a branch the wait for
// the next row has to assume it was skipped, and waits for the row before to have been written.  (8 steps of 4 channels,
// 2 x 2048 x 2048 in bf16: 10.2 us with a branch around each row's store, 8.1 without; 2 x 576 x 512 6.2 and 3.9.)
template <typename T, int W, int TT, int CV, bool SILU, bool FULL>
FLA_DEVICE void conv_fwd_tile(const ConvParams& p, int64_t b, int64_t t0, int d0, const float (*w)[CV], const float* bias) {
  typedef Chan<T, CV> C;
  typedef typename C::raw raw;
  const int64_t pitch = (int64_t)p.D * sizeof(T);
  const char* xb = (const char*)p.x + b * p.T * pitch;
  char* yb = (char*)p.y + b * p.T * pitch;
  const unsigned vo = (unsigned)d0 * sizeof(T);
  // rows t0-(W-1) .. t0+TT-1; rows outside the sequence read its first or last row
  raw rows[TT + W - 1];
#pragma unroll
  for (int s = 0; s < TT + W - 1; ++s) {
    const int64_t t = t0 - (W - 1) + s;
    const int64_t tc = s < W - 1 ? (t < 0 ? 0 : t) : FULL || t < p.T ? t : p.T - 1;
    rows[s] = load_at<raw>(row_in(xb, tc * pitch), vo);
  }
  float win[W][CV];   // win[i] = x[t - (W-1) + i]
#pragma unroll
  for (int s = 0; s < TT + W - 1; ++s) {
    const int64_t t = t0 - (W - 1) + s;
#pragma unroll
    for (int i = 0; i < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CV; ++j) win[i][j] = win[i + 1][j];
    C::to_f32(rows[s], win[W - 1]);
    if (s < W - 1) {
#pragma unroll
      for (int j = 0; j < CV; ++j) win[W - 1][j] = t >= 0 ? win[W - 1][j] : 0.f;
    }
    if (s >= W - 1 && (FULL || t < p.T)) {
      float out[CV];
#pragma unroll
      for (int j = 0; j < CV; ++j) {
        float acc = bias[j];
#pragma unroll
        for (int i = 0; i < W; ++i) acc = fmaf(w[i][j], win[i][j], acc);
        out[j] = SILU ? silu_f(acc) : acc;
      }
      store_at<raw>(row_out(yb, t * pitch), vo, C::from_f32(out));
    }
  }
}

// block (64, 4): x = channel vector, y = tile; workgroups that share rows of x are adjacent in dispatch order
template <typename T, int W, int TT, int CV, bool SILU>
__global__ __launch_bounds__(256) void conv_fwd_kernel(ConvParams p) {
  const unsigned cb = blockIdx.x % p.cblocks;
  const unsigned first = __builtin_amdgcn_readfirstlane(p.tile0 + blockIdx.x / p.cblocks * 4 + threadIdx.y);
  const int d0 = (int)(cb * 64 + threadIdx.x) * CV;
  if (d0 >= p.D) return;
  float w[W][CV], bias[CV];   // (ahead of the rows: all of them are used with the first one)
  load_weights<W, CV>(p, d0, w, bias);
  for (unsigned tile = first; tile < p.tiles; tile += gridDim.x / p.cblocks * 4) {
    const unsigned b = tile / p.tiles_per_seq;
    const int64_t t0 = (int64_t)(tile - b * p.tiles_per_seq) * TT;
    if (t0 + TT <= p.T) conv_fwd_tile<T, W, TT, CV, SILU, true>(p, b, t0, d0, w, bias);
    else conv_fwd_tile<T, W, TT, CV, SILU, false>(p, b, t0, d0, w, bias);
    if (sizeof(T) == 2) break;   // (launch_fwd)
  }
}

template <typename T, int W, int TT, int CV, bool SILU, bool BIAS, bool FULL>
FLA_DEVICE void conv_bwd_tile(const ConvParams& p, int64_t b, int64_t t0, int d0, const float (*w)[CV], const float* bias,
                              float (*dw)[CV], float* db) {
  typedef Chan<T, CV> C;
  typedef typename C::raw raw;
  const int64_t pitch = (int64_t)p.D * sizeof(T);
  const char* xb = (const char*)p.x + b * p.T * pitch;
  const char* gb = (const char*)p.dy + b * p.T * pitch;
  char* dxb = (char*)p.dx + b * p.T * pitch;
  const unsigned vo = (unsigned)d0 * sizeof(T);
  // x rows t0-(W-1) .. t0+TT+W-2 and dy rows t0 .. t0+TT+W-2 (rows outside the sequence read its first or last row and
  // count as zero)
  raw xr[TT + 2 * (W - 1)], gr[TT + W - 1];
#pragma unroll
  for (int s = 0; s < TT + 2 * (W - 1); ++s) {
    const int64_t t = t0 - (W - 1) + s;
    const int64_t tc = s < W - 1 ? (t < 0 ? 0 : t) : (FULL && s < TT + W - 1) || t < p.T ? t : p.T - 1;
    xr[s] = load_at<raw>(row_in(xb, tc * pitch), vo);
    if (s >= W - 1) gr[s - (W - 1)] = load_at<raw>(row_in(gb, tc * pitch), vo);
  }
  __builtin_amdgcn_sched_barrier(0);
  float win[W][CV];   // inputs   x[t-(W-1) .. t]
  float dpw[W][CV];   // pre-activation gradients of steps t-(W-1) .. t
#pragma unroll
  for (int j = 0; j < CV; ++j) {
#pragma unroll
    for (int i = 0; i < W; ++i) dpw[i][j] = 0.f;
#pragma unroll
    for (int i = 1; i < W; ++i) win[i][j] = t0 - W + i >= 0 ? (float)xr[i - 1][j] : 0.f;
  }
  // step s (time t0+s) forms the pre-activation gradient of its own time step; the input gradient of time t0+s-(W-1) is
  // complete once the W steps ahead of it are known
#pragma unroll
  for (int s = 0; s < TT + W - 1; ++s) {
    const int64_t t = t0 + s;
    const bool live = (FULL && s < TT) || t < p.T;
#pragma unroll
    for (int i = 0; i < W - 1; ++i)
#pragma unroll
      for (int j = 0; j < CV; ++j) {
        win[i][j] = win[i + 1][j];
        dpw[i][j] = dpw[i + 1][j];
      }
    C::to_f32(xr[s + W - 1], win[W - 1]);
    float gs[CV];
    C::to_f32(gr[s], gs);
#pragma unroll
    for (int j = 0; j < CV; ++j) {
      float dp = gs[j];
      if (SILU) {
        float pre = BIAS ? bias[j] : 0.f;
#pragma unroll
        for (int i = 0; i < W; ++i) pre = fmaf(w[i][j], win[i][j], pre);
        dp *= silu_grad(pre);
      }
      dpw[W - 1][j] = live ? dp : 0.f;
      if (s < TT && (FULL || live)) {   // own time step: weight and bias gradients
#pragma unroll
        for (int i = 0; i < W; ++i) dw[i][j] = fmaf(dpw[W - 1][j], win[i][j], dw[i][j]);
        if (BIAS) db[j] += dpw[W - 1][j];
      }
    }
    if (s >= W - 1 && (FULL || t - (W - 1) < p.T)) {
      float out[CV];
#pragma unroll
      for (int j = 0; j < CV; ++j) {
        float acc = 0.f;
        // dx[to] = sum_i w[i] dpre[to + (W-1) - i]; dpw[m] holds dpre[to + m]
#pragma unroll
        for (int i = 0; i < W; ++i) acc = fmaf(w[i][j], dpw[W - 1 - i][j], acc);
        out[j] = acc;
      }
      store_at<raw>(row_out(dxb, (t - (W - 1)) * pitch), vo, C::from_f32(out));
    }
    // the rows in order: without it a lane holds several rows' temporaries at once (135 registers instead of 126)
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Backward.  block (64, 4): x = channel vector, y = wave.  BIAS: p.bias, p.dbias or both
template <typename T, int W, int TT, int CV, bool SILU, bool BIAS>
__global__ __launch_bounds__(256) void conv_bwd_kernel(ConvParams p) {
  constexpr int SUMS = (W + BIAS) * CV;
  constexpr unsigned waves = 4;
  __shared__ float sred[waves][SUMS][64];
  const unsigned wave = __builtin_amdgcn_readfirstlane(threadIdx.y);
  const unsigned cb = blockIdx.x % p.cblocks, group = blockIdx.x / p.cblocks, groups = gridDim.x / p.cblocks;
  const int own = (int)(cb * 64 + threadIdx.x) * CV;
  const bool active = own < p.D;   // idle lanes still take part in the reduction barrier
  const int d0 = active ? own : 0;
  float w[W][CV], bias[CV], dw[W][CV], db[CV];
  load_weights<W, CV>(p, d0, w, bias);
#pragma unroll
  for (int j = 0; j < CV; ++j) {
#pragma unroll
    for (int i = 0; i < W; ++i) dw[i][j] = 0.f;
    db[j] = 0.f;
  }
  if (active) {
    // (the tiles that run at one time adjacent: 3 x 5500 x 512 in bf16 13.5 us, consecutive tiles per wave 16.2)
    for (unsigned tile = group * waves + wave; tile < p.tiles; tile += groups * waves) {
      const unsigned b = tile / p.tiles_per_seq;
      const int64_t t0 = (int64_t)(tile - b * p.tiles_per_seq) * TT;
      if (t0 + TT <= p.T) conv_bwd_tile<T, W, TT, CV, SILU, BIAS, true>(p, b, t0, d0, w, bias, dw, db);
      else conv_bwd_tile<T, W, TT, CV, SILU, BIAS, false>(p, b, t0, d0, w, bias, dw, db);
    }
  }
  // sum the workgroup's waves, then one partial per workgroup
#pragma unroll
  for (int j = 0; j < CV; ++j) {
#pragma unroll
    for (int i = 0; i < W; ++i) sred[wave][j * W + i][threadIdx.x] = dw[i][j];
    if (BIAS) sred[wave][W * CV + j][threadIdx.x] = db[j];
  }
  __syncthreads();
  if (!active) return;
  float* dwp = p.dw + ((int64_t)group * p.D + d0) * W;
  for (int e = wave; e < SUMS; e += waves) {
    const float sum = (sred[0][e][threadIdx.x] + sred[1][e][threadIdx.x]) + (sred[2][e][threadIdx.x] + sred[3][e][threadIdx.x]);
    if (e < W * CV) dwp[e] = sum;
    else if (p.dbias) p.dbias[(int64_t)group * p.D + d0 + e - W * CV] = sum;
  }
}

// single-token step: shift the cache [B,D,W] left by one, append x, y = act(bias + sum cache * w)
template <typename T, typename WT, int W>
__global__ __launch_bounds__(256) void conv_update_kernel(const T* __restrict__ x, T* __restrict__ cache,
                                                          const WT* __restrict__ w, const float* __restrict__ bias,
                                                          T* __restrict__ y, int64_t BD, int D, int silu) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= BD) return;
  const int d = (int)(i % D);
  T c[W];
#pragma unroll
  for (int k = 0; k < W; ++k) c[k] = cache[i * W + k];
#pragma unroll
  for (int k = 0; k < W - 1; ++k) c[k] = c[k + 1];
  c[W - 1] = x[i];
  float acc = bias ? bias[d] : 0.f;
#pragma unroll
  for (int k = 0; k < W; ++k) {
    acc = fmaf((float)c[k], (float)w[(int64_t)d * W + k], acc);
    cache[i * W + k] = c[k];
  }
  y[i] = (T)(silu ? silu_f(acc) : acc);
}

// Backward: few enough workgroups that the partial sums stay small, enough to fill the chip.  What bounds it: 2 x 2048 x 2048
// in bf16 is 50 MB (7 us out of the last-level cache) and 8 us of vector instructions, 12.5 us in all (14.2 with a store under a
// branch per row; 8 x 4096 x 2048 91 -> 83).
constexpr int kBwdShort = 8, kBwdLong = 16;
int64_t conv_bwd_parts(int64_t B, int64_t T) {
  const int64_t g = fla_cdiv(B * fla_cdiv(T, kBwdShort), 4);
  return g < 1 ? 1 : (g > 128 ? 128 : g);
}

// a launch has fewer than 2^32 threads in x: workgroups of 64 x 4
constexpr int64_t kMostBlocks = (1LL << 26) - 1;

template <typename T, int W, int TT, int CV, bool SILU>
int launch_fwd(ConvParams p, hipStream_t st) {
  const int64_t per = fla_cdiv(p.T, TT), tiles = p.B * per, cb = fla_cdiv(p.D / CV, 64);
  FLA_REQUIRE(tiles <= 0xffffffffLL - 0x100000 && cb <= kMostBlocks, FLA_E_UNSUPPORTED);
  p.cblocks = (unsigned)cb, p.tiles_per_seq = (unsigned)per, p.tiles = (unsigned)tiles;
  int64_t groups = fla_cdiv(tiles, 4);
  // fp32: a few tiles per wave, the weights loaded once (8 x 4096 x 2048: 96 - 98 us, a tile per wave up to 111); a tile per wave
  // in 16 bits (50 and 52 us)
  if (sizeof(T) == 4 && groups * cb > 4096) groups = fla_cdiv(4096, cb);
  const int64_t most = kMostBlocks / cb;   // rows of a few channels and 2^31 of them in 16 bits: the tiles of a launch after another's
  for (int64_t g0 = 0; g0 < groups; g0 += most) {
    p.tile0 = (unsigned)(4 * g0);
    const int64_t blocks = (groups - g0 < most ? groups - g0 : most) * cb;
    hipLaunchKernelGGL((conv_fwd_kernel<T, W, TT, CV, SILU>), dim3((unsigned)blocks), dim3(64, 4), 0, st, p);
    FLA_CHECK_LAUNCH();
  }
  return FLA_OK;
}

template <typename T, int W, int TT, int CV, bool SILU>
int launch_bwd(ConvParams p, hipStream_t st) {
  const int64_t per = fla_cdiv(p.T, TT), tiles = p.B * per, cb = fla_cdiv(p.D / CV, 64), groups = conv_bwd_parts(p.B, p.T);
  FLA_REQUIRE(tiles <= 0xffffffffLL - 0x10000 && groups * cb <= kMostBlocks, FLA_E_UNSUPPORTED);
  p.cblocks = (unsigned)cb, p.tiles_per_seq = (unsigned)per, p.tiles = (unsigned)tiles;
  const dim3 grid((unsigned)(groups * cb)), block(64, 4);   // a partial sum per workgroup of a channel block
  if (p.bias || p.dbias) hipLaunchKernelGGL((conv_bwd_kernel<T, W, TT, CV, SILU, true>), grid, block, 0, st, p);
  else hipLaunchKernelGGL((conv_bwd_kernel<T, W, TT, CV, SILU, false>), grid, block, 0, st, p);
  FLA_CHECK_LAUNCH();
  return FLA_OK;
}

template <typename T, int W, bool SILU>
int launch_conv(const ConvParams& p, bool bwd, hipStream_t st) {
  auto waves = [&](int steps, int channels) { return p.B * fla_cdiv(p.T, steps) * fla_cdiv(p.D / channels, 64); };
  if (bwd) {
    // Long tiles (3 rows of halo to recompute in 16 instead of 8) of 2 channels (4 take 230 registers: 13.8 us against 12.2 at
    // 2 x 2048 x 2048 in bf16) once they make two waves per SIMD; below that a wave's own steps are what a call waits for
    // (2 x 128 x 4096: short tiles 4.4 us, long ones 5.1).  fp32 takes 16-byte accesses where rows abound (8 x 4096 x 2048:
    // 152 us, with 8-byte ones 167 - 175).
    if (sizeof(T) == 4 && waves(kBwdShort, 4) >= 8 * 1024) return launch_bwd<T, W, kBwdShort, 4, SILU>(p, st);
    if (waves(kBwdLong, 2) < 2 * 1024) return launch_bwd<T, W, kBwdShort, 2, SILU>(p, st);
    return launch_bwd<T, W, kBwdLong, 2, SILU>(p, st);
  }
  // Little work: short tiles, a wave's own steps are what the call waits for (5 x 333 x 256: 8 x 2 3.5 us, 16 x 2 3.7).
  if (sizeof(T) == 2 && waves(16, 2) < 2 * 1024) return launch_fwd<T, W, 8, 2, SILU>(p, st);
  // 16 steps x 2 channels (39 registers: every wave of the chip's eight per SIMD) while 8 x 4 leave fewer than 16 waves per
  // SIMD to come (2 x 2048 x 2048 7.6 and 8.2 us, 7 x 642 x 4096 12.6 and 13.0); then fewer, wider loads
  // (8 x 4096 x 2048 52.3 and 50.0).  In fp32 four channels are 16 bytes.
  if (sizeof(T) == 2 && waves(8, 4) < 16 * 1024) return launch_fwd<T, W, 16, 2, SILU>(p, st);
  return launch_fwd<T, W, 8, 4, SILU>(p, st);
}

template <typename T>
int dispatch_conv(const ConvParams& p, int W, bool silu, bool bwd, hipStream_t st) {
#define C(WW) \
  if (W == WW) return silu ? launch_conv<T, WW, true>(p, bwd, st) : launch_conv<T, WW, false>(p, bwd, st);
  C(2) C(3) C(4)
#undef C
  return FLA_E_UNSUPPORTED;
}

template <typename T, typename WT>
int dispatch_update(const void* x, void* cache, const void* w, const float* bias, void* y, int64_t BD, int D, int W,
                    int silu, hipStream_t st) {
  dim3 grid((unsigned)fla_cdiv(BD, 256));
#define U(WW)                                                                                                    \
  if (W == WW) {                                                                                                 \
    hipLaunchKernelGGL((conv_update_kernel<T, WT, WW>), grid, dim3(256), 0, st, (const T*)x, (T*)cache, (const WT*)w, bias, (T*)y, \
                       BD, D, silu);                                                                             \
    FLA_CHECK_LAUNCH();                                                                                          \
    return FLA_OK;                                                                                               \
  }
  U(2) U(3) U(4)
#undef U
  return FLA_E_UNSUPPORTED;
}

}  // namespace

extern "C" int fla_causal_conv1d_fwd(const void* x, const float* weight, const float* bias, void* y, int64_t B, int64_t T,
                                     int64_t D, int64_t W, int silu, int dtype, fla_stream_t stream) {
  FLA_REQUIRE(x && weight && y && B >= 0 && T >= 0 && D > 0, FLA_E_INVALID);
  FLA_REQUIRE(D % 8 == 0 && D < (1 << 30) && W >= 2 && W <= 4, FLA_E_UNSUPPORTED);   // (a row: 32-bit byte offsets)
  FLA_REQUIRE((((uintptr_t)x) | ((uintptr_t)y)) % 16 == 0, FLA_E_ALIGNMENT);
  if (B == 0 || T == 0) return FLA_OK;
  ConvParams p{x, weight, bias, y, nullptr, nullptr, nullptr, nullptr, B, T, (int)D, 0, 0, 0, 0};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == FLA_BF16) return dispatch_conv<bf16>(p, (int)W, silu, false, st);
  if (dtype == FLA_F16) return dispatch_conv<f16>(p, (int)W, silu, false, st);
  if (dtype == FLA_F32) return dispatch_conv<float>(p, (int)W, silu, false, st);
  return FLA_E_UNSUPPORTED;
}

extern "C" int fla_causal_conv1d_bwd_partials(int64_t B, int64_t T) { return (int)conv_bwd_parts(B, T); }

extern "C" int fla_causal_conv1d_bwd(const void* x, const float* weight, const float* bias, const void* dy, void* dx,
                                     float* dw_partial, float* db_partial, int64_t B, int64_t T, int64_t D, int64_t W,
                                     int silu, int dtype, fla_stream_t stream) {
  float* dweight = dw_partial;
  float* dbias = db_partial;
  FLA_REQUIRE(x && weight && dy && dx && dweight && B >= 0 && T >= 0 && D > 0, FLA_E_INVALID);
  FLA_REQUIRE(D % 8 == 0 && D < (1 << 30) && W >= 2 && W <= 4, FLA_E_UNSUPPORTED);   // (a row: 32-bit byte offsets)
  FLA_REQUIRE((((uintptr_t)x) | ((uintptr_t)dy) | ((uintptr_t)dx)) % 16 == 0, FLA_E_ALIGNMENT);
  if (B == 0 || T == 0) return FLA_OK;
  ConvParams p{x, weight, bias, nullptr, dy, dx, dweight, dbias, B, T, (int)D, 0, 0, 0, 0};
  hipStream_t st = (hipStream_t)stream;
  if (dtype == FLA_BF16) return dispatch_conv<bf16>(p, (int)W, silu, true, st);
  if (dtype == FLA_F16) return dispatch_conv<f16>(p, (int)W, silu, true, st);
  if (dtype == FLA_F32) return dispatch_conv<float>(p, (int)W, silu, true, st);
  return FLA_E_UNSUPPORTED;
}

extern "C" int fla_causal_conv1d_update(const void* x, void* cache, const void* weight, const float* bias, void* y,
                                        int64_t B, int64_t D, int64_t W, int silu, int dtype, int weight_dtype,
                                        fla_stream_t stream) {
  FLA_REQUIRE(x && cache && weight && y && B >= 0 && D > 0, FLA_E_INVALID);
  FLA_REQUIRE(W >= 2 && W <= 4, FLA_E_UNSUPPORTED);
  if (B == 0) return FLA_OK;
  hipStream_t st = (hipStream_t)stream;
#define U(E, T, WE, WT) \
  if (dtype == E && weight_dtype == WE) return dispatch_update<T, WT>(x, cache, weight, bias, y, B * D, (int)D, (int)W, silu, st);
  U(FLA_BF16, bf16, FLA_BF16, bf16)
  U(FLA_BF16, bf16, FLA_F32, float)
  U(FLA_F16, f16, FLA_F16, f16)
  U(FLA_F16, f16, FLA_F32, float)
  U(FLA_F32, float, FLA_F32, float)
#undef U
  return FLA_E_UNSUPPORTED;
}
