// Convolutions of stride 1 (forward and backward-data) with few result tiles: one image to serve, a
// small convnet's layers.  The other families give a workgroup 64 result channels and 64 or more positions; with a few
// dozen such tiles most of the chip is idle and a tile's contraction is one long chain.  Here a tile is 32 (or 64)
// channels x 32 positions and the waves of its workgroup share the contraction, 16 channels of one window tap at a time
// ("unit"); their sums meet in LDS in wave order.
//
//   weights   copied to the order in which lanes hold them first (thin_weights_kernel): [unit][32 rows][lane][8], lane
//             (row, half h) holding the 8 channels from 8 h of its row: one contiguous read per unit, and forward and
//             backward-data are one kernel.
//   source    straight from memory: a lane holds one position; a tap is one offset (out of range where the window
//             leaves the plane: reads zero) and the unit's 8 channels are 8 loads at it.
// 16-bit storage multiplies a unit with one 32x32x16 instruction, fp32 with eight 32x32x2 (step e: channels e and 8 + e).
//
// What bounds it is the latency of two or three rounds of loads where there are few tiles, and the loads' issue
// (8 of one element per unit and 32 positions) where there are many.  Measured with the copy of the weights, us (before: the
// tapped GEMM, in 16-bit storage with fp32 arithmetic):
//   3x3, one image      f16  128 x 28 x 28  68 -> 10    256 x 14 x 14  130 -> 16    512 x 7 x 7  264 -> 27
//                       f32  128 x 28 x 28  46 -> 16    256 x 14 x 14   84 -> 25    512 x 7 x 7  162 -> 45
//   5x5, 64 -> 32 over 14 x 14, f32, batch 64, backward-data 63 -> 31
#include <algorithm>

#include "conv2d.h"
#include "conv2d_mfma.h"

namespace flhip {
namespace {

constexpr int THIN_KC = 16;      // channels of a unit
constexpr int THIN_OOB = (int)0x80000000;

struct ThinParams {
  int N, SC, SH, SW, DC, DH, DW;
  int KHW, KW;
  int sh0, sw0, shs, sws;        // source row / column of tap (0, 0) against the result's, step per window row / column
  int P;                         // result positions of all images
  int mt32;                      // blocks of 32 result channels
  int units;
  unsigned src_bytes;
};

template <typename E>
struct ThinOps {                 // 16-bit storage
  struct Src { uint16_t v[8]; };
  typedef uintx4_t Wgt;
  static __device__ __forceinline__ void load(Src& s, __amdgpu_buffer_rsrc_t r, int off, int soff, int step) {
#pragma unroll
    for (int e = 0; e < 8; ++e) s.v[e] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, off, soff + e * step, 0);
  }
  static __device__ __forceinline__ Wgt weights(const E* frag, size_t at) {
    return *reinterpret_cast<const uintx4_t*>(frag + at);
  }
  template <int RT>
  static __device__ __forceinline__ void mma(const Wgt (&w)[RT], const Src& s, floatx16 (&acc)[RT]) {
    uintx4_t b;
#pragma unroll
    for (int e = 0; e < 4; ++e) b[e] = (unsigned)s.v[2 * e] | ((unsigned)s.v[2 * e + 1] << 16);
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[i] = Lo16<E>::mma32(w[i], b, acc[i]);
  }
};
template <>
struct ThinOps<float> {
  struct Src { float v[8]; };
  struct Wgt { float v[8]; };
  static __device__ __forceinline__ void load(Src& s, __amdgpu_buffer_rsrc_t r, int off, int soff, int step) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      s.v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, off, soff + e * step, 0));
  }
  static __device__ __forceinline__ Wgt weights(const float* frag, size_t at) {
    Wgt w;
    const float4 a = *reinterpret_cast<const float4*>(frag + at), b = *reinterpret_cast<const float4*>(frag + at + 4);
    w.v[0] = a.x; w.v[1] = a.y; w.v[2] = a.z; w.v[3] = a.w;
    w.v[4] = b.x; w.v[5] = b.y; w.v[6] = b.z; w.v[7] = b.w;
    return w;
  }
  template <int RT>
  static __device__ __forceinline__ void mma(const Wgt (&w)[RT], const Src& s, floatx16 (&acc)[RT]) {
#pragma unroll
    for (int e = 0; e < 8; ++e)
#pragma unroll
      for (int i = 0; i < RT; ++i) acc[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[i].v[e], s.v[e], acc[i], 0, 0, 0);
  }
};

// grid (position tiles, channel tiles), W waves; RT blocks of 32 result channels per workgroup
template <typename E, int RT, int W>
__global__ void __launch_bounds__(W * 64)
thin_conv_kernel(ThinParams p, const E* __restrict__ src, const E* __restrict__ frag, const float* __restrict__ bias,
                 E* __restrict__ dst) {
  typedef ThinOps<E> Ops;
  constexpr int ES = (int)sizeof(E);
  constexpr int U = ES == 2 ? (RT == 1 ? 5 : 4) : 2;       // units whose loads are in flight together
  __shared__ float red[W * RT * 1024];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int plane = p.SH * p.SW, dplane = p.DH * p.DW;
  const int pos = blockIdx.x * 32 + fr;
  const int n = pos / dplane, in = pos - n * dplane, oh = in / p.DW, ow = in - oh * p.DW;
  const int ih0 = oh + p.sh0, iw0 = ow + p.sw0;
  const int base = (n * p.SC + 8 * h) * plane;
  const bool inside = pos < p.P;
  const int u0 = wave * p.units / W, u1 = (wave + 1) * p.units / W;
  const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(src, p.src_bytes);
  const E* wgt = frag + (size_t)blockIdx.y * RT * 512 + lane * 8;
  const size_t wstep = (size_t)p.mt32 * 512;
  const int cstep = plane * ES;

  floatx16 acc[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[i][r] = 0.f;

  // the unit's place: channels 16 c .., window tap t = (kh, kw)
  int c = u0 / p.KHW, t = u0 - c * p.KHW, kh = t / p.KW, kw = t - kh * p.KW;
  auto fetch = [&](int u, typename Ops::Src& s, typename Ops::Wgt (&w)[RT]) __attribute__((always_inline)) {
    const int ih = ih0 + kh * p.shs, iw = iw0 + kw * p.sws;
    const bool ok = inside && (unsigned)ih < (unsigned)p.SH && (unsigned)iw < (unsigned)p.SW && c * THIN_KC + 8 * h < p.SC;
    Ops::load(s, rsrc, ok ? (base + ih * p.SW + iw) * ES : THIN_OOB, c * THIN_KC * cstep, cstep);
#pragma unroll
    for (int i = 0; i < RT; ++i) w[i] = Ops::weights(wgt, (size_t)u * wstep + i * 512);
    if (++kw == p.KW) {
      kw = 0;
      ++kh;
    }
    if (++t == p.KHW) {
      t = kh = kw = 0;
      ++c;
    }
  };
  int u = u0;
  for (; u + U <= u1; u += U) {
    typename Ops::Src s[U];
    typename Ops::Wgt w[U][RT];
#pragma unroll
    for (int j = 0; j < U; ++j) fetch(u + j, s[j], w[j]);
#pragma unroll
    for (int j = 0; j < U; ++j) Ops::template mma<RT>(w[j], s[j], acc);
  }
  for (; u < u1; ++u) {
    typename Ops::Src s;
    typename Ops::Wgt w[RT];
    fetch(u, s, w);
    Ops::template mma<RT>(w, s, acc);
  }

  // element r of a lane: row 8 (r / 4) + 4 h + r % 4, column fr
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) red[(wave * RT + i) * 1024 + (8 * (r >> 2) + 4 * h + (r & 3)) * 32 + fr] = acc[i][r];
  __syncthreads();
  if (!inside) return;                       // (lane, and so position, is the same for all of a thread's results)
  const size_t out = (size_t)n * p.DC * dplane + in;
  for (int i = tid; i < RT * 1024; i += W * 64) {
    const int m = blockIdx.y * RT * 32 + (i >> 5);
    if (m >= p.DC) break;
    float v = red[i];
#pragma unroll
    for (int k = 1; k < W; ++k) v += red[k * RT * 1024 + i];
    if (bias) v += bias[m];
    st(dst, out + (size_t)m * dplane, v);
  }
}

// w [K][C][KHW] -> [unit][block of 32 rows][lane][8]; rows are the result channels (BWD: the input channels).  Rows
// and channels past the end are zeros.  A workgroup copies 32 rows x 16 channels x up to 16 taps through LDS: both sides
// of the copy are runs of neighbours (512 x 512 x 3 x 3 in 16-bit storage, with the convolution of one 7 x 7 image: 31 -> 27 us
// against a thread per eight values that reads memory itself; 128 x 128: 9 -> 10).  grid (block of rows, 16 channels, 16 taps)
constexpr int THIN_TAPS = 16;
template <typename E, bool BWD>
__global__ void __launch_bounds__(1024) thin_weights_kernel(const E* __restrict__ w, E* __restrict__ frag, int SC, int DC, int KHW, int mt32) {
  constexpr int THREADS = 1024, NL = 512 * THIN_TAPS / THREADS;
  __shared__ E part[512 * (THIN_TAPS + 1)];
  const int m0 = blockIdx.x * 32, c0 = blockIdx.y * THIN_KC, t0 = blockIdx.z * THIN_TAPS, nt = min(THIN_TAPS, KHW - t0);
  const float inv = 1.0f / (float)nt;
  E v[NL];                                   // all loads in flight together
  int at[NL];
#pragma unroll
  for (int j = 0; j < NL; ++j) {
    int t;
    const int i = threadIdx.x + j * THREADS, pair = fast_div(i, nt, inv, &t);
    const int m = m0 + (BWD ? pair & 31 : pair >> 4), c = c0 + (BWD ? pair >> 5 : pair & 15);
    // (row, channel) pair -> its taps in LDS, so that the rows a wave reads below lie in different banks
    at[j] = i < 512 * nt ? (BWD ? pair * (nt | 1) : pair * nt + (pair >> 4)) + t : -1;
    v[j] = E{};
    if (at[j] >= 0 && m < DC && c < SC) v[j] = w[(size_t)(BWD ? c * DC + m : m * SC + c) * KHW + t0 + t];
  }
#pragma unroll
  for (int j = 0; j < NL; ++j)
    if (at[j] >= 0) part[at[j]] = v[j];
  __syncthreads();
  for (int i = threadIdx.x; i < 64 * nt; i += THREADS) {      // (at most one each)
    const int t = i >> 6, lane = i & 63, row = lane & 31, h = lane >> 5;
    __align__(16) E u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) u[e] = part[(BWD ? ((8 * h + e) * 32 + row) * (nt | 1) : (row * 16 + 8 * h + e) * nt + row) + t];
    uint4* out = reinterpret_cast<uint4*>(frag + ((((size_t)blockIdx.y * KHW + t0 + t) * mt32 + blockIdx.x) * 64 + lane) * 8);
    const uint4* from = reinterpret_cast<const uint4*>(u);
    out[0] = from[0];
    if (sizeof(E) == 4) out[1] = from[1];
  }
}

bool thin_geom(const ConvGeom& g, int dtype, bool bwd, ThinParams* p) {
  if (g.groups != 1 || g.sy != 1 || g.sx != 1) return false;
  p->N = g.N;
  p->KHW = g.KH * g.KW; p->KW = g.KW;
  if (!bwd) {
    p->SC = g.C; p->SH = g.H; p->SW = g.W; p->DC = g.K; p->DH = g.OH; p->DW = g.OW;
    p->sh0 = -g.py; p->sw0 = -g.px; p->shs = g.dly; p->sws = g.dlx;
  } else {
    p->SC = g.K; p->SH = g.OH; p->SW = g.OW; p->DC = g.C; p->DH = g.H; p->DW = g.W;
    p->sh0 = g.py; p->sw0 = g.px; p->shs = -g.dly; p->sws = -g.dlx;
  }
  if (p->SC % 8 != 0 || p->KHW > 65535) return false;      // a lane's 8 channels are all there or none
  const long long sbytes = (long long)g.N * p->SC * p->SH * p->SW * (long long)dtype_size(dtype);
  const long long pos = (long long)g.N * p->DH * p->DW;
  const long long units = (long long)(p->SC + THIN_KC - 1) / THIN_KC * p->KHW;
  p->mt32 = (p->DC + 31) / 32;
  if (sbytes >= (1ll << 31) || pos >= (1ll << 31) - 32 || units >= (1ll << 26) || p->mt32 > 65535 ||
      units * p->mt32 >= (1ll << 20) || (p->SC + THIN_KC - 1) / THIN_KC > 65535)
    return false;
  p->src_bytes = (unsigned)sbytes;
  p->P = (int)pos;
  p->units = (int)units;
  return true;
}

size_t thin_weight_bytes(const ThinParams& p, int dtype) { return (size_t)p.units * p.mt32 * 512 * dtype_size(dtype); }

template <typename E, int RT, int W>
int thin_go(const ThinParams& p, const E* src, const E* frag, const float* bias, E* dst, hipStream_t s) {
  hipLaunchKernelGGL((thin_conv_kernel<E, RT, W>), dim3((unsigned)((p.P + 31) / 32), (unsigned)((p.mt32 + RT - 1) / RT)), dim3(W * 64),
                     0, s, p, src, frag, bias, dst);
  return check_launch("conv2d (few tiles)");
}

int thin_conv(const ConvGeom& g, int dtype, bool bwd, const void* src, const void* w, const float* bias, void* dst, void* ws,
              size_t ws_bytes, hipStream_t s) {
  ThinParams p{};
  if (!thin_geom(g, dtype, bwd, &p)) return -1;
  if (!ws || ws_bytes < thin_weight_bytes(p, dtype) || reinterpret_cast<uintptr_t>(ws) % 16 != 0) return -1;
  const dim3 wgrid((unsigned)p.mt32, (unsigned)((p.SC + THIN_KC - 1) / THIN_KC), (unsigned)((p.KHW + THIN_TAPS - 1) / THIN_TAPS));
  // Two blocks of channels per workgroup halve the source's loads; one makes twice the workgroups
  const long long tiles = (long long)((p.P + 31) / 32) * p.mt32;
  const bool two = p.mt32 % 2 == 0 && tiles / 2 >= 2 * mfma_num_cus();
  const long long wgs = two ? tiles / 2 : tiles;
  // waves that share a tile: about twelve waves for each compute unit
  const int waves = wgs * 4 >= 12 * mfma_num_cus() ? 4 : wgs * 8 >= 12 * mfma_num_cus() || two ? 8 : 16;
  return by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    T* frag = static_cast<T*>(ws);
    const T *x = static_cast<const T*>(src), *wt = static_cast<const T*>(w);
    T* y = static_cast<T*>(dst);
    if (bwd) hipLaunchKernelGGL((thin_weights_kernel<T, true>), wgrid, dim3(1024), 0, s, wt, frag, p.SC, p.DC, p.KHW, p.mt32);
    else hipLaunchKernelGGL((thin_weights_kernel<T, false>), wgrid, dim3(1024), 0, s, wt, frag, p.SC, p.DC, p.KHW, p.mt32);
    if (two) return waves == 4 ? thin_go<T, 2, 4>(p, x, frag, bias, y, s) : thin_go<T, 2, 8>(p, x, frag, bias, y, s);
    return waves == 4 ? thin_go<T, 1, 4>(p, x, frag, bias, y, s)
         : waves == 8 ? thin_go<T, 1, 8>(p, x, frag, bias, y, s) : thin_go<T, 1, 16>(p, x, frag, bias, y, s);
  });
}

}  // namespace

size_t mfma_thin_ws(const ConvGeom& g, int dtype, bool bwd) {
  ThinParams p{};
  return thin_geom(g, dtype, bwd, &p) ? thin_weight_bytes(p, dtype) : 0;
}
int mfma_thin_conv_fwd(const ConvGeom& g, int dtype, const void* x, const void* w, const float* bias, void* y, hipStream_t s, void* ws,
                       size_t ws_bytes) {
  return thin_conv(g, dtype, false, x, w, bias, y, ws, ws_bytes, s);
}
int mfma_thin_conv_bwd_data(const ConvGeom& g, int dtype, const void* dy, const void* w, void* dx, hipStream_t s, void* ws,
                            size_t ws_bytes) {
  return thin_conv(g, dtype, true, dy, w, nullptr, dx, ws, ws_bytes, s);
}

}  // namespace flhip
