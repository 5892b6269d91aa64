// Filter gradient of 3x3 windows of stride 1 and padding 1 in fp32, on the bf16 matrix cores in three parts (split_f32.h):
//   dw[k][c][kh][kw] = sum over images, rows and columns of dy[k][h][w] x[c][h + kh - 1][w + kw - 1]
// The contraction runs over positions, which are contiguous in both operands: a fragment is 8 consecutive positions of a row.
//
// The batch is one sequence of rows, H of an image and one of zeros behind them, so that what lies above and below an image needs no
// question.  A workgroup (12 waves) owns 64 filters x 64 channels x nine taps over a run of rows, a wave 32 x 32 of them for
// one kh: three taps with two accumulators each, 96 registers, three waves to a SIMD.  A stage is R rows (1, 2 or 4 by the
// length of a row).  Its rows of dy and the rows of x that it needs first are loaded as they lie in memory while the stage before
// multiplies, taken apart in registers and written to LDS [row][part][channel][positions]; rows of x stay for the three
// stages that read them.  The shifted fragments of kw = 0 and 2 are made from the aligned one and the words beside it.
//
// What bounds it is the bf16 matrix pipe (18 instructions per wave and 16 positions, 21 LDS reads and 60 vector instructions beside them).
// The partial tiles go to the workspace as [slice][tile][tap][64][64] and are added in a fixed order: that of the slices up to eight of them, else
// interleaved runs of slices, and those in pairs.
// Measured, us, both launches (before: wgrad_slab_kernel on v_mfma_f32_16x16x4_f32): 64 channels over 56 x 56, 32 / 64 images 71 / 131 -> 61 / 100, 128 over
// 28 x 28 81 / 147 -> 61 / 99, 256 over 14 x 14 97 / 177 -> 56 / 95, 512 over 7 x 7 108 / 208 -> 59 / 103.  Its products and LDS reads alone, 64
// channels over 56 x 56, take 31 us per 32 images, all of it 37: with every wave bringing in rows behind the last product of a stage it was 47.
#include <algorithm>

#include "conv2d.h"
#include "split_f32.h"

namespace flhip {
namespace {

constexpr int W3_T = 64;                       // tile side
constexpr int W3_THREADS = 768;
constexpr int W3_OOB = (int)0x80000000;

struct W3Params {
  int C, H, W, K;
  int V, G;                    // rows of the sequence, cells of 8 positions per row
  int XU, DU;                  // cells from one channel's row to the next in LDS
  int nstages, sps;            // stages, stages per slice
  int ctiles, tiles;
  unsigned x_bytes, dy_bytes;
};

// rows of x in LDS are written R at a time, in BATCHES sets in turn
constexpr int w3_batches(int R) { return R == 1 ? 4 : 3; }
constexpr int odd_cells(int n) { return n | 1; }          // (an odd number of cells: 16 rows of a read cover the banks)

template <int R>
__global__ void __launch_bounds__(W3_THREADS, 1)
wgrad3_split_kernel(W3Params p, const float* __restrict__ x, const float* __restrict__ dy, float* __restrict__ part) {
  constexpr int RING = w3_batches(R) * R;                 // rows of x
  extern __shared__ __align__(16) char w3_lds[];
  const int xrow = 3 * W3_T * p.XU * 16, drow = 3 * W3_T * p.DU * 16, xpart = W3_T * p.XU * 16, dpart = W3_T * p.DU * 16;
  char* const xs = w3_lds;
  char* const ds = w3_lds + RING * xrow;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), fb = wave & 1, cb = wave >> 1 & 1, kh = wave >> 2;
  const int slice = blockIdx.x / p.tiles, tile = blockIdx.x - slice * p.tiles, kt = tile / p.ctiles, ct = tile - kt * p.ctiles;
  const int s0 = slice * p.sps, send = min(p.nstages, s0 + p.sps);
  const int HR = p.H + 1, cells = R * p.G;
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(x, p.x_bytes), dr = make_rsrc(dy, p.dy_bytes);

  // ---- load roles: a unit is 8 positions of a channel's row; the first cells * 64 units of a stage are x, the others dy.  At most
  // two to a thread; which row a unit is of is the same for a wave
  const int per = cells * W3_T;
  int off[2], at[2], left[2];                  // bytes within a row of its image, within the stage's (batch's) rows in LDS; positions that exist
  int isdy[2], r[2], img[2];                   // the wave's next row: of dy?  where in the sequence
  bool any[2];
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const int u = tid + k * W3_THREADS, u0 = wave * 64 + k * W3_THREADS;
    isdy[k] = u0 >= per;
    any[k] = u0 < 2 * per;
    const int row = (u0 - (isdy[k] ? per : 0)) / (W3_T * p.G), e = u - (isdy[k] ? per : 0) - row * (W3_T * p.G), ch = e / p.G, g = e - ch * p.G;
    const int channel = ch + (isdy[k] ? kt : ct) * W3_T;
    off[k] = channel < (isdy[k] ? p.K : p.C) ? (channel * p.H * p.W + 8 * g) * 4 : W3_OOB;
    at[k] = isdy[k] ? row * drow + ch * p.DU * 16 + g * 16 : row * xrow + ch * p.XU * 16 + 16 + g * 16;
    left[k] = min(8, p.W - 8 * g);
    const int v = s0 * R + row - (isdy[k] ? 0 : 1);       // (the row before the first: the zeros behind an image)
    img[k] = v < 0 ? -1 : v / HR;
    r[k] = v < 0 ? p.H : v - img[k] * HR;
  }
  const int images = p.V / HR;
  // the unit's next row: loads it (zeros where there is none), and goes on to the one R further
  auto load = [&](int k, uintx4_t (&raw)[2]) __attribute__((always_inline)) {
    const bool in = any[k] && r[k] < p.H && (unsigned)img[k] < (unsigned)images;
    const int row = in ? (img[k] * (isdy[k] ? p.K : p.C) * p.H + r[k]) * p.W * 4 : 0, o = in ? off[k] : W3_OOB;
    const __amdgpu_buffer_rsrc_t rs = isdy[k] ? dr : xr;
    raw[0] = __builtin_amdgcn_raw_buffer_load_b128(rs, o, row, 0);
    raw[1] = __builtin_amdgcn_raw_buffer_load_b128(rs, o + 16, row, 0);
    r[k] += R;
    while (r[k] >= HR) {
      r[k] -= HR;
      ++img[k];
    }
  };
  // takes it apart and writes it to the rows at `to`
  auto store = [&](int k, const uintx4_t (&raw)[2], char* to) __attribute__((always_inline)) {
    if (!any[k]) return;
    float v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = e < left[k] ? __uint_as_float(raw[e >> 2][e & 3]) : 0.f;
    uintx4_t h, m, l;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const Split2 s = split2(v[2 * e], v[2 * e + 1]);
      h[e] = s.h; m[e] = s.m; l[e] = s.l;
    }
    const int step = isdy[k] ? dpart : xpart;
    char* const o = to + at[k];
    *reinterpret_cast<uintx4_t*>(o) = h;
    *reinterpret_cast<uintx4_t*>(o + step) = m;
    *reinterpret_cast<uintx4_t*>(o + 2 * step) = l;
  };
  // rows of x from ring row `slot`, rows of dy of a stage
  auto place = [&](int k, int slot, int half) __attribute__((always_inline)) -> char* { return isdy[k] ? ds + half * R * drow : xs + slot * xrow; };
  // The batches of x that the first stage reads, and its dy with the first of them; while they are on their way zeros everywhere
  // (nothing is written beside a row's cells later).  The loads of the second stage's stay in flight.
  constexpr int AHEAD = w3_batches(R) - 1;
  uintx4_t raw[2][2];
  {
    uintx4_t first[AHEAD][2][2];
#pragma unroll
    for (int b = 0; b < AHEAD; ++b)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (b == 0 || !isdy[k]) load(k, first[b][k]);
    for (int i = tid; i < (RING * xrow + 2 * R * drow) / 16; i += W3_THREADS) reinterpret_cast<uintx4_t*>(w3_lds)[i] = uintx4_t{0u, 0u, 0u, 0u};
    __syncthreads();
#pragma unroll
    for (int b = 0; b < AHEAD; ++b)
#pragma unroll
      for (int k = 0; k < 2; ++k)
        if (b == 0 || !isdy[k]) store(k, first[b][k], place(k, b * R, 0));
#pragma unroll
    for (int k = 0; k < 2; ++k) load(k, raw[k]);
  }
  __syncthreads();

  floatx16 big[3], small[3];
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) big[t][r] = small[t][r] = 0.f;
  const char* const alane = ds + (fb * 32 + fr) * p.DU * 16;
  const char* const blane = xs + (cb * 32 + fr) * p.XU * 16 + 16;
  const int steps = (cells + 1) / 2, store_at = min(kh, steps - 1);
  int base = 0;                                // ring row of the row before the stage's first
  for (int s = s0; s < send; ++s) {
    const int half = (s - s0) & 1;
    int slot = base + AHEAD * R;
    if (slot >= RING) slot -= RING;
    int i = 0, g = fg;                         // row of the stage and cell of this half wave
    if (p.G == 1) {
      i = fg;
      g = 0;
    }
#pragma unroll 1
    for (int st = 0; st < steps; ++st) {
      const int c = 2 * st + fg;
      const bool live = c < cells;             // (an odd number of cells: the last step has one)
      const int ii = live ? i : 0, gg = live ? g : 0;
      int rr = base + ii + kh;
      if (rr >= RING) rr -= RING;
      const char* const ap = alane + (half * R + ii) * drow + gg * 16;
      const char* const bp = blane + rr * xrow + gg * 16;
      uintx4_t a[3], b[3], t[3];
      uint32_t before[3], after[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        a[q] = *reinterpret_cast<const uintx4_t*>(ap + q * dpart);
        b[q] = *reinterpret_cast<const uintx4_t*>(bp + q * xpart);
        before[q] = *reinterpret_cast<const uint32_t*>(bp + q * xpart - 4);
        after[q] = *reinterpret_cast<const uint32_t*>(bp + q * xpart + 16);
      }
      if (!live) {
#pragma unroll
        for (int q = 0; q < 3; ++q) a[q] = uintx4_t{0u, 0u, 0u, 0u};
      }
      // (one shifted fragment at a time: with both of them made first they and the loads in flight did not fit the registers)
      split_mma(big[1], small[1], a, b);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        t[q] = uintx4_t{__builtin_amdgcn_alignbit(b[q].x, before[q], 16), __builtin_amdgcn_alignbit(b[q].y, b[q].x, 16),
                        __builtin_amdgcn_alignbit(b[q].z, b[q].y, 16), __builtin_amdgcn_alignbit(b[q].w, b[q].z, 16)};
      split_mma(big[0], small[0], a, t);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 0; q < 3; ++q)
        t[q] = uintx4_t{__builtin_amdgcn_alignbit(b[q].y, b[q].x, 16), __builtin_amdgcn_alignbit(b[q].z, b[q].y, 16),
                        __builtin_amdgcn_alignbit(b[q].w, b[q].z, 16), __builtin_amdgcn_alignbit(after[q], b[q].w, 16)};
      split_mma(big[2], small[2], a, t);
      // The next stage's dy and the batch of x that it reads last, and the loads of those of the stage behind it: the waves of a SIMD
      // (one of each kh) do so behind different steps, so that the others' products go on.
      if (st == store_at) {
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          store(k, raw[k], place(k, slot, half ^ 1));
          load(k, raw[k]);
        }
      }
      if (p.G == 1) {
        i += 2;
      } else {
        g += 2;
        if (g >= p.G) {
          g -= p.G;
          ++i;
        }
      }
    }
    base += R;
    if (base >= RING) base -= RING;
    __syncthreads();
  }

  bool bad = false;
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      big[t][r] += small[t][r];
      bad |= split_redo(big[t][r]);
    }
  // Once more with the operands as they are, loaded element by element.  Both launches, us, plain / one infinity in every tile of one image / of every image / all
  // results below 2^-90: 256 channels over 14 x 14, 64 images 109 / 419 / 439 / 455, 64 over 56 x 56, 32 images 66 / 335 / 334 / 344, 512 over 7 x 7, 64 images
  // 104 / 355 / 358 / 357.
  if (__builtin_amdgcn_ballot_w64(bad)) {
    const int k = kt * W3_T + fb * 32 + fr, c = ct * W3_T + cb * 32 + fr;
#pragma unroll
    for (int t = 0; t < 3; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) big[t][r] = 0.f;
#pragma unroll 1
    for (int v = s0 * R; v < min(p.V, send * R); ++v) {
      const int img = v / HR, r = v - img * HR, sr = r + kh - 1;
      if (r == p.H) continue;
#pragma unroll 1
      for (int o = fg; o < p.W + fg; o += 2) {
        const bool in = o < p.W;
        const float a = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(dr, in && k < p.K ? (((img * p.K + k) * p.H + r) * p.W + o) * 4 : W3_OOB, 0, 0));
#pragma unroll
        for (int t = 0; t < 3; ++t) {
          const int col = o + t - 1;
          const bool there = in && c < p.C && (unsigned)sr < (unsigned)p.H && (unsigned)col < (unsigned)p.W;
          const float b = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xr, there ? (((img * p.C + c) * p.H + sr) * p.W + col) * 4 : W3_OOB, 0, 0));
          big[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, big[t], 0, 0, 0);
        }
      }
    }
  }

  // element r of a block: filter 8 (r / 4) + 4 fg + r % 4, channel fr
  float* const out = part + ((size_t)(slice * p.tiles + tile) * 9 + 3 * kh) * (W3_T * W3_T) + (fb * 32 + 4 * fg) * W3_T + cb * 32 + fr;
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) out[t * (W3_T * W3_T) + (8 * (r >> 2) + (r & 3)) * W3_T] = big[t][r];
}

// dw from the partial tiles: a workgroup owns CW channels of ROWS filters, a wave one tap of them, in RUNS runs of slices that are
// added at the end: <64, 1> for few slices, <64, 4>, and <16, 16> for many slices of few filters
template <int CW, int RUNS>
__global__ void __launch_bounds__(576)
wgrad3_sum_kernel(const float* __restrict__ part, float* __restrict__ dw, int slices, int tiles, int ctiles, int K, int C) {
  constexpr int LC = CW / 4, ROWS = 64 / (LC * RUNS);
  __shared__ float out[ROWS][CW * 9];
  const int lane = threadIdx.x & 63, tap = threadIdx.x >> 6, c4 = lane % LC, run = lane / LC % RUNS, kr = lane / (LC * RUNS);
  const int piece = blockIdx.x % (W3_T / CW), rows = blockIdx.x / (W3_T / CW), tile = rows / (W3_T / ROWS), kl = (rows - tile * (W3_T / ROWS)) * ROWS;
  const int kt = tile / ctiles, ct = tile - kt * ctiles, k = kt * W3_T + kl, c0 = ct * W3_T + piece * CW;
  if (k >= K || c0 >= C) return;               // (the whole workgroup)
  const float4* const src = reinterpret_cast<const float4*>(part + ((size_t)tile * 9 + tap) * (W3_T * W3_T) + (kl + kr) * W3_T + piece * CW) + c4;
  const size_t stride = (size_t)tiles * 9 * (W3_T * W3_T) / 4;
  float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s = run; s < slices; s += 8 * RUNS) {
    float4 v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = s + j * RUNS < slices ? src[(size_t)(s + j * RUNS) * stride] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sum.x += v[j].x; sum.y += v[j].y; sum.z += v[j].z; sum.w += v[j].w;
    }
  }
#pragma unroll
  for (int o = LC; o < LC * RUNS; o *= 2) {
    sum.x += __shfl_xor(sum.x, o, 64); sum.y += __shfl_xor(sum.y, o, 64);
    sum.z += __shfl_xor(sum.z, o, 64); sum.w += __shfl_xor(sum.w, o, 64);
  }
  if (run == 0) {
    float* const o = out[kr] + 4 * c4 * 9 + tap;
    o[0] = sum.x; o[9] = sum.y; o[18] = sum.z; o[27] = sum.w;
  }
  __syncthreads();
  const int n = min(CW, C - c0) * 9;
  for (int row = 0; row < ROWS && k + row < K; ++row)
    if ((int)threadIdx.x < n) dw[((size_t)(k + row) * C + c0) * 9 + threadIdx.x] = out[row][threadIdx.x];
}

int w3_rows(int G) { return G == 1 ? 4 : G <= 3 ? 2 : 1; }
size_t w3_lds_bytes(const W3Params& p, int R) { return (size_t)16 * 3 * W3_T * (w3_batches(R) * R * p.XU + 2 * R * p.DU); }

bool wgrad3_plan(const ConvGeom& g, W3Params* p, int* R, int* slices) {
  if (!(g.KH == 3 && g.KW == 3 && g.sy == 1 && g.sx == 1 && g.py == 1 && g.px == 1 && g.dly == 1 && g.dlx == 1 && g.groups == 1)) return false;
  if (g.H < 4 || g.W < 4 || g.W > 56 || g.C < 32 || g.K < 32) return false;      // (rows of eight cells, with their pitches of 11 and 9, need 186 KB of LDS)
  const long long xb = (long long)g.N * g.C * g.H * g.W * 4, db = (long long)g.N * g.K * g.H * g.W * 4;
  if (xb >= (1ll << 31) || db >= (1ll << 31)) return false;
  p->C = g.C; p->H = g.H; p->W = g.W; p->K = g.K;
  p->G = (g.W + 7) / 8;
  *R = w3_rows(p->G);
  if (2 * *R * p->G * W3_T > 2 * W3_THREADS) return false;
  p->XU = odd_cells(p->G + 2); p->DU = odd_cells(p->G);
  if (w3_lds_bytes(*p, *R) > 156 * 1024) return false;
  if ((long long)g.N * (g.H + 1) > 0x3fffffff) return false;
  p->V = g.N * (g.H + 1);
  p->nstages = (p->V + *R - 1) / *R;
  p->ctiles = (g.C + W3_T - 1) / W3_T;
  p->tiles = p->ctiles * ((g.K + W3_T - 1) / W3_T);
  p->x_bytes = (unsigned)xb; p->dy_bytes = (unsigned)db;
  // a workgroup fills a compute unit; every slice writes and re-reads the whole gradient, and wants three stages at least
  const int cus = mfma_num_cus();
  int n = std::max(1, std::min(cus / std::max(1, std::min(p->tiles, cus)), p->nstages / 3));
  p->sps = (p->nstages + n - 1) / n;
  *slices = (p->nstages + p->sps - 1) / p->sps;
  return (long long)*slices * p->tiles <= 0x7fffffff;
}

// From 1.1 billion multiply-adds on: below, what a workgroup pays before its first product (three rows on their way, 150 KB of LDS
// cleared) and the partial tiles cost as much as the products save.  us, wgrad_slab_kernel / here: 64 channels over 56 x 56, 6 / 9 / 12 / 16 / 32
// images (0.7 to 3.7 billion) 31 / 33, 32 / 34, 39 / 39, 43 / 43, 71 / 61; 128 over 28 x 28, 4 / 9 / 16 38 / 27, 38 / 34, 51 / 42; 256 over 12 x 12, 4 / 9 26 /
// 27, 36 / 34; 512 over 7 x 7, 4 / 6 / 9 25 / 30, 31 / 33, 38 / 36.  Not where less than 5 / 8 of the tiles' products exist.
bool wgrad3_pays(const ConvGeom& g, const W3Params& p) {
  const double macs = 9.0 * g.N * g.H * g.W * g.C * g.K, all = 9.0 * p.V * 8 * p.G * p.tiles * W3_T * W3_T;
  return macs >= 1.1e9 && all <= 1.6 * macs;
}

}  // namespace

size_t mfma_wgrad3_split_ws(const ConvGeom& g) {
  W3Params p{};
  int R, slices;
  if (!wgrad3_plan(g, &p, &R, &slices) || !wgrad3_pays(g, p)) return 0;
  return (size_t)slices * p.tiles * 9 * W3_T * W3_T * sizeof(float);
}

int mfma_wgrad3_split(const ConvGeom& g, const float* x, const float* dy, float* dw, void* ws, size_t ws_bytes, hipStream_t s) {
  W3Params p{};
  int R, slices;
  if (!dw || !wgrad3_plan(g, &p, &R, &slices) || !wgrad3_pays(g, p)) return -1;
  if (!ws || ws_bytes < (size_t)slices * p.tiles * 9 * W3_T * W3_T * sizeof(float) || reinterpret_cast<uintptr_t>(ws) % 16 != 0) return -1;
  float* const part = static_cast<float*>(ws);
  const size_t lds = w3_lds_bytes(p, R);
  auto go = [&](auto kernel) {
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(slices * p.tiles)), dim3(W3_THREADS), lds, s, p, x, dy, part);
    return check_launch("conv2d_bwd_filter (3x3, fp32 in three parts)");
  };
  const int rc = R == 1 ? go(wgrad3_split_kernel<1>) : R == 2 ? go(wgrad3_split_kernel<2>) : go(wgrad3_split_kernel<4>);
  if (rc) return rc;
  auto sum = [&](auto kernel, int cw, int runs) {
    const int rows = 64 / (cw / 4 * runs);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.tiles * (W3_T / rows) * (W3_T / cw))), dim3(576), 0, s, part, dw, slices, p.tiles, p.ctiles, g.K, g.C);
  };
  if (slices <= 8) sum(wgrad3_sum_kernel<64, 1>, 64, 1);
  else if (slices <= 32) sum(wgrad3_sum_kernel<64, 4>, 64, 4);
  else sum(wgrad3_sum_kernel<16, 16>, 16, 16);
  return check_launch("conv2d_bwd_filter (3x3, sum)");
}

}  // namespace flhip
