// Windows of one row, and windows of stride 1 over planes stacked in one sequence (conv2d_mfma_tap1d.hip has both in 16-bit
// storage, the latter for 3 x 3), in fp32: operands in three bf16 parts (split_f32.h), forward and backward-data.
//
// Operands: the source as it lies in memory (PLANES), or the channels-last rows xr[sequence][position][Cs] that the forward pass of
// one-row windows leaves to their filter gradient; and the weights already taken apart, wf[block of 32 result channels][phase][chunk of 16 channels][tap][part][lane][8 channels]: the fragments in the
// order in which a wave walks them.
//
// A workgroup of 4 waves (WM along the result channels x 4 / WM along the positions) owns 32 WM channels x 32 NB (4 / WM)
// positions of one phase; a wave NB blocks of 32 x 32 with two accumulators each.  The contraction runs chunk by chunk of 16
// channels, and within a chunk over the taps:
//   * the source rows that the tile needs (its positions and the window's reach) are loaded a chunk ahead into registers (a thread
//     one or two rows of 16 channels; neighbouring lanes are neighbouring positions), taken apart once per chunk - not per tap - and written to one of two LDS buffers, a row
//     6 cells of 16 bytes ([part][half of the channels]) and 1 unused, which keeps the lanes of a pass on distinct banks;
//   * a tap shifts whole rows: a step (chunk, tap) reads 3 NB fragments and issues 6 NB products;
//   * a wave's weights go straight to registers, as many steps ahead as its registers allow (WR); the steps of all chunks are one
//     sequence.
// One barrier per chunk; two workgroups share a compute unit, and the one multiplies while the other waits.
// Channels are the rows of the instruction's tile, positions its columns: the lanes of a store are neighbouring positions.
//
// What bounds it is the bf16 matrix pipe in large layers, a workgroup's chain of steps in small ones (a step of one block 0.19 us:
// its fragments are read a step ahead, which took a third off).  Measured with the operand passes, us (before: v_mfma_f32_32x32x2_f32
// on channels-last rows, or the slab kernels), error in the 2-norm against 64 bits 4.6e-7 (before 1.3e-6) at 250 channels and 21 taps:
//   21 taps, 250 -> 250 channels, 16 x 1500 frames, forward 476 -> 294 (214 TFLOP/s), backward-data 473 -> 278; 2 x 300 frames 244 -> 68
//   3 x 3, 64 images: 64 channels over 56 x 56 131 -> 84, 256 over 14 x 14 140 -> 89, 512 over 7 x 7 234 -> 111
#include <algorithm>

#include "conv2d.h"
#include "gemm_f32.h"
#include "split_f32.h"

namespace flhip {
namespace {

constexpr int TS_CC = 16;         // channels per chunk
constexpr int TS_ROW = 112;       // bytes of a slab row
constexpr int TS_OOB = (int)0x80000000;

struct TapSplit {
  int rows, H;                    // sequences (images x rows), rows per image
  int TS, TOu, TO;                // source positions; result positions per sequence and of them per phase
  int Cs, nchunk, Mo;             // Cs: channels of the rows
  int cstride;                    // bytes from a channel to the next (planes: of the source; rows: 4)
  int SS, SR, half;               // source stride; slab rows; stride 2: row of the first odd source offset
  int nph, smin[2], ntap[2], tap0[2];      // per phase: first source position for result 0, taps, index of its first tap
  int tw, tpitch;                 // taps per window row, slab rows from one to the next
  int ptiles, mtiles, taps_total;
  unsigned src_bytes, w_bytes, dst_bytes;
  int pW, pH, pN, pY;             // stacked planes: their geometry (pW = 0: one-row windows), zero rows between two
  int Cc, Cw, KW, bwd;            // the weight tensor
  signed char tapj[64];           // weight tap of a tap
};

// weights as they lie in memory to their parts: one wave per (block, phase, chunk, tap); the tap is the index that changes
// fastest over the waves of a workgroup, so that they read the same cache lines
__global__ void __launch_bounds__(256) tap_split_weights_kernel(const float* __restrict__ w, uintx4_t* __restrict__ wf, TapSplit p, int total) {
  const int unit = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
  if (unit >= total) return;
  const int per = p.nchunk * p.taps_total, mblk = unit / per;
  int r = unit - mblk * per;
  const int q = p.nph == 2 && r >= p.nchunk * p.ntap[0] ? 1 : 0;
  if (q) r -= p.nchunk * p.ntap[0];
  const int chunk = r / p.ntap[q], tap = r - chunk * p.ntap[q];
  const int j = p.tapj[p.tap0[q] + tap];
  const int m = mblk * 32 + (lane & 31), c0 = chunk * TS_CC + 8 * (lane >> 5);
  float v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = c0 + e;
    v[e] = m < p.Mo && c < p.Cc ? w[p.bwd ? ((size_t)c * p.Cw + m) * p.KW + j : ((size_t)m * p.Cw + c) * p.KW + j] : 0.f;
  }
  uintx4_t h, m4, l;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const Split2 s = split2(v[2 * e], v[2 * e + 1]);
    h[e] = s.h; m4[e] = s.m; l[e] = s.l;
  }
  uintx4_t* const out = wf + (size_t)unit * 192 + lane;
  out[0] = h; out[64] = m4; out[128] = l;
}

// byte offset of a source position's first channel, or past every tensor
template <bool PLANES>
__device__ __forceinline__ int tap_split_src(const TapSplit& p, int row, int sp) {
  if constexpr (!PLANES) return (unsigned)sp < (unsigned)p.TS ? (row * p.TS + sp) * p.Cs * 4 : TS_OOB;
  if (!p.pW) {
    const int n = row / p.H, h = row - n * p.H;
    return (unsigned)sp < (unsigned)p.TS ? ((n * p.Cc * p.H + h) * p.TS + sp) * 4 : TS_OOB;
  }
  // position sp of the sequence = row sp / pitch (the first pY rows and as many behind every plane are zero), column sp % pitch
  // (those from pW on are zero)
  const int s0 = max(sp, 0), prow = s0 / p.tpitch, c = s0 - prow * p.tpitch, H1 = p.pH + p.pY;
  const int n = max(prow - p.pY, 0) / H1, h = max(prow - p.pY, 0) - n * H1;
  return prow >= p.pY && n < p.pN && h < p.pH && c < p.pW ? ((n * p.Cc * p.pH + h) * p.pW + c) * 4 : TS_OOB;
}

// NR: slab rows per thread
template <int NB, int WM, int NR, bool PLANES>
__global__ void __launch_bounds__(256, 2)
tap_split_kernel(TapSplit p, const float* __restrict__ xr, const uintx4_t* __restrict__ wf, const float* __restrict__ w,
                 const float* __restrict__ bias, float* __restrict__ dst) {
  extern __shared__ __align__(16) char ts_lds[];
  constexpr int WP = 4 / WM, BM = 32 * WM, TP = 32 * NB * WP;
  constexpr int WR = NB == 1 ? 8 : NB == 2 ? 6 : NB == 3 ? 4 : 3;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fg = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wp = wave / WM;
  // phases of a tile run side by side (their results share cache lines), channel tiles apart (each is a sequence of weights)
  int tile = gemm32_tile_of(blockIdx.x, gridDim.x);
  const int q = p.nph == 2 ? tile & 1 : 0;
  tile = p.nph == 2 ? tile >> 1 : tile;
  const int per = p.rows * p.ptiles, mtile = __builtin_amdgcn_readfirstlane(tile / per), rt = tile - mtile * per;
  const int row = __builtin_amdgcn_readfirstlane(rt / p.ptiles), o0 = (rt - row * p.ptiles) * TP;
  const int ntap = __builtin_amdgcn_readfirstlane(q ? p.ntap[1] : p.ntap[0]);
  const int tap0 = __builtin_amdgcn_readfirstlane(q ? p.tap0[1] : p.tap0[0]);
  const int smin = __builtin_amdgcn_readfirstlane(q ? p.smin[1] : p.smin[0]), s0 = o0 * p.SS + smin;

  // ---- the thread's slab rows
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(xr, p.src_bytes);
  int off[NR];
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int R = tid + 256 * i;
    const int sp = s0 + (p.SS == 1 ? R : R < p.half ? 2 * R : 2 * (R - p.half) + 1);
    off[i] = R < p.SR ? tap_split_src<PLANES>(p, row, sp) : TS_OOB;
  }
  uintx4_t raw[NR][4];
  auto load = [&](int chunk) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NR; ++i)
#pragma unroll
      for (int e = 0; e < (PLANES ? 16 : 4); ++e) {
        // (channels past the last meet zero weights: the last one again)
        if constexpr (PLANES) raw[i][e >> 2][e & 3] = __builtin_amdgcn_raw_buffer_load_b32(xrs, off[i], min(chunk * TS_CC + e, p.Cc - 1) * p.cstride, 0);
        else raw[i][e] = __builtin_amdgcn_raw_buffer_load_b128(xrs, off[i], chunk * (TS_CC * 4) + 16 * e, 0);
      }
  };
  const int slab = p.SR * TS_ROW;
  auto split_out = [&](int x) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      char* const at = ts_lds + x * slab + (tid + 256 * i) * TS_ROW;
      if (tid + 256 * i < p.SR) {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          uintx4_t h, m, l;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const Split2 s = split2(__uint_as_float(raw[i][2 * g + (e >> 1)][2 * (e & 1)]), __uint_as_float(raw[i][2 * g + (e >> 1)][2 * (e & 1) + 1]));
            h[e] = s.h; m[e] = s.m; l[e] = s.l;
          }
          *reinterpret_cast<uintx4_t*>(at + 16 * g) = h;
          *reinterpret_cast<uintx4_t*>(at + 32 + 16 * g) = m;
          *reinterpret_cast<uintx4_t*>(at + 64 + 16 * g) = l;
        }
      }
    }
  };

  // ---- weights: this wave's steps are consecutive
  const __amdgpu_buffer_rsrc_t wrs = make_rsrc(wf, p.w_bytes);
  const int wlane = lane * 16;
  int wpos = __builtin_amdgcn_readfirstlane(((mtile * WM + wm) * p.taps_total + tap0) * p.nchunk * 3072);
  uintx4_t wq[WR][3];
  const int total = p.nchunk * ntap;
  auto weights = [&](int r, int step) __attribute__((always_inline)) {      // (zero past the last step)
    const int at = step < total ? wlane : TS_OOB;
#pragma unroll
    for (int e = 0; e < 3; ++e) wq[r][e] = __builtin_amdgcn_raw_buffer_load_b128(wrs, at, wpos + 1024 * e, 0);
    wpos += 3072;
  };

  floatx16 big[NB], small[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) big[b][r] = small[b][r] = 0.f;

  load(0);
#pragma unroll
  for (int r = 0; r < WR; ++r) weights(r, r);
  split_out(0);
  load(min(1, p.nchunk - 1));
  __syncthreads();
  const int lrow = (wp * (32 * NB) + fr) * TS_ROW + 16 * fg;
  int chunk = 0, tap = 0, col = 0, d = 0;
  const int dmask = p.SS - 1;              // (the source stride is 1 or 2)
  constexpr bool AHEAD = NB <= 3;          // the next step's fragments are read while this one's are multiplied
  static_assert(!AHEAD || WR % 2 == 0, "the fragment sets alternate");
  uintx4_t f[AHEAD ? 2 : 1][NB][3];
  auto read = [&](int set, int at_d) __attribute__((always_inline)) {
    const char* const at = ts_lds + (chunk & 1) * slab + ((at_d & dmask) * p.half + (at_d >> dmask)) * TS_ROW + lrow;
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int e = 0; e < 3; ++e) f[set][b][e] = *reinterpret_cast<const uintx4_t*>(at + b * (32 * TS_ROW) + 32 * e);
  };
  if (AHEAD) read(0, 0);
  // (whole groups of WR steps, the last filled up with zero weights: a step that may be left out would make the compiler wait for
  // every load at the next)
#pragma unroll 1
  for (int i = 0; i < total; i += WR) {
#pragma unroll
    for (int r = 0; r < WR; ++r) {
      const int set = AHEAD ? r & 1 : 0;
      if (!AHEAD) read(0, d);
      ++d;
      if (++col == p.tw) { col = 0; d += p.tpitch - p.tw; }
      const bool last = ++tap == ntap;
      if (last) tap = col = d = 0;
      if (AHEAD) read(set ^ 1, d);         // (the next chunk's: once more behind the barrier)
#pragma unroll
      for (int b = 0; b < NB; ++b) split_mma(big[b], small[b], wq[r], f[set][b]);
      weights(r, i + r + WR);
      if (last && chunk + 1 < p.nchunk) {
        ++chunk;
        split_out(chunk & 1);              // (read last in the chunk before this one, behind the barrier at its end)
        load(min(chunk + 1, p.nchunk - 1));
        __syncthreads();
        if (AHEAD) read(set ^ 1, 0);
      }
    }
  }

  bool bad = false;
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      big[b][r] += small[b][r];
      bad |= split_redo(big[b][r]);
    }
  const int mrow = mtile * BM + wm * 32, ob = o0 + wp * (32 * NB) + fr;
  if (__builtin_amdgcn_ballot_w64(bad)) {          // once more with the operands as they are
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) big[b][r] = 0.f;
    int td = 0, tc = 0;
#pragma unroll 1
    for (int t = 0; t < ntap; ++t) {
      const int j = p.tapj[tap0 + t], m = mrow + fr;
      int at[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) at[b] = tap_split_src<PLANES>(p, row, (ob + 32 * b) * p.SS + smin + td);
#pragma unroll 1
      for (int c = fg; c < p.nchunk * TS_CC; c += 2) {
        const bool in = m < p.Mo && c < p.Cc;
        const float a = in ? w[p.bwd ? ((size_t)c * p.Cw + m) * p.KW + j : ((size_t)m * p.Cw + c) * p.KW + j] : 0.f;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const float f = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(xrs, c < p.Cc ? at[b] + c * p.cstride : TS_OOB, 0, 0));
          big[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, f, big[b], 0, 0, 0);
        }
      }
      ++td;
      if (++tc == p.tw) { tc = 0; td += p.tpitch - p.tw; }
    }
  }

  // ---- results: element r of block b: channel 8 (r / 4) + 4 fg + r % 4 of the wave's, position ob + 32 b
  const __amdgpu_buffer_rsrc_t drs = make_rsrc(dst, p.dst_bytes);
  const int pitch = (p.pW ? p.pH * p.pW : p.H * p.TOu) * 4;       // bytes from a channel to the next
  float bv[16];
  if (bias) {
#pragma unroll
    for (int r = 0; r < 16; ++r) bv[r] = bias[min(mrow + 8 * (r >> 2) + 4 * fg + (r & 3), p.Mo - 1)];
  }
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int o = ob + 32 * b;
    int at;
    bool in;
    if (p.pW) {
      const int prow = o / p.tpitch, c = o - prow * p.tpitch, H1 = p.pH + p.pY;      // (as in tap_split_src)
      const int n = max(prow - p.pY, 0) / H1, h = max(prow - p.pY, 0) - n * H1;
      in = prow >= p.pY && n < p.pN && h < p.pH && c < p.pW;
      at = ((n * p.Mo * p.pH + h) * p.pW + c) * 4;
    } else {
      const int n = row / p.H, h = row - n * p.H, u = o * p.nph + q;
      in = u < p.TOu;
      at = ((n * p.Mo * p.H + h) * p.TOu + u) * 4;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mrow + 8 * (r >> 2) + 4 * fg + (r & 3);
      const float v = bias ? big[b][r] + bv[r] : big[b][r];
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), drs, in && m < p.Mo ? at + m * pitch : TS_OOB, 0, 0);
    }
  }
}

// ---- host side ---------------------------------------------------------------------------
struct TapSplitPlan {
  TapSplit p;
  int NB, WM;
  bool planes;
  double cost;           // of the chosen tile, per step
  size_t rows_bytes, w_bytes, lds_bytes;
  int C, H, T;           // of the source tensor, for the rows pass
};

// The tile with the least estimated time: rounds of workgroups over the compute units (two share one, at the rate of one) times
// a workgroup's products in units of one block of 32 positions, and 0.4 for what a step costs besides.  A workgroup that has its
// unit for itself waits for its fragments and weights: `alone` times as long.  Fitted to every tile's time on 537 random layers
// (1 to 24 sequences of 100 to 2000 frames, 80 to 320 channels, 5 to 21 taps, both passes): the choice is 1.1 % behind the best in
// the geometric mean, at worst 25.
void tap_split_tile(TapSplitPlan* pl) {
  TapSplit& p = pl->p;
  const int span = p.pW ? 1 - 2 * p.smin[0] : std::max(p.ntap[0], p.nph == 2 ? p.ntap[1] : 0);
  const double alone[4] = {1.3, 1.2, 1.1, 1.1};
  double best = 1e30;
  for (int wm : {4, 2})
    for (int nb = 4; nb >= 1; --nb) {
      const int tp = 32 * nb * (4 / wm);
      const int half = p.SS == 2 ? ((2 * (tp - 1) + span - 1) >> 1) + 1 : 0, sr = p.SS == 2 ? 2 * half : tp + span - 1;
      const size_t lds = 2 * (size_t)sr * TS_ROW;
      if (sr > 512 || lds > 160 * 1024) continue;
      const long long pt = (p.TO + tp - 1) / tp, mt = (p.Mo + 32 * wm - 1) / (32 * wm);
      const long long wgs = p.rows * pt * mt * p.nph, rounds = (wgs + mfma_num_cus() - 1) / mfma_num_cus();
      const double cost = (double)rounds * (nb + 0.4) * (rounds == 1 ? alone[nb - 1] : 1.0);
      if (cost < best) {
        best = cost;
        pl->NB = nb; pl->WM = wm;
        p.SR = sr; p.half = half;
        p.ptiles = (int)pt; p.mtiles = (int)mt;
        pl->lds_bytes = lds;
        pl->cost = cost;
      }
    }
}

bool tap_split_finish(const ConvGeom& g, bool bwd, long long src_elems, long long dst_elems, TapSplitPlan* pl) {
  TapSplit& p = pl->p;
  p.Mo = bwd ? g.C : g.K;
  p.Cc = bwd ? g.K : g.C; p.Cw = g.C; p.KW = g.KH * g.KW; p.bwd = bwd ? 1 : 0;
  p.nchunk = (p.Cc + TS_CC - 1) / TS_CC;
  p.taps_total = p.ntap[0] + (p.nph == 2 ? p.ntap[1] : 0);
  if (p.taps_total > 64) return false;
  tap_split_tile(pl);
  if (!pl->NB) return false;
  const long long rb = pl->planes ? src_elems * 4 : (long long)p.rows * p.TS * p.Cs * 4, db = dst_elems * 4;
  const long long wb = (long long)p.mtiles * pl->WM * p.taps_total * p.nchunk * 3072;
  if (rb >= (1ll << 31) || wb >= (1ll << 31) || db >= (1ll << 31)) return false;
  p.src_bytes = (unsigned)rb; p.w_bytes = (unsigned)wb; p.dst_bytes = (unsigned)db;
  pl->rows_bytes = pl->planes ? 0 : ((size_t)rb + 255) & ~(size_t)255;
  pl->w_bytes = (size_t)wb;
  return true;
}

bool tap1d_split_plan(const ConvGeom& g, bool bwd, TapSplitPlan* pl) {
  if (g.KH != 1 || g.py != 0 || g.sy != 1 || g.dlx != 1 || g.groups != 1) return false;
  if (g.KW < 2 || g.KW > 32 || (g.sx != 1 && g.sx != 2)) return false;
  if (g.OH != g.H || (long long)g.N * g.H > 65535) return false;
  *pl = TapSplitPlan{};
  TapSplit& p = pl->p;
  const int Cc = bwd ? g.K : g.C;
  p.Cs = mfma_tap1d_cs(Cc, 4);
  if (!p.Cs || Cc < 16) return false;
  p.rows = g.N * g.H; p.H = g.H;
  p.TS = bwd ? g.OW : g.W; p.TOu = bwd ? g.W : g.OW;
  p.SS = bwd ? 1 : g.sx; p.nph = bwd ? g.sx : 1;
  p.tw = 1 << 20; p.tpitch = 0;
  if (p.nph == 1) {
    p.ntap[0] = g.KW;
    p.smin[0] = bwd ? g.px - (g.KW - 1) : -g.px;
    for (int i = 0; i < g.KW; ++i) p.tapj[i] = (signed char)(bwd ? g.KW - 1 - i : i);
  } else {
    // u = 2 v + q takes the taps j = jq + 2 i' with jq = (q + px) & 1, from dy[v + (q + px - jq) / 2 - i']
    for (int q = 0; q < 2; ++q) {
      const int jq = (q + g.px) & 1;
      p.ntap[q] = (g.KW - jq + 1) / 2;
      if (p.ntap[q] < 1) return false;
      p.tap0[q] = q ? p.ntap[0] : 0;
      p.smin[q] = (q + g.px - jq) / 2 - (p.ntap[q] - 1);
      for (int i = 0; i < p.ntap[q]; ++i) p.tapj[p.tap0[q] + i] = (signed char)(jq + 2 * (p.ntap[q] - 1 - i));
    }
  }
  p.TO = (p.TOu + p.nph - 1) / p.nph;
  pl->C = Cc; pl->H = g.H; pl->T = p.TS;
  // (the forward pass leaves its rows to the filter gradient)
  pl->planes = bwd;
  p.cstride = bwd ? g.H * p.TS * 4 : 4;
  return tap_split_finish(g, bwd, (long long)p.rows * Cc * p.TS, (long long)p.rows * (bwd ? g.C : g.K) * p.TOu, pl);
}

// Windows of several rows of stride 1 that keep the plane's size, over stacked planes: every plane of the batch in one sequence, rows
// followed by px zero columns, planes separated by py zero rows (which the next plane's windows share); the window's taps are then
// fixed offsets into it.
bool tap2d_split_plan(const ConvGeom& g, bool bwd, TapSplitPlan* pl) {
  if (g.KH < 2 || g.KH != 2 * g.py + 1 || g.KW != 2 * g.px + 1 || g.sy != 1 || g.sx != 1 || g.dly != 1 || g.dlx != 1 || g.groups != 1)
    return false;
  const int Cc = bwd ? g.K : g.C, P = g.W + g.px, taps = g.KH * g.KW;
  const long long ts = ((long long)g.N * (g.H + g.py) + g.py) * P;
  if (ts >= (1ll << 22) - 1024 || Cc < 16 || Cc > 512 || taps > 64) return false;
  *pl = TapSplitPlan{};
  TapSplit& p = pl->p;
  p.rows = 1; p.H = 1;
  pl->planes = true;
  p.cstride = g.H * g.W * 4;
  p.TS = p.TOu = (int)ts;
  p.TO = p.TS - g.py * P;          // (the last zero rows hold no result)
  p.SS = p.nph = 1;
  p.ntap[0] = taps;
  p.smin[0] = -(g.py * P + g.px);
  p.tw = g.KW; p.tpitch = P; p.pW = g.W; p.pH = g.H; p.pN = g.N; p.pY = g.py;
  for (int i = 0; i < taps; ++i) p.tapj[i] = (signed char)(bwd ? taps - 1 - i : i);
  pl->C = Cc; pl->H = g.H; pl->T = g.W;
  return tap_split_finish(g, bwd, (long long)g.N * Cc * g.H * g.W, (long long)g.N * (bwd ? g.C : g.K) * g.H * g.W, pl);
}

int launch_tap_split(const TapSplitPlan& pl, const float* src, uintx4_t* wf, const float* w, const float* bias, float* dst, hipStream_t s) {
  const TapSplit& p = pl.p;
  const int total = p.mtiles * pl.WM * p.taps_total * p.nchunk;
  hipLaunchKernelGGL(tap_split_weights_kernel, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, s, w, wf, p, total);
  if (const int rc = check_launch("conv2d (one-row windows, operand passes)")) return rc;
  auto go = [&](auto kernel) {
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), pl.lds_bytes)) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)((long long)p.rows * p.ptiles * p.mtiles * p.nph)), dim3(256), pl.lds_bytes, s, p, src, wf, w,
                       bias, dst);
    return check_launch("conv2d (one-row windows, fp32 in three parts)");
  };
  auto tile = [&](auto nb, auto planes) {
    constexpr int NB = decltype(nb)::value;
    constexpr bool PL = decltype(planes)::value;
    if (p.SR <= 256) return pl.WM == 4 ? go(tap_split_kernel<NB, 4, 1, PL>) : go(tap_split_kernel<NB, 2, 1, PL>);
    return pl.WM == 4 ? go(tap_split_kernel<NB, 4, 2, PL>) : go(tap_split_kernel<NB, 2, 2, PL>);
  };
  auto rows = [&](auto nb) { return pl.planes ? tile(nb, std::true_type{}) : tile(nb, std::false_type{}); };
  switch (pl.NB) {
    case 1: return rows(std::integral_constant<int, 1>{});
    case 2: return rows(std::integral_constant<int, 2>{});
    case 3: return rows(std::integral_constant<int, 3>{});
    default: return rows(std::integral_constant<int, 4>{});
  }
}

int run_tap_split(const TapSplitPlan& pl, const void* src, const void* w, const float* bias, void* dst, hipStream_t s, void* ws, size_t ws_bytes) {
  if (!ws || ws_bytes < pl.rows_bytes + pl.w_bytes) return -1;
  const float* from = static_cast<const float*>(src);
  if (!pl.planes) {
    mfma_tap1d_rows_f32(from, static_cast<float*>(ws), pl.C, pl.H, pl.T, pl.p.Cs, pl.p.rows, s);
    from = static_cast<const float*>(ws);
  }
  return launch_tap_split(pl, from, reinterpret_cast<uintx4_t*>(static_cast<char*>(ws) + pl.rows_bytes), static_cast<const float*>(w), bias,
                          static_cast<float*>(dst), s);
}

}  // namespace

size_t mfma_tap1d_split_ws(const ConvGeom& g, bool bwd, size_t* rows_bytes) {
  TapSplitPlan pl;
  if (!tap1d_split_plan(g, bwd, &pl)) return 0;
  if (rows_bytes) *rows_bytes = pl.rows_bytes;
  return pl.rows_bytes + pl.w_bytes;
}
int mfma_tap1d_split(const ConvGeom& g, bool bwd, const void* src, const void* w, const float* bias, void* dst, hipStream_t s, void* ws,
                     size_t ws_bytes) {
  TapSplitPlan pl;
  return tap1d_split_plan(g, bwd, &pl) ? run_tap_split(pl, src, w, bias, dst, s, ws, ws_bytes) : -1;
}
// Whether they are faster than the kernels on the fp32 instructions (slab, few tiles, tapped), by estimate in us: 9 and 0.105 per
// step and unit of the tile's cost here; there 8, the products at 112 TFLOP/s (result channels in whole blocks of 32) and 0.055 per
// contraction channel and 9 taps, 20 more where the channels are not whole pieces of 8 (the kernel for few tiles declines them).
// Measured on 12828 random 3x3 layers (1 to 64 planes of 4 x 4 to 112 x 112, 16 to 512 channels), backward-data: the choice is 0.6 %
// behind the better one in the geometric mean and takes 0.82 of the time without these kernels; of the layers it takes 0.9 % are
// more than 6 % slower here, nearly all of 16 contraction channels, which it leaves out.  64 images, here / there: 64 channels over
// 56 x 56 84 / 131 us, 256 over 14 x 14 89 / 140, 512 over 7 x 7 111 / 234; 4 images: 16 / 21, 35 / 25, 63 / 43.
bool mfma_tap2d_split_pays(const ConvGeom& g, bool bwd) {
  TapSplitPlan pl;
  const int Cc = bwd ? g.K : g.C, Mo = bwd ? g.C : g.K;
  if (Cc < 32 || !tap2d_split_plan(g, bwd, &pl)) return false;
  const double taps = pl.p.ntap[0], flops = 2.0 * taps * Cc * ((Mo + 31) / 32 * 32) * g.N * g.H * g.W;
  const double here = 9.0 + 0.105 * pl.cost * pl.p.nchunk * taps;
  const double there = 8.0 + flops / 112e6 + 0.055 * Cc * taps / 9.0 + (Cc % 8 ? 20.0 : 0.0);
  return here < 1.05 * there;
}
size_t mfma_tap2d_split_ws(const ConvGeom& g, bool bwd) {
  TapSplitPlan pl;
  return tap2d_split_plan(g, bwd, &pl) ? pl.w_bytes : 0;
}
int mfma_tap2d_split(const ConvGeom& g, bool bwd, const void* src, const void* w, const float* bias, void* dst, hipStream_t s, void* ws,
                     size_t ws_bytes) {
  TapSplitPlan pl;
  return tap2d_split_plan(g, bwd, &pl) ? run_tap_split(pl, src, w, bias, dst, s, ws, ws_bytes) : -1;
}

}  // namespace flhip
