// Convolutions with one-row windows (KH = 1, KW taps along the contiguous axis: the 21 x 1
// windows of a wav2letter-style speech stack) on the matrix cores, forward, backward-data and
// filter gradient, column stride 1 or 2; 16-bit storage on v_mfma_f32_32x32x16 (bf16 and IEEE half), and the filter gradient in fp32
// too (its forward and backward-data: conv2d_mfma_tap_split.hip).
//
//   forward        y[m][o]  = sum_c sum_j w[m][c][j]  x[c][o*s + j - p]   (+ bias[m])
//   backward-data  dx[c][u] = sum_m sum_j w[m][c][j] dy[m][(u + p - j) / s]   where s divides
//
// A matrix instruction wants consecutive contraction channels of one position per lane, and
// every tap shifts the positions by one element: with the tensors as they lie in memory
// (channel-major rows of positions) a shifted 16-byte fragment would start on any element
// boundary.  So two small passes first bring the operands into the order the instruction reads:
//   rows     xr[sequence][position][Cs]: the source with its channels last, Cs = the channel
//            count padded with zeros (tap1d_rows_block; a sequence is one (image, row) pair); a
//            tap then shifts whole 16-byte cells (8 channels of one position);
//   weights  wf[block of 32 result channels][tap][stage of 2 cells][lane][cell]: the fragment
//            of every (tap, stage) exactly as the 64 lanes hold it, in the order the kernel walks
//            (tap1d_weights_block); padded channels and taps are zero.
// A stage is 16 channels, one matrix instruction per block.
// Backward-data over a stride of 2 is two interleaved stride-1 problems (the results of even
// and of odd index take the taps of one parity each): "phases" of one workgroup, which
// writes both so that its stores cover whole runs of dx.
//
// A workgroup (4 waves) owns 32 NB result positions (per phase; NB = 3, or 2 where the slab of 3
// would not fit) of one sequence x 128 result channels; wave w owns channels 32 w .. 32 w + 31:
// NB (2 NB) accumulator blocks of 32 x 32.  NB = 1: 64 positions x 64 channels, two waves to either half of both: for layers of so few
// tiles that a compute unit has one, where a wave's walk over the taps is the whole time.  What that walk waits for is the
// fragments' way through the vector cache (4 KB a stage and compute unit at some 40 bytes a clock), not the matrix pipe: a
// stage takes 95 clocks with one block, 103 with two and 135 with three, of which 32, 64 and 96 are matrix instructions.  (Neither the
// fragments of a stage next to each other for all four waves, nor touching them all for the die's second-level cache first, nor
// reading positions three or six stages ahead changes it.)
//   * The source rows the tile needs (its positions + the window's reach, every channel) are
//     copied to LDS once, by buffer loads with the LDS modifier (no registers, no vector
//     instructions); a row of the slab is its cells + 1 unused cell, which puts the eight
//     lanes of a 16-byte read cycle on distinct banks.  With a forward stride of 2 the slab
//     keeps even and odd source positions apart, so a tap's 32 positions are consecutive rows.
//   * The weights never pass through LDS: a wave's fragment of a (tap, stage) is 1 KiB of
//     contiguous memory, fetched straight into registers RW stages ahead of its use.  No other
//     wave needs it, so the main loop has no barrier.
//   * Per stage a wave reads NB position fragments from LDS (two stages ahead of their use) and
//     issues NB matrix instructions.
// Positions are the rows of the instruction tile: a lane holds 4 consecutive positions of one
// result channel (8 with two phases), stored as one piece.
#include <algorithm>
#include <cmath>
#include <cmath>
#include <cstring>

#include "conv2d_mfma.h"
#include "lds_direct.h"
#include "split_f32.h"

namespace flhip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
#if defined(__HIP_DEVICE_COMPILE__)
typedef __attribute__((address_space(3))) const uintx4_t* lds_cell_t;
#else
typedef const uintx4_t* lds_cell_t;
#endif

// a workgroup's four waves: blocks of 32 result channels x groups of positions, with NB blocks of 32 positions in a wave
__host__ __device__ constexpr int t1_wm(int NB) { return NB == 1 ? 2 : 4; }
__host__ __device__ constexpr int t1_positions(int NB) { return 32 * NB * 4 / t1_wm(NB); }
constexpr int T1_KW = 32;        // taps of a window
constexpr int T1_MAXTAPS = 64;   // taps over both phases, padding included
constexpr int T1_OOB = (int)0x80000000;

// element type -> channels per 16-byte cell; a stage is two cells
template <typename T> struct Tap1Elem;
template <> struct Tap1Elem<bf16_t> { static constexpr int CELL = 8; };
template <> struct Tap1Elem<f16_t> { static constexpr int CELL = 8; };
template <> struct Tap1Elem<float> { static constexpr int CELL = 4; };

// one stage of one block: acc += a (positions x stage channels) * w (stage channels x result channels)
__device__ __forceinline__ void tap1d_mma(floatx16& acc, const uintx4_t& a, const uintx4_t& w, const bf16_t*) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, w), acc, 0, 0, 0);
}
__device__ __forceinline__ void tap1d_mma(floatx16& acc, const uintx4_t& a, const uintx4_t& w, const f16_t*) {
  acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, w), acc, 0, 0, 0);
}
// two results rounded to the storage type, the first in the low half
__device__ __forceinline__ uint32_t tap1d_pack(float a, float b, const bf16_t*) { return pack_bf16(a, b); }
__device__ __forceinline__ uint32_t tap1d_pack(float a, float b, const f16_t*) { return pack_f16(a, b); }

struct Tap1Params {
  int rows, H;           // sequences (images x rows), rows per image
  int TS, TO, TOu;       // source positions, result indices per phase, result positions per sequence
  int Cs, KS;            // padded contraction channels, stages per tap
  int Mo;                // result channels
  int nph;               // phases (1; 2: results u = 2 o + q)
  int ntaps[2];          // taps per phase as stored (a multiple of the kernel's tap group)
  int nreal[2];          // taps per phase that exist (the others carry zero weights)
  int d0[2];             // source offset of tap 0 of a phase, relative to the slab's first position
  int smin;              // slab's first source position for result 0
  int SR, half;          // slab rows; stride 2: row of the first odd source offset
  int taps_total;        // ntaps[0] + ntaps[1]
  int ptiles, mtiles;
  unsigned src_bytes, w_bytes, dst_bytes;
  // two-dimensional windows over stacked planes (tap2d_*): taps per window row, slab rows per window row = the
  // pitch of a plane's row, and the plane's geometry for the results
  int tw, tpitch, pW, pH, pN;
  int zcells;            // cells of zeros behind the slab's rows, for the taps that do not exist (0: there are none)
};

// ---- operand passes ------------------------------------------------------------------------
// two neighbouring 16-bit values from any address, the second one only where it exists
struct __attribute__((packed, aligned(2))) Pair16 {
  uint32_t v;
};
template <typename T>
__device__ __forceinline__ uint32_t pair_at(const T* p, int left) {
  return left >= 2 ? reinterpret_cast<const Pair16*>(p)->v : left == 1 ? (uint32_t)__builtin_bit_cast(uint16_t, *p) : 0u;
}

// x[n][c][h][t] -> xr[n * H + h][t][Cs], channels c >= C zero.  A block transposes 64 channels x 64
// positions through LDS: (16-bit storage: pairs of positions in;) whole 16-byte cells out.
template <typename T>
__device__ __forceinline__ void tap1d_rows_block(const T* __restrict__ x, T* __restrict__ xr, int C, int H, int Tn, int Cs, int bx, int by,
                                                 int row, void* lds) {
  constexpr int CELL = Tap1Elem<T>::CELL;
  T(*tile)[sizeof(T) == 2 ? 66 : 65] = reinterpret_cast<T(*)[sizeof(T) == 2 ? 66 : 65]>(lds);
  const int t0 = bx * 64, c0 = by * 64;
  const int n = row / H, h = row - n * H;
  if constexpr (sizeof(T) == 2) {
    const int tp = threadIdx.x & 31, cy = threadIdx.x >> 5;      // pair of positions, channel (+ 8 i)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int c = c0 + cy + 8 * i, t = t0 + 2 * tp;
      *reinterpret_cast<uint32_t*>(&tile[cy + 8 * i][2 * tp]) = pair_at(x + (((size_t)n * C + c) * H + h) * Tn + t, c < C ? Tn - t : 0);
    }
  } else {
    const int tx = threadIdx.x & 63, cy = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int c = c0 + cy + 4 * i, t = t0 + tx;
      tile[cy + 4 * i][tx] = (c < C && t < Tn) ? x[(((size_t)n * C + c) * H + h) * Tn + t] : T{};
    }
  }
  __syncthreads();
  constexpr int CPT = 64 / CELL;                // cells per position of the tile
#pragma unroll
  for (int i = 0; i < CPT * 64 / 256; ++i) {
    const int item = threadIdx.x + 256 * i, cell = item % CPT, tl = item / CPT;
    const int t = t0 + tl, c = c0 + CELL * cell;
    if (t < Tn && c < Cs) {
      __attribute__((aligned(16))) T v[CELL];
#pragma unroll
      for (int e = 0; e < CELL; ++e) v[e] = tile[CELL * cell + e][tl];
      *reinterpret_cast<uintx4_t*>(xr + ((size_t)row * Tn + t) * Cs + c) = *reinterpret_cast<const uintx4_t*>(v);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256)
tap1d_rows_kernel(const T* __restrict__ x, T* __restrict__ xr, int C, int H, int Tn, int Cs) {
  __shared__ __align__(16) T tile[64][sizeof(T) == 2 ? 66 : 65];
  tap1d_rows_block(x, xr, C, H, Tn, Cs, blockIdx.x, blockIdx.y, blockIdx.z, tile);
}

static dim3 rows_grid(int Tn, int Cs, int rows) { return dim3((unsigned)((Tn + 63) / 64), (unsigned)((Cs + 63) / 64), (unsigned)rows); }

template <typename T>
static void launch_rows(const T* x, T* xr, int C, int H, int Tn, int Cs, int rows, hipStream_t s) {
  hipLaunchKernelGGL((tap1d_rows_kernel<T>), rows_grid(Tn, Cs, rows), dim3(256), 0, s, x, xr, C, H, Tn, Cs);
}

struct Tap1Weights {
  int Mo, Cc;            // result / contraction channels that exist
  int KS, taps_total;
  int bwd;               // 0: w[m][c][j], 1: w[c][m][j] (contraction over the filters)
  int Cw, KW;            // channels per filter and taps of the weight tensor
  int mblocks;
  signed char tapj[T1_MAXTAPS];   // weight tap of stored tap i (-1: padding)
};

// The fragments of 32 result channels x 16 contraction channels, every tap: 32 (or, over the filters, 16) runs of 16 (32) channels'
// taps come in as pairs of neighbours and leave LDS tap by tap.
template <typename T>
__device__ __forceinline__ void tap1d_weights_block(const T* __restrict__ w, uintx4_t* __restrict__ wf, const Tap1Weights& p, int block, T* lds) {
  const int mblk = block / p.KS, ks = block - mblk * p.KS, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = mblk * 32, c0 = ks * 16;
  // a row of the runs: its threads, pairs between two of a thread, the source's first element and how many follow in range
  const int per = p.bwd ? 16 : 8, r = tid / per, q = tid % per, pitch = (p.bwd ? 34 : 16) * p.KW + 2;
  // (neighbouring lanes read elements KW apart over the filters: two unused ones after every 32 keep even KW off one bank)
  const auto at = [&](int e) { return p.bwd ? e + 2 * (e >> 5) : e; };
  const int first = (p.bwd ? m0 : c0) * p.KW, row = (p.bwd ? c0 : m0) + r;
  const int left = row < (p.bwd ? p.Cc : p.Mo) ? p.Cw * p.KW - first : 0;
  const T* const src = w + (size_t)(left > 0 ? row : 0) * p.Cw * p.KW + first;
  uint32_t in[T1_KW];                     // (all of a thread's loads before the first value is waited for)
#pragma unroll
  for (int k = 0; k < T1_KW; ++k) {
    const int e = 2 * (q + per * k);
    if (k < p.KW) in[k] = pair_at(src + e, left - e);
  }
#pragma unroll
  for (int k = 0; k < T1_KW; ++k)
    if (k < p.KW) *reinterpret_cast<uint32_t*>(lds + r * pitch + at(2 * (q + per * k))) = in[k];
  __syncthreads();
  const int fr = lane & 31, fh = lane >> 5;
  const T* const mine = lds + (p.bwd ? 8 * fh : fr) * pitch;
  const int run = (p.bwd ? fr : 8 * fh) * p.KW, step = p.bwd ? pitch : p.KW;
#pragma unroll 4
  for (int tap = wave; tap < p.taps_total; tap += 4) {
    const int j = p.tapj[tap];
    const T* const from = mine + at(run + max(j, 0));
    __attribute__((aligned(16))) T v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = from[e * step];
    if (j < 0)
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = T{};
    wf[(((size_t)mblk * p.taps_total + tap) * p.KS + ks) * 64 + lane] = *reinterpret_cast<const uintx4_t*>(v);
  }
}

// The same, one wave per fragment (`unit`: the tap fastest, so that a workgroup's waves read the same lines).
template <typename T>
__device__ __forceinline__ void tap1d_weights_gather(const T* __restrict__ w, uintx4_t* __restrict__ wf, const Tap1Weights& p, int unit) {
  const int lane = threadIdx.x & 63, block = unit / p.taps_total, tap = unit - block * p.taps_total, mblk = block / p.KS, ks = block - mblk * p.KS;
  if (mblk >= p.mblocks) return;
  const int m = mblk * 32 + (lane & 31), c0 = ks * 16 + 8 * (lane >> 5), j = p.tapj[tap];
  __attribute__((aligned(16))) T v[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = c0 + e;
    v[e] = j >= 0 && m < p.Mo && c < p.Cc ? w[p.bwd ? ((size_t)c * p.Cw + m) * p.KW + j : ((size_t)m * p.Cw + c) * p.KW + j] : T{};
  }
  wf[(((size_t)mblk * p.taps_total + tap) * p.KS + ks) * 64 + lane] = *reinterpret_cast<const uintx4_t*>(v);
}
// Up to so many blocks of tap1d_weights_block: they leave most of the chip idle, and each is a chain of loads, LDS and its taps.
// us of a layer (blocks / fragments; before either 15.5, 11.9, 26.9, 46.5, 55.6): 256 channels to 29 over 6 x 491 frames, 29 taps,
// backward (8 blocks) 15.0 / 12.4; 80 to 28 over 3 x 300, 21 taps, backward (8) 11.5 / 9.4; 80 to 250 over 7 x 1111, 21 taps (48) 22.1 / 21.3;
// 250 to 250 (128), weights not in the caches, 33.4 / 35.3; 250 to 1000 over 4 x 400 (512) 35.0 / 42.7.
constexpr int T1_FEW_BLOCKS = 64;

// Both operands of a layer in 16-bit storage in one launch: neither pass fills the chip, and each is a few microseconds of latency
// (loads, LDS, stores).  The first blocks take the rows, the others the weights.  Rows one element at a time where they are odd, and
// weights gathered fragment by fragment (every line met once per tap) in a launch of their own: 8.2 + 8.8 us for 250 -> 250 channels, 21 taps
// over 7 x 1111 frames, and a launch more for the host; the layer's passes replayed from a graph 48.6 -> 44.6 and 45.5 -> 44.2; 240
// random layers in bf16 and f16, both passes, 0.82 of the time, the slowest 1.01.
template <typename T>
__global__ void __launch_bounds__(256)
tap1d_operands_kernel(const T* __restrict__ x, T* __restrict__ xr, int C, int H, int Tn, int Cs, int tblocks, int cblocks, int rblocks,
                      const T* __restrict__ w, uintx4_t* __restrict__ wf, Tap1Weights p, bool gather) {
  extern __shared__ uintx4_t t1_operands[];
  const int b = blockIdx.x;
  if (b < rblocks) {
    const int t = b / tblocks;
    tap1d_rows_block(x, xr, C, H, Tn, Cs, b - t * tblocks, t % cblocks, t / cblocks, t1_operands);
  } else if (gather) {
    tap1d_weights_gather(w, wf, p, (b - rblocks) * 4 + (int)(threadIdx.x >> 6));
  } else {
    tap1d_weights_block(w, wf, p, b - rblocks, reinterpret_cast<T*>(t1_operands));
  }
}

// ---- the convolution ---------------------------------------------------------------------
// KS stages per tap; DT taps per unrolled group; RW stages between a weight fragment's load and its use (RW divides
// DT * KS); SS source stride;
// NPH phases; NB blocks of 32 positions.
// TD: the taps form a two-dimensional window over planes stacked in one sequence (see tap2d_plan); only the slab
// offset of a tap and the addresses of the results differ.
template <typename T, int KS, int DT, int RW, int SS, int NPH, int NB, bool TD>
__device__ __forceinline__ void
tap_conv_body(const Tap1Params& p, const T* __restrict__ xr, const uintx4_t* __restrict__ wf,
              const float* __restrict__ bias, T* __restrict__ dst) {
  extern __shared__ uintx4_t t1_slab[];
  constexpr int CELL = Tap1Elem<T>::CELL;
  constexpr int ESZ = (int)sizeof(T);
  constexpr int CPR = 2 * KS + 1;               // cells per slab row
  constexpr int WM = t1_wm(NB), TP = t1_positions(NB), BM = 32 * WM;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave % WM, wp = wave / WM;
  const int ptile = __builtin_amdgcn_readfirstlane(blockIdx.x % p.ptiles);
  const int row = __builtin_amdgcn_readfirstlane(blockIdx.x / p.ptiles);
  const int mtile = blockIdx.y;
  const int o0 = ptile * TP;
  const int s0 = o0 * SS + p.smin;              // source position of slab offset 0

  // ---- the slab: load instruction ii fills cells ii * 64 .. + 63, cell L = slab row L / CPR, cell L % CPR
  {
    const intx4_t xrs = pd_rsrc(xr, p.src_bytes);
    const unsigned base = pd_lds_addr(t1_slab);
    const int ncell = p.SR * CPR + (DT > 1 ? p.zcells : 0), ninstr = (ncell + 63) >> 6;
    const float inv = 1.0f / (float)CPR;
    for (int ii = wave; ii < ninstr; ii += 4) {
      const int L = ii * 64 + lane;
      int c;
      const int R = fast_div(L, CPR, inv, &c);
      const int off = SS == 1 ? R : (R < p.half ? 2 * R : 2 * (R - p.half) + 1);
      const int sp = s0 + off;
      int voff = T1_OOB;
      if (R < p.SR && c < 2 * KS && (unsigned)sp < (unsigned)p.TS) voff = ((row * p.TS + sp) * p.Cs + CELL * c) * ESZ;
      pd_load_lds(xrs, base + ii * 1024, voff, 0);
    }
  }

  // ---- weights: this wave's stream of fragments, RW stages ahead
  constexpr int NS = DT * KS;
  static_assert(NS % 4 == 0 && NS % RW == 0 && KS >= 2, "fragment sets and the weight ring rotate with the unrolled group");
  const __amdgpu_buffer_rsrc_t wrs = make_rsrc(wf, p.w_bytes);
  const int mblk = mtile * WM + wm;
  int wpos = mblk * p.taps_total * KS * 1024;   // byte offset of the stage RW ahead of the group's first
  const int wlane = lane * 16;
  uintx4_t bq[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) bq[i] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wlane, wpos + i * 1024, 0);
  wpos += RW * 1024;

  floatx16 acc[NPH][NB];
#pragma unroll
  for (int q = 0; q < NPH; ++q)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[q][b][r] = 0.f;

  const int fr = lane & 31, fg = lane >> 5;
  lds_cell_t ap[NB];                            // this lane's cell of a tap's first row
#pragma unroll
  for (int b = 0; b < NB; ++b) ap[b] = (lds_cell_t)t1_slab + (((wp * NB + b) * 32 + fr) * CPR + fg);

  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the slab (and the first weight fragments) have landed
  __syncthreads();

  // The position fragments of a stage are read two stages ahead of their use (four sets of registers in rotation;
  // a group's stage count is a multiple of four).
  auto run = [&](floatx16 (&ac)[NB], int q) __attribute__((always_inline)) {
    const int groups = p.ntaps[q] / DT;
    const int dq = p.d0[q], last = p.nreal[q] - 1;
    // slab offset (cells) of a tap's rows.  Taps that do not exist (DT > 1) read zeros, every lane the same (`rows` takes its place in the slab off):
    // zero weights times rows that exist would make NaN of an infinity.  (Behind the last group, where nothing is multiplied: any rows.)
    const int real = p.zcells ? last : 1 << 30;
    auto toff_of = [&](int tap) {
      if (DT > 1 && tap > real) return p.SR * CPR;
      const int tl = min(tap, last);
      const int d = dq + (TD ? (tl / p.tw) * p.tpitch + tl % p.tw : tl);
      const int trow = SS == 1 ? d : (d & 1) * p.half + (d >> 1);
      return trow * CPR;
    };
    auto rows = [&](int b, int off) __attribute__((always_inline)) {
      return (DT > 1 && off == p.SR * CPR ? (lds_cell_t)t1_slab : ap[b]) + off;
    };
    uintx4_t af[4][NB];
    int tcur[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) tcur[dt] = toff_of(dt);
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int b = 0; b < NB; ++b) af[i][b] = rows(b, tcur[i / KS])[2 * (i % KS)];
    for (int g = 0; g < groups; ++g) {
      int tnext[DT];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) tnext[dt] = toff_of((g + 1) * DT + dt);
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int i2 = i + 2;
        const int o2 = i2 < NS ? tcur[(i2 % NS) / KS] : tnext[(i2 % NS) / KS];
#pragma unroll
        for (int b = 0; b < NB; ++b) af[i2 % 4][b] = rows(b, o2)[2 * ((i2 % NS) % KS)];
        const uintx4_t w8 = bq[i % RW];
        bq[i % RW] = __builtin_amdgcn_raw_buffer_load_b128(wrs, wlane, wpos + i * 1024, 0);
#pragma unroll
        for (int b = 0; b < NB; ++b) tap1d_mma(ac[b], af[i % 4][b], w8, static_cast<const T*>(nullptr));
        __builtin_amdgcn_sched_barrier(0);     // (the scheduler would otherwise move every read down to its use)
      }
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) tcur[dt] = tnext[dt];
      wpos += NS * 1024;
    }
  };
  run(acc[0], 0);
  if (NPH == 2) run(acc[NPH - 1], 1);

  // ---- results: element r of block b: result index o0 + 32 b + 8 (r / 4) + 4 fg + r % 4 of channel m
  const int m = mtile * BM + wm * 32 + fr;
  if constexpr (TD) {
    // Results through LDS (the slab is done with): every wave parks its 32 channels x 32 NB positions at storage size,
    // then threads walk positions (consecutive lanes = consecutive positions = consecutive addresses inside a plane's
    // row, and across row ends too: the zero column has no address) with the position's plane / row / column worked
    // out once per thread.  Position o of the sequence = row o / pitch (row 0 and every (pH + 1)-th after it are the
    // zero rows between the planes), column o % pitch (the last one of a row is the zero column).
    constexpr int TPOS = TP, CG = 256 / TPOS;     // (CG: groups of threads, a channel each at a time)
    constexpr int SPT = TPOS + 4;                 // staging pitch (elements): 8-byte rows, lanes on distinct banks
    T* const stage = reinterpret_cast<T*>(t1_slab);
    const float bvt = (bias && m < p.Mo) ? bias[m] : 0.f;
    __syncthreads();
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int g4 = 0; g4 < 4; ++g4) {
        T* const at = stage + (wm * 32 + fr) * SPT + (wp * NB + b) * 32 + g4 * 8 + fg * 4;
#pragma unroll
        for (int e = 0; e < 4; ++e) st(at, e, acc[0][b][4 * g4 + e] + bvt);
      }
    __syncthreads();
    if (tid >= CG * TPOS) return;
    const int pos = tid % TPOS, cg = tid / TPOS;
    const int o = o0 + pos;
    const int P = p.tpitch, H1 = p.pH + 1;
    const int prow = o / P, col = o - prow * P;
    const int n = max(prow - 1, 0) / H1, h = max(prow - 1, 0) - n * H1;
    if (!(prow >= 1 && n < p.pN && h < p.pH && col < p.pW)) return;
    const int mlim = min(BM, p.Mo - mtile * BM);
    const size_t plane = (size_t)p.pH * p.pW;
    T* const out = dst + ((size_t)n * p.Mo + mtile * BM) * plane + (size_t)h * p.pW + col;
    for (int c = cg; c < mlim; c += CG) out[(size_t)c * plane] = stage[c * SPT + pos];
    return;
  }
  if (m >= p.Mo) return;
  const float bv = bias ? bias[m] : 0.f;
  const int n = row / p.H, h = row - n * p.H;
  const long long rbase = (((long long)n * p.Mo + m) * p.H + h) * p.TOu;     // element offset of the result row
  const __amdgpu_buffer_rsrc_t drs = make_rsrc(dst, p.dst_bytes);
  const bool aligned = (rbase & 1) == 0;     // pieces start on 4-byte boundaries
#pragma unroll
  for (int b = 0; b < NB; ++b)
#pragma unroll
    for (int g4 = 0; g4 < 4; ++g4) {
      const int o = o0 + (wp * NB + b) * 32 + g4 * 8 + fg * 4;
      float v[8];
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int q = 0; q < NPH; ++q) v[e * NPH + q] = acc[q][b][4 * g4 + e] + bv;
      const int u = o * NPH;
      if (aligned && u + 4 * NPH <= p.TOu) {      // (u is a multiple of 4)
        const int at = (int)((rbase + u) * ESZ);
        if (NPH == 1) {
          const T* const tt = nullptr;
          const uintx2_t t = {tap1d_pack(v[0], v[1], tt), tap1d_pack(v[2], v[3], tt)};
          __builtin_amdgcn_raw_buffer_store_b64(t, drs, at, 0, 0);
        } else {
          const T* const tt = nullptr;
          const uintx4_t t = {tap1d_pack(v[0], v[1], tt), tap1d_pack(v[2], v[3], tt), tap1d_pack(v[4], v[5], tt), tap1d_pack(v[6], v[7], tt)};
          __builtin_amdgcn_raw_buffer_store_b128(t, drs, at, 0, 0);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4 * NPH; ++e)
          if (u + e < p.TOu) st(dst, (size_t)(rbase + u + e), v[e]);
      }
    }
}

template <typename T, int KS, int DT, int RW, int SS, int NPH, int NB>
__global__ void __launch_bounds__(256, 1)
tap1d_conv_kernel(Tap1Params p, const T* __restrict__ xr, const uintx4_t* __restrict__ wf,
                  const float* __restrict__ bias, T* __restrict__ dst) {
  tap_conv_body<T, KS, DT, RW, SS, NPH, NB, false>(p, xr, wf, bias, dst);
}

// 3 x 3 windows of stride 1 over small planes (the 14 x 14 and 7 x 7 layers of a residual network): the same loop
// over a sequence that holds every plane of the batch, rows pH + 1 apart with a zero row between two planes, a row's
// pW positions followed by one zero column (tap2d_rows_block writes it so) - the window's taps are then nine fixed
// offsets into the sequence, and the zero row / column are the padding.  Results at the zero positions are not stored.
template <typename T, int KS, int DT, int RW, int NB>
__global__ void __launch_bounds__(256, 1)
tap2d_conv_kernel(Tap1Params p, const T* __restrict__ xr, const uintx4_t* __restrict__ wf,
                  const float* __restrict__ bias, T* __restrict__ dst) {
  tap_conv_body<T, KS, DT, RW, 1, 1, NB, true>(p, xr, wf, bias, dst);
}

// x[n][c][h][w] -> xr[position][Cs] with position = ((n (H + 1) + 1 + h) P + w), P = W + 1; the zero rows, the zero
// column and channels c >= C are written as zeros.  A block transposes 64 channels x 64 positions through LDS.
template <typename T>
__device__ __forceinline__ void tap2d_rows_block(const T* __restrict__ x, T* __restrict__ xr, int C, int H, int W, int N, int TS, int Cs, int bx,
                                                 int by, void* lds) {
  constexpr int CELL = Tap1Elem<T>::CELL;
  T(*tile)[66] = reinterpret_cast<T(*)[66]>(lds);
  const int t0 = bx * 64, c0 = by * 64;
  const int P = W + 1, H1 = H + 1;
  {
    const int tx = threadIdx.x & 63, cy = threadIdx.x >> 6;
    const int t = t0 + tx;
    const int prow = t / P, col = t - prow * P;
    const int n = (prow - 1) / H1, h = (prow - 1) - n * H1;
    const bool ok = t < TS && prow >= 1 && n < N && h < H && col < W;
    const size_t at = ok ? ((size_t)n * C * H + h) * W + col : 0;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int c = c0 + cy + 4 * i;
      tile[cy + 4 * i][tx] = (ok && c < C) ? x[at + (size_t)c * H * W] : T{};
    }
  }
  __syncthreads();
  constexpr int CPT = 64 / CELL;
#pragma unroll
  for (int i = 0; i < CPT * 64 / 256; ++i) {
    const int item = threadIdx.x + 256 * i, cell = item % CPT, tl = item / CPT;
    const int t = t0 + tl, c = c0 + CELL * cell;
    if (t < TS && c < Cs) {
      __attribute__((aligned(16))) T v[CELL];
#pragma unroll
      for (int e = 0; e < CELL; ++e) v[e] = tile[CELL * cell + e][tl];
      *reinterpret_cast<uintx4_t*>(xr + (size_t)t * Cs + c) = *reinterpret_cast<const uintx4_t*>(v);
    }
  }
}

// Both operands in one launch, the first blocks the positions', the others the weights', through LDS (tap1d_weights_block): two launches, and weights
// gathered element by element, took 7 us more (512 channels over 7 x 7, 20 images 33.5 -> 26.5 us; 256 channels over 8 x 8, 64 images 27.5 -> 22.9).
template <typename T>
__global__ void __launch_bounds__(256)
tap2d_operands_kernel(const T* __restrict__ x, T* __restrict__ xr, int C, int H, int W, int N, int TS, int Cs, int tblocks, int rblocks,
                      const T* __restrict__ w, uintx4_t* __restrict__ wf, Tap1Weights p) {
  extern __shared__ uintx4_t t1_operands[];
  const int b = blockIdx.x;
  if (b < rblocks) tap2d_rows_block(x, xr, C, H, W, N, TS, Cs, b % tblocks, b / tblocks, t1_operands);
  else tap1d_weights_block(w, wf, p, b - rblocks, reinterpret_cast<T*>(t1_operands));
}

// ---- host side ---------------------------------------------------------------------------
struct Tap1Plan {
  Tap1Params p;
  Tap1Weights w;
  int SS, DT, NB;
  size_t rows_bytes, w_bytes, lds_bytes;
  int C, H, T;           // of the source tensor, for the rows pass
};

// channels of the channels-last rows: the count padded to one the 16-bit convolution kernels are compiled for (the fp32 ones take
// any whole chunk).  Compiled for every 32 up to 256, in 16-bit storage also for every 64 up to 512.  Before, 16-bit layers of more than
// 256 channels ran on the general kernels (us, 320 -> 320 channels, 21 taps over 4 x 1200 frames, forward / backward / filter gradient
// 76.7 / 77.4 / 417 -> 38.0 / 38.3 / 56, stride 2 363 / 247 / 216 -> 34.2 / 31.2 / 46), and 200 channels as 256 (3 x 1300 frames 31.9 -> 24.7).
int tap1d_cs(int C, int esz) {
  if (esz == 4) {
    for (int c : {32, 64, 96, 128, 256})
      if (C <= c) return c;
    return C <= 512 ? (C + 31) / 32 * 32 : 0;
  }
  return C <= 256 ? (C + 31) / 32 * 32 : C <= 512 ? (C + 63) / 64 * 64 : 0;
}

int t1_mtiles(int Mo, int NB) { return (Mo + 32 * t1_wm(NB) - 1) / (32 * t1_wm(NB)); }

// taps per unrolled group: so that its stages are a multiple of four
int dt_of(int KS) { return KS % 4 != 0 ? (KS == 2 ? 8 : 2) : KS >= 12 ? 1 : KS == 8 ? 2 : 4; }

// bwd = false: forward; true: backward-data.
bool tap1d_plan(const ConvGeom& g, bool bwd, Tap1Plan* pl) {
  constexpr int esz = 2;
  if (g.KH != 1 || g.py != 0 || g.sy != 1 || g.dlx != 1 || g.groups != 1) return false;
  if (g.KW < 2 || g.KW > 32 || (g.sx != 1 && g.sx != 2)) return false;
  if (g.OH != g.H || (long long)g.N * g.H > 65535) return false;
  const int Cc = bwd ? g.K : g.C, Mo = bwd ? g.C : g.K;
  // contraction channels padded to a count the kernel is compiled for
  const int Cs = tap1d_cs(Cc, esz);
  if (!Cs || Cc < 16) return false;
  const int KS = Cs / 16, DT = dt_of(KS);
  Tap1Params& p = pl->p;
  Tap1Weights& w = pl->w;
  std::memset(&p, 0, sizeof p);
  std::memset(&w, 0, sizeof w);
  p.rows = g.N * g.H; p.H = g.H;
  p.Cs = Cs; p.KS = KS; p.Mo = Mo;
  int soff[2] = {0, 0};
  if (!bwd) {
    pl->SS = g.sx; p.nph = 1;
    p.TS = g.W; p.TOu = g.OW;
    p.nreal[0] = g.KW; soff[0] = -g.px;
    for (int i = 0; i < g.KW; ++i) w.tapj[i] = (signed char)i;
  } else if (g.sx == 1) {
    pl->SS = 1; p.nph = 1;
    p.TS = g.OW; p.TOu = g.W;
    p.nreal[0] = g.KW; soff[0] = g.px - (g.KW - 1);
    for (int i = 0; i < g.KW; ++i) w.tapj[i] = (signed char)(g.KW - 1 - i);
  } else {
    // u = 2 v + q takes the taps j = jq + 2 i' with jq = (q + px) & 1, from dy[v + (q + px - jq) / 2 - i']
    pl->SS = 1; p.nph = 2;
    p.TS = g.OW; p.TOu = g.W;
    for (int q = 0; q < 2; ++q) {
      const int jq = (q + g.px) & 1;
      p.nreal[q] = (g.KW - jq + 1) / 2;
      if (p.nreal[q] < 1) return false;
      soff[q] = (q + g.px - jq) / 2 - (p.nreal[q] - 1);
    }
  }
  p.TO = (p.TOu + p.nph - 1) / p.nph;
  int stored = 0;
  for (int q = 0; q < p.nph; ++q) {
    p.ntaps[q] = (p.nreal[q] + DT - 1) / DT * DT;
    if (bwd && g.sx == 2) {
      const int jq = (q + g.px) & 1;
      for (int i = 0; i < p.ntaps[q]; ++i) w.tapj[stored + i] = (signed char)(i < p.nreal[q] ? jq + 2 * (p.nreal[q] - 1 - i) : -1);
    } else {
      for (int i = p.nreal[q]; i < p.ntaps[q]; ++i) w.tapj[stored + i] = -1;
    }
    stored += p.ntaps[q];
  }
  if (stored > T1_MAXTAPS) return false;
  p.taps_total = stored;
  p.smin = p.nph == 2 ? std::min(soff[0], soff[1]) : soff[0];
  int span = 0;
  for (int q = 0; q < p.nph; ++q) {
    p.d0[q] = soff[q] - p.smin;
    span = std::max(span, p.d0[q] + p.nreal[q]);
    if (p.ntaps[q] != p.nreal[q]) p.zcells = 2 * KS;
  }
  const int CPR = 2 * KS + 1;
  // three blocks of positions per wave; two, or one with half the channels, where the workgroups still fit the compute units at once, so that
  // more of the chip works on shorter tiles (us of a layer with its copies; three / two: 250 -> 250 channels over 7 x 1111 frames, 168
  // and 252 workgroups, 49.7 / 46.2, stride 2, 84 and 126, 45.8 / 41.6; but 12 x 900 frames, 240 and 360, 47.5 / 51.6.  Two / one, 21 taps:
  // 320 -> 320 over 12 x 254, 144 and 240 workgroups, 35.9 / 32.5, over 4 x 1200, stride 2, 37.1 / 34.2, backward 35.4 / 31.2, 250 -> 250 over 7 x
  // 1111, stride 2, backward 34.7 / 31.1; one where it is more than the compute units: 7 x 1111, 504 workgroups, 38.0 / 43.9)
  const auto wgs = [&](int nb) { return (long long)p.rows * ((p.TO + t1_positions(nb) - 1) / t1_positions(nb)) * t1_mtiles(Mo, nb); };
  pl->NB = 0;
  for (int nb = wgs(1) <= mfma_num_cus() ? 1 : wgs(2) <= mfma_num_cus() ? 2 : 3; nb >= 1 && !pl->NB; --nb) {
    const int tp = t1_positions(nb);
    if (pl->SS == 1) {
      p.SR = tp + span - 1;
      p.half = 0;
    } else {
      p.half = ((2 * (tp - 1) + span - 1) >> 1) + 1;
      p.SR = 2 * p.half;
    }
    pl->lds_bytes = (size_t)(((long long)p.SR * CPR + p.zcells + 63) / 64) * 1024;
    if (pl->lds_bytes <= 160 * 1024) pl->NB = nb;
  }
  if (!pl->NB) return false;
  p.ptiles = (p.TO + t1_positions(pl->NB) - 1) / t1_positions(pl->NB);
  p.mtiles = t1_mtiles(Mo, pl->NB);
  const long long rb = (long long)p.rows * p.TS * Cs * esz;
  const long long wb = (long long)p.mtiles * t1_wm(pl->NB) * stored * KS * 1024;
  const long long db = (long long)g.N * Mo * g.H * p.TOu * esz;
  if (rb >= (1ll << 31) || wb >= (1ll << 31) || db >= (1ll << 31)) return false;
  p.src_bytes = (unsigned)rb; p.w_bytes = (unsigned)wb; p.dst_bytes = (unsigned)db;
  pl->rows_bytes = ((size_t)rb + 255) & ~(size_t)255;
  pl->w_bytes = (size_t)wb;
  w.Mo = Mo; w.Cc = Cc; w.KS = KS; w.taps_total = stored; w.bwd = bwd ? 1 : 0;
  w.Cw = g.C; w.KW = g.KW; w.mblocks = p.mtiles * t1_wm(pl->NB);
  pl->DT = DT;
  pl->C = Cc; pl->H = g.H; pl->T = p.TS;
  return true;
}

template <typename T, int KS, int DT, int RW>
int launch_conv(const Tap1Plan& pl, const T* xr, const uintx4_t* wf, const float* bias, T* dst, hipStream_t s) {
  const dim3 grid((unsigned)(pl.p.rows * pl.p.ptiles), (unsigned)pl.p.mtiles);
  auto go = [&](auto kernel) {
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), pl.lds_bytes)) return -1;
    hipLaunchKernelGGL(kernel, grid, dim3(256), pl.lds_bytes, s, pl.p, xr, wf, bias, dst);
    return check_launch("conv2d (one-row windows)");
  };
  if (pl.NB == 1) {
    if (pl.p.nph == 2) return go(tap1d_conv_kernel<T, KS, DT, RW, 1, 2, 1>);
    return pl.SS == 2 ? go(tap1d_conv_kernel<T, KS, DT, RW, 2, 1, 1>) : go(tap1d_conv_kernel<T, KS, DT, RW, 1, 1, 1>);
  }
  if (pl.NB == 2) {
    if (pl.p.nph == 2) return go(tap1d_conv_kernel<T, KS, DT, RW, 1, 2, 2>);
    return pl.SS == 2 ? go(tap1d_conv_kernel<T, KS, DT, RW, 2, 1, 2>) : go(tap1d_conv_kernel<T, KS, DT, RW, 1, 1, 2>);
  }
  if (pl.p.nph == 2) return go(tap1d_conv_kernel<T, KS, DT, RW, 1, 2, 3>);
  if (pl.SS == 2) return go(tap1d_conv_kernel<T, KS, DT, RW, 2, 1, 3>);
  return go(tap1d_conv_kernel<T, KS, DT, RW, 1, 1, 3>);
}

template <typename T>
int run_conv(const ConvGeom& g, bool bwd, const void* src, const void* w, const float* bias, void* dst, hipStream_t s,
             void* ws, size_t ws_bytes) {
  Tap1Plan pl;
  if (!tap1d_plan(g, bwd, &pl)) return -1;
  if (!ws || ws_bytes < pl.rows_bytes + pl.w_bytes) return -1;
  T* xr = static_cast<T*>(ws);
  uintx4_t* wf = reinterpret_cast<uintx4_t*>(static_cast<char*>(ws) + pl.rows_bytes);
  {
    const dim3 rg = rows_grid(pl.T, pl.p.Cs, pl.p.rows);
    const size_t rblocks = (size_t)rg.x * rg.y * rg.z, wblocks = (size_t)pl.w.mblocks * pl.w.KS;
    const bool gather = wblocks <= T1_FEW_BLOCKS;
    const size_t blocks = rblocks + (gather ? (wblocks * pl.w.taps_total + 3) / 4 : wblocks);
    const size_t lds = std::max<size_t>(64 * 66 * sizeof(T), gather ? 0 : (544 * (size_t)pl.w.KW + 64) * sizeof(T));
    hipLaunchKernelGGL((tap1d_operands_kernel<T>), dim3((unsigned)blocks), dim3(256), lds, s, static_cast<const T*>(src), xr, pl.C, pl.H, pl.T,
                       pl.p.Cs, (int)rg.x, (int)rg.y, (int)rblocks, static_cast<const T*>(w), wf, pl.w, gather);
  }
  if (const int rc = check_launch("conv2d (one-row windows, operand passes)")) return rc;
  T* out = static_cast<T*>(dst);
  switch (pl.p.KS) {
    case 2: return launch_conv<T, 2, 8, 16>(pl, xr, wf, bias, out, s);
    case 4: return launch_conv<T, 4, 4, 16>(pl, xr, wf, bias, out, s);
    case 6: return launch_conv<T, 6, 2, 12>(pl, xr, wf, bias, out, s);
    case 8: return launch_conv<T, 8, 2, 16>(pl, xr, wf, bias, out, s);
    case 10: return launch_conv<T, 10, 2, 20>(pl, xr, wf, bias, out, s);
    case 12: return launch_conv<T, 12, 1, 12>(pl, xr, wf, bias, out, s);
    case 14: return launch_conv<T, 14, 2, 14>(pl, xr, wf, bias, out, s);
    case 16: return launch_conv<T, 16, 1, 16>(pl, xr, wf, bias, out, s);
    case 20: return launch_conv<T, 20, 1, 20>(pl, xr, wf, bias, out, s);
    case 24: return launch_conv<T, 24, 1, 24>(pl, xr, wf, bias, out, s);
    case 28: return launch_conv<T, 28, 1, 14>(pl, xr, wf, bias, out, s);
    default: return launch_conv<T, 32, 1, 16>(pl, xr, wf, bias, out, s);
  }
}

// ---- 3 x 3 windows over small planes -------------------------------------------------------
// The sequence of tap2d_conv_kernel: N planes of H x W, each row followed by one zero column (pitch P = W + 1), one
// zero row before every plane and one after the last: TS = (N (H + 1) + 1) P positions.  Result position o takes tap
// (r, s) from position o + (r - 1) P + (s - 1): the slab of a tile starts P + 1 positions before its first result and
// tap 3 r + s sits r P + s rows into it.  Backward-data is the same walk over dy with the taps in reverse order and
// the roles of the two channel counts exchanged.  (H + 1)(W + 1) / (H W) of the positions are computed: 1.15 for
// 14 x 14 planes, 1.31 for 7 x 7.
bool tap2d_plan(const ConvGeom& g, bool bwd, Tap1Plan* pl) {
  constexpr int esz = 2;
  if (g.KH != 3 || g.KW != 3 || g.sy != 1 || g.sx != 1 || g.py != 1 || g.px != 1 || g.dly != 1 || g.dlx != 1 || g.groups != 1)
    return false;
  const int Cc = bwd ? g.K : g.C, Mo = bwd ? g.C : g.K;
  // contraction channels padded to a count the two-dimensional kernel is compiled for
  int Cs = 0;
  for (int c : {128, 256, 512})
    if (!Cs && Cc <= c) Cs = c;
  if (!Cs || Cc <= Cs / 2) return false;
  const int KS = Cs / 16, DT = dt_of(KS);
  Tap1Params& p = pl->p;
  Tap1Weights& w = pl->w;
  std::memset(&p, 0, sizeof p);
  std::memset(&w, 0, sizeof w);
  const int P = g.W + 1;
  const long long ts = ((long long)g.N * (g.H + 1) + 1) * P;
  if (ts >= (1ll << 22) - 256) return false;
  p.rows = 1; p.H = 1;
  p.Cs = Cs; p.KS = KS; p.Mo = Mo;
  p.nph = 1;
  p.TS = (int)ts; p.TOu = p.TS; p.TO = p.TS;
  p.nreal[0] = 9;
  p.ntaps[0] = (9 + DT - 1) / DT * DT;
  p.taps_total = p.ntaps[0];
  p.d0[0] = 0;
  p.smin = -(P + 1);
  p.tw = 3; p.tpitch = P; p.pW = g.W; p.pH = g.H; p.pN = g.N;
  for (int i = 0; i < p.ntaps[0]; ++i) w.tapj[i] = (signed char)(i < 9 ? (bwd ? 8 - i : i) : -1);
  const int CPR = 2 * KS + 1;
  // three blocks of positions per wave; two where three would leave compute units without a workgroup
  // (7 x 7 x 512 at batch 64: 172 workgroups of three blocks 43.0 / 40.9 us, 256 of two 41.3 / 39.1); one with half the channels where those
  // fit the compute units at once (two / one: 20 images 36.2 / 33.1, 8 x 8 x 512, 12 images 36.1 / 32.3, 7 x 7 x 256, 40 images 24.6 / 22.8)
  pl->SS = 1; pl->DT = DT;
  const auto tiles = [&](int nb) { return (ts - P + t1_positions(nb) - 1) / t1_positions(nb); };      // (the last zero row holds no result)
  pl->NB = tiles(1) * t1_mtiles(Mo, 1) <= mfma_num_cus() ? 1 : tiles(3) * t1_mtiles(Mo, 3) < mfma_num_cus() ? 2 : 3;
  const int tp = t1_positions(pl->NB);
  p.SR = tp + 2 * P + 2;
  if (p.ntaps[0] != p.nreal[0]) p.zcells = 2 * KS;
  // the slab; the results are staged in the same memory afterwards
  pl->lds_bytes = std::max((size_t)(((long long)p.SR * CPR + p.zcells + 63) / 64) * 1024, (size_t)32 * t1_wm(pl->NB) * (tp + 4) * esz);
  if (pl->lds_bytes > 160 * 1024) return false;
  p.half = 0;
  p.ptiles = (int)tiles(pl->NB);
  p.mtiles = t1_mtiles(Mo, pl->NB);
  const long long rb = ts * Cs * esz;
  const long long wb = (long long)p.mtiles * t1_wm(pl->NB) * p.taps_total * KS * 1024;
  const long long db = (long long)g.N * Mo * g.H * g.W * esz;
  if (rb >= (1ll << 31) || wb >= (1ll << 31) || db >= (1ll << 31)) return false;
  p.src_bytes = (unsigned)rb; p.w_bytes = (unsigned)wb; p.dst_bytes = (unsigned)db;
  pl->rows_bytes = ((size_t)rb + 255) & ~(size_t)255;
  pl->w_bytes = (size_t)wb;
  w.Mo = Mo; w.Cc = Cc; w.KS = KS; w.taps_total = p.taps_total; w.bwd = bwd ? 1 : 0;
  w.Cw = g.C; w.KW = 9; w.mblocks = p.mtiles * t1_wm(pl->NB);
  pl->C = Cc; pl->H = g.H; pl->T = g.W;
  return true;
}

template <typename T, int KS, int DT, int RW>
int launch_conv2d(const Tap1Plan& pl, const T* xr, const uintx4_t* wf, const float* bias, T* dst, hipStream_t s) {
  const dim3 grid((unsigned)pl.p.ptiles, (unsigned)pl.p.mtiles);
  auto go = [&](auto kernel) {
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), pl.lds_bytes)) return -1;
    hipLaunchKernelGGL(kernel, grid, dim3(256), pl.lds_bytes, s, pl.p, xr, wf, bias, dst);
    return check_launch("conv2d (3x3 windows over stacked planes)");
  };
  if (pl.NB == 1) return go(tap2d_conv_kernel<T, KS, DT, RW, 1>);
  return pl.NB == 2 ? go(tap2d_conv_kernel<T, KS, DT, RW, 2>) : go(tap2d_conv_kernel<T, KS, DT, RW, 3>);
}

template <typename T>
int run_conv2d(const ConvGeom& g, bool bwd, const void* src, const void* w, const float* bias, void* dst, hipStream_t s,
               void* ws, size_t ws_bytes) {
  Tap1Plan pl;
  if (!tap2d_plan(g, bwd, &pl)) return -1;
  if (!ws || ws_bytes < pl.rows_bytes + pl.w_bytes) return -1;
  T* xr = static_cast<T*>(ws);
  uintx4_t* wf = reinterpret_cast<uintx4_t*>(static_cast<char*>(ws) + pl.rows_bytes);
  {
    const int tblocks = (pl.p.TS + 63) / 64, rblocks = tblocks * ((pl.p.Cs + 63) / 64), wblocks = pl.w.mblocks * pl.w.KS;
    const size_t lds = std::max<size_t>(64 * 66, 544 * (size_t)pl.w.KW + 64) * sizeof(T);
    hipLaunchKernelGGL(tap2d_operands_kernel<T>, dim3((unsigned)(rblocks + wblocks)), dim3(256), lds, s, static_cast<const T*>(src), xr, pl.C,
                       g.H, g.W, g.N, pl.p.TS, pl.p.Cs, tblocks, rblocks, static_cast<const T*>(w), wf, pl.w);
  }
  if (const int rc = check_launch("conv2d (3x3 windows over stacked planes, operand passes)")) return rc;
  T* out = static_cast<T*>(dst);
  switch (pl.p.KS) {
    case 8: return launch_conv2d<T, 8, 2, 16>(pl, xr, wf, bias, out, s);
    case 16: return launch_conv2d<T, 16, 1, 16>(pl, xr, wf, bias, out, s);
    default: return launch_conv2d<T, 32, 1, 16>(pl, xr, wf, bias, out, s);
  }
}

// ---- the filter gradient -------------------------------------------------------------------
//   dw[k][c][j] = sum over sequences and positions o of dy[k][o] x[c][o*s + j - p],  db[k] = sum dy[k][o]
// The contraction runs over positions, 16 per matrix instruction.  dy is read as it lies in
// memory (a lane's 8 consecutive positions of one filter are 16 contiguous bytes, fetched
// straight into registers a few steps ahead); x comes from the channels-last rows through LDS:
// a tap shifts whole slab rows, and transposing reads (ds_read_b64_tr_b16) hand every lane its
// 8 positions of one channel.  A workgroup (4 waves) owns 64 filters x 32 channels x every tap
// over a range of positions of one sequence (or several such ranges in turn); wave w owns the
// slots w TQ .. w TQ + TQ - 1 of both filter blocks, slot g being tap g for g < KW, the bias
// gradient (dy times a tile of ones) for g = KW and unused beyond: 2 x TQ accumulator blocks
// per wave (at most 192 registers, so they stay in the accumulator file), one slab fragment
// per two matrix instructions.
// The slab of a range (its positions and the window's reach, 32 channels) is copied to LDS by
// the loads themselves before the range's first step; rows are 6 cells apart for stride 1 and
// 5 for stride 2, which keeps the four rows of a transposing read on distinct banks.
// 16-bit rows of an odd length start on 2-byte boundaries every other row: such a fragment (ODD) is fetched from the
// 4-byte boundary below it with one word more, and shifted by the lane's 0 or 16 bits while the step before multiplies.
// Before, odd rows went to the kernels that widen their operands: the speech stack's training pass (three 21-tap layers,
// 250 channels, 7 sequences of 1111 frames, bf16) took 787 us, 484 of them in two such filter gradients; now 407 us.
// The workgroups' tiles go to the workspace as [range set][tile][slot][64 filters][32 channels]
// and tap1d_wgrad_reduce_kernel adds them in a fixed order into dw's memory order.
typedef short shortx4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4_t* lds_tr_t;

struct Tap1WParams {
  int rows, H;          // sequences, rows per image
  int OW, TS;           // positions of dy / of the source per sequence
  int Cs;               // channels of the channels-last source rows
  int K, C, KW, px;
  int tsplit, TL;       // ranges per sequence, positions per range (a multiple of 16)
  int units, upw;       // ranges over all sequences, ranges per workgroup
  int ktiles, ctiles;
  int SRW;              // slab rows
  unsigned src_bytes, dy_bytes;
};

template <typename T, int TQ, int SS, bool ODD>
__global__ void __launch_bounds__(256, 1)
tap1d_wgrad_kernel(Tap1WParams p, const T* __restrict__ xr, const T* __restrict__ dy, float* __restrict__ part) {
  extern __shared__ uintx4_t t1_slab[];
  constexpr int CELL = 8, ESZ = 2;
  constexpr int STEP = 2 * CELL;                // positions per step: a lane half holds CELL consecutive ones
  constexpr int RC = 32 / CELL;                 // cells of a slab row in use (32 channels)
  constexpr int PC = SS == 1 ? 6 : 5;           // cells per slab row
  constexpr int PE = PC * CELL;                 // the same in elements
  constexpr int RD = 4;                         // steps between a dy fragment's load and its use
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = blockIdx.x, tile = blockIdx.y;
  const int kt = tile / p.ctiles, ct = tile - kt * p.ctiles;
  const intx4_t xrs = pd_rsrc(xr, p.src_bytes);
  // (ODD: the buffer is whole words; the 2 bytes a word may reach beyond dy lie in dy's own first or last word)
  const unsigned dy_low = ODD ? (unsigned)(reinterpret_cast<uintptr_t>(dy) & 2u) : 0u;
  const __amdgpu_buffer_rsrc_t drs = make_rsrc(reinterpret_cast<const char*>(dy) - dy_low,
                                               ODD ? (p.dy_bytes + dy_low + 3u) & ~3u : p.dy_bytes);
  const unsigned slab_addr = pd_lds_addr(t1_slab);
  const int fr = lane & 31, fg = lane >> 5, fq = (lane >> 4) & 1, fs = lane & 15;

  floatx16 acc[2][TQ];
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int t = 0; t < TQ; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[a][t][r] = 0.f;
  // a tile of ones for the bias slot
  const uint32_t one = std::is_same<T, f16_t>::value ? 0x3c003c00u : 0x3f803f80u;
  const uintx4_t ones = {one, one, one, one};
  const int bias_slot = p.KW - wave * TQ;       // this wave's slot index of the bias gradient (outside 0 .. TQ - 1: none)

  // this lane's first (transposing) read of a step at the wave's first tap: row SS * (fs / 4) (+ 8 SS fg), channels
  // 16 fq + 4 (fs % 4) .. + 3
  const T* const slabT = reinterpret_cast<const T*>(t1_slab);
  const int blane = ((8 * fg + (fs >> 2)) * SS + wave * TQ) * PE + 16 * fq + 4 * (fs & 3);

  const int u0 = split * p.upw, u1 = min(u0 + p.upw, p.units);
  for (int u = u0; u < u1; ++u) {
    const int seq = u / p.tsplit, tr = u - seq * p.tsplit;
    const int t0 = tr * p.TL, oend = min(p.OW, t0 + p.TL);
    if (t0 >= oend) continue;
    const int nsteps = (oend - t0 + STEP - 1) / STEP;
    const int tailn = (oend - t0) % STEP, nwhole = nsteps - (tailn != 0);       // positions of a last, partial step (0: none); steps before it
    if (u != u0) __syncthreads();                // every wave is done with the previous slab
    // ---- slab: row R holds source position t0 * SS - px + R, channels 32 ct .. + 31
    {
      const int ncell = p.SRW * PC, ninstr = (ncell + 63) >> 6;
      const float inv = 1.0f / (float)PC;
      const int sp0 = t0 * SS - p.px;
      for (int ii = wave; ii < ninstr; ii += 4) {
        const int L = ii * 64 + lane;
        int c;
        const int R = fast_div(L, PC, inv, &c);
        const int sp = sp0 + R;
        int voff = T1_OOB;
        if (R < p.SRW && c < RC && (unsigned)sp < (unsigned)p.TS) voff = ((seq * p.TS + sp) * p.Cs + ct * 32 + CELL * c) * ESZ;
        pd_load_lds(xrs, slab_addr + ii * 1024, voff, 0);
      }
    }
    // ---- dy: filters kt * 64 + 32 a + fr, positions t0 + STEP step + CELL fg .. + CELL - 1
    const int n = seq / p.H, h = seq - n * p.H;
    int aoff[2];
    unsigned ashift[2] = {0u, 0u};
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int k = kt * 64 + a * 32 + fr;
      aoff[a] = k < p.K ? ((((n * p.K + k) * p.H + h) * p.OW) + t0 + CELL * fg) * ESZ : T1_OOB;
      if (ODD && k < p.K) {
        aoff[a] += dy_low;
        ashift[a] = (unsigned)(aoff[a] & 2) * 8u;
        aoff[a] &= ~3;
      }
    }
    // the partial step's mask: elements at and past oend are zero
    uint32_t tmask[4];
    {
      const int cnt = tailn ? tailn - CELL * fg : CELL;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        tmask[d] = cnt >= 2 * d + 2 ? 0xffffffffu : cnt == 2 * d + 1 ? 0x0000ffffu : 0u;
    }
    uintx4_t aq[RD + 1][2];                       // (the last: the partial step's)
    uint32_t ax[ODD ? RD + 1 : 1][2];             // ODD: the word behind each fragment
    auto dy_load = [&](int i, int a, int st) __attribute__((always_inline)) {
      const int off = st < nsteps ? aoff[a] : T1_OOB;
      aq[i][a] = __builtin_amdgcn_raw_buffer_load_b128(drs, off, st * 32, 0);
      if constexpr (ODD) ax[i][a] = __builtin_amdgcn_raw_buffer_load_b32(drs, off, st * 32 + 16, 0);
    };
    auto dy_take = [&](int i, int a) __attribute__((always_inline)) {
      uintx4_t v = aq[i][a];
      if constexpr (ODD) {
        const uint32_t w4 = ax[i][a], sh = ashift[a];
        v = uintx4_t{__builtin_amdgcn_alignbit(v.y, v.x, sh), __builtin_amdgcn_alignbit(v.z, v.y, sh),
                     __builtin_amdgcn_alignbit(v.w, v.z, sh), __builtin_amdgcn_alignbit(w4, v.w, sh)};
      }
      return v;
    };
#pragma unroll
    for (int a = 0; a < 2; ++a) {
#pragma unroll
      for (int i = 0; i < RD; ++i) dy_load(i, a, i);
      if (tailn) dy_load(RD, a, nwhole);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();                              // the slab has landed for every wave

    // the slab fragment of slot t + 1 is read while slot t is multiplied (the first slot of a step behind the last
    // of the step before)
    auto bread = [&](const T* at) __attribute__((always_inline)) {
      const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)at);
      const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + 4 * SS * PE));
      const uintx2_t l2 = __builtin_bit_cast(uintx2_t, lo), h2 = __builtin_bit_cast(uintx2_t, hi);
      return uintx4_t{l2.x, l2.y, h2.x, h2.y};
    };
    uintx4_t bnext = bread(slabT + blane);
#define T1W_STEP(I)                                                                                       \
  {                                                                                                       \
    const int st = st0 + I;                                                                               \
    if (st < nwhole) {                                                                                    \
      const uintx4_t a0 = dy_take(I, 0), a1 = dy_take(I, 1);                                              \
      _Pragma("unroll") for (int a = 0; a < 2; ++a) dy_load(I, a, st + RD);                               \
      const T* bp = slabT + blane + st * (STEP * SS * PE);                                                \
      _Pragma("unroll") for (int t = 0; t < TQ; ++t) {                                                    \
        uintx4_t b4 = bnext;                                                                              \
        bnext = bread(t + 1 < TQ ? bp + (t + 1) * PE : bp + STEP * SS * PE);                              \
        if (t == bias_slot) b4 = ones;                                                                    \
        tap1d_mma(acc[0][t], a0, b4, static_cast<const T*>(nullptr));                                     \
        tap1d_mma(acc[1][t], a1, b4, static_cast<const T*>(nullptr));                                     \
        __builtin_amdgcn_sched_barrier(0);                                                                \
      }                                                                                                   \
    }                                                                                                     \
  }
    for (int st0 = 0; st0 < nwhole; st0 += RD) {
      T1W_STEP(0) T1W_STEP(1) T1W_STEP(2) T1W_STEP(3)
    }
#undef T1W_STEP
    // The partial step: rows past the range count for nothing either, as they are other taps' positions within it and need not be finite.
    // (In the loop the rows' masks took up to 1.19 of the time, a branch there up to 2.1.)
    if (tailn) {
      uintx4_t a0 = dy_take(RD, 0), a1 = dy_take(RD, 1);
      const T* bp = slabT + blane + nwhole * (STEP * SS * PE);
#pragma unroll
      for (int d = 0; d < 4; ++d) { a0[d] &= tmask[d]; a1[d] &= tmask[d]; }
#pragma unroll
      for (int t = 0; t < TQ; ++t) {
        uintx4_t b4 = bnext;
        if (t + 1 < TQ) bnext = bread(bp + (t + 1) * PE);
#pragma unroll
        for (int d = 0; d < 4; ++d) b4[d] &= tmask[d];
        if (t == bias_slot) b4 = ones;
        tap1d_mma(acc[0][t], a0, b4, static_cast<const T*>(nullptr));
        tap1d_mma(acc[1][t], a1, b4, static_cast<const T*>(nullptr));
      }
    }
  }

  // ---- the tile: element r of block (a, t): filter 32 a + 8 (r / 4) + 4 fg + r % 4, channel fr
  float* out = part + ((size_t)(split * (p.ktiles * p.ctiles) + tile) * (4 * TQ) + wave * TQ) * 2048;
#pragma unroll
  for (int t = 0; t < TQ; ++t) {
    if (wave * TQ + t > p.KW) continue;          // an unused slot
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int kl = a * 32 + (r >> 2) * 8 + fg * 4 + (r & 3);
        out[t * 2048 + kl * 32 + fr] = acc[a][t][r];
      }
  }
}

// The same in fp32: dy and the rows in three bf16 parts (split_f32.h), six products in place of one, two accumulators.
// A workgroup owns one of the tile's two blocks of 32 filters (TQ slots per wave: 32 TQ registers of accumulators, and two workgroups
// still share a compute unit, so that one multiplies while the other brings in its slab).  The slab's rows are taken apart when
// they go to LDS, [row][part][32 channels] - 12 cells a row, 14 for stride 2, which keeps the four rows of a transposing read on
// distinct banks - and dy in registers, by each wave for itself (44 vector instructions to 6 TQ products).
// Measured, us with the sum of the tiles (before: v_mfma_f32_32x32x2_f32, 0.7 of its pipe), 21 taps: 250 -> 250 channels, 16 x 1500 frames
// 592 -> 363, stride 2 315 -> 197, 80 -> 250 318 -> 163; error in the 2-norm 9.8e-7 -> 3.4e-7.
constexpr int t1ws_cells(int SS) { return SS == 1 ? 12 : 14; }

template <int TQ, int SS>
__global__ void __launch_bounds__(256, 2)
tap1d_wgrad_split_kernel(Tap1WParams p, const float* __restrict__ xr, const float* __restrict__ dy, float* __restrict__ part) {
  extern __shared__ uintx4_t t1_slab[];
  constexpr int ROW = t1ws_cells(SS) * 16;      // bytes
  constexpr int RD = 2;                         // steps between a dy fragment's load and its use
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int split = blockIdx.x, tile = blockIdx.y >> 1, fb = blockIdx.y & 1;
  const int kt = tile / p.ctiles, ct = tile - kt * p.ctiles;
  const __amdgpu_buffer_rsrc_t xrs = make_rsrc(xr, p.src_bytes), drs = make_rsrc(dy, p.dy_bytes);
  const int fr = lane & 31, fg = lane >> 5, fq = (lane >> 4) & 1, fs = lane & 15;
  if (kt * 64 + fb * 32 >= p.K) return;         // (nobody reads that half of the tile)
  const int k = kt * 64 + fb * 32 + fr;

  floatx16 big[TQ], small[TQ];
#pragma unroll
  for (int t = 0; t < TQ; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) big[t][r] = small[t][r] = 0.f;
  const int bias_slot = p.KW - wave * TQ;
  char* const slab = reinterpret_cast<char*>(t1_slab);
  // this lane's first read of a step at the wave's first tap: row SS * (fs / 4) (+ 8 SS fg), channels 16 fq + 4 (fs % 4) .. + 3
  const int blane = ((8 * fg + (fs >> 2)) * SS + wave * TQ) * ROW + 32 * fq + 8 * (fs & 3);

  const int u0 = split * p.upw, u1 = min(u0 + p.upw, p.units);
  for (int u = u0; u < u1; ++u) {
    const int seq = u / p.tsplit, tr = u - seq * p.tsplit;
    const int t0 = tr * p.TL, oend = min(p.OW, t0 + p.TL);
    if (t0 >= oend) continue;
    const int nsteps = (oend - t0 + 15) / 16, tailn = (oend - t0) % 16;
    const int n = seq / p.H, h = seq - n * p.H;
    const int aoff = k < p.K ? ((((n * p.K + k) * p.H + h) * p.OW) + t0 + 8 * fg) * 4 : T1_OOB;
    uintx4_t raw[RD][2];
    auto dy_load = [&](int i, int st) __attribute__((always_inline)) {
      const int off = st < nsteps ? aoff : T1_OOB;
      raw[i][0] = __builtin_amdgcn_raw_buffer_load_b128(drs, off, st * 64, 0);
      raw[i][1] = __builtin_amdgcn_raw_buffer_load_b128(drs, off, st * 64 + 16, 0);
    };
#pragma unroll
    for (int i = 0; i < RD; ++i) dy_load(i, i);
    if (u != u0) __syncthreads();                // every wave is done with the previous slab
    // ---- slab: row R holds source position t0 * SS - px + R, channels 32 ct .. + 31; a thread takes 8 channels of a row
    for (int i = tid; i < p.SRW * 4; i += 256) {
      const int R = i >> 2, c = i & 3, sp = t0 * SS - p.px + R;
      const int off = (unsigned)sp < (unsigned)p.TS ? ((seq * p.TS + sp) * p.Cs + ct * 32 + 8 * c) * 4 : T1_OOB;
      const uintx4_t v0 = __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 0, 0), v1 = __builtin_amdgcn_raw_buffer_load_b128(xrs, off, 16, 0);
      const Split2 s0 = split2(__uint_as_float(v0.x), __uint_as_float(v0.y)), s1 = split2(__uint_as_float(v0.z), __uint_as_float(v0.w));
      const Split2 s2 = split2(__uint_as_float(v1.x), __uint_as_float(v1.y)), s3 = split2(__uint_as_float(v1.z), __uint_as_float(v1.w));
      char* const at = slab + R * ROW + 16 * c;
      *reinterpret_cast<uintx4_t*>(at) = uintx4_t{s0.h, s1.h, s2.h, s3.h};
      *reinterpret_cast<uintx4_t*>(at + 64) = uintx4_t{s0.m, s1.m, s2.m, s3.m};
      *reinterpret_cast<uintx4_t*>(at + 128) = uintx4_t{s0.l, s1.l, s2.l, s3.l};
    }
    __syncthreads();
    const char* bp = slab + blane;
    for (int st0 = 0; st0 < nsteps; st0 += RD) {
#pragma unroll
      for (int i = 0; i < RD; ++i) {
        const int st = st0 + i;                  // (a step past the last: dy reads zero there, the rows are those of the last)
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(raw[i][e >> 2][e & 3]);
        if (tailn && st == nsteps - 1) {
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = 8 * fg + e < tailn ? v[e] : 0.f;
        }
        uintx4_t a[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const Split2 s = split2(v[2 * e], v[2 * e + 1]);
          a[0][e] = s.h; a[1][e] = s.m; a[2][e] = s.l;
        }
        dy_load(i, st + RD);
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
          uintx4_t b[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            const char* const at = bp + t * ROW + 64 * q;
            const uintx2_t lo = __builtin_bit_cast(uintx2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)at));
            const uintx2_t hi = __builtin_bit_cast(uintx2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + 4 * SS * ROW)));
            b[q] = uintx4_t{lo.x, lo.y, hi.x, hi.y};
          }
          if (t == bias_slot) {                  // dy times ones
            b[0] = uintx4_t{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};
            b[1] = b[2] = uintx4_t{0u, 0u, 0u, 0u};
          }
          split_mma(big[t], small[t], a, b);
        }
        if (st + 1 < nsteps) bp += 16 * SS * ROW;
      }
    }
  }

  bool bad = false;
#pragma unroll
  for (int t = 0; t < TQ; ++t)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      big[t][r] += small[t][r];
      bad |= split_redo(big[t][r]);
    }
  if (__builtin_amdgcn_ballot_w64(bad)) {          // once more with the operands as they are
#pragma unroll
    for (int t = 0; t < TQ; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) big[t][r] = 0.f;
#pragma unroll 1
    for (int u = u0; u < u1; ++u) {
      const int seq = u / p.tsplit, t0 = (u - seq * p.tsplit) * p.TL, oend = min(p.OW, t0 + p.TL);
      const int n = seq / p.H, h = seq - n * p.H;
#pragma unroll 1
      for (int o = t0 + fg; o < oend + fg; o += 2) {
        const bool in = o < oend;
        const float a = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(drs, in && k < p.K ? (((n * p.K + k) * p.H + h) * p.OW + o) * 4 : T1_OOB, 0, 0));
#pragma unroll
        for (int t = 0; t < TQ; ++t) {
          const int sp = o * SS - p.px + wave * TQ + t;
          const float x = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
              xrs, in && (unsigned)sp < (unsigned)p.TS ? ((seq * p.TS + sp) * p.Cs + ct * 32 + fr) * 4 : T1_OOB, 0, 0));
          big[t] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, t == bias_slot ? 1.f : x, big[t], 0, 0, 0);
        }
      }
    }
  }

  // ---- the tile: element r of slot t: filter 32 fb + 8 (r / 4) + 4 fg + r % 4, channel fr
  float* out = part + ((size_t)(split * (p.ktiles * p.ctiles) + tile) * (4 * TQ) + wave * TQ) * 2048;
#pragma unroll
  for (int t = 0; t < TQ; ++t) {
    if (wave * TQ + t > p.KW) continue;          // an unused slot
#pragma unroll
    for (int r = 0; r < 16; ++r) out[t * 2048 + (fb * 32 + (r >> 2) * 8 + fg * 4 + (r & 3)) * 32 + fr] = big[t][r];
  }
}

// dw[k][c][j] and db[k] from the tiles of nsplit range sets, added in the order of the sets.
// Slot g of a tile: tap g for g < KW, the bias gradient for g = KW.
__global__ void __launch_bounds__(256)
tap1d_wgrad_reduce_kernel(const float* __restrict__ part, int nsplit, int tiles, int ctiles, int slots, int K, int C, int KW,
                            float* __restrict__ dw, float* __restrict__ db) {
  const int e = blockIdx.x * 256 + threadIdx.x;   // element of a slot: filter e / 32, channel e % 32
  const int g = blockIdx.y, tile = blockIdx.z;
  const int kt = tile / ctiles, ct = tile - kt * ctiles;
  const int k = kt * 64 + (e >> 5), c = ct * 32 + (e & 31);
  const bool is_bias = g == KW;
  if (k >= K) return;
  if (is_bias ? (ct != 0 || (e & 31) != 0 || !db) : (c >= C || !dw)) return;
  const size_t stride = (size_t)tiles * slots * 2048;
  const float* src = part + ((size_t)tile * slots + g) * 2048 + e;
  float sum = 0.f;
  int s = 0;
  for (; s + 4 <= nsplit; s += 4) {
    const float v0 = src[(size_t)s * stride], v1 = src[(size_t)(s + 1) * stride], v2 = src[(size_t)(s + 2) * stride],
                v3 = src[(size_t)(s + 3) * stride];
    sum += v0; sum += v1; sum += v2; sum += v3;
  }
  for (; s < nsplit; ++s) sum += src[(size_t)s * stride];
  if (is_bias) db[k] = sum;
  else dw[((size_t)k * C + c) * KW + g] = sum;
}

struct Tap1WPlan {
  Tap1WParams p;
  int TQ, SS, nsplit;
  bool odd;             // 16-bit rows of dy that start on 2-byte boundaries
  size_t rows_bytes, part_bytes, lds_bytes;
};

bool tap1d_wgrad_plan(const ConvGeom& g, int esz, Tap1WPlan* pl) {
  if (g.KH != 1 || g.py != 0 || g.sy != 1 || g.dlx != 1 || g.groups != 1) return false;
  if (g.KW < 6 || g.KW > 23 || (g.sx != 1 && g.sx != 2)) return false;
  if (g.OH != g.H || (long long)g.N * g.H > 65535 || g.C < 16 || g.K < 32) return false;
  Tap1WParams& p = pl->p;
  std::memset(&p, 0, sizeof p);
  const int TQ = (g.KW + 1 + 3) / 4;            // KW taps and the bias gradient over four waves
  pl->TQ = TQ; pl->SS = g.sx;
  pl->odd = esz == 2 && g.OW % 2 != 0;
  p.rows = g.N * g.H; p.H = g.H; p.OW = g.OW; p.TS = g.W;
  p.Cs = tap1d_cs(g.C, esz);
  if (!p.Cs) return false;
  p.K = g.K; p.C = g.C; p.KW = g.KW; p.px = g.px;
  p.ktiles = (g.K + 63) / 64; p.ctiles = (g.C + 31) / 32;
  const long long rb = (long long)p.rows * p.TS * p.Cs * esz;
  const long long yb = (long long)g.N * g.K * g.H * g.OW * esz;
  if (rb >= (1ll << 31) || yb >= (1ll << 31)) return false;
  const int tiles = p.ktiles * p.ctiles;
  if (esz == 4 && tiles > 65535 / 2) return false;      // (two workgroups of the grid's second dimension to a tile)
  // 16-bit storage over more than 256 channels, the general kernels / here: 320 channels, 21 taps over 60 frames to 32 filters (13 million multiply-adds)
  // 10.8 / 16.9, 384 to 80 over 200 (129 million) 16.3 / 21.5, over 4 x 300 (774) 52 / 29, 512 to 512, 11 taps over 60 (173) 20 / 27, over 200 (577) 32 /
  // 30, 320 to 320 over 200 (225) 22.3 / 22.0, to 32 over 4 x 300 (135) 24 / 20.
  if (esz == 2 && g.C > 256) {
    const long long pos = (long long)p.rows * g.OW;
    if (pos < 64 || pos * g.C * g.K * g.KW < (pos >= 512 ? 100000000 : 200000000)) return false;
  }
  // fp32 over more than 256 channels: from 800 million multiply-adds on; below, the general kernel's two launches are ahead of the copy of the
  // rows, the tiles and their sums.  us general / here: 320 channels, 21 taps over 1 x 200 frames to 80 filters (110 million) 15 / 36, to 320 (430) 40 / 43,
  // over 1 x 800 (1700) 70 / 64, 4 x 700 183 / 104.  Of 840 random layers 1 % behind the better one in the geometric mean, at worst 1.38.
  if (esz == 4 && g.C > 256 && (long long)p.rows * g.OW * g.C * g.K * g.KW < 800000000) return false;
  const int PC = esz == 2 ? (g.sx == 1 ? 6 : 5) : t1ws_cells(g.sx), most = esz == 2 ? 150 * 1024 : 80 * 1024;
  const int cus = mfma_num_cus();
  // ranges of ceil(OW / tsplit) positions; false: the slab of one does not fit in LDS
  auto split = [&](int tsplit) {
    p.TL = ((g.OW + tsplit - 1) / tsplit + 15) / 16 * 16;
    p.SRW = (p.TL - 1) * g.sx + 4 * TQ;
    pl->lds_bytes = (size_t)(((long long)p.SRW * PC + 63) / 64) * 1024;
    p.tsplit = (g.OW + p.TL - 1) / p.TL;
    p.units = p.rows * p.tsplit;
    return pl->lds_bytes <= (size_t)most;
  };
  if (esz == 4) {
    // fp32 is bound by the matrix pipe: enough workgroups for the chip (a tile is two of them, and two share a compute unit), rather
    // with a last round that is half full than of twice the length ...
    const int want = (cus + tiles - 1) / tiles;
    auto fill = [&](auto fits) {
      for (int tsplit = std::max(1, (want + p.rows - 1) / p.rows); !fits(tsplit); ++tsplit)
        if (p.TL <= 16) return 0;
      p.upw = std::max(1, p.units / want);
      return (p.units + p.upw - 1) / p.upw;
    };
    // ... but no more partial tiles than with a slab of 9 cells a row and 150 KB, the fp32 instruction's kernel: the parts' smaller one makes
    // ranges shorter, as many of them per workgroup then up to twice the tiles, and geometries that fit the static buffer no longer did
    // (250 -> 250 channels over 4 x 1100 frames, 9 taps 31.5 -> 42.3 MB; 80 -> 250 over 11 x 1134, 15 taps 39.4 -> 56.7).
    const int most_splits = fill([&](int tsplit) {
      split(tsplit);
      return ((long long)p.SRW * 9 + 63) / 64 * 1024 <= 150 * 1024;
    });
    const int splits = fill(split);
    if (!most_splits || !splits) return false;
    // Where it would be more, the range's length and ranges per workgroup with the least estimated time under that bound: 1.8 us and
    // 0.021 per four taps and position for a range, 0.7 of it where a workgroup has its compute unit for itself, rounds of 512
    // workgroups, 0.01 per four taps and tile and 0.11 for each set of partial tiles.  Fitted to 5900 times of 220 random geometries (1 to 24 x
    // 100 to 2200 frames, 16 to 320 channels, 7 to 21 taps); of 150 others those that the bound reaches take 0.86 to 1.00 of their time
    // without it (17 x 39 -> 250 channels, 1993 frames, 15 taps 120 -> 104 us; 2 x 250 -> 256, 1624 frames, 21 taps 91 -> 81).
    if (splits > most_splits) {
      double best = 1e30;
      int best_split = 0, best_upw = 0;
      const double set = 0.01 * TQ * tiles + 0.11;
      for (int tsplit = 1;; tsplit += std::max(1, tsplit / 4)) {
        if (split(tsplit)) {
          const double each = 1.8 + 0.021 * TQ * p.TL;
          const int even = (int)(p.units / std::max(1.0, std::sqrt(p.units * set / each)));
          for (int n : {most_splits, cus / tiles, cus / tiles / 2, even}) {
            const int upw = (p.units - 1) / std::max(1, std::min(n, most_splits)) + 1, ns = (p.units + upw - 1) / upw;
            const int wgs = 2 * tiles * ns, rounds = (wgs + 2 * cus - 1) / (2 * cus);
            const double cost = rounds * upw * each * (wgs <= cus ? 0.7 : 1.0) + ns * set;
            if (cost < best) { best = cost; best_split = tsplit; best_upw = upw; }
          }
        }
        if (p.TL <= 16) break;
      }
      if (!best_split) return false;
      split(best_split);
      p.upw = best_upw;
    }
  } else {
    // 16-bit storage is bound by what surrounds the products.  The length of a range and the ranges per workgroup with the least
    // estimated time: a workgroup's ranges follow each other, about 1 us each and 0.012 + 0.002 per four taps for a position; its partial
    // tiles (TQ times 32 KB, written and read) take 0.013 us per four taps of the whole, and the reduction 0.05 for each that it adds.
    // No more workgroups than compute units, but for windows of up to 11 taps, whose registers leave room for two on a unit:
    // up to twice as many with one range each, of which those that share a unit take 1.2 times as long.  (Constants fitted to
    // 14292 times of 1175 random geometries; taking the estimate's choice costs 1 % over the best of those measured, at worst 15.
    // Filling the chip whatever the partial tiles cost, as before, 19 %, at worst 126: 16 -> 64 channels over 31 x 193 frames, 7 taps,
    // 27 -> 14 us; 64 -> 40 over 4 x 1017, 15 taps, stride 2, 26 -> 12; 250 -> 250 over 7 x 1111, 21 taps, 56 -> 55.)
    double best = 1e30;
    int best_split = 0, best_upw = 0;
    const double set = 0.013 * TQ * tiles + 0.05;
    for (int tsplit = 1;; tsplit += std::max(1, tsplit / 4)) {
      const bool fits = split(tsplit);
      const double each = 1.0 + p.TL * (0.012 + 0.002 * TQ);
      auto consider = [&](int upw, double slower) {
        const double cost = (double)((p.units + upw - 1) / upw) * set + upw * each * slower;
        if (cost < best) { best = cost; best_split = tsplit; best_upw = upw; }
      };
      if (fits) {
        const int least = (p.units - 1) / std::max(1, cus / tiles) + 1;
        const int upw = (int)std::sqrt(p.units * set / each);
        consider(std::max(least, upw), 1.0);
        consider(std::max(least, upw + 1), 1.0);
        if (TQ <= 3 && pl->lds_bytes <= 80 * 1024 && least == 2 && (long long)p.units * tiles < 2 * cus) consider(1, 1.2);
      }
      if (p.TL <= 16) break;
    }
    if (!best_split) return false;
    split(best_split);
    p.upw = best_upw;
  }
  pl->nsplit = (p.units + p.upw - 1) / p.upw;
  p.src_bytes = (unsigned)rb; p.dy_bytes = (unsigned)yb;
  pl->rows_bytes = ((size_t)rb + 255) & ~(size_t)255;
  pl->part_bytes = (size_t)pl->nsplit * tiles * (4 * TQ) * 2048 * sizeof(float);
  return true;
}

template <typename T, int TQ>
int launch_wgrad(const Tap1WPlan& pl, const T* xr, const T* dy, float* part, hipStream_t s) {
  const dim3 grid((unsigned)pl.nsplit, (unsigned)(pl.p.ktiles * pl.p.ctiles));
  auto go = [&](auto kernel) {
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), pl.lds_bytes)) return -1;
    hipLaunchKernelGGL(kernel, grid, dim3(256), pl.lds_bytes, s, pl.p, xr, dy, part);
    return check_launch("conv2d_bwd_filter (one-row windows)");
  };
  if constexpr (sizeof(T) == 4) {
    const dim3 halves(grid.x, 2 * grid.y);
    auto go32 = [&](auto kernel) {
      if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), pl.lds_bytes)) return -1;
      hipLaunchKernelGGL(kernel, halves, dim3(256), pl.lds_bytes, s, pl.p, xr, dy, part);
      return check_launch("conv2d_bwd_filter (one-row windows, fp32 in three parts)");
    };
    return pl.SS == 2 ? go32(tap1d_wgrad_split_kernel<TQ, 2>) : go32(tap1d_wgrad_split_kernel<TQ, 1>);
  } else {
    if (pl.odd) return pl.SS == 2 ? go(tap1d_wgrad_kernel<T, TQ, 2, true>) : go(tap1d_wgrad_kernel<T, TQ, 1, true>);
    return pl.SS == 2 ? go(tap1d_wgrad_kernel<T, TQ, 2, false>) : go(tap1d_wgrad_kernel<T, TQ, 1, false>);
  }
}

template <typename T>
int run_wgrad(const ConvGeom& g, const void* x, const void* dy, float* dw, float* db, void* ws, size_t ws_bytes, hipStream_t s,
              const void* rows) {
  Tap1WPlan pl;
  if (!tap1d_wgrad_plan(g, (int)sizeof(T), &pl)) return -1;
  if (!ws || ws_bytes < pl.rows_bytes + pl.part_bytes) return -1;
  const T* xr = static_cast<const T*>(rows ? rows : ws);
  float* part = reinterpret_cast<float*>(static_cast<char*>(ws) + pl.rows_bytes);
  if (!rows) {
    launch_rows(static_cast<const T*>(x), static_cast<T*>(ws), g.C, g.H, g.W, pl.p.Cs, pl.p.rows, s);
    if (const int rc = check_launch("conv2d_bwd_filter (one-row windows, rows pass)")) return rc;
  }
  const T* dyp = static_cast<const T*>(dy);
  int rc;
  switch (pl.TQ) {
    case 2: rc = launch_wgrad<T, 2>(pl, xr, dyp, part, s); break;
    case 3: rc = launch_wgrad<T, 3>(pl, xr, dyp, part, s); break;
    case 4: rc = launch_wgrad<T, 4>(pl, xr, dyp, part, s); break;
    case 5: rc = launch_wgrad<T, 5>(pl, xr, dyp, part, s); break;
    default: rc = launch_wgrad<T, 6>(pl, xr, dyp, part, s); break;
  }
  if (rc) return rc;
  const int tiles = pl.p.ktiles * pl.p.ctiles;
  hipLaunchKernelGGL(tap1d_wgrad_reduce_kernel, dim3(8, (unsigned)(g.KW + 1), (unsigned)tiles), dim3(256), 0, s, part, pl.nsplit,
                     tiles, pl.p.ctiles, 4 * pl.TQ, g.K, g.C, g.KW, dw, db);
  return check_launch("conv2d_bwd_filter (one-row windows, sum)");
}

int esz_of(int dtype) { return dtype == FLHIP_F32 ? 4 : dtype == FLHIP_BF16 || dtype == FLHIP_F16 ? 2 : 0; }

}  // namespace

int mfma_tap1d_cs(int C, int esz) { return tap1d_cs(C, esz); }
void mfma_tap1d_rows_f32(const float* x, float* xr, int C, int H, int T, int Cs, int rows, hipStream_t s) {
  launch_rows(x, xr, C, H, T, Cs, rows, s);
}

size_t mfma_tap1d_conv_ws(const ConvGeom& g, int dtype, bool bwd) {
  if (dtype == FLHIP_F32) return mfma_tap1d_split_ws(g, bwd, nullptr);
  Tap1Plan pl;
  return esz_of(dtype) && tap1d_plan(g, bwd, &pl) ? pl.rows_bytes + pl.w_bytes : 0;
}

int mfma_tap1d_conv_fwd(const ConvGeom& g, int dtype, const void* x, const void* w, const float* bias, void* y, hipStream_t s,
                        void* ws, size_t ws_bytes) {
  if (dtype == FLHIP_F32) return mfma_tap1d_split(g, false, x, w, bias, y, s, ws, ws_bytes);
  if (dtype == FLHIP_BF16) return run_conv<bf16_t>(g, false, x, w, bias, y, s, ws, ws_bytes);
  if (dtype == FLHIP_F16) return run_conv<f16_t>(g, false, x, w, bias, y, s, ws, ws_bytes);
  return -1;
}

int mfma_tap1d_conv_bwd_data(const ConvGeom& g, int dtype, const void* dy, const void* w, void* dx, hipStream_t s, void* ws,
                             size_t ws_bytes) {
  if (dtype == FLHIP_F32) return mfma_tap1d_split(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  if (dtype == FLHIP_BF16) return run_conv<bf16_t>(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  if (dtype == FLHIP_F16) return run_conv<f16_t>(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  return -1;
}

size_t mfma_tap2d_conv_ws(const ConvGeom& g, int dtype, bool bwd) {
  if (dtype == FLHIP_F32) return mfma_tap2d_split_ws(g, bwd);
  Tap1Plan pl;
  return esz_of(dtype) && tap2d_plan(g, bwd, &pl) ? pl.rows_bytes + pl.w_bytes : 0;
}

int mfma_tap2d_conv_fwd(const ConvGeom& g, int dtype, const void* x, const void* w, const float* bias, void* y, hipStream_t s,
                        void* ws, size_t ws_bytes) {
  if (dtype == FLHIP_F32) return mfma_tap2d_split(g, false, x, w, bias, y, s, ws, ws_bytes);
  if (dtype == FLHIP_BF16) return run_conv2d<bf16_t>(g, false, x, w, bias, y, s, ws, ws_bytes);
  if (dtype == FLHIP_F16) return run_conv2d<f16_t>(g, false, x, w, bias, y, s, ws, ws_bytes);
  return -1;
}

int mfma_tap2d_conv_bwd_data(const ConvGeom& g, int dtype, const void* dy, const void* w, void* dx, hipStream_t s, void* ws,
                             size_t ws_bytes) {
  if (dtype == FLHIP_F32) return mfma_tap2d_split(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  if (dtype == FLHIP_BF16) return run_conv2d<bf16_t>(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  if (dtype == FLHIP_F16) return run_conv2d<f16_t>(g, true, dy, w, nullptr, dx, s, ws, ws_bytes);
  return -1;
}

size_t mfma_tap1d_wgrad_ws(const ConvGeom& g, int dtype) {
  Tap1WPlan pl;
  return esz_of(dtype) && tap1d_wgrad_plan(g, esz_of(dtype), &pl) ? pl.rows_bytes + pl.part_bytes : 0;
}

size_t mfma_tap1d_rows_bytes(const ConvGeom& g, int dtype) {
  Tap1Plan f;
  Tap1WPlan w;
  const int esz = esz_of(dtype);
  if (dtype == FLHIP_F32) {
    size_t rows = 0;
    return mfma_tap1d_split_ws(g, false, &rows) && tap1d_wgrad_plan(g, esz, &w) && rows == w.rows_bytes ? rows : 0;
  }
  return esz && tap1d_plan(g, false, &f) && tap1d_wgrad_plan(g, esz, &w) && f.rows_bytes == w.rows_bytes ? w.rows_bytes : 0;
}

int mfma_tap1d_wgrad(const ConvGeom& g, int dtype, const void* x, const void* dy, float* dw, float* db, void* ws, size_t ws_bytes,
                     hipStream_t s, const void* rows) {
  if (dtype == FLHIP_F32) return run_wgrad<float>(g, x, dy, dw, db, ws, ws_bytes, s, rows);
  if (dtype == FLHIP_BF16) return run_wgrad<bf16_t>(g, x, dy, dw, db, ws, ws_bytes, s, rows);
  if (dtype == FLHIP_F16) return run_wgrad<f16_t>(g, x, dy, dw, db, ws, ws_bytes, s, rows);
  return -1;
}

}  // namespace flhip
