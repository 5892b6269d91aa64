// Large products in 16-bit storage on tiles of 256 x 256 (or 256 x 128): 1x1 convolutions of stride 1, forward and backward-data, and
// the three products of fl::linear, where the kernels of conv2d_mfma_pointwise_dma_bf16.hip (128 x 128) would run for several rounds.
//
// What bounds those is the way from the caches to LDS: a compute unit gets 50 to 55 bytes per ns of tiles that most of the
// time come from beyond its die's L2, and a 128 x 128 tile needs 1/64 byte per operation: 600 to 700 TFLOP/s (4000 x 2000 -> 9998 in
// bf16: 265 us; the loads and barriers alone, nothing multiplied, 212; the products alone 130).  A 256 x 256 tile needs half of that.
//
// Eight waves; a stage is 32 contraction indexes of both operands, copied to a ring of 4 stages in LDS by the loads themselves (the
// same cells, offsets and range checks as in the smaller kernel), 3 stages ahead.  A wave owns 64 positions x 128 (64) channels: 2 x 4
// (2 x 2) blocks of 32 x 32.  Within a stage it reads the fragments of one half (16 indexes) while it multiplies the other; the
// barrier of a stage stands between its halves, when every wave has read the slot that the next loads go to.
// Measured, us (smaller kernels / here), bf16: A B 4000 x 2000 -> 9998 241 / 175 (914 TFLOP/s; its products alone 135), A B^T
// 9998 x 2000 over 4000 220 / 180, A^T B 4000 x 2000 over 9998 249 / 195; 4096 x 4096 x 4096 155 / 124 (1109 TFLOP/s).
#include <algorithm>

#include "conv2d_mfma.h"
#include "lds_direct.h"

namespace flhip {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short shortx4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4_t* lds_tr_t;

constexpr int BG_KC = 32, BG_NS = 4, BG_D = BG_NS - 1, BG_THREADS = 512;
constexpr int BG_CELLS = 32;                       // cells of 8 positions per workgroup
constexpr int BG_OOB = (int)0x80000000;

// rows r0 .. r0+7 of column c0 + s of a 16-bit tile stored [row][column]
__device__ __forceinline__ bf16x8 bg_gather8(const uint16_t* tile, int pitch, int r0, int c0, int s) {
  const uint16_t* t = tile + (r0 + (s >> 2)) * pitch + c0 + 4 * (s & 3);
  const shortx4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)t);
  const shortx4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(t + 4 * pitch));
  const uintx2_t l = __builtin_bit_cast(uintx2_t, lo), h = __builtin_bit_cast(uintx2_t, hi);
  return __builtin_bit_cast(bf16x8, uintx4_t{l.x, l.y, h.x, h.y});
}

// this wave's loads of all but the last STAGES stages have landed; it issues FEW or FEW + 1 (more) per stage
template <int FEW, int STAGES>
__device__ __forceinline__ void bg_wait(bool more) {
  if (more) asm volatile("s_waitcnt vmcnt(%0)" :: "n"((FEW + 1) * STAGES) : "memory");
  else asm volatile("s_waitcnt vmcnt(%0)" :: "n"(FEW * STAGES) : "memory");
}

// Tile t of columns x rows tiles, in panels of `panel` columns (the last one maybe fewer), row after row within a panel.  The 32 tiles
// that a die computes at a time then need 8 + 4 source tiles at once; column after column it was up to 32 + 1.
// Measured, us (column after column / here), bf16: A B 4000 x 2000 -> 9998 174 / 172, its two backward products 408 / 396 together, of 4096 x
// 4096 x 4096 285 / 275, forward 124 / 123, 6000 x 1024 -> 4001 67.2 / 65.7.  Panels of 4 to 8 columns are level, 16 are no better than none.
__device__ __forceinline__ void bg_panel(int t, int columns, int rows, int panel, int& column, int& row) {
  const int first = t / (panel * rows) * panel, width = min(panel, columns - first), r = t - first * rows;
  row = r / width;
  column = first + r - row * width;
}

struct BigParams {
  int Kc, Mo;           // contraction channels, result channels
  int P, Pc;            // positions and cells per plane
  int ncells, nstages, mtiles, ctiles;
  int panel;            // channel tiles side by side (bg_panel)
  int halves;           // of the last tiles, computed as two of 128 channels each
  unsigned src_bytes, w_bytes, dst_bytes;
};

template <bool BWD, int BM>
constexpr int big16_stage() { return BG_KC * (BG_CELLS + 2) + (BWD ? BG_KC * (BM / 8 + 2) : BM * 5); }     // cells

// The tile of 256 positions from cell0 x BM channels from m0.  forward: w[m][c]; BWD: w[c][m].  pos_bias: one value per position (one
// image), or null
template <typename E, bool BWD, int BM>
__device__ __forceinline__ void big16_tile(const BigParams& p, int m0, int cell0, const E* __restrict__ src, const E* __restrict__ wgt,
                                           const float* __restrict__ bias, const float* __restrict__ pos_bias, E* __restrict__ dst,
                                           const E* __restrict__ addend) {
  constexpr int XC = BG_CELLS + 2, XP = XC * 8, XCELLS = BG_KC * XC;             // source tile [32][256 positions], two unused cells a row
  constexpr int WC = 5, WP = WC * 8;                                             // forward weights [BM][32], one unused cell
  constexpr int WXC = BM / 8 + 2, WXP = WXC * 8;                                 // backward weights [32][BM]
  constexpr int WCELLS = BWD ? BG_KC * WXC : BM * WC, STAGE = big16_stage<BWD, BM>();
  constexpr int NXI = XCELLS / 64, NI = (XCELLS + WCELLS) / 64, PER = (NI + 7) / 8, FEW = NI / 8;
  static_assert(XCELLS % 64 == 0 && WCELLS % 64 == 0, "whole load instructions");
  constexpr int NB = BM / 64;                      // blocks of 32 channels per wave
  constexpr int YP = 8 * BG_CELLS + 8;             // result staging pitch (elements)
  static_assert(BM * YP * 2 <= BG_NS * STAGE * 16, "the staged results fit in the ring");
  extern __shared__ __align__(16) uint4 bg_ring[];
  uint16_t* const ys = reinterpret_cast<uint16_t*>(bg_ring);

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const intx4_t xrs = pd_rsrc(src, p.src_bytes), wrs = pd_rsrc(wgt, p.w_bytes);

  // ---- load roles: instruction ii = wave + 8 n of a stage; lane -> LDS cell ii * 64 + lane
  int voff[PER], klim[PER];            // klim: contraction channels from the lane's cell to the end of its row (forward weights)
  intx4_t lrs[PER];
  int loff[PER], lstep[PER];
#pragma unroll
  for (int n = 0; n < PER; ++n) {
    const int ii = wave + 8 * n;
    const bool isx = ii < NXI;
    lrs[n] = isx ? xrs : wrs;
    loff[n] = ii * 1024;
    lstep[n] = isx ? BG_KC * 2 * p.P : BWD ? BG_KC * 2 * p.Mo : BG_KC * 2;
    voff[n] = BG_OOB;
    klim[n] = 0x7fffffff;
    if (isx) {
      const int L = ii * 64 + lane, row = L / XC, c = L - row * XC, cell = cell0 + c;
      if (c < BG_CELLS && cell < p.ncells) {
        const int img = cell / p.Pc, j = cell - img * p.Pc;
        voff[n] = ((img * p.Kc + row) * p.P + min(8 * j, p.P - 8)) * 2;
      }
      klim[n] = p.Kc - row;            // rows past the last channel would lie in the next image
    } else if (ii < NI) {
      const int L = (ii - NXI) * 64 + lane;
      if (BWD) {
        const int row = L / WXC, c = L - row * WXC, mo = m0 + 8 * c;
        if (c < BM / 8 && mo < p.Mo) voff[n] = (row * p.Mo + mo) * 2;
        klim[n] = p.Kc - row;
      } else {
        const int m = L / WC, c = L - m * WC;
        if (c < 4 && m0 + m < p.Mo) voff[n] = ((m0 + m) * p.Kc + 8 * c) * 2;
        klim[n] = p.Kc - 8 * c;        // cells past the row's end fetch nothing
      }
    }
  }
  const bool more = wave < NI % 8;
  const int nst = p.nstages;
  auto issue = [&](int t) __attribute__((always_inline)) {
    const unsigned base = pd_lds_addr(bg_ring) + (unsigned)(t & (BG_NS - 1)) * (STAGE * 16);
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if (k < FEW || more) pd_load_lds(lrs[k], base + loff[k], t * BG_KC < klim[k] ? voff[k] : BG_OOB, t * lstep[k]);
  };

  // ---- fragments: wave = (position quarter, channel half)
  const int pos0 = (wave & 3) * 64, mw0 = (wave >> 2) * (BM / 2);
  const int fh = lane >> 5, fq = (lane >> 4) & 1, fs = lane & 15, fr = lane & 31;
  bf16x8 fa[2][2], fb[2][NB];          // [half of the stage][block]
  floatx16 acc[2][NB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto read = [&](int t, int ks) __attribute__((always_inline)) {
    const uint4* const ring = bg_ring + (t & (BG_NS - 1)) * STAGE;
    const uint16_t* const X = reinterpret_cast<const uint16_t*>(ring);
    const uint16_t* const W = reinterpret_cast<const uint16_t*>(ring + XCELLS);
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[ks][i] = bg_gather8(X, XP, ks * 16 + 8 * fh, pos0 + i * 32 + 16 * fq, fs);
#pragma unroll
    for (int j = 0; j < NB; ++j)
      fb[ks][j] = BWD ? bg_gather8(W, WXP, ks * 16 + 8 * fh, mw0 + j * 32 + 16 * fq, fs)
                      : __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4_t*>(&W[(mw0 + j * 32 + fr) * WP + ks * 16 + 8 * fh]));
  };
  auto multiply = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = Lo16<E>::mma32(fa[ks][i], fb[ks][j], acc[i][j]);
    // reads among the products (the compiler would put them behind, and wait for them in the next half)
    constexpr int READS = 4 + (BWD ? 2 : 1) * NB, MULTS = 2 * NB;
#pragma unroll
    for (int q = 0; q < MULTS; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, (READS + MULTS - 1) / MULTS, 0);
    }
  };

#pragma unroll
  for (int st = 0; st < BG_NS; ++st)
    if (st < nst) issue(st);
  if (nst >= BG_NS) bg_wait<FEW, BG_D>(more);
  else PD_WAIT_VM(0);
  __syncthreads();
  read(0, 0);
#pragma unroll 1
  for (int t = 0; t < nst; ++t) {
    read(t, 1);
    multiply(0);
    // stage t + 1 has landed: this wave's loads, then (the barrier) everybody's; and everybody has read stage t
    if (t + BG_D < nst) bg_wait<FEW, BG_D - 1>(more);
    else PD_WAIT_VM(0);
    __syncthreads();
    if (t + BG_NS < nst) issue(t + BG_NS);
    read(t + 1 < nst ? t + 1 : t, 0);
    multiply(1);
  }
  __syncthreads();                     // the ring becomes the staging tile

  // ---- results: element r of block (i, j): slot pos0 + i*32 + (r/4)*8 + fh*4 + r%4 of channel mw0 + j*32 + fr.
  // [channel][slot] in LDS, then whole cells to memory.
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int ml = mw0 + j * 32 + fr;
    const float bv = bias && m0 + ml < p.Mo ? bias[m0 + ml] : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        float v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[i][j][4 * g + e] + bv;
        if (pos_bias) {                // one image: slot 8 c + e of the tile is position min(8 (cell0 + c), P - 8) + e
          const int cell = cell0 + (pos0 + i * 32) / 8 + g;
          if (cell < p.ncells) {
            const float* pb = pos_bias + min(8 * cell, p.P - 8) + fh * 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += pb[e];
          }
        }
        *reinterpret_cast<uintx2_t*>(&ys[ml * YP + pos0 + i * 32 + g * 8 + fh * 4]) = uintx2_t{Lo16<E>::pack(v[0], v[1]), Lo16<E>::pack(v[2], v[3])};
      }
  }
  __syncthreads();
  {
    const int c = tid & (BG_CELLS - 1), cell = cell0 + c;
    if (cell < p.ncells) {
      const int img = cell / p.Pc, j = cell - img * p.Pc;
      const int base = (img * p.Mo + m0) * p.P + min(8 * j, p.P - 8);
      const __amdgpu_buffer_rsrc_t drs = make_rsrc(dst, p.dst_bytes);
      const __amdgpu_buffer_rsrc_t ars = make_rsrc(addend ? addend : dst, p.dst_bytes);
      for (int ml = tid / BG_CELLS; ml < BM && m0 + ml < p.Mo; ml += BG_THREADS / BG_CELLS) {
        uintx4_t v = *reinterpret_cast<const uintx4_t*>(&ys[ml * YP + 8 * c]);
        const int off = (base + ml * p.P) * 2;
        if (addend) {
          const uintx4_t a = __builtin_amdgcn_raw_buffer_load_b128(ars, off, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = Lo16<E>::pack(Lo16<E>::lo(v[e]) + Lo16<E>::lo(a[e]), Lo16<E>::hi(v[e]) + Lo16<E>::hi(a[e]));
        }
        __builtin_amdgcn_raw_buffer_store_b128(v, drs, off, 0, 0);
      }
    }
  }
}

// The tiles in the order in which workgroups start: whole ones (256 channels) first, then `halves` of them as two of 128 channels each,
// which fill the compute units' last round.  Consecutive workgroups go to the eight dies in turn; a die takes runs of tiles
// (bg_panel).
template <typename E, bool BWD>
__global__ void __launch_bounds__(BG_THREADS, 2)
big16_conv_kernel(BigParams p, const E* __restrict__ src, const E* __restrict__ wgt, const float* __restrict__ bias,
                  const float* __restrict__ pos_bias, E* __restrict__ dst, const E* __restrict__ addend) {
  const int id = blockIdx.x, tiles = p.ctiles * p.mtiles, whole = tiles - p.halves;
  auto at = [&](int n, int i) { return (n >> 3) * (i & 7) + min(n & 7, i & 7) + (i >> 3); };       // the i-th of n tiles, run by run
  if (id < whole) {
    const int t = __builtin_amdgcn_readfirstlane(at(whole, id));
    int mt, ct;
    bg_panel(t, p.mtiles, p.ctiles, p.panel, mt, ct);
    big16_tile<E, BWD, 256>(p, mt * 256, ct * BG_CELLS, src, wgt, bias, pos_bias, dst, addend);
  } else {
    const int h = __builtin_amdgcn_readfirstlane(at(2 * p.halves, id - whole)), t = whole + (h >> 1);
    int mt, ct;
    bg_panel(t, p.mtiles, p.ctiles, p.panel, mt, ct);
    const int m0 = mt * 256 + (h & 1) * 128;
    if (m0 >= p.Mo) return;
    big16_tile<E, BWD, 128>(p, m0, ct * BG_CELLS, src, wgt, bias, pos_bias, dst, addend);
  }
}

template <typename E, bool BWD>
int big16_go(const BigParams& p, const void* src, const void* w, const float* bias, const float* pos_bias, void* dst, const void* addend, hipStream_t s) {
  const long long tiles = (long long)p.ctiles * p.mtiles;
  const size_t lds = (size_t)BG_NS * 16 * (p.halves < tiles ? big16_stage<BWD, 256>() : big16_stage<BWD, 128>());
  auto kernel = big16_conv_kernel<E, BWD>;
  if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return -1;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles + p.halves)), dim3(BG_THREADS), lds, s, p, static_cast<const E*>(src), static_cast<const E*>(w),
                     bias, pos_bias, static_cast<E*>(dst), static_cast<const E*>(addend));
  return check_launch("1x1 / matmul (16-bit mfma, 256-wide tiles)");
}

// ---- both operands contiguous along the contraction: out[m][c] = sum_k a[m][k] b[c][k] (+ bias[c]) ------------------------------
// A tile is 256 rows of a x 128 of b, a stage 64 contraction indexes (whole cache lines of a row), a ring of 3.
// LDS [row][8 cells of 8 k], 128 bytes a row; cell c of row r lies at c ^ (r & 7), so that the rows of a fragment read spread over
// the banks.  A row's last cell ends at its last element and so repeats up to 7 of the cell before it: in both tiles those become
// zeros (an infinity must meet no zero of the other tile), written by the lanes that loaded them between the wait for their loads and the barrier.
struct BigNtParams {
  int M, C, K, Kcells;
  int nstages, mtiles, ctiles, panel, dup;
  unsigned a_bytes, b_bytes;
};
constexpr int BN_A = 256, BN_B = 128, BN_STAGE = (BN_A + BN_B) * 128, BN_NS = 3;

template <typename E>
__global__ void __launch_bounds__(BG_THREADS, 2)
big16_nt_kernel(BigNtParams p, const E* __restrict__ a, const E* __restrict__ b, const float* __restrict__ bias, uint16_t* __restrict__ out) {
  constexpr int INSTR = BN_STAGE / 1024 / 8, AI = BN_A / 64;       // load instructions per wave, and of a's rows
  constexpr int NB = BN_B / 64;
  extern __shared__ __align__(16) uint4 bg_ring[];
  char* const ring = reinterpret_cast<char*>(bg_ring);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, fh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // runs of tiles on one die
  const int tiles = p.mtiles * p.ctiles, id = blockIdx.x;
  const int t0 = __builtin_amdgcn_readfirstlane((tiles >> 3) * (id & 7) + min(tiles & 7, id & 7) + (id >> 3));
  int mt, ct;
  bg_panel(t0, p.ctiles, p.mtiles, p.panel, ct, mt);
  const int m0 = mt * BN_A, c0 = ct * BN_B;
  const intx4_t ars = pd_rsrc(a, p.a_bytes), brs = pd_rsrc(b, p.b_bytes);

  // ---- load roles: instruction wave + 8 k fills rows 8 (wave + 8 k) .. + 7 (the first AI: a's rows); lane -> row lane / 8, slot lane % 8
  const int lcell = (lane & 7) ^ (lane >> 3);
  int rowoff[INSTR];
#pragma unroll
  for (int k = 0; k < INSTR; ++k) {
    const int r = 8 * (wave + 8 * k) + (lane >> 3);
    rowoff[k] = k < AI ? (m0 + r < p.M ? (m0 + r) * p.K * 2 : BG_OOB) : (c0 + r - BN_A < p.C ? (c0 + r - BN_A) * p.K * 2 : BG_OOB);
  }
  const int nst = p.nstages;
  auto issue = [&](int t, int slot) __attribute__((always_inline)) {
    const unsigned base = pd_lds_addr(bg_ring) + (unsigned)slot * BN_STAGE + wave * 1024;
    const int cell = 8 * t + lcell, col = min(8 * cell, p.K - 8) * 2;
#pragma unroll
    for (int k = 0; k < INSTR; ++k)
      pd_load_lds(k < AI ? ars : brs, base + k * 8192, rowoff[k] == BG_OOB || cell >= p.Kcells ? BG_OOB : rowoff[k] + col, 0);
  };
  // zeros over what the last cell of this lane's rows repeats (its loads have landed)
  auto fix_tail = [&](int t, int slot) __attribute__((always_inline)) {
    if (p.dup && t == nst - 1 && 8 * t + lcell == p.Kcells - 1) {
#pragma unroll
      for (int k = 0; k < INSTR; ++k) {
        uint16_t* const q = reinterpret_cast<uint16_t*>(ring + slot * BN_STAGE + (wave + 8 * k) * 1024 + lane * 16);
        for (int e = 0; e < p.dup; ++e) q[e] = 0;
      }
    }
  };

  // ---- fragments: wave = (row quarter of a, half of b's rows)
  const int ar0 = (wave & 3) * 64, br0 = (wave >> 2) * (BN_B / 2);
  const int arow = (ar0 + fr) * 128, brow = (BN_A + br0 + fr) * 128, sw = fr & 7;
  bf16x8 fa[2][2], fb[2][NB];          // [sixteen indexes, in turn][block]
  floatx16 acc[2][NB];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  auto read = [&](int slot, int ks) __attribute__((always_inline)) {
    const char* const st = ring + slot * BN_STAGE + ((2 * ks + fh) ^ sw) * 16;
#pragma unroll
    for (int i = 0; i < 2; ++i) fa[ks & 1][i] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4_t*>(st + arow + i * 4096));
#pragma unroll
    for (int j = 0; j < NB; ++j) fb[ks & 1][j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uintx4_t*>(st + brow + j * 4096));
  };
  auto multiply = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = Lo16<E>::mma32(fa[ks & 1][i], fb[ks & 1][j], acc[i][j]);
#pragma unroll
    for (int q = 0; q < 2 * NB; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
  };
#pragma unroll
  for (int st = 0; st < BN_NS; ++st)
    if (st < nst) issue(st, st);
  if (nst >= BN_NS) bg_wait<INSTR, BN_NS - 1>(false);
  else PD_WAIT_VM(0);
  fix_tail(0, 0);
  __syncthreads();
  read(0, 0);
  int slot = 0;
#pragma unroll 1
  for (int t = 0; t < nst; ++t) {
    const int next = slot == BN_NS - 1 ? 0 : slot + 1;
#pragma unroll
    for (int ks = 0; ks < 3; ++ks) {
      read(slot, ks + 1);
      multiply(ks);
    }
    if (t + BN_NS - 1 < nst) bg_wait<INSTR, BN_NS - 2>(false);
    else PD_WAIT_VM(0);
    fix_tail(t + 1, next);
    __syncthreads();
    if (t + BN_NS < nst) issue(t + BN_NS, slot);
    read(next, 0);                     // (behind the last stage: what is there, for nobody)
    multiply(3);
    slot = next;
  }

  // element r of block (i, j): row m0 + ar0 + i*32 + (r/4)*8 + fh*4 + r%4, column c0 + br0 + j*32 + fr
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int c = c0 + br0 + j * 32 + fr;
    if (c >= p.C) continue;
    const float bv = bias ? bias[c] : 0.f;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + ar0 + i * 32 + (r >> 2) * 8 + fh * 4 + (r & 3);
        if (m < p.M) out[(size_t)m * p.C + c] = Lo16<E>::narrow(acc[i][j][r] + bv);
      }
  }
}

}  // namespace

// equal panels of at most eight columns
static int bg_panel_width(int columns) {
  const int panels = (columns + 7) / 8;
  return (columns + panels - 1) / panels;
}

// Whether the tiles here are the faster ones, and how many of them, the last, should be computed as two halves (< 0: the smaller
// kernels).  In rounds of the smaller kernels, which compute a tile of 128 x 128 per unit and round: a round of whole tiles takes 2.8
// (convolutions 3.0), one of at most 128 tiles in halves 2.0 (2.5); the medians over 32473 random products and layers are 2.3 to 2.9
// (2.7 to 3.2) and 1.6 to 2.1 (1.9 to 2.6).  Where the rule takes the tiles here they need 0.70 to 0.87 of the smaller kernels' time (geometric
// means for matrix products by length of the contraction, 95 % at most 1.00; convolutions 0.82 to 0.89, 95 % at most 1.06); those with 8 stages and
// fewer, 1.0 to 1.2 of it, stay where they were, as do products of at most half a chip of tiles (0.9 to 1.4 by how they fill their last tiles).
int mfma_big16_halves(bool conv, long long images, int Kc, int Mo, int P) {
  const long long cells = images * ((P + 7) / 8), ct = (cells + BG_CELLS - 1) / BG_CELLS, tiles = ct * ((Mo + 255) / 256);
  const int cus = mfma_num_cus();
  if (tiles > 0x3fffffff || (conv && (Kc + BG_KC - 1) / BG_KC <= 8)) return -1;
  const int last = (int)(tiles % cus);
  const bool halved = tiles > cus && last && 2 * last <= cus;
  const float whole = conv ? 3.f : 2.8f, half = conv ? 2.5f : 2.f;
  const long long small = ((cells + 15) / 16 * ((Mo + 127) / 128) + cus - 1) / cus;      // rounds of the smaller kernels
  if ((tiles / cus) * whole + (!last ? 0.f : halved ? half : whole) >= small) return -1;
  return halved ? last : 0;
}

// halves: how many of the tiles (256 positions x 256 channels) are computed in two
int mfma_big16(int dtype, bool bwd, long long images, int Kc, int Mo, int P, const void* src, const void* w, const float* bias,
               const float* pos_bias, void* dst, const void* addend, int halves, hipStream_t s) {
  BigParams p{};
  p.Kc = Kc; p.Mo = Mo; p.P = P;
  p.Pc = (P + 7) / 8;
  p.src_bytes = (unsigned)(images * Kc * P * 2); p.dst_bytes = (unsigned)(images * Mo * P * 2); p.w_bytes = (unsigned)((long long)Kc * Mo * 2);
  p.ncells = (int)(images * p.Pc);
  p.nstages = (Kc + BG_KC - 1) / BG_KC;
  p.ctiles = (p.ncells + BG_CELLS - 1) / BG_CELLS;
  p.mtiles = (Mo + 255) / 256;
  p.panel = bg_panel_width(p.mtiles);
  p.halves = halves;
  return by_lo16(dtype, [&](auto* e_) {
    using E = FLHIP_T_OF(e_);
    return bwd ? big16_go<E, true>(p, src, w, bias, pos_bias, dst, addend, s) : big16_go<E, false>(p, src, w, bias, pos_bias, dst, addend, s);
  });
}

// The same for A^T B: a round of 256 x 128 tiles takes 1.1 to 1.3 of the smaller kernel's; taken, 0.65 to 0.72 of its time (95 % at most
// 0.89), not taken 0.98 to 1.22.
bool mfma_big16_nt_pays(int M, int C) {
  const long long ct = (C + BN_B - 1) / BN_B, cus = mfma_num_cus(), big = ((M + BN_A - 1) / BN_A * ct + cus - 1) / cus;
  return 1.25f * big < ((M + 127) / 128 * ct + cus - 1) / cus;
}
// out[m][c] = sum over k of a[m][k] b[c][k] (+ bias[c])
int mfma_big16_nt(int dtype, int M, int C, int K, const void* a, const void* b, const float* bias, void* out, hipStream_t s) {
  BigNtParams p{};
  p.M = M; p.C = C; p.K = K;
  p.Kcells = (K + 7) / 8;
  p.dup = (8 - K % 8) % 8;
  p.nstages = (p.Kcells + 7) / 8;
  p.mtiles = (M + BN_A - 1) / BN_A;
  p.ctiles = (C + BN_B - 1) / BN_B;
  p.panel = bg_panel_width(p.ctiles);
  p.a_bytes = (unsigned)((long long)M * K * 2); p.b_bytes = (unsigned)((long long)C * K * 2);
  return by_lo16(dtype, [&](auto* e_) {
    using E = FLHIP_T_OF(e_);
    constexpr size_t lds = (size_t)BN_NS * BN_STAGE;
    auto kernel = big16_nt_kernel<E>;
    if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return -1;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(p.mtiles * p.ctiles)), dim3(BG_THREADS), lds, s, p, static_cast<const E*>(a),
                       static_cast<const E*>(b), bias, static_cast<uint16_t*>(out));
    return check_launch("matmul (A^T * B, 16-bit mfma, 256-wide tiles)");
  });
}

}  // namespace flhip
