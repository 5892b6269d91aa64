// fp32 matrix products on the bf16 matrix cores, each operand in three parts (split_f32.h); column-major, modes as in
// gemm_f32.hip:
//   mode 0  C [M x N] = A [M x K]   * B [K x N]
//   mode 1  C [M x N] = A [K x M]^T * B [K x N]
//   mode 2  C [M x N] = A [M x K]   * B [N x K]^T
// (Products whose fp32 sums have to stay, gemm32's fp32_sums, run on gemm_f32.hip whatever their size: 2000 x 4000 x 2000 forward 232 us, here 160.)
//
// A workgroup (4 waves, 2 x 2) owns a TM x TN tile of C, a wave RT x CT instruction tiles of 32 x 32 with two accumulators each.
// The contraction runs in stages of 16.  A stage's values pass through registers, where they are taken apart: loaded two stages
// ahead, split and written to LDS one stage ahead (two buffers, one barrier per stage), read as fragments in their own.  (One
// loop of whole stages, its loads unchecked, and a last stage of fewer indexes behind it: with a second loop for the checked
// stages the compiler kept registers of both and spilled.)
//   LDS  [part][row][2 cells of 8 k], 16 bytes a cell; cell c of row r lies at slot c ^ ((r >> 2 ^ r >> 3) & 1), so that the
//        lanes of a read or write pass touch distinct banks whether 8 or 16 of them make a pass.
//   An operand that is contiguous along k comes in 16-byte pieces, four neighbouring lanes 64 contiguous bytes; one that is
//   contiguous along the rows comes as one value per lane and k, neighbouring lanes neighbouring rows: the conversion takes its
//   two values from any two registers, so transposing costs nothing.
//
// What bounds it is the bf16 matrix pipe (768 cycles of it per stage and 128 x 128 tile, for 1500 taken) with what shares its
// cycles: 12 fragment reads and about 100 vector instructions per wave and stage.  Measured, us (before: v_mfma_f32_32x32x2_f32
// from LDS, 0.8 of its pipe at best), and the 2-norm of the error:
//   mode 0  2000 x 4000 x 2000  256 -> 157 (204 TFLOP/s)  8.0e-7 -> 2.7e-7    1024 x 6400 x 3072  312 -> 205
//   mode 1  2000 x 4000 x 2000  256 -> 160                8.0e-7 -> 2.7e-7    2048 x 6400 x 512   113 -> 82
//   mode 2  2000 x 2000 x 4000  265 -> 164 (2 slices)     1.1e-6 -> 2.7e-7    1024 x 2048 x 6400  200 -> 135 (4 slices)
//
// Layers of 1x1 windows are the same products with the positions of all images as A's and C's rows (modes 0 and 2) or as the contraction
// (mode 1): only where a thread's values lie differs (PL), a position being looked up once per workgroup.  Over large planes memory bounds
// them: four small tiles to a compute unit (128 registers, A B with one value kept in memory over its loop; three at 129; A^T B on 64 x
// 128 tiles needs 132) and tiles that share positions one after the other on one die, us: 64 -> 256 channels over 56 x 56, 32 images 47 -> 39 (129 MB), the addend's loads in front of the stores 70 -> 38; filter
// gradient of 256 x 64, a slice's tiles on one die, 45 -> 39.  (The general kernels' times stand at the rule, conv2d_mfma_pointwise.hip.)
#include <algorithm>

#include "conv2d.h"
#include "gemm_f32.h"
#include "split_f32.h"

namespace flhip {
namespace {

constexpr int ST = 256;                        // threads
constexpr int S_OOB = (int)0x80000000;

__device__ __forceinline__ int split_slot(int row, int cell) { return cell ^ ((row >> 2 ^ row >> 3) & 1); }

// One operand's share of a stage: T rows x 16 k.
template <bool KROWS, int T>
struct SplitSide {
  static constexpr int EL = T * G32_KC / ST;   // values per thread: 8 or 4
  static constexpr int PART = T * 32;          // bytes of a part
  static constexpr int BYTES = 3 * PART;
  // k rows: EL / 4 pieces of 4 k, rows 64 apart; m rows: EL consecutive k of one row
  int off[KROWS ? EL / 4 : 1];
  int at;                                      // where in a part the thread's first piece goes
  int k0;                                      // its first contraction index within a stage
  int step, rowstep;

  __device__ __forceinline__ void init(int r0, int R, int K, int tid) {
    if (KROWS) {
      const int row = tid >> 2, q = tid & 3;
      k0 = 4 * q;
#pragma unroll
      for (int i = 0; i < EL / 4; ++i) off[i] = r0 + row + 64 * i < R ? ((r0 + row + 64 * i) * K + k0) * 4 : S_OOB;
      at = row * 32 + split_slot(row, q >> 1) * 16 + (q & 1) * 8;       // (64 rows further: 2048 bytes, the same slot)
      step = G32_KC * 4;
      rowstep = 0;
    } else {
      const int row = tid % T, g = tid / T;    // EL = 8: g = cell; EL = 4: g = half of a cell
      k0 = EL * g;
      off[0] = r0 + row < R ? (k0 * R + r0 + row) * 4 : S_OOB;
      at = EL == 8 ? row * 32 + split_slot(row, g) * 16 : row * 32 + split_slot(row, g >> 1) * 16 + (g & 1) * 8;
      step = G32_KC * R * 4;
      rowstep = R * 4;
    }
  }
  // rows that are positions of planes (contiguous along the rows): where the first value of position r0 + row lies
  __device__ __forceinline__ void init_positions(int r0, const Gemm32& p, int tid) {
    init(r0, p.M, p.K, tid);
    if constexpr (!KROWS) {
      const int r = r0 + tid % T, img = r / p.P, pos = r - img * p.P, row = pos / p.OW;
      if (r < p.M) off[0] = ((img * p.K + k0) * p.SP + row * p.rowstep + (pos - row * p.OW) * p.colstep) * 4;
      step = G32_KC * p.SP * 4;
      rowstep = p.SP * 4;
    }
  }
  // rows that are channels, the contraction their positions, one image after the other: pieces of 4 positions, which a plane
  // holds whole.  (Past the last image a piece lies past the tensor.)
  int piece, pieces, jump;
  __device__ __forceinline__ void init_channels(int r0, int R, const Gemm32& p, int s0, int tid) {
    init(r0, R, p.SP, tid);
    pieces = p.SP / 4;
    jump = (R - 1) * p.SP * 4;
    const int at0 = s0 * (G32_KC / 4) + (tid & 3), img = at0 / pieces;
    piece = at0 - img * pieces;
#pragma unroll
    for (int i = 0; i < (KROWS ? EL / 4 : 1); ++i)
      if (off[i] != S_OOB) off[i] += (img * R * p.SP + 4 * piece - k0) * 4;
  }
  __device__ __forceinline__ void load_next(float (&v)[EL], __amdgpu_buffer_rsrc_t rsrc) {
    load<false>(v, rsrc, 0, G32_KC);
    piece += G32_KC / 4;
    const int by = G32_KC * 4 + (piece >= pieces ? jump : 0);
    if (piece >= pieces) piece -= pieces;
#pragma unroll
    for (int i = 0; i < (KROWS ? EL / 4 : 1); ++i) off[i] += by;       // (a row that is none: past every tensor all the same)
  }
  // the stage at byte offset `stage` of every row.  CHECKED: only its first `left` contraction indexes exist, the others read
  // zero (a piece that the row ends in holds the next row's first values)
  template <bool CHECKED>
  __device__ __forceinline__ void load(float (&v)[EL], __amdgpu_buffer_rsrc_t rsrc, int stage, int left) const {
    if constexpr (KROWS) {
#pragma unroll
      for (int i = 0; i < EL / 4; ++i) {
        const uintx4_t f = __builtin_amdgcn_raw_buffer_load_b128(rsrc, CHECKED && k0 >= left ? S_OOB : off[i], stage, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * i + e] = !CHECKED || k0 + e < left ? __uint_as_float(f[e]) : 0.f;
      }
    } else {
      const int at0 = off[0] + stage;          // (past the last row: still past every tensor)
#pragma unroll
      for (int e = 0; e < EL; ++e)
        v[e] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rsrc, CHECKED && k0 + e >= left ? S_OOB : at0, e * rowstep, 0));
    }
  }
  __device__ __forceinline__ void store(const float (&v)[EL], char* lds) const {
    if constexpr (EL == 8 && !KROWS) {
      uintx4_t h, m, l;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const Split2 s = split2(v[2 * e], v[2 * e + 1]);
        h[e] = s.h; m[e] = s.m; l[e] = s.l;
      }
      *reinterpret_cast<uintx4_t*>(lds + at) = h;
      *reinterpret_cast<uintx4_t*>(lds + PART + at) = m;
      *reinterpret_cast<uintx4_t*>(lds + 2 * PART + at) = l;
    } else {
#pragma unroll
      for (int i = 0; i < EL / 4; ++i) {
        const Split2 s = split2(v[4 * i], v[4 * i + 1]), t = split2(v[4 * i + 2], v[4 * i + 3]);
        char* const o = lds + at + 2048 * i;
        *reinterpret_cast<uintx2_t*>(o) = uintx2_t{s.h, t.h};
        *reinterpret_cast<uintx2_t*>(o + PART) = uintx2_t{s.m, t.m};
        *reinterpret_cast<uintx2_t*>(o + 2 * PART) = uintx2_t{s.l, t.l};
      }
    }
  }
};

template <int MODE, int TM, int TN, bool PL>
__global__ void __launch_bounds__(ST, PL && TM * TN < 128 * 128 && !(MODE == 1 && TM == 64) ? 4 : 2)
gemm32_split_kernel(Gemm32 p, const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
                    const float* addend, float* C) {
  constexpr bool AK = MODE == 1, BK = MODE != 2;
  constexpr int RT = TM / 64, CT = TN / 64;
  // Whether the next loads go out before the products (behind the conversions) or where the compiler puts them, among the
  // products: 128 x 128 tiles with an operand that is contiguous along the rows, 1024 x 6400 x 3072 225 -> 205 us, A * B^T
  // 2000 x 2000 x 4000 170 -> 164; the others lose by it (A^T B 3072 x 6400 x 1024 204 -> 221, 512 x 6400 x 2048 on 128 x 64 tiles 86 -> 97)
  constexpr bool PINNED = MODE != 1 && TM * TN == 128 * 128;
  typedef SplitSide<AK, TM> SA;
  typedef SplitSide<BK, TN> SB;
  constexpr int STAGE = SA::BYTES + SB::BYTES;
  __shared__ __align__(16) char lds[2 * STAGE];
  if (!PL && blockIdx.z) A = p.A2, B = p.B2, bias = p.bias2, C = p.C2;
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  int tile, slice = blockIdx.y;
  if constexpr (PL && MODE == 1) {
    // the tiles of a slice follow each other on one die, whose cache holds the slice's rows (slices past the last full eight: as they come)
    const int tiles = p.mtiles * p.ntiles, at = blockIdx.x, full8 = p.slices / 8 * 8;
    if (at < full8 * tiles) {
      tile = (at >> 3) % tiles;
      slice = (at >> 3) / tiles * 8 + (at & 7);
    } else {
      tile = at % tiles;
      slice = at / tiles;
    }
  } else {
    tile = gemm32_tile_of(blockIdx.x, p.mtiles * p.ntiles);
  }
  // (over planes the weights are the small operand: the tiles that share positions follow each other)
  const bool nfast = PL && MODE != 1;
  const int m0 = (nfast ? tile / p.ntiles : tile % p.mtiles) * TM, n0 = (nfast ? tile % p.ntiles : tile / p.mtiles) * TN;
  const int s0 = slice * p.sps, send = min(p.nstages, s0 + p.sps);

  SA sa;
  SB sb;
  if constexpr (PL && MODE == 1) {
    sa.init_channels(m0, p.M, p, s0, tid);
    sb.init_channels(n0, p.N, p, s0, tid);
  } else {
    if constexpr (PL) sa.init_positions(m0, p, tid);
    else sa.init(m0, p.M, p.K, tid);
    sb.init(n0, p.N, p.K, tid);
  }
  const __amdgpu_buffer_rsrc_t ar = make_rsrc(A, p.a_bytes), br = make_rsrc(B, p.b_bytes);
  float va[SA::EL], vb[SB::EL];
  // end of the slice's whole stages (the contraction has one at least; a last slice may have none, only the stage of fewer indexes, and then
  // loads one of the slice before it for nobody; of planes every stage is whole: what lies past them reads zero)
  const int full = PL && MODE == 1 ? send : min(send, p.K / G32_KC);
  auto stage_in = [&](int s) __attribute__((always_inline)) {
    if constexpr (PL && MODE == 1) {
      sa.load_next(va, ar);
      sb.load_next(vb, br);
      return;
    }
    s = min(s, full - 1);
    sa.template load<false>(va, ar, s * sa.step, G32_KC);
    sb.template load<false>(vb, br, s * sb.step, G32_KC);
  };
  floatx16 big[RT][CT], small[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) big[i][j][r] = small[i][j][r] = 0.f;

  // where the wave's fragments lie within a part (row blocks 32 rows = 1024 bytes apart)
  const int fa = (wm * 32 * RT + fr) * 32 + split_slot(fr, h) * 16, fb = (wn * 32 * CT + fr) * 32 + split_slot(fr, h) * 16;
  auto split_out = [&](int x) __attribute__((always_inline)) {
    sa.store(va, lds + x * STAGE);
    sb.store(vb, lds + x * STAGE + SA::BYTES);
  };
  uintx4_t a[RT][3], b[CT][3];
  auto read = [&](int x) __attribute__((always_inline)) {
    const char* const la = lds + x * STAGE;
    const char* const lb = la + SA::BYTES;
#pragma unroll
    for (int q = 0; q < 3; ++q) {
#pragma unroll
      for (int i = 0; i < RT; ++i) a[i][q] = *reinterpret_cast<const uintx4_t*>(la + q * SA::PART + i * 1024 + fa);
#pragma unroll
      for (int c = 0; c < CT; ++c) b[c][q] = *reinterpret_cast<const uintx4_t*>(lb + q * SB::PART + c * 1024 + fb);
    }
  };
  auto multiply = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int c = 0; c < CT; ++c) split_mma(big[i][c], small[i][c], b[c], a[i]);
  };
  stage_in(s0);
  split_out(0);
  stage_in(s0 + 1);
  // (past the last whole stage it is loaded and written once more, and read by nobody: no load needs a check)
#pragma unroll 1
  for (int s = s0; s < full; ++s) {
    const int x = (s - s0) & 1;
    __syncthreads();             // stage s is in its buffer, and every wave is done with the other
    read(x);
    split_out(x ^ 1);
    if constexpr (PINNED) __builtin_amdgcn_sched_barrier(0);
    stage_in(s + 2);
    if constexpr (PINNED) __builtin_amdgcn_sched_barrier(0);
    multiply();
  }
  if (send > full) {             // the last stage of all, of fewer indexes
    sa.template load<true>(va, ar, full * sa.step, p.K - full * G32_KC);
    sb.template load<true>(vb, br, full * sb.step, p.K - full * G32_KC);
    __syncthreads();
    split_out(0);
    __syncthreads();
    read(0);
    multiply();
  }

  bool bad = false;
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        big[i][c][r] += small[i][c][r];
        bad |= split_redo(big[i][c][r]);
      }
  // once more with the operands as they are (rows, columns and contraction indexes past the last as zero)
  if (__builtin_amdgcn_ballot_w64(bad)) {
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int c = 0; c < CT; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) big[i][c][r] = 0.f;
    const int kend = min(p.K, send * G32_KC);
    size_t arow[RT];                           // positions of planes: a row's first value
    if constexpr (PL && MODE != 1) {
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int m = m0 + wm * 32 * RT + 32 * i + fr, img = m / p.P, pos = m - img * p.P;
        arow[i] = (size_t)img * p.K * p.SP + pos / p.OW * p.rowstep + pos % p.OW * p.colstep;
      }
    }
    auto index = [&](int img, int pos, int row, int rows) { return ((size_t)img * rows + row) * p.SP + pos; };
#pragma unroll 1
    for (int k = s0 * G32_KC + h; k < ((kend + 1) & ~1); k += 2) {
      float a[RT], b[CT];
      const int img = PL && MODE == 1 ? k / p.SP : 0, pos = PL && MODE == 1 ? k - img * p.SP : 0;
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int m = m0 + wm * 32 * RT + 32 * i + fr;
        const size_t at = !PL ? (AK ? (size_t)m * p.K + k : (size_t)k * p.M + m)
                        : MODE == 1 ? index(img, pos, m, p.M) : arow[i] + (size_t)k * p.SP;
        a[i] = k < kend && m < p.M ? A[at] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int n = n0 + wn * 32 * CT + 32 * c + fr;
        const size_t at = PL && MODE == 1 ? index(img, pos, n, p.N) : BK ? (size_t)n * p.K + k : (size_t)k * p.N + n;
        b[c] = k < kend && n < p.N ? B[at] : 0.f;
      }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int c = 0; c < CT; ++c) big[i][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[c], a[i], big[i][c], 0, 0, 0);
    }
  }

  // B's columns are the rows of the instruction's tiles, so that the lanes of a store are neighbours along C's contiguous
  // dimension: element r of a lane is column 8 (r / 4) + 4 h + r % 4 and row fr of C's tile.  (A store past the last column is
  // out of the buffer's range, one past the last row is put there.)
  const int m = m0 + wm * 32 * RT + fr, nl = wn * 32 * CT + 4 * h;
  constexpr bool PC = PL && MODE != 1;         // C in planes: columns P apart, a column past the last is looked for (the next image is there)
  const int ldc = PC ? p.P : p.M, cols = p.N - n0 - nl;
  const size_t origin = (size_t)n0 * ldc, left = ((size_t)(PC ? p.M / p.P * p.N : p.N) * ldc - origin) * 4;
  const unsigned range = left < 0x7fffffffu ? (unsigned)left : 0x7fffffffu;
  const __amdgpu_buffer_rsrc_t orsrc = make_rsrc(C + (size_t)slice * p.slice + origin, range);
  int at[RT];
  float bv[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const bool in = m + i * 32 < p.M;
    const int img = PC ? (m + i * 32) / p.P : 0;
    at[i] = !in ? S_OOB : (PC ? (img * p.N + nl) * p.P + m + i * 32 - img * p.P : nl * p.M + m + i * 32) * 4;
    bv[i] = bias && !PC && in ? bias[m + i * 32] : 0.f;
  }
  // f(element, byte offset, whether the column exists) over the lane's elements
  auto each = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int col = c * 32 + 8 * (r >> 2) + (r & 3);
        const bool is = !PC || col < cols;
        const float bc = PC && bias && is ? bias[n0 + nl + col] : 0.f;
#pragma unroll
        for (int i = 0; i < RT; ++i) f(big[i][c][r], PC ? bc : bv[i], is ? at[i] + col * ldc * 4 : S_OOB);
      }
  };
  if (addend) {                  // (all of its loads before the first store, behind which they could not move)
    const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(addend + origin, range);
    float add[RT * CT * 16];
    int e = 0;
    each([&](float, float, int o) { add[e++] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(arsrc, o, 0, 0)); });
    e = 0;
    each([&](float v, float b, int o) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v + b + add[e++]), orsrc, o, 0, 0); });
  } else {
    each([&](float v, float b, int o) { __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v + b), orsrc, o, 0, 0); });
  }
}

template <int MODE, int TM, int TN, bool PL>
int split_go(const Gemm32& p, int slices, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  hipLaunchKernelGGL((gemm32_split_kernel<MODE, TM, TN, PL>), PL && MODE == 1 ? dim3((unsigned)(p.mtiles * p.ntiles * slices)) : dim3((unsigned)(p.mtiles * p.ntiles), (unsigned)slices, !PL && p.C2 ? 2 : 1), dim3(ST), 0, s, p, A, B,
                     bias, addend, C);
  return check_launch("matmul (fp32 in three parts)");
}
template <int MODE, bool PL>
int split_tile(int tm, int tn, const Gemm32& p, int slices, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  if constexpr (!PL || MODE == 1) {
    if (tm == 128 && tn == 128) return split_go<MODE, 128, 128, PL>(p, slices, A, B, bias, addend, C, s);
    if (tm == 64) return split_go<MODE, 64, 128, PL>(p, slices, A, B, bias, addend, C, s);
  }
  return split_go<MODE, 128, 64, PL>(p, slices, A, B, bias, addend, C, s);
}
template <bool PL>
int split_mode(int mode, int tm, int tn, const Gemm32& p, int slices, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  return mode == 0 ? split_tile<0, PL>(tm, tn, p, slices, A, B, bias, addend, C, s)
       : mode == 1 ? split_tile<1, PL>(tm, tn, p, slices, A, B, bias, addend, C, s)
                   : split_tile<2, PL>(tm, tn, p, slices, A, B, bias, addend, C, s);
}

}  // namespace

int gemm32_split(int mode, int tm, int tn, int slices, const Gemm32& p, const float* A, const float* B, const float* bias,
                 const float* addend, float* C, hipStream_t s) {
  if (tm * tn < 128 * 64) return -1;
  return split_mode<false>(mode, tm, tn, p, slices, A, B, bias, addend, C, s);
}
int gemm32_split_planes(int mode, int tm, int tn, int slices, const Gemm32& p, const float* A, const float* B, const float* bias,
                        const float* addend, float* C, hipStream_t s) {
  return split_mode<true>(mode, tm, tn, p, slices, A, B, bias, addend, C, s);
}

}  // namespace flhip
