// fp32 matrix products on the bf16 matrix cores, each operand in three parts (split_f32.h); column-major, modes as in
// gemm_f32.hip:
//   mode 0  C [M x N] = A [M x K]   * B [K x N]
//   mode 1  C [M x N] = A [K x M]^T * B [K x N]
//   mode 2  C [M x N] = A [M x K]   * B [N x K]^T
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
  // the stage at byte offset `stage` of every row.  CHECKED: only its first `left` contraction indexes exist, the others read
  // zero
  template <bool CHECKED>
  __device__ __forceinline__ void load(float (&v)[EL], __amdgpu_buffer_rsrc_t rsrc, int stage, int left) const {
    if constexpr (KROWS) {
#pragma unroll
      for (int i = 0; i < EL / 4; ++i) {
        const uintx4_t f = __builtin_amdgcn_raw_buffer_load_b128(rsrc, CHECKED && k0 >= left ? S_OOB : off[i], stage, 0);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * i + e] = __uint_as_float(f[e]);
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

template <int MODE, int TM, int TN>
__global__ void __launch_bounds__(ST, 2)
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
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  const int tile = gemm32_tile_of(blockIdx.x, p.mtiles * p.ntiles);
  const int m0 = (tile % p.mtiles) * TM, n0 = (tile / p.mtiles) * TN;
  const int s0 = blockIdx.y * p.sps, send = min(p.nstages, s0 + p.sps);

  SA sa;
  SB sb;
  sa.init(m0, p.M, p.K, tid);
  sb.init(n0, p.N, p.K, tid);
  const __amdgpu_buffer_rsrc_t ar = make_rsrc(A, p.a_bytes), br = make_rsrc(B, p.b_bytes);
  float va[SA::EL], vb[SB::EL];
  const int full = min(send, p.K / G32_KC);    // end of the slice's whole stages (there is one at least)
  auto stage_in = [&](int s) __attribute__((always_inline)) {
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
        bad |= not_finite(big[i][c][r]);
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
#pragma unroll 1
    for (int k = s0 * G32_KC + h; k < ((kend + 1) & ~1); k += 2) {
      float a[RT], b[CT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int m = m0 + wm * 32 * RT + 32 * i + fr;
        a[i] = k < kend && m < p.M ? A[AK ? (size_t)m * p.K + k : (size_t)k * p.M + m] : 0.f;
      }
#pragma unroll
      for (int c = 0; c < CT; ++c) {
        const int n = n0 + wn * 32 * CT + 32 * c + fr;
        b[c] = k < kend && n < p.N ? B[BK ? (size_t)n * p.K + k : (size_t)k * p.N + n] : 0.f;
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
  const size_t origin = (size_t)n0 * p.M, left = ((size_t)(p.N - n0) * p.M) * 4;
  const unsigned range = left < 0x7fffffffu ? (unsigned)left : 0x7fffffffu;
  const __amdgpu_buffer_rsrc_t orsrc = make_rsrc(C + (size_t)blockIdx.y * p.slice + origin, range);
  int at[RT];
  float bv[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const bool in = m + i * 32 < p.M;
    at[i] = in ? (nl * p.M + m + i * 32) * 4 : S_OOB;
    bv[i] = bias && in ? bias[m + i * 32] : 0.f;
  }
  auto store = [&](auto added) __attribute__((always_inline)) {
    constexpr bool ADD = decltype(added)::value;
    const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(ADD ? addend + origin : nullptr, range);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int o = (c * 32 + 8 * (r >> 2) + (r & 3)) * p.M * 4;
#pragma unroll
        for (int i = 0; i < RT; ++i) {
          float v = big[i][c][r] + bv[i];
          if (ADD) v += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(arsrc, at[i] + o, 0, 0));
          __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), orsrc, at[i] + o, 0, 0);
        }
      }
  };
  if (addend) store(std::true_type{});
  else store(std::false_type{});
}

template <int MODE, int TM, int TN>
int split_go(const Gemm32& p, int slices, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  hipLaunchKernelGGL((gemm32_split_kernel<MODE, TM, TN>), dim3((unsigned)(p.mtiles * p.ntiles), (unsigned)slices), dim3(ST), 0, s, p, A, B,
                     bias, addend, C);
  return check_launch("matmul (fp32 in three parts)");
}
template <int MODE>
int split_tile(int tm, int tn, const Gemm32& p, int slices, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  if (tm == 128 && tn == 128) return split_go<MODE, 128, 128>(p, slices, A, B, bias, addend, C, s);
  if (tm == 128) return split_go<MODE, 128, 64>(p, slices, A, B, bias, addend, C, s);
  return split_go<MODE, 64, 128>(p, slices, A, B, bias, addend, C, s);
}

}  // namespace

int gemm32_split(int mode, int tm, int tn, int slices, const Gemm32& p, const float* A, const float* B, const float* bias,
                 const float* addend, float* C, hipStream_t s) {
  if (tm * tn < 128 * 64) return -1;
  return mode == 0 ? split_tile<0>(tm, tn, p, slices, A, B, bias, addend, C, s)
       : mode == 1 ? split_tile<1>(tm, tn, p, slices, A, B, bias, addend, C, s)
                   : split_tile<2>(tm, tn, p, slices, A, B, bias, addend, C, s);
}

}  // namespace flhip
