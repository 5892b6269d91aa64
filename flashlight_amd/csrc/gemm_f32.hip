// fp32 matrix products on the matrix cores, column-major:
//   mode 0  C [M x N] = A [M x K]   * B [K x N]
//   mode 1  C [M x N] = A [K x M]^T * B [K x N]
//   mode 2  C [M x N] = A [M x K]   * B [N x K]^T            (+ bias[m])
// the three products of fl::linear, and those of the recurrent layers over all time steps.  gemm32_plan chooses between the kernel
// here (v_mfma_f32_32x32x2_f32) and that of gemm_f32_split.hip.
//
// A workgroup (4 waves, 2 x 2) owns a TM x TN tile of C, a wave TM/2 x TN/2 of it: RT x CT instruction tiles of 32 x 32.
// The contraction runs in stages of 16; both operands' stages are copied to LDS by the loads themselves (buffer loads with
// the LDS modifier: no registers, no vector instructions - on these cores those would wait for the matrix pipe), RING - 1
// stages ahead of their use, one barrier per stage.
//
// An operand is contiguous either along the contraction ("k rows": B of modes 0 and 1, A of mode 1) or along the surviving
// dimension ("m rows").  The lane of an instruction holds one row and, by lane half h, one of two contraction indexes; the
// order of the indexes is free as long as both operands have it, and step e of group j takes k = 8 j + 4 h + e:
//   k rows  LDS [row][4 pieces of 4 k]: a 16-byte read is a lane's operand of four steps.  Piece p of row r lies at slot
//           p ^ ((r >> 2) & 3), so that the 16 lanes of a read pass touch distinct banks; four neighbouring lanes of a
//           load still cover 64 contiguous bytes.
//   m rows  LDS [k][row]: with RT = 2 a lane reads two neighbouring rows at once, which are its rows of the two instruction
//           tiles (tile t of a wave has the rows 2 r + t).
// Two workgroups fit a compute unit (64 KB of LDS each at 128 x 128), so one wave multiplies while its neighbour waits.
//
// What bounds it in large products is the matrix pipe, and the last round of tiles that does not fill the chip (128 x 128 tiles: 2048 x
// 6400 is 3.1 tiles per compute unit, so at most 78 % of the pipe's 153 TFLOP/s); in small ones waits (a tile's few stages, each a trip to
// memory) and the launch; over a short contraction the stores of C: with lanes along C's contiguous dimension they are whole
// cache lines wherever a column starts (lanes along the other one, 16 bytes each: 4002 x 132 x 20 5.8 -> 3.9 us).  Measured, us (before: the
// 1x1 convolution kernels with a matrix as one image's plane, thin products on the vector ALUs):
//   mode 0  2000 x 4000 x 2000  286 -> 240 (133 TFLOP/s)    1024 x 6400 x 2048  286 -> 237    1024 x 64 x 3136  42 -> 12
//   mode 1  2000 x 4000 x 2000  268 -> 235                  3072 x 6400 x 1024  353 -> 297    3136 x 64 x 1024  30 -> 10
#include <algorithm>

#include "conv2d.h"
#include "conv2d_mfma.h"
#include "gemm_f32.h"
#include "lds_direct.h"

namespace flhip {
namespace {

constexpr int KC = G32_KC, RING = 4, GTHREADS = 256;
constexpr int G32_OOB = (int)0x80000000;

// One operand's share of a stage: INSTR load instructions per wave, each 64 lanes x 16 bytes.
template <bool KROWS, int T>
struct Side {
  static constexpr int INSTR = T * KC * 4 / 1024 / 4;
  static constexpr int BYTES = T * KC * 4;
  int off[INSTR];              // byte offset of a lane's piece at stage 0 (or out of range)
  int kidx[INSTR];             // contraction index of that piece within a stage
  int step;                    // bytes from a stage to the next

  __device__ __forceinline__ void init(int r0, int R, int K, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < INSTR; ++i) {
      const int ii = wave * INSTR + i;
      if (KROWS) {
        const int row = ii * 16 + (lane >> 2), p = (lane & 3) ^ ((row >> 2) & 3);
        kidx[i] = 4 * p;
        off[i] = r0 + row < R ? ((r0 + row) * K + 4 * p) * 4 : G32_OOB;
      } else {
        const int piece = ii * 64 + lane, k = piece / (T / 4), m = 4 * (piece % (T / 4));
        kidx[i] = k;
        off[i] = r0 + m < R ? (k * R + r0 + m) * 4 : G32_OOB;
      }
    }
    step = KROWS ? KC * 4 : KC * R * 4;
  }
  // the stage at byte offset `at` of every row, to the ring slot at lds (workgroup address).  CHECKED: only its first
  // `left` contraction indexes exist (none of them, or fewer), the others read zero
  template <bool CHECKED>
  __device__ __forceinline__ void load(intx4_t rsrc, unsigned lds, int at, int left, int wave) const {
#pragma unroll
    for (int i = 0; i < INSTR; ++i)
      pd_load_lds(rsrc, lds + (wave * INSTR + i) * 1024, CHECKED && kidx[i] >= left ? G32_OOB : off[i], at);
  }
};

// the operands of one group of 8 contraction indexes: v[t][e] for instruction tile t and step e
template <bool KROWS, int T, int NT>
__device__ __forceinline__ void read_group(const float* lds, int j, int w, int fr, int h, float (&v)[NT][4]) {
  if constexpr (KROWS) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = w * 32 * NT + t * 32 + fr;
      const float4 f = *reinterpret_cast<const float4*>(lds + row * KC + 4 * ((2 * j + h) ^ ((row >> 2) & 3)));
      v[t][0] = f.x; v[t][1] = f.y; v[t][2] = f.z; v[t][3] = f.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float* at = lds + (8 * j + 4 * h + e) * T + w * 32 * NT + NT * fr;
      if constexpr (NT == 2) {
        const float2 f = *reinterpret_cast<const float2*>(at);
        v[0][e] = f.x; v[1][e] = f.y;
      } else {
        v[0][e] = *at;
      }
    }
  }
}

template <int MODE, int TM, int TN>
__global__ void __launch_bounds__(GTHREADS, 2)
gemm32_kernel(Gemm32 p, const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
              const float* addend, float* C) {
  constexpr bool AK = MODE == 1, BK = MODE != 2;
  constexpr int RT = TM / 64, CT = TN / 64;
  typedef Side<AK, TM> SA;
  typedef Side<BK, TN> SB;
  constexpr int STAGE = SA::BYTES + SB::BYTES;
  extern __shared__ __align__(16) float g32_lds[];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  if (blockIdx.z) A = p.A2, B = p.B2, bias = p.bias2, C = p.C2;
  const int tile = gemm32_tile_of(blockIdx.x, p.mtiles * p.ntiles);
  const int m0 = (tile % p.mtiles) * TM, n0 = (tile / p.mtiles) * TN;
  const int s0 = blockIdx.y * p.sps, send = min(p.nstages, s0 + p.sps);

  SA sa;
  SB sb;
  sa.init(m0, p.M, p.K, wave, lane);
  sb.init(n0, p.N, p.K, wave, lane);
  const intx4_t ar = pd_rsrc(A, p.a_bytes), br = pd_rsrc(B, p.b_bytes);
  const unsigned lds0 = pd_lds_addr(g32_lds);
  // stages from `send` on are not fetched, but every stage counts the same number of loads
  auto stage_in = [&](auto checked, int slot, int s) __attribute__((always_inline)) {
    constexpr bool CHECKED = decltype(checked)::value;
    const int left = s < send ? p.K - s * KC : 0, at = CHECKED && s >= send ? 0 : s;
    const unsigned lds = lds0 + (unsigned)slot * STAGE;
    sa.template load<CHECKED>(ar, lds, at * sa.step, left, wave);
    sb.template load<CHECKED>(br, lds + SA::BYTES, at * sb.step, left, wave);
  };
  constexpr std::integral_constant<bool, true> checked{};
  constexpr std::integral_constant<bool, false> whole{};
  floatx16 acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) stage_in(checked, s, s0 + s);
  auto stage = [&](auto checked_, int slot, int s) __attribute__((always_inline)) {
    // this stage has landed when at most the two behind it are still in flight
    if constexpr (SA::INSTR + SB::INSTR == 4) PD_WAIT_VM(8);
    else if constexpr (SA::INSTR + SB::INSTR == 3) PD_WAIT_VM(6);
    else PD_WAIT_VM(4);
    __syncthreads();                         // ... for every wave, and every wave is done with the slot of stage s - 1
    const float* la = g32_lds + slot * (STAGE / 4);
    const float* lb = la + SA::BYTES / 4;
    float a[KC / 8][RT][4], b[KC / 8][CT][4];
#pragma unroll
    for (int j = 0; j < KC / 8; ++j) {
      read_group<AK, TM, RT>(la, j, wm, fr, h, a[j]);
      read_group<BK, TN, CT>(lb, j, wn, fr, h, b[j]);
      if (j == 0) stage_in(checked_, (slot + RING - 1) % RING, s + RING - 1);
    }
#pragma unroll
    for (int j = 0; j < KC / 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int c = 0; c < CT; ++c)
            acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j][c][e], a[j][i][e], acc[i][c], 0, 0, 0);
  };
  int s = s0;
  // rounds of the ring whose look-ahead is whole stages
  const int sfull = min(send, p.K / KC) - (RING - 1);
  for (; s + RING <= sfull; s += RING) {
#pragma unroll
    for (int x = 0; x < RING; ++x) stage(whole, x, s + x);
  }
  for (; s < send; s += RING) {
#pragma unroll
    for (int x = 0; x < RING; ++x)
      if (s + x < send) stage(checked, x, s + x);
  }
  PD_WAIT_VM(0);                             // nothing may land in LDS after the workgroup has ended

  // B's columns are the rows of the instruction's tiles, so that the lanes of a store are neighbours along C's contiguous
  // dimension, wherever its columns start: element r of a lane is column 8 (r / 4) + 4 h + r % 4 and row fr of C's tile
  // (M is below 2^22: a tile's columns lie within 2 GiB.  A store past the last column is out of the buffer's range, one past the
  // last row is put there, and so neither needs a branch around it.)
  const int m = m0 + wm * 32 * RT + (AK ? fr : RT * fr);      // and 32 (AK) or one row further for the second tile
  constexpr int MSTEP = AK ? 32 : 1;
  const int nl = wn * 32 * CT + (BK ? 4 * h : CT * 4 * h);
  const size_t origin = (size_t)n0 * p.M, left = ((size_t)(p.N - n0) * p.M) * 4;
  const unsigned range = left < 0x7fffffffu ? (unsigned)left : 0x7fffffffu;
  const __amdgpu_buffer_rsrc_t orsrc = make_rsrc(C + (size_t)blockIdx.y * p.slice + origin, range);
  int at[RT];
  float bv[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const bool in = m + i * MSTEP < p.M;
    at[i] = in ? (nl * p.M + m + i * MSTEP) * 4 : G32_OOB;
    bv[i] = bias && in ? bias[m + i * MSTEP] : 0.f;
  }
  auto store = [&](auto added) __attribute__((always_inline)) {
    constexpr bool ADD = decltype(added)::value;
    const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(ADD ? addend + origin : nullptr, range);
#pragma unroll
    for (int c = 0; c < CT; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int col = 8 * (r >> 2) + (r & 3), o = (BK ? c * 32 + col : CT * col + c) * p.M * 4;
        if constexpr (RT == 2 && !AK) {          // (M is a multiple of 4)
          float2 v = make_float2(acc[0][c][r] + bv[0], acc[1][c][r] + bv[1]);
          if (ADD) {
            const uintx2_t f = __builtin_amdgcn_raw_buffer_load_b64(arsrc, at[0] + o, 0, 0);
            v.x += __uint_as_float(f.x); v.y += __uint_as_float(f.y);
          }
          __builtin_amdgcn_raw_buffer_store_b64(uintx2_t{__float_as_uint(v.x), __float_as_uint(v.y)}, orsrc, at[0] + o, 0, 0);
        } else {
#pragma unroll
          for (int i = 0; i < RT; ++i) {
            float v = acc[i][c][r] + bv[i];
            if (ADD) v += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(arsrc, at[i] + o, 0, 0));
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), orsrc, at[i] + o, 0, 0);
          }
        }
      }
  };
  if (addend) store(std::true_type{});
  else store(std::false_type{});
}

// out = sum of the slices (+ bias[row]) (+ addend, which may be out); rows of M4 pieces, M a multiple of 4 where there is
// a bias.  blockIdx.y = 1: those of a second product behind them, with bias2, to out2
__global__ void __launch_bounds__(256) gemm32_sum_kernel(const float4* __restrict__ part, const float* __restrict__ bias,
                                                         const float4* addend, float4* out, size_t n4, int M4, int slices, const float* bias2, float4* out2) {
  if (blockIdx.y) part += slices * n4, bias = bias2, out = out2;
  for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n4; i += (size_t)gridDim.x * 256) {
    float4 v = part[i];
#pragma unroll 4
    for (int k = 1; k < slices; ++k) {       // loads in flight together, sums in slice order
      const float4 w = part[(size_t)k * n4 + i];
      v.x += w.x; v.y += w.y; v.z += w.z; v.w += w.w;
    }
    if (bias) {
      const float* b = bias + 4 * (i % (size_t)M4);
      v.x += b[0]; v.y += b[1]; v.z += b[2]; v.w += b[3];
    }
    if (addend) {
      const float4 f = addend[i];
      v.x += f.x; v.y += f.y; v.z += f.z; v.w += f.w;
    }
    out[i] = v;
  }
}

struct Gemm32Plan {
  Gemm32 p;
  int tm, tn, slices;
  bool parts;                  // on the kernel of gemm_f32_split.hip
};

// The tile and the number of contraction slices with the least estimated time.  64 x 64 tiles run on the fp32 instruction, larger
// ones in three bf16 parts (gemm_f32_split.hip).  A tile's workgroup takes `stage` (in units of 1.5 us) per stage of 16 while its
// compute unit is shared, `alone` times that where it has the unit for itself, and `more` stages' time around its loop; slices cost
// their partial results' traffic and a second launch.  Fitted to 1067 random products (16 to 8192 a side, 2 MFLOP to 60 GFLOP) with every tile
// and 1 to 16 slices timed: the choice is 1.9 % behind the fastest of them in the geometric mean.  Where the fastest was 64 x 64
// is three quarters of them, from 0.1 GFLOP down nearly all: few tiles, short contractions.
struct Gemm32Tile {
  int tm, tn;
  double stage, alone, more;
};
constexpr Gemm32Tile G32_TILES[] = {{64, 64, 0.17, 1.07, 5}, {128, 64, 0.24, 1.47, 6}, {64, 128, 0.27, 1.47, 6}, {128, 128, 0.40, 1.25, 8}};
// fp32_sums (modes 0 and 1): every tile on the fp32 instruction, in units of a 128 x 128 stage (2048 matrix cycles): a smaller
// tile reads more LDS per product (64 x 64 tiles reach about 0.85 of the rate of 128 x 128), and one alone on its unit has nobody to hide its
// waits behind.
constexpr Gemm32Tile G32_FP32_TILES[] = {{128, 128, 1.0, 1.25, 6}, {128, 64, 0.5 / 0.93, 1.25, 6}, {64, 128, 0.5 / 0.93, 1.25, 6}, {64, 64, 0.25 / 0.85, 1.25, 6}};

// Rows of no whole pieces: the kernels in three parts alone, which load what is contiguous along the rows one by one and ask a row's
// last piece for its end.  us, the 1x1 layers' kernels on the fp32 instruction (which stay where the fp32 instruction's sums do) / here: A^T B 2000 x
// 4000 x 9998 1681 / 856, 2000 x 1500 x 4001 263 / 150, 256 x 500 x 4001 188 / 18, 256 x 150 x 29 5.9 / 5.3; A B^T 9998 x 2000 x 4000 1631 / 921, 4001 x 768
// x 1500 107 / 69, 1001 x 256 x 500 15 / 13, 130 x 768 x 150 8.9 / 8.7, but 29 x 768 x 150 7.9 / 8.9, 29 x 768 x 4000 16.2 / 17.9.
bool gemm32_ragged(int mode, int M, int N, int K, bool fp32_sums) {
  const double macs = (double)M * N * K;
  if (fp32_sums || options().matmul_fp32_cores || K < KC) return false;
  return mode == 2 ? macs >= 1e7 && (K <= 3000 || macs >= 2e8) : macs >= 1e6;
}

// pair > 0: for two such products in a launch, whose slices fit `pair` bytes
bool gemm32_plan(int mode, int M, int N, int K, bool sliced, bool fp32_sums, Gemm32Plan* best, size_t pair = 0) {
  const bool ak = mode == 1, bk = mode != 2;
  const bool pieces = (ak ? K : M) % 4 == 0 && (bk ? K : N) % 4 == 0;      // rows of whole 16-byte pieces
  if (!pieces && !gemm32_ragged(mode, M, N, K, fp32_sums)) return false;
  const long long ab = (long long)M * K * 4, bb = (long long)N * K * 4;
  if (ab >= (1ll << 31) || bb >= (1ll << 31) || (long long)M * N >= (1ll << 31) || M >= 1 << 22) return false;
  const int cus = mfma_num_cus(), nst = (K + KC - 1) / KC;
  const bool whole = mode != 2 && (fp32_sums || options().matmul_fp32_cores);      // tiles of every size on the fp32 instruction
  const double unit = whole ? 2048.0 / 2.4e9 * 4e12 : 8e6, second = whole ? 3.0 : 1.6;
  double best_cost = 1e30;
  for (const Gemm32Tile& t : whole ? G32_FP32_TILES : G32_TILES) {
    if (!whole && t.tm * t.tn > 64 * 64 && (K < KC || options().matmul_fp32_cores)) continue;
    if (!pieces && t.tm * t.tn == 64 * 64) continue;
    const int mt = (M + t.tm - 1) / t.tm, nt = (N + t.tn - 1) / t.tn;
    for (int ns = 1; ns <= (sliced ? 16 : 1); ++ns) {
      if (ns > 1 && (nst / ns < 8 || ((size_t)M * N) % 4 != 0 || (pair && (size_t)8 * ns * M * N > pair))) break;
      const int sps = (nst + ns - 1) / ns;
      if ((nst + sps - 1) / sps != ns) continue;
      const long long wgs = (long long)mt * nt * ns * (pair ? 2 : 1), rounds = (wgs + cus - 1) / cus;
      double cost = (double)rounds * (sps + t.more) * t.stage * (rounds == 1 ? t.alone : 1.0);
      if (ns > 1) cost += (double)(ns + 1) * M * N * (pair ? 8 : 4) / unit + second;
      if (cost < best_cost) {
        best_cost = cost;
        best->tm = t.tm; best->tn = t.tn; best->slices = ns; best->parts = !whole && t.tm * t.tn > 64 * 64;
        best->p.mtiles = mt; best->p.ntiles = nt; best->p.sps = sps;
      }
    }
  }
  best->p.M = M; best->p.N = N; best->p.K = K;
  best->p.nstages = nst;
  best->p.a_bytes = (unsigned)ab; best->p.b_bytes = (unsigned)bb;
  best->p.slice = (size_t)M * N;
  return best_cost < 1e30;
}

template <int MODE, int TM, int TN>
int gemm32_go(const Gemm32Plan& pl, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  constexpr size_t lds = (size_t)RING * (TM + TN) * KC * 4;
  auto kernel = gemm32_kernel<MODE, TM, TN>;
  if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return -1;
  hipLaunchKernelGGL(kernel, dim3((unsigned)(pl.p.mtiles * pl.p.ntiles), (unsigned)pl.slices, pl.p.C2 ? 2 : 1), dim3(GTHREADS), lds, s, pl.p, A, B,
                     bias, addend, C);
  return check_launch("matmul (fp32)");
}
template <int MODE>
int gemm32_tile(const Gemm32Plan& pl, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  if constexpr (MODE == 2) return gemm32_go<2, 64, 64>(pl, A, B, bias, addend, C, s);
  if (pl.tm == 128) return pl.tn == 128 ? gemm32_go<MODE, 128, 128>(pl, A, B, bias, addend, C, s) : gemm32_go<MODE, 128, 64>(pl, A, B, bias, addend, C, s);
  return pl.tn == 128 ? gemm32_go<MODE, 64, 128>(pl, A, B, bias, addend, C, s) : gemm32_go<MODE, 64, 64>(pl, A, B, bias, addend, C, s);
}

}  // namespace

// bytes of workspace with which gemm32 may cut the contraction (0: it does not, or declines)
size_t gemm32_ws_bytes(int mode, int M, int N, int K, bool fp32_sums) {
  Gemm32Plan pl{};
  if (!gemm32_plan(mode, M, N, K, true, fp32_sums, &pl) || pl.slices == 1) return 0;
  return (size_t)pl.slices * M * N * sizeof(float);
}

int gemm32(int mode, const float* A, const float* B, float* C, int M, int N, int K, const float* bias, void* ws, size_t ws_bytes,
           hipStream_t s, const float* addend, bool (*take)(int, int, int, bool), bool fp32_sums) {
  Gemm32Plan pl{};
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
       reinterpret_cast<uintptr_t>(addend)) % 16 != 0)
    return -1;
  if (take && ((mode == 1 ? K : M) % 4 != 0 || (mode != 2 ? K : N) % 4 != 0)) return -1;      // (a thin product of such rows stays on the kernels for those)
  const bool can = ws != nullptr && (!bias || M % 4 == 0);
  if (!gemm32_plan(mode, M, N, K, can || take, fp32_sums, &pl)) return -1;
  const bool fits = can && ws_bytes >= (size_t)pl.slices * M * N * sizeof(float);
  if (take && ((pl.slices > 1 && !fits) || !take(M, N, K, pl.slices > 1))) return -1;
  if (pl.slices > 1 && !fits && !gemm32_plan(mode, M, N, K, false, fp32_sums, &pl)) return -1;
  float* dst = pl.slices > 1 ? static_cast<float*>(ws) : C;
  const float *b = pl.slices > 1 ? nullptr : bias, *a = pl.slices > 1 ? nullptr : addend;
  const int rc = pl.parts  ? gemm32_split(mode, pl.tm, pl.tn, pl.slices, pl.p, A, B, b, a, dst, s)
               : mode == 0 ? gemm32_tile<0>(pl, A, B, b, a, dst, s)
               : mode == 1 ? gemm32_tile<1>(pl, A, B, b, a, dst, s)
                           : gemm32_tile<2>(pl, A, B, b, a, dst, s);
  if (rc || pl.slices == 1) return rc;
  const size_t n4 = (size_t)M * N / 4;
  hipLaunchKernelGGL(gemm32_sum_kernel, dim3((unsigned)std::min<size_t>((n4 + 255) / 256, 4096)), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(ws), bias,
                     reinterpret_cast<const float4*>(addend), reinterpret_cast<float4*>(C), n4, M / 4, pl.slices, (const float*)nullptr, (float4*)nullptr);
  return check_launch("matmul (fp32, slices added)");
}

// gemm32 of two products of one shape in a launch (and one that adds both's slices, where the workspace holds them); -1: one after the other.
// Thin ones (N <= 128) too.  The pass with pairs against one product after the other, 170 random layers of two directions, 64 to 1024 units, 8 to
// 9200 columns of all steps: forward 0.75 to 1.00 (N <= 128 0.75 to 0.97, 3 to 31 us less a pass), weight gradients 0.85 to 1.00 (LSTM of 768
// units over 2873 columns 1.01, less than its runs differ), input gradients 0.69 to 1.01.
int gemm32_pair(int mode, const float* A, const float* A2, const float* B, const float* B2, float* C, float* C2, int M, int N, int K, const float* bias, const float* bias2,
                void* ws, size_t ws_bytes, hipStream_t s) {
  Gemm32Plan pl{};
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(A2) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(B2) |
       reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(C2)) % 16 != 0)
    return -1;
  if (bias && M % 4 != 0) return -1;
  if (mode != 2 && (options().matmul_valu || options().matmul_planes >= 0)) return -1;      // (the kernels that matmul chooses by them)
  if (!gemm32_plan(mode, M, N, K, ws != nullptr, false, &pl, std::max<size_t>(ws_bytes, 1))) return -1;
  const bool cut = pl.slices > 1;
  float* const part = static_cast<float*>(ws);
  pl.p.A2 = A2; pl.p.B2 = B2; pl.p.bias2 = cut ? nullptr : bias2;
  pl.p.C2 = cut ? part + (size_t)pl.slices * M * N : C2;
  float* const dst = cut ? part : C;
  const float* const b = cut ? nullptr : bias;
  const int rc = pl.parts  ? gemm32_split(mode, pl.tm, pl.tn, pl.slices, pl.p, A, B, b, nullptr, dst, s)
               : mode == 0 ? gemm32_tile<0>(pl, A, B, b, nullptr, dst, s)
               : mode == 1 ? gemm32_tile<1>(pl, A, B, b, nullptr, dst, s)
                           : gemm32_tile<2>(pl, A, B, b, nullptr, dst, s);
  if (rc || !cut) return rc;
  const size_t n4 = (size_t)M * N / 4;
  hipLaunchKernelGGL(gemm32_sum_kernel, dim3((unsigned)std::min<size_t>((n4 + 255) / 256, 4096), 2), dim3(256), 0, s, reinterpret_cast<const float4*>(ws),
                     bias, (const float4*)nullptr, reinterpret_cast<float4*>(C), n4, M / 4, pl.slices, bias2, reinterpret_cast<float4*>(C2));
  return check_launch("matmul (fp32, two products' slices added)");
}

}  // namespace flhip
