// fp32 matrix products on the matrix cores, column-major:
//   mode 0  C [M x N] = A [M x K]   * B [K x N]
//   mode 1  C [M x N] = A [K x M]^T * B [K x N]
//   mode 2  C [M x N] = A [M x K]   * B [N x K]^T            (+ bias[m])
// the three products of fl::linear, and those of the recurrent layers over all time steps.  gemm32_plan chooses between the kernel
// here (v_mfma_f32_32x32x2_f32 on 64 x 64 tiles, for few tiles or short contractions) and that of gemm_f32_split.hip.
//
// A workgroup (4 waves, 2 x 2) owns a 64 x 64 tile of C, a wave an instruction tile of 32 x 32 of it.
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
//   m rows  LDS [k][row]
//
// What bounds it: waits (a tile's few stages, each a trip to memory) and the launch; over a short contraction the stores of C: with
// lanes along C's contiguous dimension they are whole cache lines wherever a column starts (lanes along the other one, 16 bytes
// each: 4002 x 132 x 20 5.8 -> 3.9 us).  Thin products: 1024 x 64 x 3136 42 -> 12 us, 3136 x 64 x 1024 30 -> 10 (before: on the vector ALUs).
#include <algorithm>

#include "conv2d.h"
#include "conv2d_mfma.h"
#include "gemm_f32.h"
#include "lds_direct.h"

namespace flhip {
namespace {

constexpr int KC = G32_KC, RING = 4, GTHREADS = 256, T = 64;      // T: rows and columns of a tile
constexpr int G32_OOB = (int)0x80000000;

// One operand's share of a stage: INSTR load instructions per wave, each 64 lanes x 16 bytes.
template <bool KROWS>
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

// the operands of one group of 8 contraction indexes: v[e] for step e
template <bool KROWS>
__device__ __forceinline__ void read_group(const float* lds, int j, int w, int fr, int h, float (&v)[4]) {
  const int row = w * 32 + fr;
  if constexpr (KROWS) {
    const float4 f = *reinterpret_cast<const float4*>(lds + row * KC + 4 * ((2 * j + h) ^ ((row >> 2) & 3)));
    v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = lds[(8 * j + 4 * h + e) * T + row];
  }
}

template <int MODE>
__global__ void __launch_bounds__(GTHREADS, 2)
gemm32_kernel(Gemm32 p, const float* __restrict__ A, const float* __restrict__ B, const float* __restrict__ bias,
              const float* addend, float* C) {
  constexpr bool AK = MODE == 1, BK = MODE != 2;
  typedef Side<AK> SA;
  typedef Side<BK> SB;
  constexpr int STAGE = SA::BYTES + SB::BYTES;
  extern __shared__ __align__(16) float g32_lds[];
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave & 1, wn = wave >> 1;
  const int tile = gemm32_tile_of(blockIdx.x, p.mtiles * p.ntiles);
  const int m0 = (tile % p.mtiles) * T, n0 = (tile / p.mtiles) * T;
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
  floatx16 acc;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = 0.f;
#pragma unroll
  for (int s = 0; s < RING - 1; ++s) stage_in(checked, s, s0 + s);
  auto stage = [&](auto checked_, int slot, int s) __attribute__((always_inline)) {
    // this stage has landed when at most the two behind it are still in flight
    PD_WAIT_VM(4);
    static_assert(SA::INSTR + SB::INSTR == 2, "loads of two stages");
    __syncthreads();                         // ... for every wave, and every wave is done with the slot of stage s - 1
    const float* la = g32_lds + slot * (STAGE / 4);
    const float* lb = la + SA::BYTES / 4;
    float a[KC / 8][4], b[KC / 8][4];
#pragma unroll
    for (int j = 0; j < KC / 8; ++j) {
      read_group<AK>(la, j, wm, fr, h, a[j]);
      read_group<BK>(lb, j, wn, fr, h, b[j]);
      if (j == 0) stage_in(checked_, (slot + RING - 1) % RING, s + RING - 1);
    }
#pragma unroll
    for (int j = 0; j < KC / 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j][e], a[j][e], acc, 0, 0, 0);
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

  // B's columns are the rows of the instruction's tile, so that the lanes of a store are neighbours along C's contiguous
  // dimension, wherever its columns start: element r of a lane is column 8 (r / 4) + 4 h + r % 4 and row fr of C's tile
  // (M is below 2^22: a tile's columns lie within 2 GiB.  A store past the last column is out of the buffer's range, one past the
  // last row is put there, and so neither needs a branch around it.)
  const int m = m0 + wm * 32 + fr, nl = wn * 32 + 4 * h;
  const size_t origin = (size_t)n0 * p.M, left = ((size_t)(p.N - n0) * p.M) * 4;
  const unsigned range = left < 0x7fffffffu ? (unsigned)left : 0x7fffffffu;
  const __amdgpu_buffer_rsrc_t orsrc = make_rsrc(C + (size_t)blockIdx.y * p.slice + origin, range);
  const bool in = m < p.M;
  const int at = in ? (nl * p.M + m) * 4 : G32_OOB;
  const float bv = bias && in ? bias[m] : 0.f;
  auto store = [&](auto added) __attribute__((always_inline)) {
    constexpr bool ADD = decltype(added)::value;
    const __amdgpu_buffer_rsrc_t arsrc = make_rsrc(ADD ? addend + origin : nullptr, range);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int o = (8 * (r >> 2) + (r & 3)) * p.M * 4;
      float v = acc[r] + bv;
      if (ADD) v += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(arsrc, at + o, 0, 0));
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), orsrc, at + o, 0, 0);
    }
  };
  if (addend) store(std::true_type{});
  else store(std::false_type{});
}

// out = sum of the slices (+ bias[row]) (+ addend, which may be out); rows of M4 pieces, M a multiple of 4 where there is
// a bias
__global__ void __launch_bounds__(256) gemm32_sum_kernel(const float4* __restrict__ part, const float* __restrict__ bias,
                                                         const float4* addend, float4* out, size_t n4, int M4, int slices) {
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

bool gemm32_plan(int mode, int M, int N, int K, bool sliced, Gemm32Plan* best) {
  const bool ak = mode == 1, bk = mode != 2;
  if ((ak ? K : M) % 4 != 0 || (bk ? K : N) % 4 != 0) return false;      // rows of whole 16-byte pieces
  const long long ab = (long long)M * K * 4, bb = (long long)N * K * 4;
  if (ab >= (1ll << 31) || bb >= (1ll << 31) || (long long)M * N >= (1ll << 31) || M >= 1 << 22) return false;
  const int cus = mfma_num_cus(), nst = (K + KC - 1) / KC;
  double best_cost = 1e30;
  for (const Gemm32Tile& t : G32_TILES) {
    if (t.tm * t.tn > 64 * 64 && (K < KC || options().matmul_fp32_cores)) continue;
    const int mt = (M + t.tm - 1) / t.tm, nt = (N + t.tn - 1) / t.tn;
    for (int ns = 1; ns <= (sliced ? 16 : 1); ++ns) {
      if (ns > 1 && (nst / ns < 8 || ((size_t)M * N) % 4 != 0)) break;
      const int sps = (nst + ns - 1) / ns;
      if ((nst + sps - 1) / sps != ns) continue;
      const long long wgs = (long long)mt * nt * ns, rounds = (wgs + cus - 1) / cus;
      double cost = (double)rounds * (sps + t.more) * t.stage * (rounds == 1 ? t.alone : 1.0);
      if (ns > 1) cost += (double)(ns + 1) * M * N * 4 / 8e6 + 1.6;
      if (cost < best_cost) {
        best_cost = cost;
        best->tm = t.tm; best->tn = t.tn; best->slices = ns;
        best->p.mtiles = mt; best->p.ntiles = nt; best->p.sps = sps;
      }
    }
  }
  best->p.M = M; best->p.N = N; best->p.K = K;
  best->p.nstages = nst;
  best->p.a_bytes = (unsigned)ab; best->p.b_bytes = (unsigned)bb;
  best->p.slice = (size_t)M * N;
  return true;
}

template <int MODE>
int gemm32_small(const Gemm32Plan& pl, const float* A, const float* B, const float* bias, const float* addend, float* C, hipStream_t s) {
  hipLaunchKernelGGL((gemm32_kernel<MODE>), dim3((unsigned)(pl.p.mtiles * pl.p.ntiles), (unsigned)pl.slices), dim3(GTHREADS),
                     RING * 2 * T * KC * 4, s, pl.p, A, B, bias, addend, C);
  return check_launch("matmul (fp32)");
}

}  // namespace

// bytes of workspace with which gemm32 may cut the contraction (0: it does not, or declines)
size_t gemm32_ws_bytes(int mode, int M, int N, int K) {
  Gemm32Plan pl{};
  if (!gemm32_plan(mode, M, N, K, true, &pl) || pl.slices == 1) return 0;
  return (size_t)pl.slices * M * N * sizeof(float);
}

int gemm32(int mode, const float* A, const float* B, float* C, int M, int N, int K, const float* bias, void* ws, size_t ws_bytes,
           hipStream_t s, const float* addend, bool (*take)(int, int, int, bool)) {
  Gemm32Plan pl{};
  if ((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B) | reinterpret_cast<uintptr_t>(C) |
       reinterpret_cast<uintptr_t>(addend)) % 16 != 0)
    return -1;
  const bool can = ws != nullptr && (!bias || M % 4 == 0);
  if (!gemm32_plan(mode, M, N, K, can || take, &pl)) return -1;
  const bool fits = can && ws_bytes >= (size_t)pl.slices * M * N * sizeof(float);
  if (take && ((pl.slices > 1 && !fits) || !take(M, N, K, pl.slices > 1))) return -1;
  if (pl.slices > 1 && !fits && !gemm32_plan(mode, M, N, K, false, &pl)) return -1;
  float* dst = pl.slices > 1 ? static_cast<float*>(ws) : C;
  const float *b = pl.slices > 1 ? nullptr : bias, *a = pl.slices > 1 ? nullptr : addend;
  const int rc = pl.tm * pl.tn > 64 * 64 ? gemm32_split(mode, pl.tm, pl.tn, pl.slices, pl.p, A, B, b, a, dst, s)
               : mode == 0               ? gemm32_small<0>(pl, A, B, b, a, dst, s)
               : mode == 1               ? gemm32_small<1>(pl, A, B, b, a, dst, s)
                                         : gemm32_small<2>(pl, A, B, b, a, dst, s);
  if (rc || pl.slices == 1) return rc;
  const size_t n4 = (size_t)M * N / 4;
  hipLaunchKernelGGL(gemm32_sum_kernel, dim3((unsigned)std::min<size_t>((n4 + 255) / 256, 4096)), dim3(256), 0, s,
                     reinterpret_cast<const float4*>(ws), bias,
                     reinterpret_cast<const float4*>(addend), reinterpret_cast<float4*>(C), n4, M / 4, pl.slices);
  return check_launch("matmul (fp32, slices added)");
}

}  // namespace flhip
