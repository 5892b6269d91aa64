// rnn / rnnBackward: ReLU / tanh RNN, LSTM and GRU, stacked and bidirectional, with the
// semantics and the flat weight order of the cuDNN calls the reference makes
// (flashlight/fl/autograd/tensor/backend/cudnn/RNN.cpp:62-375): per pseudo-layer
// (layer-major, forward direction first) the input matrices of every gate
// ([hidden][in], row-major) then the recurrent ones; after all matrices, per
// pseudo-layer the input biases then the recurrent biases.  Gates: LSTM i, f, g, o;
// GRU r, z, n with n = tanh(W_n x + b_Wn + r * (R_n h + b_Rn)), h' = (1-z)*n + z*h.
//
// Structure: the input projections of all time steps of a pseudo-layer are one matrix
// product; the recurrence is one launch per layer where the hidden size allows and the sequence
// is long enough to gain by it, else a launch per step, or a loop over time of (recurrent product, gate kernel).
// The products go through flhip_matmul (matrix cores where the shapes allow).  The
// forward pass keeps, per pseudo-layer and in step order, the state before every step,
// the gate activations and (GRU) R_n h + b_Rn in the reserve buffer; the backward pass
// walks the steps in reverse, writes the pre-activation gradients of all steps, and
// turns them into dx, dW, dR and the bias gradients with four products / reductions.
// Layouts follow Flashlight: x [input, B, T] column-major = memory [T][B][input], etc.
// fp32 only; no dropout between layers (the closure's dropProb must be 0).
#include <algorithm>
#include <atomic>

#include "common.h"
#include "conv2d.h"
#include "conv2d_mfma.h"

extern "C" int flhip_sum_columns_ws(const void* x, float* out, int32_t rows, int32_t cols, int dtype, void* ws,
                                    size_t ws_bytes, void* stream);
extern "C" size_t flhip_sum_columns_workspace_bytes(int32_t rows, int32_t cols, int dtype);

namespace flhip {
namespace {

enum { RNN_RELU = 0, RNN_TANH = 1, RNN_LSTM = 2, RNN_GRU = 3 };

struct RnnGeom {
  int I, H, L, D, mode, T, B, G;
  size_t BH, GH;
  size_t nparams;
  float dropout;
  uint32_t seed_lo, seed_hi;
};

constexpr int gates_of(int mode) { return mode == RNN_LSTM ? 4 : mode == RNN_GRU ? 3 : 1; }

// widest layer input, in whole 16-byte pieces so that what follows in the workspace stays aligned
inline size_t widest_input(const RnnGeom& g) { return (std::max<size_t>(g.I, (size_t)g.D * g.H) + 3) & ~(size_t)3; }

int make_geom(const flhip_rnn_desc* d, RnnGeom* g) {
  FLHIP_REQUIRE(d, "rnn: null descriptor");
  FLHIP_REQUIRE(d->input_size > 0 && d->hidden_size > 0 && d->num_layers > 0 && d->seq_len > 0 &&
                    d->batch > 0,
                "rnn: sizes must be positive");
  FLHIP_REQUIRE(d->mode >= RNN_RELU && d->mode <= RNN_GRU, "rnn: unknown mode");
  FLHIP_REQUIRE(d->dtype == FLHIP_F32, "rnn: f32 only");
  FLHIP_REQUIRE(d->dropout >= 0.f && d->dropout < 1.f, "rnn: dropout must be in [0, 1)");
  g->dropout = d->dropout; g->seed_lo = d->seed_lo; g->seed_hi = d->seed_hi;
  g->I = d->input_size; g->H = d->hidden_size; g->L = d->num_layers; g->D = d->bidirectional ? 2 : 1;
  g->mode = d->mode; g->T = d->seq_len; g->B = d->batch; g->G = gates_of(d->mode);
  g->BH = (size_t)g->B * g->H;
  g->GH = (size_t)g->G * g->H;
  size_t n = 0;
  for (int l = 0; l < g->L; ++l) {
    const size_t in = l == 0 ? g->I : (size_t)g->D * g->H;
    n += g->D * (g->GH * (in + g->H) + 2 * g->GH);
  }
  g->nparams = n;
  FLHIP_REQUIRE((size_t)g->T * g->B * std::max<size_t>(g->GH, (size_t)g->D * g->H) < (1u << 30) &&
                    n < (1u << 30),
                "rnn: problem too large for 32-bit indices");
  return FLHIP_OK;
}

struct Offsets {
  size_t W, R, bW, bR;
};
Offsets offsets(const RnnGeom& g, int pl) {
  Offsets o{};
  size_t off = 0;
  for (int p = 0; p < g.L * g.D; ++p) {
    const size_t in = p / g.D == 0 ? g.I : (size_t)g.D * g.H;
    if (p == pl) {
      o.W = off;
      o.R = off + g.GH * in;
    }
    off += g.GH * (in + g.H);
  }
  o.bW = off + (size_t)pl * 2 * g.GH;
  o.bR = o.bW + g.GH;
  return o;
}

// reserve buffer, in floats: per pseudo-layer {HP [(T+1)*BH], CP [(T+1)*BH] (LSTM),
// GT [T*B*GH], RN [T*BH] (GRU)}, then the outputs of layers 0 .. L-2 ([T*B*D*H] each)
struct Reserve {
  size_t per_pl, hp, cp, gt, rn, acts, total;
};
Reserve reserve_layout(const RnnGeom& g) {
  Reserve r{};
  size_t o = 0;
  r.hp = o; o += (size_t)(g.T + 1) * g.BH;
  r.cp = o; if (g.mode == RNN_LSTM) o += (size_t)(g.T + 1) * g.BH;
  r.gt = o; o += (size_t)g.T * g.B * g.GH;
  r.rn = o; if (g.mode == RNN_GRU) o += (size_t)g.T * g.BH;
  r.per_pl = o;
  r.acts = r.per_pl * g.L * g.D;
  r.total = r.acts + (size_t)(g.L - 1) * g.T * g.B * g.D * g.H;
  return r;
}

// workspace, in floats (one call): forward {XP [T*B*GH], RP [B*GH], bias [GH]};
// backward {dGW [T*B*GH], dGR [T*B*GH], gout [T*B*D*H], gin [T*B*inmax], tmp [T*B*inmax],
// dh_dir [2*BH], dc [BH], dh_rec [slices*BH]}
// The recurrent products of one time step are small (batch columns): their contraction is
// cut into slices so that enough workgroups run, and the gate kernels add the partial
// products.  Slices for a product with M rows, N columns, contraction K:
int step_slices(size_t M, size_t N, size_t K, int* ksplit) {
  const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64), chunks = (long long)(K + 31) / 32;
  // from 32 tiles on, one step is bound by its two launches, not by the product
  long long k = tiles >= 32 ? 1 : 256 / tiles;
  if (k > chunks / 4) k = chunks / 4;   // at least four chunks of 32 per slice
  if (k > 32) k = 32;
  if (k < 1) k = 1;
  *ksplit = (int)k;
  return mfma_gemm_slices((int)K, (int)k);
}

// The fused path (one launch per time step for both directions) keeps the projections
// and gradients of both directions at once: forward {XP [D][T*B*GH], bias [D][GH]};
// backward = the layout above, then for the second direction {dGW, dGR, dh_dir [2*BH], dc [BH]}.
// slices of the contraction for the weight-gradient products (A * B^T over all time steps
// and batch columns): enough 64 x 64 tiles times slices to fill the machine several
// times over, at least eight chunks of 32 per slice
int wgrad_slices(size_t M, size_t N, size_t K) {
  const long long tiles = (long long)((M + 63) / 64) * ((N + 63) / 64), chunks = (long long)(K + 31) / 32;
  long long ns = 1024 / tiles;
  if (ns > chunks / 8) ns = chunks / 8;
  if (ns > 16) ns = 16;
  if (ns < 1) ns = 1;
  const long long cps = (chunks + ns - 1) / ns;
  return (int)((chunks + cps - 1) / cps);
}

// the products over all time steps and the column sums may use the scratch at the end of the workspace
struct Scratch {
  void* p = nullptr;
  size_t bytes = 0;
};

int mm(const float* A, const float* B, float* C, size_t M, size_t N, size_t K, int ta, int tb,
       const float* bias, hipStream_t s, Scratch w = Scratch(), bool fp32_sums = false) {
  // A thin product A * B that gemm_f32.hip cuts into slices is faster there from the shortest such contraction on (512 x 64 x 512 7.4 /
  // 8.5 us).  flhip_matmul_ws leaves it to the other kernel up to a contraction of 704 for the second launch's host time,
  // which a layer's queued launches hide: GRU of 320 units, 3 layers, backward over 13 steps, 7 columns 321 -> 272 us.
  if (!ta && !tb && N <= 128 && !options().matmul_valu && options().matmul_planes < 0) {
    const int rc = gemm32(0, A, B, C, (int)M, (int)N, (int)K, bias, w.p, w.bytes, s, nullptr,
                          [](int, int, int, bool slices) { return slices; });
    if (rc >= 0) return rc;
  }
  return matmul(A, B, C, (int)M, (int)N, (int)K, ta, tb, bias, FLHIP_F32, w.p, w.bytes, s, fp32_sums);
}

// C = op(A) B in `*slices` partial products at C + k*M*N (see step_slices)
int mm_sliced(const float* A, const float* B, float* C, size_t M, size_t N, size_t K, int ta, int* slices,
              hipStream_t s) {
  int ksplit;
  const int ns = step_slices(M, N, K, &ksplit);
  if (ns > 1 && mfma_gemm(FLHIP_F32, ta ? 1 : 0, A, B, C, (int)M, (int)N, (int)K, nullptr, s, ksplit) >= 0) {
    *slices = ns;
    return check_launch("rnn (recurrent product)");
  }
  *slices = 1;
  return mm(A, B, C, M, N, K, ta, 0, nullptr, s);
}


// ... and at the end the partial products of the sliced weight-gradient products
size_t wgrad_scratch(const RnnGeom& g) {
  const size_t TB = (size_t)g.T * g.B, inmax = widest_input(g);
  size_t n = 0;
  for (size_t M : {(size_t)g.I, inmax, (size_t)g.H}) {
    const int ns = wgrad_slices(M, g.GH, TB);
    if (ns > 1) n = std::max(n, (size_t)ns * M * g.GH);
  }
  return n;
}

size_t wgrad_scratch_offset(const RnnGeom& g) {
  const size_t TB = (size_t)g.T * g.B, inmax = widest_input(g);
  int k;
  const size_t sb = step_slices(g.H, g.B, g.GH, &k);
  return 2 * TB * g.GH + TB * g.D * g.H + 2 * TB * inmax + (3 + sb) * g.BH +
         (size_t)(g.D - 1) * (2 * TB * g.GH + 3 * g.BH);
}

size_t workspace_core(const RnnGeom& g) {
  const size_t TB = (size_t)g.T * g.B;
  int k;
  const size_t sf = step_slices(g.GH, g.B, g.H, &k);
  const size_t fwd = std::max(TB * g.GH + sf * g.B * g.GH + g.GH, (size_t)g.D * (TB * g.GH + g.GH));
  const size_t bwd = wgrad_scratch_offset(g) + wgrad_scratch(g);
  return ((std::max(fwd, bwd) + 67) & ~(size_t)3) + 4;
}
// whether whole sequences may be launched: 16-byte pieces of the state, recurrent matrices in registers
bool seq_holds(const RnnGeom& g) { return g.H % 4 == 0 && g.H <= 1024; }
// floats of a step of the exchange
size_t seq_row(const RnnGeom& g, size_t K) { return (size_t)g.B * ((K + 15) & ~(size_t)15); }

// whether a wait inside one of the call's sequence launches has given up (one word before the scratch)
uint32_t* seq_status(const RnnGeom& g, float* ws) { return reinterpret_cast<uint32_t*>(ws + workspace_core(g) - 4); }
Scratch scratch_of(const RnnGeom& g, float* ws) {
  const int TB = g.T * g.B, GH = (int)g.GH;
  size_t n = flhip_sum_columns_workspace_bytes(GH, TB, FLHIP_F32);
  for (int in : {g.I, g.D * g.H}) {
    n = std::max(n, gemm32_ws_bytes(1, GH, TB, in, g.mode == RNN_RELU));
    n = std::max(n, gemm32_ws_bytes(0, in, TB, GH));
    n = std::max(n, gemm32_ws_bytes(2, in, GH, TB));
  }
  n = std::max(n, gemm32_ws_bytes(2, g.H, GH, TB));
  return Scratch{ws + workspace_core(g), (n + 15) & ~(size_t)15};
}
// the fused step kernels tile the hidden state by 16 and hold at most 64 batch columns
bool fused_applies(const RnnGeom& g) {
  return !options().rnn_unfused && g.H % 16 == 0 && g.B <= 64;
}

__device__ __forceinline__ float sigm(float v) {
#pragma clang fp contract(off)
  return 1.f / (1.f + expf(-v));
}

// Dropout between layers: x[i] *= keep(i) / (1 - p) over the output sequence of `layer`, with the
// counter-based mask of (seed, layer, i): two rounds of a 32-bit finaliser, the top 24 bits as
// a uniform number in [0, 1).  The backward pass applies the same mask to the gradient.
__global__ void __launch_bounds__(256) rnn_dropout_kernel(float* __restrict__ x, size_t n, uint32_t seed_lo,
                                                          uint32_t seed_hi, uint32_t layer, float p, float scale) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  uint32_t h = (uint32_t)i * 0x9E3779B1u ^ seed_lo;
  h ^= h >> 16; h *= 0x85EBCA6Bu; h ^= h >> 13; h *= 0xC2B2AE35u; h ^= h >> 16;
  h += seed_hi + layer * 0x632BE5ABu;
  h ^= h >> 16; h *= 0x85EBCA6Bu; h ^= h >> 13; h *= 0xC2B2AE35u; h ^= h >> 16;
  const bool keep = (float)(h >> 8) * (1.0f / 16777216.0f) >= p;
  x[i] = keep ? x[i] * scale : 0.f;
}

__global__ void __launch_bounds__(256) rnn_init_kernel(const float* __restrict__ src, float* __restrict__ dst, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) dst[i] = src ? src[i] : 0.f;
}

// out = a + sum of nb slices of b (either may be null); out may be a
__global__ void __launch_bounds__(256) rnn_add2_kernel(const float* a, const float* __restrict__ b, int nb,
                                                       float* out, size_t n) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v = a ? a[i] : 0.f;
  if (b)
    for (int k = 0; k < nb; ++k) v += b[(size_t)k * n + i];
  out[i] = v;
}

constexpr int SEQ_COLS = 16;
constexpr int RNN_OOB = (int)0x80000000;
// Where the values of a step are that the workgroups of a cluster hand to each other (the state, the gate gradients): an exchange
// (where it lies: seq_place), in chunks of 16 contraction indexes, and in a chunk in the order of the lanes that read it, [4][columns][4], so
// that a wave's load is one piece of 1 KB.  Read from the rows of the reserve buffer / workspace it was 16 pieces of 64 bytes, a
// row apart (8 KB: all in one channel of the caches): the 128 KB of a step of an LSTM of 512 units' backward pass took 10000 cycles of
// its 13600.
struct SeqRow {
  int K, nc;            // contraction, columns of the cluster
  int lane;             // byte offset of this lane's piece in a chunk, or RNN_OOB
  size_t step;          // floats between steps
  float* base;
  __device__ __forceinline__ SeqRow(float* X, int K, int B, int b0) : K(K), nc(min(SEQ_COLS, B - b0)) {
    const int Kp = (K + 15) & ~15, fr = threadIdx.x & 15, fg = threadIdx.x >> 4 & 3;
    lane = fr < nc ? (fg * nc + fr) * 16 : RNN_OOB;
    step = (size_t)B * Kp;
    base = X + (size_t)b0 * Kp;
  }
  __device__ __forceinline__ int at(int k, int col) const { return (k >> 4) * (nc * 16) + ((k >> 2 & 3) * nc + col) * 4 + (k & 3); }
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(int st) const {
    return make_rsrc(base + st * step, (unsigned)(K * nc * 4));      // (the last chunk's pieces beyond K are the buffer's end)
  }
};

struct CellFwd {
  const float* xp;    // [B][GH] input projection (+ biases) of this time step
  const float* rp;    // [nrp][B][GH] recurrent projection, in nrp partial products (two-kernel path)
  int nrp;
  const float* R;     // [GH][H] recurrent matrices (fused path)
  const float* bRn;   // GRU: recurrent bias of the n gate [H]
  const float* hp;    // [B][H] state before the step
  const float* cp;    // LSTM
  float* hn;          // [B][H] state after the step
  float* cn;
  float* gt;          // [B][GH] gate activations kept for the backward pass
  float* rn;          // GRU: R_n h + b_Rn
  float* out;         // layer output at this time step, this direction's slice; row pitch ldo
  float* hy;          // final state of the pseudo-layer (written at the last step) or null
  float* cy;
  int ldo;
};

// (The gate math below leaves no choice of fused or separate multiply-adds to the compiler, and the step kernels add in the
// sequence kernels' order: hidden sizes that are multiples of 16 with at most 64 columns give the same bits captured and eager, as do stacked
// layers of one direction that rnn_stack_fwd takes, which runs both ways.
// The two-kernel steps, which others run on where a sequence launch is not made, add their products in another order.)
// gate math of one (batch b, hidden h) element, in two halves so that a kernel can issue
// the loads before it computes the recurrent projections rp (one per gate)
template <int MODE>
struct CellFwdIn {
  float xp[MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1];
  float prev;   // LSTM: c before the step; GRU: h before the step
  float bRn;
};

template <int MODE>
__device__ __forceinline__ CellFwdIn<MODE> cell_fwd_load(const CellFwd& a, int b, int h, int H) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1;
  const size_t e = (size_t)b * H + h, q = (size_t)b * G * H + h;
  CellFwdIn<MODE> in;
#pragma unroll
  for (int gq = 0; gq < G; ++gq) in.xp[gq] = a.xp[q + (size_t)gq * H];
  in.prev = MODE == RNN_LSTM ? a.cp[e] : MODE == RNN_GRU ? a.hp[e] : 0.f;
  in.bRn = MODE == RNN_GRU ? a.bRn[h] : 0.f;
  return in;
}

// Values that another workgroup of the same launch waits for (the sequence kernels below): every element starts as
// RNN_UNSET, a NaN that no element is stored as, and is written once, past the caches that the readers do not share.
// RNN_LOST, another one, is stored by a workgroup that has given up waiting.
constexpr uint32_t RNN_UNSET = 0xffffffffu, RNN_LOST = 0xfffffffeu;
__device__ __forceinline__ float rnn_value(float v) { return __float_as_uint(v) >= RNN_LOST ? __uint_as_float(0x7fc00000u) : v; }
__device__ __forceinline__ void rnn_publish(float* p, float v, bool lost) {
  __hip_atomic_store(p, lost ? __uint_as_float(RNN_LOST) : rnn_value(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// SEQ: the state goes to the other workgroups of the launch; returns what the element's thread keeps for the next step
// (LSTM: c, else h).  lost (rp is NaN then): so are the state and what follows from it, also where the ReLU of a NaN is zero
template <int MODE, bool SEQ = false>
__device__ __forceinline__ float cell_fwd_finish(const CellFwd& a, int b, int h, int H, const CellFwdIn<MODE>& in,
                                                 const float* rp, bool lost = false, float* pub = nullptr) {
#pragma clang fp contract(off)
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1;
  const size_t e = (size_t)b * H + h, q = (size_t)b * G * H + h;
  float hv, keep = 0.f;
  if (MODE == RNN_RELU || MODE == RNN_TANH) {
    const float pre = in.xp[0] + rp[0];
    hv = MODE == RNN_RELU ? (pre > 0.f || (SEQ && lost) ? pre : 0.f) : tanhf(pre);
    if (SEQ && pub) rnn_publish(pub, hv, lost);
    a.gt[q] = hv;
  } else if (MODE == RNN_LSTM) {
    const float ig = sigm(in.xp[0] + rp[0]), fg = sigm(in.xp[G > 1 ? 1 : 0] + rp[G > 1 ? 1 : 0]);
    const float gg = tanhf(in.xp[G > 2 ? 2 : 0] + rp[G > 2 ? 2 : 0]), og = sigm(in.xp[G > 3 ? 3 : 0] + rp[G > 3 ? 3 : 0]);
    const float c = fmaf(fg, in.prev, ig * gg);
    keep = c;
    hv = og * tanhf(c);
    if (SEQ && pub) rnn_publish(pub, hv, lost);
    a.cn[e] = c;
    if (a.cy) a.cy[e] = c;
    a.gt[q] = ig; a.gt[q + H] = fg; a.gt[q + 2 * H] = gg; a.gt[q + 3 * H] = og;
  } else {
    const float rg = sigm(in.xp[0] + rp[0]), zg = sigm(in.xp[G > 1 ? 1 : 0] + rp[G > 1 ? 1 : 0]);
    const float rn = rp[G > 2 ? 2 : 0] + in.bRn;
    const float ng = tanhf(fmaf(rg, rn, in.xp[G > 2 ? 2 : 0]));
    hv = fmaf(1.f - zg, ng, zg * in.prev);
    keep = hv;
    if (SEQ && pub) rnn_publish(pub, hv, lost);
    a.rn[e] = rn;
    a.gt[q] = rg; a.gt[q + H] = zg; a.gt[q + 2 * H] = ng;
  }
  a.hn[e] = hv;
  a.out[(size_t)b * a.ldo + h] = hv;
  if (a.hy) a.hy[e] = hv;
  return keep;
}

template <int MODE>
__global__ void __launch_bounds__(256) rnn_cell_fwd(CellFwd a, int B, int H) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= B * H) return;
  const int b = e / H, h = e - b * H;
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1;
  const size_t q = (size_t)b * G * H + h;
  const CellFwdIn<MODE> in = cell_fwd_load<MODE>(a, b, h, H);
  float rp[G];
#pragma unroll
  for (int gq = 0; gq < G; ++gq) rp[gq] = 0.f;
  for (int k = 0; k < a.nrp; ++k) {
    const float* r = a.rp + (size_t)k * B * G * H + q;
#pragma unroll
    for (int gq = 0; gq < G; ++gq) rp[gq] += r[gq * H];
  }
  cell_fwd_finish<MODE>(a, b, h, H, in, rp);
}

// One time step of up to two directions in one launch: recurrent product and gate math.
// A workgroup owns four hidden units (blockIdx.x) of one direction (blockIdx.y): its
// 16-row matrix-core tile is {gate g, unit hh} = row 4*g + hh of the recurrent
// matrices, its columns are the batch (NBT tiles of 16, batch <= 64), and the contraction
// over the hidden state is split over eight groups in interleaved chunks of 16, whether four waves
// or eight hold them (as the sequence kernels do: a captured launch sequence and an eager one add
// in the same order).  A
// lane's 16-byte load supplies the operands of four 16x16x4 products (the k index of a
// lane group is permuted the same way on both operands).  The partial tiles meet in
// LDS, then one thread per (batch, unit) applies the gates; those threads issue the
// loads of their gate inputs before the product, so that the two latencies overlap.
// Needs H % 16 == 0.
struct StepFwd {
  CellFwd d[2];
  int B, H;
};
constexpr int STEP_GROUPS = 8;
constexpr int step_fwd_chunks(int nbt) { return nbt == 4 ? 4 : 8; }      // in flight per wave

template <int MODE, int NBT, int W>
__global__ void __launch_bounds__(64 * W) rnn_step_fwd(StepFwd p) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1, NB = NBT * 16, S = STEP_GROUPS / W;
  __shared__ float red[STEP_GROUPS][16][NB + 1];
  const CellFwd& a = p.d[blockIdx.y];
  const int H = p.H, B = p.B, h0 = blockIdx.x * 4;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const bool cell = tid < 4 * B;
  const int cb = tid >> 2, ch = h0 + (tid & 3);
  CellFwdIn<MODE> cin{};
  if (cell) cin = cell_fwd_load<MODE>(a, cb, ch, H);
  const int gate = fr >> 2;
  const bool av = gate < G;
  const float* ap = a.R + ((size_t)(av ? gate : 0) * H + h0 + (fr & 3)) * H + 4 * fg;
  const float* bp[NBT];
  bool bv[NBT];
#pragma unroll
  for (int nt = 0; nt < NBT; ++nt) {
    const int b = nt * 16 + fr;
    bv[nt] = b < B;
    bp[nt] = a.hp + (size_t)(bv[nt] ? b : 0) * H + 4 * fg;
  }
  floatx4_t acc[S][NBT];                  // group wave + W * s of the contraction: every S-th of the wave's chunks
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int nt = 0; nt < NBT; ++nt) acc[s][nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
  // U chunks are in flight per wave at a time: the loop is bound by the latency of
  // its loads, not by the products
  constexpr int U = step_fwd_chunks(NBT);
  const int chunks = H >> 4;
  const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int c0 = wave; c0 < chunks; c0 += W * U) {
    float4 ra[U], rb[U][NBT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // every load is issued (from a clamped, valid address) before any is used
      const int c = min(c0 + W * u, chunks - 1);
      ra[u] = *reinterpret_cast<const float4*>(ap + c * 16);
#pragma unroll
      for (int nt = 0; nt < NBT; ++nt) rb[u][nt] = *reinterpret_cast<const float4*>(bp[nt] + c * 16);
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bool in = c0 + W * u < chunks;
      if (!(in && av)) ra[u] = zero4;
#pragma unroll
      for (int nt = 0; nt < NBT; ++nt)
        if (!(in && bv[nt])) rb[u][nt] = zero4;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const float av4[4] = {ra[u].x, ra[u].y, ra[u].z, ra[u].w};
#pragma unroll
      for (int nt = 0; nt < NBT; ++nt) {
        const float bv4[4] = {rb[u][nt].x, rb[u][nt].y, rb[u][nt].z, rb[u][nt].w};
#pragma unroll
        for (int m = 0; m < 4; ++m)
          acc[u % S][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(av4[m], bv4[m], acc[u % S][nt], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int s = 0; s < S; ++s)
#pragma unroll
    for (int nt = 0; nt < NBT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[wave + W * s][4 * fg + r][nt * 16 + fr] = acc[s][nt][r];
  __syncthreads();
  if (cell) {
    const int hh = tid & 3;
    float rp[G];
#pragma unroll
    for (int gq = 0; gq < G; ++gq) {
      float v = 0.f;
#pragma unroll
      for (int k = 0; k < STEP_GROUPS; ++k) v += red[k][gq * 4 + hh][cb];
      rp[gq] = v;
    }
    cell_fwd_finish<MODE>(a, cb, ch, H, cin, rp);
  }
}

struct CellBwd {
  const float* gout;  // gradient of the layer output at this time step, this direction's slice; pitch ldo (may be null)
  const float* dh_a;  // gradient reaching h through the recurrence: direct part ...
  const float* dh_b;  // ... and the part through the recurrent matrices, in ndhb partial products
  int ndhb;           //     (either pointer may be null)
  const float* R;         // fused path: recurrent matrices [GH][H] and the recurrent-side
  const float* dgr_next;  // pre-activation gradients [B][GH] of the step walked before (or null)
  float* dc;          // LSTM: in = gradient of c after the step, out = of c before it
  const float* gt;    // gate activations of the step
  const float* cp;    // LSTM: c before the step
  const float* cn;    //       c after the step
  const float* hp;    // state before the step
  const float* rn;    // GRU
  float* dgw;         // [B][GH] pre-activation gradients seen by the input side
  float* dgr;         // [B][GH] ... by the recurrent side
  float* dh_dir;      // [B][H] direct gradient towards the previous state (GRU: go * z, else 0)
  float* dhx;         // fused path: only the gradient of the initial state, no step (else null)
  int ldo;
};

// gradient math of one (batch b, hidden h) element in two halves (loads, then math and
// stores); rec = gradient arriving through the recurrent matrices
template <int MODE>
struct CellBwdIn {
  float go;     // gradient of the output + direct recurrent part
  float gt[MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1];
  float cn, cp, dc;   // LSTM
  float hp, rn;       // GRU
};

template <int MODE>
__device__ __forceinline__ CellBwdIn<MODE> cell_bwd_load(const CellBwd& a, int b, int h, int H) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1;
  const size_t e = (size_t)b * H + h, q = (size_t)b * G * H + h;
  CellBwdIn<MODE> in{};
  in.go = a.gout ? a.gout[(size_t)b * a.ldo + h] : 0.f;
  if (a.dh_a) in.go += a.dh_a[e];
#pragma unroll
  for (int gq = 0; gq < G; ++gq) in.gt[gq] = a.gt[q + (size_t)gq * H];
  if (MODE == RNN_LSTM) {
    in.cn = a.cn[e]; in.cp = a.cp[e]; in.dc = a.dc[e];
  }
  if (MODE == RNN_GRU) {
    in.hp = a.hp[e]; in.rn = a.rn[e];
  }
  return in;
}

// SEQ: the recurrent-side gradients go to the other workgroups of the launch, and what the element's thread hands to its
// next step stays in *dc and *dir.  lost: as in the forward pass (rec is NaN)
template <int MODE, bool SEQ = false>
__device__ __forceinline__ void cell_bwd_finish(const CellBwd& a, int b, int h, int H, const CellBwdIn<MODE>& in,
                                                float rec, float* dc_out = nullptr, float* dir_out = nullptr, bool lost = false,
                                                float* pub = nullptr, const SeqRow* row = nullptr, int col = 0) {
#pragma clang fp contract(off)
  auto put = [&](int g, float v) {
    if (SEQ) rnn_publish(pub + row->at(g * H + h, col), v, lost);
  };
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1;
  const size_t e = (size_t)b * H + h, q = (size_t)b * G * H + h;
  const float go = in.go + rec;
  float direct = 0.f;
  if (MODE == RNN_RELU || MODE == RNN_TANH) {
    const float hv = in.gt[0];
    const float gp = MODE == RNN_RELU ? (hv > 0.f || (SEQ && lost) ? go : 0.f) : go * fmaf(-hv, hv, 1.f);
    put(0, gp);
    a.dgr[q] = gp;
    a.dgw[q] = gp;
  } else if (MODE == RNN_LSTM) {
    const float ig = in.gt[0], fg = in.gt[G > 1 ? 1 : 0], gg = in.gt[G > 2 ? 2 : 0], og = in.gt[G > 3 ? 3 : 0];
    const float tc = tanhf(in.cn);
    const float dc = fmaf(go * og, fmaf(-tc, tc, 1.f), in.dc);
    const float v0 = dc * gg * ig * (1.f - ig), v1 = dc * in.cp * fg * (1.f - fg);
    const float v2 = dc * ig * fmaf(-gg, gg, 1.f), v3 = go * tc * og * (1.f - og);
    put(0, v0); put(1, v1); put(2, v2); put(3, v3);
    a.dgr[q] = v0; a.dgr[q + H] = v1; a.dgr[q + 2 * H] = v2; a.dgr[q + 3 * H] = v3;
    a.dgw[q] = v0; a.dgw[q + H] = v1; a.dgw[q + 2 * H] = v2; a.dgw[q + 3 * H] = v3;
    if (SEQ) *dc_out = dc * fg;
    else a.dc[e] = dc * fg;
  } else {
    const float rg = in.gt[0], zg = in.gt[G > 1 ? 1 : 0], ng = in.gt[G > 2 ? 2 : 0], rn = in.rn;
    const float dn = go * (1.f - zg) * fmaf(-ng, ng, 1.f);
    const float v0 = dn * rn * rg * (1.f - rg), v1 = go * (in.hp - ng) * zg * (1.f - zg);
    put(0, v0); put(1, v1); put(2, dn * rg);
    a.dgr[q] = v0; a.dgr[q + H] = v1; a.dgr[q + 2 * H] = dn * rg;
    a.dgw[q] = v0; a.dgw[q + H] = v1; a.dgw[q + 2 * H] = dn;
    direct = go * zg;
  }
  if (SEQ) *dir_out = direct;
  else a.dh_dir[e] = direct;
}

template <int MODE>
__global__ void __launch_bounds__(256) rnn_cell_bwd(CellBwd a, int B, int H) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= B * H) return;
  const int b = e / H, h = e - b * H;
  const CellBwdIn<MODE> in = cell_bwd_load<MODE>(a, b, h, H);
  float rec = 0.f;
  if (a.dh_b)
    for (int k = 0; k < a.ndhb; ++k) rec += a.dh_b[(size_t)k * B * H + e];
  cell_bwd_finish<MODE>(a, b, h, H, in, rec);
}

// One backward time step of up to two directions in one launch.  A workgroup owns 16
// hidden units of one direction: rows of its matrix-core tile are the units (columns
// of the recurrent matrices, 64 contiguous bytes per contraction index), columns the
// batch.  Its eight waves split the contraction over the gate rows (G*H) in
// interleaved chunks of 16 (with four batch tiles: eight groups of two waves, each wave
// two of the tiles); the partial tiles meet in LDS and one thread per (unit, batch)
// applies the gate gradients of the step, which become the next launch's operand.
// Those threads issue their loads before the product.  H % 16 == 0.
// A last launch with no step of its own (dhx) adds up the gradient of the initial state.
struct StepBwd {
  CellBwd d[2];
  int B, H;
};
constexpr int step_bwd_waves(int nbt) { return nbt == 4 ? 2 * STEP_GROUPS : STEP_GROUPS; }

template <int MODE, int NBT>
__global__ void __launch_bounds__(64 * step_bwd_waves(NBT)) rnn_step_bwd(StepBwd p) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1, NB = NBT * 16;
  constexpr int NW = NBT == 4 ? 2 : NBT;      // batch tiles per wave
  constexpr int KG = STEP_GROUPS;             // wave groups along the contraction
  __shared__ float red[KG][16][NB + 1];
  const CellBwd& a = p.d[blockIdx.y];
  const int H = p.H, B = p.B, h0 = blockIdx.x * 16, GH = G * H;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const bool cell = tid < 16 * B;
  const int cb = tid >> 4, ch = h0 + (tid & 15);
  CellBwdIn<MODE> cin{};
  if (cell && !a.dhx) cin = cell_bwd_load<MODE>(a, cb, ch, H);
  const bool have = a.dgr_next != nullptr;
  if (have) {
    const int kg = wave % KG, nt0 = (wave / KG) * NW;
    const float* ap = a.R + (size_t)(4 * fg) * H + h0 + fr;
    const float* bp[NW];
    bool bv[NW];
#pragma unroll
    for (int nt = 0; nt < NW; ++nt) {
      const int b = (nt0 + nt) * 16 + fr;
      bv[nt] = b < B;
      bp[nt] = a.dgr_next + (size_t)(bv[nt] ? b : 0) * GH + 4 * fg;
    }
    floatx4_t acc[NW];
#pragma unroll
    for (int nt = 0; nt < NW; ++nt) acc[nt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    constexpr int U = NW == 2 ? 4 : 8;   // chunks in flight per wave (registers: 128 per thread)
    const int chunks = GH >> 4;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int c0 = kg; c0 < chunks; c0 += KG * U) {
      float ra[U][4];
      float4 rb[U][NW];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = min(c0 + KG * u, chunks - 1);
#pragma unroll
        for (int m = 0; m < 4; ++m) ra[u][m] = ap[((size_t)c * 16 + m) * H];
#pragma unroll
        for (int nt = 0; nt < NW; ++nt) rb[u][nt] = *reinterpret_cast<const float4*>(bp[nt] + c * 16);
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const bool in = c0 + KG * u < chunks;
#pragma unroll
        for (int m = 0; m < 4; ++m)
          if (!in) ra[u][m] = 0.f;
#pragma unroll
        for (int nt = 0; nt < NW; ++nt)
          if (!(in && bv[nt])) rb[u][nt] = zero4;
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int nt = 0; nt < NW; ++nt) {
          const float bv4[4] = {rb[u][nt].x, rb[u][nt].y, rb[u][nt].z, rb[u][nt].w};
#pragma unroll
          for (int m = 0; m < 4; ++m)
            acc[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(ra[u][m], bv4[m], acc[nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nt = 0; nt < NW; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r) red[kg][4 * fg + r][(nt0 + nt) * 16 + fr] = acc[nt][r];
  }
  __syncthreads();
  if (cell) {
    float rec = 0.f;
    if (have) {
#pragma unroll
      for (int k = 0; k < KG; ++k) rec += red[k][tid & 15][cb];
    }
    if (a.dhx) a.dhx[(size_t)cb * H + ch] = a.dh_a[(size_t)cb * H + ch] + rec;
    else cell_bwd_finish<MODE>(a, cb, ch, H, cin, rec);
  }
}

// ---- a layer's whole recurrence in one launch -----------------------------------------------------------------------
// The steps of a sequence depend on each other, so a launch per step costs a launch's latency and one trip of the
// recurrent matrices from the caches per step (LSTM of 512 units, two directions, 32 columns: 8.2 us forward, 12.4 us
// backward per step, where the products need 0.9 and 1.7).  Here the workgroups stay: each keeps its part of the
// recurrent matrices in registers for all steps, and only the state (forward) or the pre-activation gradients (backward)
// of a step travel between workgroups.  Per step, forward / backward: that LSTM 8.2 -> 2.9 / 12.4 -> 4.1 us; GRU of 1024
// units, 64 columns 16.2 -> 5.0 / 29.7 -> 5.7 us (products 2.6, exchange of 64 / 192 KB per workgroup); LSTM of 320 units,
// 5 columns 5.1 -> 1.8 us forward.  What bounds them: the products (fp32 matrix pipe), the exchange's trip and volume, and the
// gates' math between two barriers (0.6 us of the LSTM's step).  Batch columns do not depend on each other: a cluster of workgroups
// is one direction of 16 columns, and clusters never wait for one another.
//
// The exchange needs no flags and no barrier over the grid: its buffer (SeqRow; a row for every step, none is used twice) is filled with
// RNN_UNSET before the launch, the owner of an element stores it once with
// agent scope, and a reader repeats its 16-byte loads (agent scope as well: they pass by the caches that the eight dies
// do not share) until none of its elements is unset.  (A cluster's workgroups on one die, found by its number, with loads and stores that its
// cache answers, gained nothing on that: LSTM of 512 units, two directions, 32 columns over 200 steps backward 1167 -> 1219 us.)
//
// All workgroups of the launch have to be resident at once: the launch is cooperative, and a launch covers as many
// clusters as the compute units hold, the rest follow in further launches.  A wait that does not end (it would take a
// device that lost workgroups) stops after RNN_WAIT loads, some seconds.  Its workgroup then goes on with NaN in every mode
// (RNN_LOST in ReLU layers), which is what the others' next steps read, and sets a word in the workspace with which the launches
// of the call's other layers begin; so every output that depends on the missing values is NaN.
constexpr int SEQ_WAVES = STEP_GROUPS, SEQ_THREADS = 64 * SEQ_WAVES;
constexpr int AUX_AGENT = 16;      // buffer loads: sc1, agent scope

struct SeqFwd {
  struct Dir {
    const float *xp, *R, *bRn;
    float *HP, *CP, *GT, *RN, *out, *hy, *cy, *X;
  } d[2];
  int B, H, T, ldo;
  int groups;        // of 16 batch columns
  int nwg;           // workgroups of a cluster
  int cluster0;      // first cluster of this launch; cluster = direction * groups + group
  int wait;          // options().rnn_wait
  int pause;         // of seq_pause
  uint32_t* status;  // the layer (from 1) whose launch first gave up
  uint32_t layer;
};

// What a wave knows of waits that gave up.  One that has (dead) leaves RNN_LOST in its partial sums, a NaN, and so NaN in all
// elements of its workgroup and, from the next step on, of its cluster.  ReLU layers turn a NaN sum into zero: there the thread
// of an element whose sum is NaN looks for RNN_LOST, among the partial sums and in the row that they came from (seq_lost), and
// stores it where it has found it.
struct SeqLost {
  uint32_t *status, layer;
  int limit;         // loads of a wait; negative: `first` has given up from the start
  // before: *status.  -> whether another layer's launch has given up (what this layer's other clusters do is no matter: they don't
  // depend on each other, and a word that another layer has set is left as it is)
  __device__ __forceinline__ int begin(uint32_t before, bool first) {
    before = __builtin_amdgcn_readfirstlane(before);
    int dead = before != 0 && before != layer;
    if (dead) status = nullptr;
    if (limit < 0) {
      if (first) dead = 1;
      limit = 1 << 22;
    }
    return dead;
  }
  template <int N>
  __device__ __forceinline__ void tell(int dead, floatx4_t (&acc)[N]) const {
    if (__builtin_expect(dead, 0)) {
      const float nan = __uint_as_float(RNN_LOST);
#pragma unroll
      for (int i = 0; i < N; ++i) acc[i] = floatx4_t{nan, nan, nan, nan};
      if (status && (threadIdx.x & 63) == 0) __hip_atomic_store(status, layer, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
};
// every load so far has arrived: what a loop carries from before it then needs no wait inside it (that wait would be one
// for the stores of the step before)
__device__ __forceinline__ void seq_drain() { __builtin_amdgcn_s_waitcnt(0x0f70); }

// Between two steps: every wave waits until the workgroup's own elements are on their way, and as long again as such a
// store travels (about 150 cycles for each of n), before it asks for the others'.  Asked earlier, the loads come back unset and
// are repeated, and their traffic holds up the very stores they wait for; asked later, every step waits: seq_pause_fwd.
__device__ __forceinline__ void seq_pause(int n) {
  __syncthreads();
  for (; n > 0; --n) __builtin_amdgcn_s_sleep(2);
}

// 16 bytes per lane of each of the chunks c0, c0 + SEQ_WAVES, ...: N of them.  What does not exist is out of the buffer's
// range and reads zero.
template <int N>
__device__ __forceinline__ void seq_load(__amdgpu_buffer_rsrc_t r, const SeqRow& row, int c0, uintx4_t (&v)[N]) {
  int lane = row.lane;
  asm volatile("" : "+v"(lane) : : "memory");      // memory may have changed since the last load; and N sums in each step cost less
                                                   // than registers that hold them over all steps
#pragma unroll
  for (int i = 0; i < N; ++i)
    v[i] = __builtin_amdgcn_raw_buffer_load_b128(r, lane + (c0 + SEQ_WAVES * i) * (row.nc * 64), 0, AUX_AGENT);
}
template <int N>
__device__ __forceinline__ bool seq_unset(const uintx4_t (&v)[N]) {
  uint32_t m = 0;                    // (RNN_UNSET is the largest word)
#pragma unroll
  for (int i = 0; i < N; ++i) m = max(max(m, max(v[i].x, v[i].y)), max(v[i].z, v[i].w));
  return __builtin_amdgcn_ballot_w64(m == RNN_UNSET) != 0;
}
// Repeats the loads until every element is set.  -> whether the wave has given up, now or before (dead).  One question in the
// loop: where it looked for RNN_LOST too the compiler kept a second copy of v, whose moves every step paid for (LSTM of 1024
// units over 156 steps, 4 columns, forward 479 -> 585 us).  RNN_LOST goes through the products by itself.
template <int N>
__device__ __forceinline__ int seq_wait(__amdgpu_buffer_rsrc_t r, const SeqRow& row, int c0, uintx4_t (&v)[N], int dead, int limit) {
  if (__builtin_amdgcn_readfirstlane(dead) || !seq_unset(v)) return dead;
  for (int spin = 0; spin < limit; ++spin) {
    seq_load(r, row, c0, v);
    if (!seq_unset(v)) return 0;
  }
  return 1;
}

// whether one of the partial sums part[i * stride] or of column col of the row is RNN_LOST
__device__ __forceinline__ bool seq_lost(const float* part, int stride, const SeqRow& row, int st, int col) {
  bool lost = false;
#pragma unroll 1
  for (int w = 0; w < STEP_GROUPS; ++w) lost |= __float_as_uint(part[w * stride]) == RNN_LOST;
#pragma unroll 1
  for (int k = 0; k < row.K && !lost; ++k)
    lost = __float_as_uint(__hip_atomic_load(row.base + st * row.step + row.at(k, col), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == RNN_LOST;
  return lost;
}

// A workgroup owns HU hidden units of its cluster: row gate * HU + unit of its RT tiles of 16 rows.  The eight waves split
// the contraction over the state in interleaved chunks of 16 (NC at most per wave, the recurrent matrices' fragments in
// 4 RT NC registers); the partial tiles meet in LDS (two buffers in turn, so one barrier per step) and one thread per
// (column, unit) applies the gates.  HU is the smallest for which a layer's clusters fit the compute units.
template <int MODE, int HU, int NC>
__global__ void __launch_bounds__(SEQ_THREADS, 2) rnn_seq_fwd(SeqFwd p) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1, RT = (G * HU + 15) / 16, W = SEQ_WAVES;
  extern __shared__ float seq_red[];      // [2][W][16 RT][17]
  const uint32_t status = *p.status;
  const int cl = blockIdx.x / p.nwg, cluster = p.cluster0 + cl, h0 = (blockIdx.x - cl * p.nwg) * HU;
  const int dir = __builtin_amdgcn_readfirstlane(cluster / p.groups), b0 = (cluster - dir * p.groups) * SEQ_COLS;
  const SeqFwd::Dir q = dir ? p.d[1] : p.d[0];
  float* const HP = q.HP;
  const int H = p.H, B = p.B, GH = G * H, T = p.T;
  const SeqRow row(q.X, H, B, b0);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  float a[RT][NC][4];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int k = (wave + W * i) * 16 + 4 * fg;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int row = rt * 16 + fr, gate = row / HU, h = h0 + row % HU;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
      if (gate < G && h < H && k < H) v = *reinterpret_cast<const float4*>(q.R + ((size_t)gate * H + h) * H + k);
      a[rt][i][0] = v.x; a[rt][i][1] = v.y; a[rt][i][2] = v.z; a[rt][i][3] = v.w;
    }
  }
  const int unit = tid % HU, col = tid / HU, ch = h0 + unit, cb = b0 + col;
  const bool cell = tid < HU * SEQ_COLS && cb < B && ch < H;
  const size_t BH = (size_t)B * H, e = (size_t)cb * H + ch;
  CellFwd c{};
  c.bRn = q.bRn;
  c.ldo = p.ldo;
  float keep = 0.f;
  if (cell) keep = MODE == RNN_LSTM ? q.CP[e] : MODE == RNN_GRU ? HP[e] : 0.f;
  seq_drain();
  SeqLost lost{p.status, p.layer, p.wait};
  int dead = lost.begin(status, h0 == 0);
  for (int sv = 0; sv < T; ++sv) {
    const int st = __builtin_amdgcn_readfirstlane(sv), t = dir ? T - 1 - st : st;
    c.xp = q.xp + (size_t)t * B * GH;
    CellFwdIn<MODE> in{};
    if (cell) {
#pragma unroll
      for (int g = 0; g < G; ++g) in.xp[g] = c.xp[(size_t)cb * GH + (size_t)g * H + ch];
      in.bRn = MODE == RNN_GRU ? c.bRn[ch] : 0.f;
      in.prev = keep;
    }
    if (st > 0) seq_pause(p.pause);
    const __amdgpu_buffer_rsrc_t r = row.rsrc(st);
    uintx4_t v[NC];
    seq_load(r, row, wave, v);
    dead = __builtin_amdgcn_readfirstlane(seq_wait(r, row, wave, v, dead, lost.limit));
    seq_drain();
    floatx4_t acc[RT];
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) acc[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if ((wave + W * i) * 16 < H)
#pragma unroll
        for (int m = 0; m < 4; ++m)
#pragma unroll
          for (int rt = 0; rt < RT; ++rt)
            acc[rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[rt][i][m], __uint_as_float(v[i][m]), acc[rt], 0, 0, 0);
    lost.tell(dead, acc);
    float* red = seq_red + (st & 1) * (W * RT * 16 * 17);
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
      for (int x = 0; x < 4; ++x) red[(wave * RT * 16 + rt * 16 + 4 * fg + x) * 17 + fr] = acc[rt][x];
    __syncthreads();
    if (cell) {
      float rp[G];
#pragma unroll
      for (int g = 0; g < G; ++g) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < W; ++w) sum += red[(w * RT * 16 + g * HU + unit) * 17 + col];
        rp[g] = sum;
      }
      const bool gone = MODE == RNN_RELU && __builtin_expect(rp[0] != rp[0], 0) &&
                        seq_lost(red + unit * 17 + col, RT * 16 * 17, row, st, col);
      c.hn = HP + (st + 1) * BH;
      float* const pub = st + 1 < T ? row.base + (st + 1) * row.step + row.at(ch, col) : nullptr;
      c.cn = q.CP + (st + 1) * BH;
      c.gt = q.GT + (size_t)st * B * GH;
      c.rn = q.RN + st * BH;
      c.out = q.out + (size_t)t * B * p.ldo;
      c.hy = st == T - 1 ? q.hy : nullptr;
      c.cy = st == T - 1 ? q.cy : nullptr;
      keep = cell_fwd_finish<MODE, true>(c, cb, ch, H, in, rp, gone, pub);
    }
  }
}

// Stacked layers of one direction in one launch: clusters of all layers run side by side, and a layer's step waits for the same step of
// the layer below (its row of the exchange) as it does for its own step before.  So T + L - 1 steps follow each other instead
// of L T, there is one cooperative launch instead of L, and the products between the layers are part of the steps: the recurrent
// and the input matrix lie in registers side by side, and add to one tile (GRU, whose W_n x and R_n h stay apart: to one each).  The
// lowest layer's projections are made before, as ever.
// Forward, us, a launch per layer / one for all: LSTM of 320 units, 3 layers, 5 columns, over 25 steps 225 / 84, over 100 steps 600 / 215; of
// 512 units, 2 layers, 16 columns over 50 steps 268 / 147; of 1024 units, 2 layers, 3 columns over 30 steps 224 / 190; of 256 units, 2
// layers, 64 columns over 60 steps 289 / 167; GRU of 384 units, 2 layers, 64 columns over 40 steps 257 / 187.  The recurrent and the input
// product have an accumulator each and the waves' sums are added in pairs: against 64 bits the outputs are off by (a launch per layer, whose
// products between layers may run in three bf16 parts / one for all) 1.2e-7 / 1.0e-7 for the first of these, 2.4e-7 / 1.6e-7 for the second, 1.8e-7 /
// 1.9e-7 for the GRU, 3.7e-7 / 2.3e-7 for tanh layers of 200 units over 200 steps.
constexpr int STACK_LAYERS = 4;
struct SeqStack {
  struct Layer {
    const float *xp, *W, *R, *bsum, *bRn;      // xp: the lowest layer's projections; W: the others' input matrix
    float *HP, *CP, *GT, *RN, *out, *hy, *cy, *X;
  } d[STACK_LAYERS];
  int B, H, T, L;
  int groups, nwg;
  int cluster0;      // 0: one launch holds them all
  int diagonal;      // the launch runs step diagonal - l of layer l; -1: all steps
  int wait, pause;
  uint32_t* status;
};
constexpr size_t stack_lds(int mode, int RT) { return (size_t)2 * SEQ_WAVES * (mode == RNN_GRU ? 2 : 1) * RT * 16 * 17 * sizeof(float); }

template <int MODE, int HU, int NC>
__global__ void __launch_bounds__(SEQ_THREADS, 2) rnn_stack_fwd(SeqStack p) {
  constexpr int G = gates_of(MODE), RT = (G * HU + 15) / 16, W = SEQ_WAVES;
  constexpr bool APART = MODE == RNN_GRU;
  constexpr int TILES = APART ? 2 * RT : RT;
  extern __shared__ float seq_red[];      // [2][W][16 TILES][17]
  const uint32_t status = *p.status;
  const int cluster = blockIdx.x / p.nwg, h0 = (blockIdx.x - cluster * p.nwg) * HU;
  const int layer = __builtin_amdgcn_readfirstlane(cluster / p.groups), b0 = (cluster - layer * p.groups) * SEQ_COLS;
  const SeqStack::Layer q = p.d[layer];
  const bool upper = layer > 0;
  float* const HP = q.HP;
  const int H = p.H, B = p.B, GH = G * H, T = p.T;
  const int first = p.diagonal < 0 ? 0 : p.diagonal - layer, end = p.diagonal < 0 ? T : first + 1;
  if (first < 0 || end > T) return;       // (the whole workgroup)
  const SeqRow row(q.X, H, B, b0), below(upper ? p.d[upper ? layer - 1 : 0].X : q.X, H, B, b0);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  float a[RT][NC][4], aw[RT][NC][4];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int k = (wave + W * i) * 16 + 4 * fg;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
      const int r = rt * 16 + fr, gate = r / HU, h = h0 + r % HU;
      float4 v = make_float4(0.f, 0.f, 0.f, 0.f), u = v;
      if (gate < G && h < H && k < H) {
        const size_t at = ((size_t)gate * H + h) * H + k;
        v = *reinterpret_cast<const float4*>(q.R + at);
        if (upper) u = *reinterpret_cast<const float4*>(q.W + at);
      }
      a[rt][i][0] = v.x; a[rt][i][1] = v.y; a[rt][i][2] = v.z; a[rt][i][3] = v.w;
      aw[rt][i][0] = u.x; aw[rt][i][1] = u.y; aw[rt][i][2] = u.z; aw[rt][i][3] = u.w;
    }
  }
  const int unit = tid % HU, col = tid / HU, ch = h0 + unit, cb = b0 + col;
  const bool cell = tid < HU * SEQ_COLS && cb < B && ch < H;
  const size_t BH = (size_t)B * H, e = (size_t)cb * H + ch;
  CellFwd c{};
  c.ldo = H;
  CellFwdIn<MODE> in{};
  float keep = 0.f, x0[G];
#pragma unroll
  for (int g = 0; g < G; ++g) x0[g] = 0.f;
  if (cell) {
    keep = MODE == RNN_LSTM ? q.CP[first * BH + e] : MODE == RNN_GRU ? HP[first * BH + e] : 0.f;
    in.bRn = MODE == RNN_GRU ? q.bRn[ch] : 0.f;
    if (upper)
#pragma unroll
      for (int g = 0; g < G; ++g) x0[g] = q.bsum[(size_t)g * H + ch];
  }
  seq_drain();
  const SeqLost lost{p.status, 1u, p.wait};
  int dead = SeqLost(lost).begin(status, h0 == 0);
  const int limit = lost.limit < 0 ? 1 << 22 : lost.limit;
  const bool publish_last = layer + 1 < p.L;      // the layer above reads the last state too
  for (int sv = first; sv < end; ++sv) {
    const int st = __builtin_amdgcn_readfirstlane(sv);
    const __amdgpu_buffer_rsrc_t r = row.rsrc(st), rb = below.rsrc(st + 1);
    uintx4_t v[NC], u[NC];
    if (upper) seq_load(rb, below, wave, u);
    if (cell) {
      if (!upper)
#pragma unroll
        for (int g = 0; g < G; ++g) x0[g] = q.xp[((size_t)st * B + cb) * GH + (size_t)g * H + ch];
      in.prev = keep;
    }
    if (st > first) seq_pause(p.pause);
    seq_load(r, row, wave, v);
    floatx4_t acc[2 * RT];               // the recurrent products, the input's
#pragma unroll
    for (int rt = 0; rt < 2 * RT; ++rt) acc[rt] = floatx4_t{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const float (&m)[RT][NC][4], const uintx4_t (&x)[NC], int to) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NC; ++i)
        if ((wave + W * i) * 16 < H)
#pragma unroll
          for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int rt = 0; rt < RT; ++rt)
              acc[to + rt] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[rt][i][k], __uint_as_float(x[i][k]), acc[to + rt], 0, 0, 0);
    };
    if (upper) {
      dead = __builtin_amdgcn_readfirstlane(seq_wait(rb, below, wave, u, dead, limit));
      multiply(aw, u, RT);
    }
    dead = __builtin_amdgcn_readfirstlane(seq_wait(r, row, wave, v, dead, limit));
    seq_drain();
    multiply(a, v, 0);
    lost.tell(dead, acc);
    if (!APART)
#pragma unroll
      for (int rt = 0; rt < RT; ++rt) acc[rt] += acc[RT + rt];
    float* red = seq_red + (st & 1) * (W * TILES * 16 * 17);
#pragma unroll
    for (int rt = 0; rt < TILES; ++rt)
#pragma unroll
      for (int x = 0; x < 4; ++x) red[(wave * TILES * 16 + rt * 16 + 4 * fg + x) * 17 + fr] = acc[rt][x];
    __syncthreads();
    if (cell) {
      float rp[G];
      auto sum = [&](int row) __attribute__((always_inline)) {
        float v[W];
#pragma unroll
        for (int w = 0; w < W; ++w) v[w] = red[(w * TILES * 16 + row) * 17 + col];
#pragma unroll
        for (int n = W / 2; n > 0; n /= 2)
#pragma unroll
          for (int w = 0; w < n; ++w) v[w] += v[w + n];
        return v[0];
      };
#pragma unroll
      for (int g = 0; g < G; ++g) {
        rp[g] = sum(g * HU + unit);
        in.xp[g] = x0[g];
        if (APART && upper) in.xp[g] += sum(RT * 16 + g * HU + unit);
      }
      c.hn = HP + (st + 1) * BH;
      float* const pub = st + 1 < T || publish_last ? row.base + (st + 1) * row.step + row.at(ch, col) : nullptr;
      c.cn = q.CP + (st + 1) * BH;
      c.gt = q.GT + (size_t)st * B * GH;
      c.rn = q.RN + st * BH;
      c.out = q.out + (size_t)st * BH;
      c.hy = st == T - 1 ? q.hy : nullptr;
      c.cy = st == T - 1 ? q.cy : nullptr;
      keep = cell_fwd_finish<MODE, true>(c, cb, ch, H, in, rp, false, pub);
    }
  }
}

struct SeqBwd {
  struct Dir {
    const float *gout, *dhy, *dcy, *R, *HP, *CP, *GT, *RN;
    float *dGW, *dGR, *dhx, *dcx, *X;
  } d[2];
  int B, H, T, ldo;
  int groups, nwg, cluster0, wait, pause;
  uint32_t *status, layer;
};

// The same for the backward pass: a workgroup owns 16 hidden units (rows of one tile: columns of the recurrent matrices,
// 4 NC registers) and reads the gate gradients of all units of its cluster, U chunks in flight while U are multiplied.
// What the next step needs of the reserve buffer is asked for as soon as this step's exchange has arrived: asked for at the step's
// begin, from HBM, it held up the exchange's loads behind it (LSTM of 512 units, two directions, 32 columns over 200 steps 1289 -> 1167 us;
// forward, with fewer such loads, the registers' moves cost more than that gained, 706 -> 745).
// After the last step the gradient of the initial state is one more product.
template <int MODE, int NC>
__global__ void __launch_bounds__(SEQ_THREADS, 2) rnn_seq_bwd(SeqBwd p) {
  constexpr int G = MODE == RNN_LSTM ? 4 : MODE == RNN_GRU ? 3 : 1, W = SEQ_WAVES, U = NC < 8 ? NC : 8, NB = NC / U;
  __shared__ float red2[2][W][16][17];
  const uint32_t status = *p.status;
  const int cl = blockIdx.x / p.nwg, cluster = p.cluster0 + cl, h0 = (blockIdx.x - cl * p.nwg) * 16;
  const int dir = __builtin_amdgcn_readfirstlane(cluster / p.groups), b0 = (cluster - dir * p.groups) * SEQ_COLS;
  const SeqBwd::Dir q = dir ? p.d[1] : p.d[0];
  float* const dGR = q.dGR;
  const int H = p.H, B = p.B, GH = G * H, T = p.T;
  const SeqRow row(q.X, GH, B, b0);
  const int tid = threadIdx.x, lane = tid & 63, fr = lane & 15, fg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  float a[NC][4];
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const int k = (wave + W * i) * 16 + 4 * fg;
#pragma unroll
    for (int m = 0; m < 4; ++m) a[i][m] = (h0 + fr < H && k < GH) ? q.R[(size_t)(k + m) * H + h0 + fr] : 0.f;
  }
  const int unit = tid & 15, col = tid >> 4, ch = h0 + unit, cb = b0 + col;
  const bool cell = tid < 16 * SEQ_COLS && cb < B && ch < H;
  const size_t BH = (size_t)B * H, e = (size_t)cb * H + ch;
  CellBwd c{};
  c.ldo = p.ldo;
  float direct = cell && q.dhy ? q.dhy[e] : 0.f, dc = cell && MODE == RNN_LSTM && q.dcy ? q.dcy[e] : 0.f;
  SeqLost lost{p.status, p.layer, p.wait};
  int dead = lost.begin(status, h0 == 0);
  if (dead) direct = __builtin_nanf("");          // (the first step waits for nobody)
  seq_drain();
  CellBwdIn<MODE> nx{};
  auto fetch = [&](int st) __attribute__((always_inline)) {
    if (cell && st >= 0) {
      const size_t qe = (size_t)cb * GH + ch;
      nx.go = q.gout ? q.gout[((size_t)(dir ? T - 1 - st : st) * B + cb) * p.ldo + ch] : 0.f;
#pragma unroll
      for (int g = 0; g < G; ++g) nx.gt[g] = q.GT[(size_t)st * B * GH + qe + (size_t)g * H];
      if (MODE == RNN_LSTM) {
        nx.cn = q.CP[(st + 1) * BH + e]; nx.cp = q.CP[st * BH + e];
      }
      if (MODE == RNN_GRU) {
        nx.hp = q.HP[st * BH + e]; nx.rn = q.RN[st * BH + e];
      }
    }
  };
  fetch(T - 1);
  for (int sv = T - 1; sv >= (q.dhx ? -1 : 0); --sv) {
    const int st = __builtin_amdgcn_readfirstlane(sv), t = dir ? T - 1 - st : st;
    CellBwdIn<MODE> in = nx;
    float (*red)[16][17] = red2[st & 1];
    if (st < T - 1) {
      seq_pause(p.pause);
      const __amdgpu_buffer_rsrc_t r = row.rsrc(st + 1);
      floatx4_t acc[1] = {{0.f, 0.f, 0.f, 0.f}};
      // (more chunks than there are scalar registers for their offsets and for whether they exist: both in each step, not once, where the
      // compiler moved 37 to 75 of them to vector registers and back; up to 16 chunks once is the faster one, by 2 to 3 %)
      SeqRow now = row;
      int rows = GH;
      if constexpr (NC > 16) asm volatile("" : "+s"(now.nc), "+s"(rows));
      uintx4_t v[2][U];
      seq_load(r, now, wave, v[0]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        if (b + 1 < NB) seq_load(r, now, wave + W * (b + 1) * U, v[(b + 1) & 1]);
        dead = __builtin_amdgcn_readfirstlane(seq_wait(r, now, wave + W * b * U, v[b & 1], dead, lost.limit));
        if (b == NB - 1) {
          seq_drain();
          fetch(st - 1);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
          if ((wave + W * (b * U + u)) * 16 < rows)
#pragma unroll
            for (int m = 0; m < 4; ++m)
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[b * U + u][m], __uint_as_float(v[b & 1][u][m]), acc[0], 0, 0, 0);
      }
      lost.tell(dead, acc);
#pragma unroll
      for (int x = 0; x < 4; ++x) red[wave][4 * fg + x][fr] = acc[0][x];
      __syncthreads();
    } else {
      fetch(st - 1);
    }
    if (cell) {
      float rec = 0.f;
      if (st < T - 1) {
#pragma unroll
        for (int w = 0; w < W; ++w) rec += red[w][unit][col];
      }
      if (st < 0) {
        q.dhx[e] = direct + rec;
      } else {
        bool gone = st == T - 1 && dead;
        if (MODE == RNN_RELU && __builtin_expect(rec != rec, 0))
          gone = seq_lost(&red[0][unit][col], 16 * 17, row, st + 1, col);
        in.go += direct;
        in.dc = dc;
        c.dgw = q.dGW + (size_t)t * B * GH;
        c.dgr = dGR + (size_t)st * B * GH;
        cell_bwd_finish<MODE, true>(c, cb, ch, H, in, rec, &dc, &direct, gone, row.base + st * row.step, &row, col);
      }
    }
  }
  if (cell && MODE == RNN_LSTM && q.dcx) q.dcx[e] = dc;
}

// What a recurrence finds in place: forward, per direction or stacked layer (blockIdx.y), the initial states and the summed biases (the GRU's
// n gate apart, whose recurrent bias stays inside r * (R_n h + b_Rn)), and for a sequence launch the initial state and
// RNN_UNSET in the exchange; backward, RNN_UNSET in all of it.
struct SeqInit {
  struct Dir {
    const float *hx, *cx, *bW, *bR;
    float *HP, *CP, *bsum, *X;
  } d[STACK_LAYERS];
  size_t BH, n;       // elements of a state / of the exchange to be filled
  int B;
  int GH, H, mode;
  uint32_t* status;   // to be cleared, or null
};
__global__ void __launch_bounds__(256) rnn_seq_init_kernel(SeqInit p) {
  const SeqInit::Dir& q = p.d[blockIdx.y];
  const size_t stride = (size_t)gridDim.x * 256, i0 = (size_t)blockIdx.x * 256 + threadIdx.x;
  const uintx4_t unset = {RNN_UNSET, RNN_UNSET, RNN_UNSET, RNN_UNSET};
  if (p.status && blockIdx.y == 0 && i0 == 0) *p.status = 0;
  const size_t first = p.BH ? (size_t)p.B * ((p.H + 15) & ~15) : 0;     // forward: the initial state, below
  for (size_t i = i0 + first / 4; i < p.n / 4; i += stride) reinterpret_cast<uintx4_t*>(q.X)[i] = unset;
  if (p.BH == 0) return;                      // backward: nothing but the fill
  for (size_t i = i0; i < p.BH; i += stride) {
    const float h = q.hx ? rnn_value(q.hx[i]) : 0.f;
    q.HP[i] = h;
    if (p.n) {
      const int b = (int)(i / p.H), k = (int)(i - (size_t)b * p.H), b0 = b & ~(SEQ_COLS - 1);
      const SeqRow row(q.X, p.H, p.B, b0);
      row.base[row.at(k, b - b0)] = h;
    }
    if (p.mode == RNN_LSTM) q.CP[i] = q.cx ? q.cx[i] : 0.f;
  }
  for (size_t i = i0; i < (size_t)p.GH; i += stride)
    q.bsum[i] = (p.mode == RNN_GRU && i >= (size_t)2 * p.H) ? q.bW[i] : q.bW[i] + q.bR[i];
}

// one launch for all directions or stacked layers
void launch_init(const SeqInit& p, int D, hipStream_t s) {
  const size_t most = std::max<size_t>(std::max<size_t>(p.n / 4, p.BH), p.GH);
  hipLaunchKernelGGL(rnn_seq_init_kernel, dim3((unsigned)std::min<size_t>((most + 255) / 256, 2048), D), dim3(256), 0, s, p);
}

inline unsigned nblocks(size_t n) { return (unsigned)((n + 255) / 256); }

// dst [M x N] = A [M x K] * B^T, through `scratch` when the contraction is cut into slices
int mm_nt(const float* A, const float* B, float* dst, size_t M, size_t N, size_t K, float* scratch, Scratch w, hipStream_t s) {
  if (const int rc = gemm32(2, A, B, dst, (int)M, (int)N, (int)K, nullptr, w.p, w.bytes, s); rc >= 0) return rc;
  const int ns = wgrad_slices(M, N, K);
  if (ns <= 1) return gemm_nt(FLHIP_F32, A, B, dst, (int)M, (int)N, (int)K, 1, s);
  if (const int rc = gemm_nt(FLHIP_F32, A, B, scratch, (int)M, (int)N, (int)K, ns, s)) return rc;
  hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(M * N)), dim3(256), 0, s, (const float*)nullptr, scratch, ns, dst,
                     M * N);
  return FLHIP_OK;
}

// The bias gradients of up to four sums in a launch, column sums of x [TB][GH]: a workgroup takes 32 columns, its threads every 32nd row.
struct BiasSums {
  const float* x[4];
  float *a[4], *b[4];      // where a sum goes, and where else (or null)
};
// Up to 1024 rows, 32 additions one after the other in a thread: 0.81 to 1.00 of the pass with the column sums' own launches (72 random layers, 0 to 28 us less).
// (Above it would still be up to 55 us less, GRU of 768 units, two directions, 2 layers, 1379 rows 2311 / 2256, but the chains of additions grow with the rows.)
constexpr int BIAS_ROWS = 1024;
__global__ void __launch_bounds__(1024) rnn_bias_kernel(BiasSums p, int GH, int TB) {
  __shared__ float sums[32][33];
  const int c = blockIdx.x * 32 + (threadIdx.x & 31), r0 = threadIdx.x >> 5;
  const float* const x = p.x[blockIdx.y];
  float v = 0.f;
  if (c < GH)
#pragma unroll 8
    for (int r = r0; r < TB; r += 32) v += x[(size_t)r * GH + c];
  sums[r0][threadIdx.x & 31] = v;
  __syncthreads();
  if (threadIdx.x >= 32 || c >= GH) return;
  v = sums[0][threadIdx.x];
#pragma unroll
  for (int r = 1; r < 32; ++r) v += sums[r][threadIdx.x];
  p.a[blockIdx.y][c] = v;
  if (p.b[blockIdx.y]) p.b[blockIdx.y][c] = v;
}

// dW [GH][in] row-major = column-major in x GH = IN [in x TB] * dGW^T; dR likewise with the states before each step; the
// bias gradients are the row sums (one sum for both but for the GRU: its n gate's recurrent side differs).  o, HP, dGW, dGR: of D directions
// over one input.  Those of two directions share their launches, and up to BIAS_ROWS rows the bias sums are one: every one of these launches is
// some 5 us of waiting, 14 of them behind a layer of two directions (tanh, 200 units, 3 layers, two directions, 65 steps of 10 columns, training: 968 us,
// now 859; GRU of 128 units, 3 layers, two directions, 16 steps of 8 columns 517, now 427).
int weight_gradients(const RnnGeom& g, int D, const Offsets* o, const float* in, size_t inl, const float* const* HP, const float* const* dGW,
                     const float* const* dGR, float* dw, float* ws, hipStream_t s) {
  const size_t TB = (size_t)g.T * g.B;
  float* scratch = ws + wgrad_scratch_offset(g);
  const Scratch w = scratch_of(g, ws);
  for (int r = 0; r < 2; ++r) {      // the input's matrix, the recurrent one
    const int M = r ? g.H : (int)inl;
    const float *a[2], *b[2];
    float* c[2];
    for (int d = 0; d < D; ++d) a[d] = r ? HP[d] : in, b[d] = r ? dGR[d] : dGW[d], c[d] = dw + (r ? o[d].R : o[d].W);
    const int both = D == 2 ? gemm32_pair(2, a[0], a[1], b[0], b[1], c[0], c[1], M, (int)g.GH, (int)TB, nullptr, nullptr, w.p, w.bytes, s) : -1;
    if (both > 0) return both;
    if (both < 0)
      for (int d = 0; d < D; ++d)
        if (const int rc = mm_nt(a[d], b[d], c[d], M, g.GH, TB, scratch, w, s)) return rc;
  }
  if (TB <= BIAS_ROWS) {
    BiasSums p{};
    int n = 0;
    for (int d = 0; d < D; ++d) {
      p.x[n] = dGW[d], p.a[n] = dw + o[d].bW, p.b[n] = g.mode == RNN_GRU ? nullptr : dw + o[d].bR, ++n;
      if (g.mode == RNN_GRU) p.x[n] = dGR[d], p.a[n] = dw + o[d].bR, ++n;
    }
    hipLaunchKernelGGL(rnn_bias_kernel, dim3((unsigned)((g.GH + 31) / 32), (unsigned)n), dim3(1024), 0, s, p, (int)g.GH, (int)TB);
    return check_launch("rnn_bwd");
  }
  for (int d = 0; d < D; ++d) {
    if (const int rc = flhip_sum_columns_ws(dGW[d], dw + o[d].bW, (int32_t)g.GH, (int32_t)TB, FLHIP_F32, w.p, w.bytes, s)) return rc;
    if (g.mode == RNN_GRU) {
      if (const int rc = flhip_sum_columns_ws(dGR[d], dw + o[d].bR, (int32_t)g.GH, (int32_t)TB, FLHIP_F32, w.p, w.bytes, s)) return rc;
    } else {
      hipLaunchKernelGGL(rnn_init_kernel, dim3(nblocks(g.GH)), dim3(256), 0, s, dw + o[d].bW, dw + o[d].bR, g.GH);
    }
  }
  return check_launch("rnn_bwd");
}

template <int MODE>
int forward_pl(const RnnGeom& g, int pl, const float* in, size_t inl, const float* w, const float* hx,
               const float* cx, float* out, float* hy, float* cy, float* res, float* ws, hipStream_t s) {
  const Reserve r = reserve_layout(g);
  const Offsets o = offsets(g, pl);
  const int dir = pl % g.D;
  const size_t TB = (size_t)g.T * g.B;
  float* HP = res + (size_t)pl * r.per_pl + r.hp;
  float* CP = res + (size_t)pl * r.per_pl + r.cp;
  float* GT = res + (size_t)pl * r.per_pl + r.gt;
  float* RN = res + (size_t)pl * r.per_pl + r.rn;
  float* XP = ws;
  float* RP = XP + TB * g.GH;
  int kdummy;
  float* bsum = RP + (size_t)step_slices(g.GH, g.B, g.H, &kdummy) * g.B * g.GH;
  SeqInit ip{};
  ip.BH = g.BH; ip.GH = (int)g.GH; ip.H = g.H; ip.mode = g.mode;
  ip.d[0] = {hx ? hx + (size_t)pl * g.BH : nullptr, cx ? cx + (size_t)pl * g.BH : nullptr, w + o.bW, w + o.bR, HP, CP, bsum};
  launch_init(ip, 1, s);
  // XP [GH x TB] = W [GH x in] (row-major = a column-major in x GH matrix, transposed) * IN [in x TB]
  if (const int rc = mm(w + o.W, in, XP, g.GH, TB, inl, 1, 0, bsum, s, scratch_of(g, ws), MODE == RNN_RELU)) return rc;
  for (int st = 0; st < g.T; ++st) {
    const int t = dir ? g.T - 1 - st : st;
    int nrp = 1;
    if (const int rc = mm_sliced(w + o.R, HP + (size_t)st * g.BH, RP, g.GH, g.B, g.H, 1, &nrp, s)) return rc;
    CellFwd a{};
    a.xp = XP + (size_t)t * g.B * g.GH;
    a.rp = RP;
    a.nrp = nrp;
    a.bRn = w + o.bR + 2 * g.H;
    a.hp = HP + (size_t)st * g.BH;
    a.cp = CP + (size_t)st * g.BH;
    a.hn = HP + (size_t)(st + 1) * g.BH;
    a.cn = CP + (size_t)(st + 1) * g.BH;
    a.gt = GT + (size_t)st * g.B * g.GH;
    a.rn = RN + (size_t)st * g.BH;
    a.ldo = g.D * g.H;
    a.out = out + (size_t)t * g.B * a.ldo + (size_t)dir * g.H;
    const bool last = st == g.T - 1;
    a.hy = last ? hy + (size_t)pl * g.BH : nullptr;
    a.cy = (last && cy && MODE == RNN_LSTM) ? cy + (size_t)pl * g.BH : nullptr;
    hipLaunchKernelGGL((rnn_cell_fwd<MODE>), dim3(nblocks(g.BH)), dim3(256), 0, s, a, g.B, g.H);
  }
  return check_launch("rnn_fwd");
}

// hidden units per workgroup of rnn_seq_fwd: the fewest for which a layer's clusters fit the compute units
int seq_units(const RnnGeom& g) {
  const int clusters = g.D * ((g.B + SEQ_COLS - 1) / SEQ_COLS), cus = mfma_num_cus();
  if (g.mode == RNN_LSTM || g.mode == RNN_GRU) {
    if (clusters * ((g.H + 3) / 4) <= cus) return 4;
    if (clusters * ((g.H + 7) / 8) <= cus) return 8;
  }
  return 16;
}

// The pause of seq_pause.  Too short costs up to a tenth of a step, too long some 60 ns per step and unit.  Forward it follows from
// what all workgroups of a layer ask for in a step (V, MB).  Measured, us with pauses of 2 / 4 / 6 / 8: LSTM of 320 units, 5 columns over
// 100 steps (V 0.5) 214 / 218 / 228 / 238; GRU of 256 units, two directions, 20 columns (2.6) 204 / 208 / 216 / 228; tanh of 384 units, two
// directions, 64 columns (4.7) 231 / 215 / 227 / 233; LSTM of 512 units, two directions, 32 columns over 200 steps (8.4) 686 / 642 / 639 /
// 648; GRU of 1024 units, 64 columns (16.8) 580 / 568 / 572 / 583.  With 4 units to a workgroup every workgroup's loads are many for the few
// columns that this many clusters have; 60 steps, 2 / 3 / 4: LSTM of 1024 units, 1 column 200 / 179 / 177, 2 columns 187 / 177 / 179, of 768,
// 1 column 185 / 163 / 164, of 512, 8 columns 145 / 145 / 148; GRU of 640, 1 column 162 / 150 / 153; but LSTM of 320 units, 1 column 133 / 132 / 132, 16
// 135 / 136 / 139, and with 8 units to a workgroup (LSTM of 1024, two directions, 1 column) 241 / 245 / 246.
int seq_pause_fwd(const RnnGeom& g, int units) {
  const double V = (double)g.D * ((g.H + units - 1) / units) * g.B * g.H * 4e-6;
  return V >= 4 ? 4 : units == 4 && g.H >= 512 ? 3 : 2;
}
// Backward a step has more to load and to do between its stores and the next step's loads: 0 / 1 / 2 / 4 1372 / 1375 / 1382 / 1405 us
// (that LSTM of 512 units), 338 / 337 / 343 / 352 (LSTM of 128 units, 16 columns over 100 steps).  Over 42 layers of up to 4 columns each 0
// takes 0.987 of the time with 1 (at worst 1.004), over 5 to 16 columns 0.994 (1.024), over more 1.004.
int seq_pause_bwd(const RnnGeom& g) { return g.B <= 4 ? 0 : 1; }

// Does a pass gain by sequence launches?  One costs some 20 us more than a step's launch does (the cooperative queue, on both
// sides), and saves on each step, the more so the more a step has to do.  Sequence / steps, of the time:
//   Against the step kernels, over 4 / 6 / 8 steps: LSTM of 128 units forward 1.07, 0.93, 0.80 with 16 columns, 0.94, 0.76, 0.65
//   with 32, 0.92, 0.75, 0.64 with 64; of 512 units, two directions, 1.01, 1.00, 0.91 with 16, 0.86, 0.73, 0.66 with 64; of 1024 units,
//   two directions, 32 columns, over 2 / 4 steps 0.99 and 0.80; GRU of 512 units, training, 16 columns 1.27, 1.09, 0.99.
//   Against the two-kernel steps (two launches per step and direction), over 2 / 4 steps: LSTM of 512 units, 128 columns 0.71, 0.47;
//   of 200 units 1.08, 0.84, ReLU of 200 units 1.13, 0.85; of 128 units, two directions 0.77, 0.56.
//   Backward the steps cost more: GRU of 768 units, 3 layers, 51 columns, over 3 steps 0.81; against the two-kernel steps, one step, LSTM
//   of 768 units, 70 columns 0.75, of 1000 units, 1 column 0.83, GRU of 768 units, 2 layers, 66 columns 0.87.
//   Clusters beyond the compute units go in further launches, so that with many columns the estimates (us per step, from 32 to
//   1024 units, ReLU to LSTM) decide: LSTM of 512 units over 20 steps, 256 columns (2 launches) 0.77, 512 columns (4) 1.19; 1024
//   units, 256 columns (4) 1.23, backward 0.8.
bool seq_pays(const RnnGeom& g, bool bwd) {
  const int tiles = (g.B + SEQ_COLS - 1) / SEQ_COLS;
  if (fused_applies(g)) {
    const int weight = g.D * g.H * tiles * (g.G == 1 ? 5 : 2 * g.G + 2) / 10;
    return g.T >= (weight >= (bwd ? 2000 : 3500) ? 3 : weight >= 1500 ? 4 : g.B > 32 ? 5 : weight >= 600 || g.B > 16 ? 6 : 8);
  }
  const int units = bwd ? 16 : seq_units(g), nwg = (g.H + units - 1) / units, per = std::max(1, mfma_num_cus() / nwg);
  const int launches = (g.D * tiles + per - 1) / per;
  if (launches == 1) return g.T >= (bwd && g.GH >= 2000 ? 1 : g.D == 2 || g.GH >= 1000 ? 2 : 3);
  const double H = g.H, step = bwd ? 5.5 + H * (0.006 + 0.016 * g.G * (1.0 + g.B / 750.0)) : 5.0 + H * (0.012 + 0.0053 * g.G);
  const double seq = bwd ? 1.6 + H * (0.0048 * g.G - 0.0003) : 1.1 + H * (0.0015 + 0.0019 * g.G);
  return g.T * (g.D * step - launches * seq) > 22.0 * launches;
}

// ---- launching whole sequences: the hidden size a multiple of 4 (16-byte pieces of the state) and at most 1024
// (registers), a step's gates within what a buffer load addresses (2 GiB: an LSTM of 1024 units up to 131071
// columns) ...
bool seq_asked(const RnnGeom& g, bool bwd) {
  const int asked = options().rnn_sequences;
  return !options().rnn_unfused && asked != Options::SEQ_NEVER && seq_holds(g) && (size_t)g.B * g.GH * 4 < ((size_t)1 << 31) &&
         (asked != Options::SEQ_AUTO || seq_pays(g, bwd));
}
// ... and a stream that is not being captured (a cooperative launch is not recorded)
bool seq_uncaptured(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(s, &st) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  return st == hipStreamCaptureStatusNone;
}
bool seq_applies(const RnnGeom& g, bool bwd, hipStream_t s) { return seq_asked(g, bwd) && seq_uncaptured(s); }

// Where the exchange of a layer's sequence launch lies in the workspace, in floats (the layers use it in turn): in what the pass leaves idle
// while the launch runs, so that it costs nothing but for the lower ones of stacked GRU layers, which need 3 H per position and direction where 2 H to 4 H are idle
// (3 layers of 512 units, 64 columns over 100 steps 144 -> 159 MiB).
//   forward   behind the projections and biases: the backward pass' buffers
//   backward  not GRU, forward direction: in place of dGR[0], which is dGW[0] there (the same values in the same order; rows of whole
//             chunks only); else gin, tmp and the step kernels' buffers behind them (the topmost layer: gout in front of them too, it reads
//             the caller's); else the weight gradients' scratch, or behind everything from the products' scratch on
// (A buffer of its own in every call: LSTM of 512 units, 2 x 2 layers, 32 columns over 200 steps 324 -> 424 MiB of workspace.)
struct SeqPlace {
  size_t at[2];
  size_t end;          // floats of workspace that it takes
  bool shared;         // dGR[0] is dGW[0]
};
SeqPlace seq_place(const RnnGeom& g, bool bwd, bool top) {
  const size_t TB = (size_t)g.T * g.B, core = workspace_core(g), need = (size_t)g.T * seq_row(g, bwd ? g.GH : g.H);
  SeqPlace p{};
  size_t from[2] = {}, to[2] = {};
  if (bwd) {
    const size_t gout = 2 * TB * g.GH, scratch = wgrad_scratch_offset(g);
    from[0] = top ? gout : gout + TB * g.D * g.H;
    to[0] = g.D == 1 ? scratch + wgrad_scratch(g) : scratch - 2 * TB * g.GH - 3 * g.BH;
    from[1] = scratch;
    to[1] = g.D == 1 ? scratch : scratch + wgrad_scratch(g);
  } else {
    from[0] = (size_t)g.D * (TB * g.GH + g.GH);
    to[0] = core - 4;
  }
  for (int dir = 0; dir < g.D; ++dir) {
    if (bwd && dir == 0 && g.mode != RNN_GRU && g.GH % 16 == 0) {
      p.at[0] = TB * g.GH;
      p.shared = true;
      continue;
    }
    bool placed = false;
    for (int i = 0; i < 2 && !placed; ++i) {
      const size_t at = (from[i] + 63) & ~(size_t)63;
      if (at + need > to[i]) continue;
      p.at[dir] = at;
      from[i] = at + need;
      placed = true;
    }
    if (placed) continue;
    // (forward the projections use the scratch after the exchange is filled)
    p.at[dir] = p.end ? p.end : core + (bwd ? 0 : scratch_of(g, nullptr).bytes / sizeof(float));
    p.end = p.at[dir] + need;
  }
  return p;
}
// floats of workspace that the exchanges of a pass end at
size_t seq_end(const RnnGeom& g, bool bwd) {
  const size_t top = seq_place(g, bwd, true).end;
  return bwd && g.L > 1 ? std::max(top, seq_place(g, true, false).end) : top;
}

// what a call cannot do without, and with what its sequence launches take where they may be launched
size_t base_bytes(const RnnGeom& g) { return workspace_core(g) * sizeof(float) + scratch_of(g, nullptr).bytes; }
size_t workspace_bytes(const RnnGeom& g) {
  size_t end = 0;
  for (const bool bwd : {false, true})
    if (seq_asked(g, bwd)) end = std::max(end, seq_end(g, bwd));
  return std::max(base_bytes(g), end * sizeof(float));
}

std::atomic<uint64_t> g_seq_launches{0};

// FLHIP_DECLINED where the runtime refuses the first launch (nothing has run then): the device does not hold it, or the
// process gets no cooperative queue (a program started by a process that had launched cooperatively on the same card was
// told 'illegal state'; by itself it launches)
template <typename P>
int seq_launch(void (*kernel)(P), P& p, int clusters, size_t lds, hipStream_t s) {
  if (options().rnn_sequences == Options::SEQ_REFUSED) return FLHIP_DECLINED;
  if (!mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return FLHIP_DECLINED;
  const int per = std::max(1, mfma_num_cus() / p.nwg);
  for (p.cluster0 = 0; p.cluster0 < clusters; p.cluster0 += per) {
    void* args[] = {&p};
    const unsigned grid = (unsigned)(std::min(per, clusters - p.cluster0) * p.nwg);
    const hipError_t e = hipLaunchCooperativeKernel(reinterpret_cast<const void*>(kernel), dim3(grid), dim3(SEQ_THREADS), args,
                                                    (unsigned)lds, s);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      if (p.cluster0 == 0 && (e == hipErrorCooperativeLaunchTooLarge || e == hipErrorIllegalState || e == hipErrorNotSupported))
        return FLHIP_DECLINED;
      return fail(FLHIP_RUNTIME_ERROR, std::string("rnn: ") + hipGetErrorString(e));
    }
    g_seq_launches.fetch_add(1, std::memory_order_relaxed);
  }
  return FLHIP_OK;
}

template <int MODE, int HU>
int seq_fwd_hu(const RnnGeom& g, SeqFwd& p, hipStream_t s) {
  constexpr int RT = (gates_of(MODE) * HU + 15) / 16;
  p.nwg = (g.H + HU - 1) / HU;
  const size_t lds = (size_t)2 * SEQ_WAVES * RT * 16 * 17 * sizeof(float);
  const int nc = ((g.H + 15) / 16 + SEQ_WAVES - 1) / SEQ_WAVES;
  if (nc <= 2) return seq_launch(rnn_seq_fwd<MODE, HU, 2>, p, g.D * p.groups, lds, s);
  if (nc <= 4) return seq_launch(rnn_seq_fwd<MODE, HU, 4>, p, g.D * p.groups, lds, s);
  return seq_launch(rnn_seq_fwd<MODE, HU, 8>, p, g.D * p.groups, lds, s);
}
template <int MODE>
int seq_fwd(const RnnGeom& g, SeqFwd& p, hipStream_t s) {
  if constexpr (MODE == RNN_LSTM || MODE == RNN_GRU) {
    const int units = seq_units(g);
    if (units == 4) return seq_fwd_hu<MODE, 4>(g, p, s);
    if (units == 8) return seq_fwd_hu<MODE, 8>(g, p, s);
  }
  return seq_fwd_hu<MODE, 16>(g, p, s);
}

// Hidden units per workgroup of rnn_stack_fwd, or 0: one direction, nothing between the layers, all their clusters in one
// launch, both matrices' fragments in 128 registers; not ReLU layers, whose input products stay the fp32 instruction's (the same
// sums in another order put its inputs on the other side of zero).  One launch is the faster one from three steps of a layer on (us, a launch
// per step / one for all: 2 layers over 1 / 2 / 3 steps, LSTM of 512 units, 16 columns 39 / 36, 46 / 39, 53 / 42, GRU of 256 units, 40 columns 34
// / 35, 43 / 37, 53 / 40; 3 layers over 1 step, LSTM of 320 units, 5 columns 51 / 38).
int stack_units(const RnnGeom& g) {
  const int asked = options().rnn_sequences;
  if (options().rnn_unfused || asked == Options::SEQ_ALWAYS || asked == Options::SEQ_NEVER) return 0;
  if (asked == Options::SEQ_AUTO && g.L * g.T < 3) return 0;
  if (g.D != 1 || g.L < 2 || g.L > STACK_LAYERS || g.mode == RNN_RELU || g.dropout > 0.f || !seq_holds(g)) return 0;
  const int clusters = g.L * ((g.B + SEQ_COLS - 1) / SEQ_COLS), nc = ((g.H + 15) / 16 + SEQ_WAVES - 1) / SEQ_WAVES;
  const int chunks = nc <= 2 ? 2 : nc <= 4 ? 4 : 8;
  for (int units = g.G == 1 ? 16 : 4; units <= 16; units *= 2)
    if ((long long)clusters * ((g.H + units - 1) / units) <= mfma_num_cus()) return (g.G * units + 15) / 16 * chunks <= 16 ? units : 0;
  return 0;
}
// where the exchanges of the layers lie, (T + 1) steps each (floats into the workspace, behind the projections and biases; 0: no room)
size_t stack_place(const RnnGeom& g) {
  const size_t at = ((size_t)g.T * g.B * g.GH + g.L * g.GH + 63) & ~(size_t)63;
  return at + g.L * (g.T + 1) * seq_row(g, g.H) <= workspace_core(g) - 4 ? at : 0;
}
// All steps in one cooperative launch, or, on a stream that is being captured, a launch for each diagonal of layers and steps: what a step waits for is
// there when it starts, so that such a launch needs none of the others, and the same kernel gives the same bits.  In a graph, forward, us, a launch per
// layer and step with the products between layers apart / these: LSTM of 320 units, 3 layers, 5 columns, over 25 steps 398 / 158, over 100 steps 1556 / 564; of
// 512 units, 2 layers, 16 columns over 50 steps 576 / 342; of 256 units, 4 layers, 64 columns over 20 steps 642 / 228; of 768 units, 2 layers, 16 columns over 30
// steps 494 / 398; GRU of 384 units, 2 layers, 64 columns over 40 steps 800 / 424; tanh of 1020 units, 2 layers, 5 columns over 30 steps 1172 / 266.  What bounds
// large ones is the matrices, fetched in every launch, the input's too: level at 896 units (LSTM, 2 layers, 3 columns over 30 steps 429 / 412, GRU 395 / 386), and the
// slower ones at 1024 over few columns (48 MB a launch: LSTM, 2 layers over 30 steps, 1 / 8 / 16 columns 414 / 483, 477 / 501, 516 / 524, GRU 1 / 16 columns 378 / 427, 493 /
// 469).  (With the states asked for before the matrices, and the input product while the recurrent matrix is on its way, nothing.)
int stack_launch(void (*kernel)(SeqStack), SeqStack& p, int clusters, size_t lds, bool captured, hipStream_t s) {
  p.diagonal = -1;
  if (!captured) return seq_launch(kernel, p, clusters, lds, s);
  if (options().rnn_sequences == Options::SEQ_REFUSED || !mfma_allow_lds(reinterpret_cast<const void*>(kernel), lds)) return FLHIP_DECLINED;
  for (p.diagonal = 0; p.diagonal < p.T + p.L - 1; ++p.diagonal) hipLaunchKernelGGL(kernel, dim3((unsigned)(clusters * p.nwg)), dim3(SEQ_THREADS), lds, s, p);
  return FLHIP_OK;
}
template <int MODE, int HU>
int stack_fwd_hu(const RnnGeom& g, SeqStack& p, bool captured, hipStream_t s) {
  constexpr int RT = (gates_of(MODE) * HU + 15) / 16;
  p.nwg = (g.H + HU - 1) / HU;
  const size_t lds = stack_lds(MODE, RT);
  const int nc = ((g.H + 15) / 16 + SEQ_WAVES - 1) / SEQ_WAVES, clusters = g.L * p.groups;
  if (nc <= 2) return stack_launch(rnn_stack_fwd<MODE, HU, 2>, p, clusters, lds, captured, s);
  if (nc <= 4) return stack_launch(rnn_stack_fwd<MODE, HU, 4>, p, clusters, lds, captured, s);
  if constexpr (RT <= 2) return stack_launch(rnn_stack_fwd<MODE, HU, 8>, p, clusters, lds, captured, s);
  return FLHIP_DECLINED;
}
// all layers of a stack; FLHIP_DECLINED: not run
template <int MODE>
int forward_stack(const RnnGeom& g, const float* x, const float* w, const float* hx, const float* cx, float* y, float* hy, float* cy,
                  float* res, float* ws, bool captured, hipStream_t s) {
  const int units = stack_units(g);
  const size_t place = stack_place(g), TB = (size_t)g.T * g.B, act = TB * g.H;
  if (!units || !place) return FLHIP_DECLINED;
  const Reserve r = reserve_layout(g);
  SeqInit ip{};
  SeqStack p{};
  p.B = g.B; p.H = g.H; p.T = g.T; p.L = g.L;
  p.groups = (g.B + SEQ_COLS - 1) / SEQ_COLS;
  p.wait = options().rnn_wait; p.pause = 2; p.status = seq_status(g, ws);
  ip.BH = g.BH; ip.n = (size_t)(g.T + 1) * seq_row(g, g.H); ip.B = g.B; ip.GH = (int)g.GH; ip.H = g.H; ip.mode = g.mode;
  ip.status = p.status;
  for (int l = 0; l < g.L; ++l) {
    const Offsets o = offsets(g, l);
    float* const base = res + (size_t)l * r.per_pl;
    float* const bsum = ws + TB * g.GH + l * g.GH;
    p.d[l] = {ws, w + o.W, w + o.R, bsum, w + o.bR + 2 * g.H, base + r.hp, base + r.cp, base + r.gt, base + r.rn,
              l == g.L - 1 ? y : res + r.acts + (size_t)l * act, hy + l * g.BH, cy && MODE == RNN_LSTM ? cy + l * g.BH : nullptr,
              ws + place + l * ip.n};
    ip.d[l] = {hx ? hx + l * g.BH : nullptr, cx ? cx + l * g.BH : nullptr, w + o.bW, w + o.bR, p.d[l].HP, p.d[l].CP, bsum, p.d[l].X};
  }
  launch_init(ip, g.L, s);
  if (const int rc = mm(w + offsets(g, 0).W, x, ws, g.GH, TB, g.I, 1, 0, ip.d[0].bsum, s, scratch_of(g, ws), false)) return rc;
  int rc = FLHIP_DECLINED;
  if constexpr (MODE == RNN_LSTM || MODE == RNN_GRU) {
    if (units == 4) rc = stack_fwd_hu<MODE, 4>(g, p, captured, s);
    else if (units == 8) rc = stack_fwd_hu<MODE, 8>(g, p, captured, s);
    else rc = stack_fwd_hu<MODE, 16>(g, p, captured, s);
  } else if constexpr (MODE == RNN_TANH) {
    rc = stack_fwd_hu<MODE, 16>(g, p, captured, s);
  }
  return rc == FLHIP_OK ? check_launch("rnn_fwd") : rc;
}

template <int MODE>
int seq_bwd(const RnnGeom& g, SeqBwd& p, hipStream_t s) {
  p.nwg = (g.H + 15) / 16;
  const int nc = ((int)((g.GH + 15) / 16) + SEQ_WAVES - 1) / SEQ_WAVES, clusters = g.D * p.groups;
  if (nc <= 4) return seq_launch(rnn_seq_bwd<MODE, 4>, p, clusters, 0, s);
  if (nc <= 8) return seq_launch(rnn_seq_bwd<MODE, 8>, p, clusters, 0, s);
  if constexpr (MODE == RNN_LSTM || MODE == RNN_GRU) {
    if (nc <= 16) return seq_launch(rnn_seq_bwd<MODE, 16>, p, clusters, 0, s);
    if (nc <= 24) return seq_launch(rnn_seq_bwd<MODE, 24>, p, clusters, 0, s);
    if (MODE == RNN_LSTM && nc <= 32) return seq_launch(rnn_seq_bwd<MODE, MODE == RNN_LSTM ? 32 : 24>, p, clusters, 0, s);
  }
  return FLHIP_DECLINED;
}

// Four or eight waves to a workgroup of rnn_step_fwd: as many chunks are asked for as fill whole rounds of the workgroup (past
// the last one, again), so the number with the smaller rounds wins where the other's ask for more (20 steps of an LSTM in a
// captured graph, us with 4 / 8 waves: 512 units, 32 columns 164 / 221, two directions 192 / 246; 1536 units 33 % more with 8;
// 640 units, 64 columns 17 % more).  Equal rounds: eight where they need only one and the chip holds a workgroup to a compute unit
// (1024 units, 1 column 143 / 135, two directions 199 / 227; 512 units, 64 columns 238 / 225), else four.
template <int NBT>
bool step_fwd_eight(int H, int D) {
  constexpr int U = step_fwd_chunks(NBT);
  const int chunks = H / 16, four = (chunks + 4 * U - 1) / (4 * U), eight = (chunks + 8 * U - 1) / (8 * U);
  return four == 2 * eight && eight == 1 && (NBT == 4 || D * H <= 1024);
}

template <int MODE, int NBT>
void launch_step_fwd(const StepFwd& p, int D, hipStream_t s) {
  const dim3 grid(p.H / 4, D);
  if (step_fwd_eight<NBT>(p.H, D)) hipLaunchKernelGGL((rnn_step_fwd<MODE, NBT, 8>), grid, dim3(512), 0, s, p);
  else hipLaunchKernelGGL((rnn_step_fwd<MODE, NBT, 4>), grid, dim3(256), 0, s, p);
}

// one layer, all directions: per direction the input projection of all steps, then the recurrence: one launch for the whole
// sequence (seq), or one per time step for both directions
template <int MODE>
int forward_layer_fused(const RnnGeom& g, int l, const float* in, size_t inl, const float* w, const float* hx,
                        const float* cx, float* out, float* hy, float* cy, float* res, float* ws, bool& seq, hipStream_t s) {
  const Reserve r = reserve_layout(g);
  const size_t TB = (size_t)g.T * g.B;
  // the initial states and the input projections
  SeqInit ip{};
  SeqFwd p{};
  const SeqPlace place = seq ? seq_place(g, false, true) : SeqPlace{};
  p.B = g.B; p.H = g.H; p.T = g.T; p.ldo = g.D * g.H;
  p.groups = (g.B + SEQ_COLS - 1) / SEQ_COLS;
  p.wait = options().rnn_wait; p.pause = seq_pause_fwd(g, seq_units(g)); p.status = seq_status(g, ws); p.layer = (uint32_t)l + 1;
  ip.BH = g.BH; ip.n = seq ? (size_t)g.T * seq_row(g, g.H) : 0; ip.B = g.B; ip.GH = (int)g.GH; ip.H = g.H; ip.mode = g.mode;
  ip.status = l == 0 ? p.status : nullptr;
  for (int dir = 0; dir < g.D; ++dir) {
    const int pl = l * g.D + dir;
    const Offsets o = offsets(g, pl);
    float* base = res + (size_t)pl * r.per_pl;
    SeqFwd::Dir& q = p.d[dir];
    q.xp = ws + (size_t)dir * TB * g.GH;
    q.R = w + o.R; q.bRn = w + o.bR + 2 * g.H;
    q.HP = base + r.hp; q.CP = base + r.cp; q.GT = base + r.gt; q.RN = base + r.rn;
    q.out = out + (size_t)dir * g.H;
    q.X = ws + place.at[dir];
    q.hy = hy + (size_t)pl * g.BH;
    q.cy = cy && MODE == RNN_LSTM ? cy + (size_t)pl * g.BH : nullptr;
    ip.d[dir] = {hx ? hx + (size_t)pl * g.BH : nullptr, cx ? cx + (size_t)pl * g.BH : nullptr, w + o.bW, w + o.bR, q.HP, q.CP,
                 ws + (size_t)g.D * TB * g.GH + (size_t)dir * g.GH, q.X};
  }
  launch_init(ip, g.D, s);
  int both = -1;      // the projections of two directions in a launch (but a ReLU layer's, whose sums stay what they are)
  if (g.D == 2 && MODE != RNN_RELU) {
    const Scratch sc = scratch_of(g, ws);
    both = gemm32_pair(1, w + offsets(g, l * 2).W, w + offsets(g, l * 2 + 1).W, in, in, const_cast<float*>(p.d[0].xp), const_cast<float*>(p.d[1].xp),
                       (int)g.GH, (int)TB, (int)inl, ip.d[0].bsum, ip.d[1].bsum, sc.p, sc.bytes, s);
    if (both > 0) return both;
  }
  for (int dir = 0; both < 0 && dir < g.D; ++dir)
    if (const int rc = mm(w + offsets(g, l * g.D + dir).W, in, const_cast<float*>(p.d[dir].xp), g.GH, TB, inl, 1, 0,
                          ip.d[dir].bsum, s, scratch_of(g, ws), MODE == RNN_RELU))
      return rc;
  if (seq) {
    const int rc = seq_fwd<MODE>(g, p, s);
    if (rc != FLHIP_DECLINED) return rc == FLHIP_OK ? check_launch("rnn_fwd") : rc;
    seq = false;              // nor the layers that follow
    if (!fused_applies(g)) return FLHIP_DECLINED;
  }
  for (int st = 0; st < g.T; ++st) {
    StepFwd p{};
    p.B = g.B;
    p.H = g.H;
    for (int dir = 0; dir < g.D; ++dir) {
      const int pl = l * g.D + dir, t = dir ? g.T - 1 - st : st;
      const Offsets o = offsets(g, pl);
      float* base = res + (size_t)pl * r.per_pl;
      CellFwd& a = p.d[dir];
      a.xp = ws + (size_t)dir * TB * g.GH + (size_t)t * g.B * g.GH;
      a.R = w + o.R;
      a.bRn = w + o.bR + 2 * g.H;
      a.hp = base + r.hp + (size_t)st * g.BH;
      a.cp = base + r.cp + (size_t)st * g.BH;
      a.hn = base + r.hp + (size_t)(st + 1) * g.BH;
      a.cn = base + r.cp + (size_t)(st + 1) * g.BH;
      a.gt = base + r.gt + (size_t)st * g.B * g.GH;
      a.rn = base + r.rn + (size_t)st * g.BH;
      a.ldo = g.D * g.H;
      a.out = out + (size_t)t * g.B * a.ldo + (size_t)dir * g.H;
      const bool last = st == g.T - 1;
      a.hy = last ? hy + (size_t)pl * g.BH : nullptr;
      a.cy = (last && cy && MODE == RNN_LSTM) ? cy + (size_t)pl * g.BH : nullptr;
    }
    if (g.B <= 16) launch_step_fwd<MODE, 1>(p, g.D, s);
    else if (g.B <= 32) launch_step_fwd<MODE, 2>(p, g.D, s);
    else launch_step_fwd<MODE, 4>(p, g.D, s);
  }
  return check_launch("rnn_fwd");
}

template <int MODE>
int backward_pl(const RnnGeom& g, int pl, const float* in, size_t inl, const float* w, const float* gout,
                const float* dhy, const float* dcy, float* gin, bool first_dir, float* dhx, float* dcx,
                float* dw, const float* res, float* ws, hipStream_t s) {
  const Reserve r = reserve_layout(g);
  const Offsets o = offsets(g, pl);
  const int dir = pl % g.D;
  const size_t TB = (size_t)g.T * g.B, inmax = widest_input(g);
  const float* HP = res + (size_t)pl * r.per_pl + r.hp;
  const float* CP = res + (size_t)pl * r.per_pl + r.cp;
  const float* GT = res + (size_t)pl * r.per_pl + r.gt;
  const float* RN = res + (size_t)pl * r.per_pl + r.rn;
  float* dGW = ws;
  float* dGR = dGW + TB * g.GH;
  float* tmp = dGR + TB * g.GH + TB * g.D * g.H + TB * inmax;   // behind gout and gin
  float* dh_dir = tmp + TB * inmax;                               // two buffers, alternating
  float* dc = dh_dir + 2 * g.BH;
  float* dh_rec = dc + g.BH;                                      // as many slices as step_slices says
  if (MODE == RNN_LSTM)
    hipLaunchKernelGGL(rnn_init_kernel, dim3(nblocks(g.BH)), dim3(256), 0, s,
                       dcy ? dcy + (size_t)pl * g.BH : nullptr, dc, g.BH);
  const float* dha = dhy ? dhy + (size_t)pl * g.BH : nullptr;   // direct part for the first step walked
  const float* dhb = nullptr;
  int ndhb = 1;
  for (int st = g.T - 1; st >= 0; --st) {
    const int t = dir ? g.T - 1 - st : st;
    CellBwd a{};
    a.ldo = g.D * g.H;
    a.gout = gout ? gout + (size_t)t * g.B * a.ldo + (size_t)dir * g.H : nullptr;
    a.dh_a = dha;
    a.dh_b = dhb;
    a.ndhb = ndhb;
    a.dc = dc;
    a.gt = GT + (size_t)st * g.B * g.GH;
    a.cp = CP + (size_t)st * g.BH;
    a.cn = CP + (size_t)(st + 1) * g.BH;
    a.hp = HP + (size_t)st * g.BH;
    a.rn = RN + (size_t)st * g.BH;
    a.dgw = dGW + (size_t)t * g.B * g.GH;
    a.dgr = dGR + (size_t)st * g.B * g.GH;
    a.dh_dir = dh_dir + (size_t)(st & 1) * g.BH;
    hipLaunchKernelGGL((rnn_cell_bwd<MODE>), dim3(nblocks(g.BH)), dim3(256), 0, s, a, g.B, g.H);
    // gradient through the recurrent matrices: dh_rec [H x B] = R^T [H x GH] * dGR[st] [GH x B]
    if (const int rc = mm_sliced(w + o.R, a.dgr, dh_rec, g.H, g.B, g.GH, 0, &ndhb, s)) return rc;
    dha = a.dh_dir;
    dhb = dh_rec;
  }
  if (dhx)
    hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(g.BH)), dim3(256), 0, s, dha, dhb, ndhb, dhx + (size_t)pl * g.BH,
                       g.BH);
  if (dcx && MODE == RNN_LSTM)
    hipLaunchKernelGGL(rnn_init_kernel, dim3(nblocks(g.BH)), dim3(256), 0, s, dc, dcx + (size_t)pl * g.BH, g.BH);
  // gradient of the layer input: gin [in x TB] (+)= W^T [in x GH] * dGW [GH x TB]
  float* gdst = first_dir ? gin : tmp;
  if (const int rc = mm(w + o.W, dGW, gdst, inl, TB, g.GH, 0, 0, nullptr, s, scratch_of(g, ws))) return rc;
  if (!first_dir)
    hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(TB * inl)), dim3(256), 0, s, gin, tmp, 1, gin, TB * inl);
  const float *hp = HP, *gw = dGW, *gr = dGR;
  return weight_gradients(g, 1, &o, in, inl, &hp, &gw, &gr, dw, ws, s);
}

template <int MODE, int NBT>
void launch_step_bwd(const StepBwd& p, int D, hipStream_t s) {
  hipLaunchKernelGGL((rnn_step_bwd<MODE, NBT>), dim3(p.H / 16, D), dim3(64 * step_bwd_waves(NBT)), 0, s, p);
}

template <int MODE>
int backward_layer_fused(const RnnGeom& g, int l, const float* in, size_t inl, const float* w, const float* gout,
                         const float* dhy, const float* dcy, float* gin, float* dhx, float* dcx, float* dw,
                         const float* res, float* ws, bool& seq, hipStream_t s) {
  const Reserve r = reserve_layout(g);
  const size_t TB = (size_t)g.T * g.B, inmax = widest_input(g);
  int kdummy;
  const size_t sb = step_slices(g.H, g.B, g.GH, &kdummy);
  float* tmp = ws + 2 * TB * g.GH + TB * g.D * g.H + TB * inmax;
  float* dh_rec = tmp + TB * inmax + 3 * g.BH;
  float* second = dh_rec + sb * g.BH;
  float *dGW[2], *dGR[2], *dh_dir[2], *dc[2];
  dGW[0] = ws; dGR[0] = ws + TB * g.GH; dh_dir[0] = tmp + TB * inmax; dc[0] = dh_dir[0] + 2 * g.BH;
  dGW[1] = second; dGR[1] = second + TB * g.GH; dh_dir[1] = second + 2 * TB * g.GH; dc[1] = dh_dir[1] + 2 * g.BH;
  if (seq) {
    SeqInit ip{};
    SeqBwd p{};
    const SeqPlace place = seq_place(g, true, l == g.L - 1);
    p.B = g.B; p.H = g.H; p.T = g.T; p.ldo = g.D * g.H;
    p.groups = (g.B + SEQ_COLS - 1) / SEQ_COLS;
    p.wait = options().rnn_wait; p.pause = seq_pause_bwd(g); p.status = seq_status(g, ws); p.layer = (uint32_t)l + 1;
    ip.n = (size_t)g.T * seq_row(g, g.GH);
    ip.status = l == g.L - 1 ? p.status : nullptr;
    for (int dir = 0; dir < g.D; ++dir) {
      const int pl = l * g.D + dir;
      const float* base = res + (size_t)pl * r.per_pl;
      SeqBwd::Dir& q = p.d[dir];
      q.gout = gout ? gout + (size_t)dir * g.H : nullptr;
      q.dhy = dhy ? dhy + (size_t)pl * g.BH : nullptr;
      q.dcy = dcy ? dcy + (size_t)pl * g.BH : nullptr;
      q.R = w + offsets(g, pl).R;
      q.HP = base + r.hp; q.CP = base + r.cp; q.GT = base + r.gt; q.RN = base + r.rn;
      q.dGW = dGW[dir]; q.dGR = place.shared && dir == 0 ? dGW[0] : dGR[dir];
      q.dhx = dhx ? dhx + (size_t)pl * g.BH : nullptr;
      q.dcx = dcx ? dcx + (size_t)pl * g.BH : nullptr;
      q.X = ws + place.at[dir];
      ip.d[dir].X = q.X;
    }
    launch_init(ip, g.D, s);
    const int rc = seq_bwd<MODE>(g, p, s);
    if (rc != FLHIP_OK && rc != FLHIP_DECLINED) return rc;
    seq = rc == FLHIP_OK;
    if (!seq && !fused_applies(g)) return FLHIP_DECLINED;
    if (seq && place.shared) dGR[0] = dGW[0];
  }
  if (!seq) {
  if (MODE == RNN_LSTM)
    for (int dir = 0; dir < g.D; ++dir)
      hipLaunchKernelGGL(rnn_init_kernel, dim3(nblocks(g.BH)), dim3(256), 0, s,
                         dcy ? dcy + (size_t)(l * g.D + dir) * g.BH : nullptr, dc[dir], g.BH);
  auto step = [&](const StepBwd& p) {
    if (g.B <= 16) launch_step_bwd<MODE, 1>(p, g.D, s);
    else if (g.B <= 32) launch_step_bwd<MODE, 2>(p, g.D, s);
    else launch_step_bwd<MODE, 4>(p, g.D, s);
  };
  for (int st = g.T - 1; st >= 0; --st) {
    StepBwd p{};
    p.B = g.B;
    p.H = g.H;
    for (int dir = 0; dir < g.D; ++dir) {
      const int pl = l * g.D + dir, t = dir ? g.T - 1 - st : st;
      const Offsets o = offsets(g, pl);
      const float* base = res + (size_t)pl * r.per_pl;
      CellBwd& a = p.d[dir];
      a.ldo = g.D * g.H;
      a.gout = gout ? gout + (size_t)t * g.B * a.ldo + (size_t)dir * g.H : nullptr;
      const bool first = st == g.T - 1;
      a.dh_a = first ? (dhy ? dhy + (size_t)pl * g.BH : nullptr) : dh_dir[dir] + (size_t)((st + 1) & 1) * g.BH;
      a.R = w + o.R;
      a.dgr_next = first ? nullptr : dGR[dir] + (size_t)(st + 1) * g.B * g.GH;
      a.dc = dc[dir];
      a.gt = base + r.gt + (size_t)st * g.B * g.GH;
      a.cp = base + r.cp + (size_t)st * g.BH;
      a.cn = base + r.cp + (size_t)(st + 1) * g.BH;
      a.hp = base + r.hp + (size_t)st * g.BH;
      a.rn = base + r.rn + (size_t)st * g.BH;
      a.dgw = dGW[dir] + (size_t)t * g.B * g.GH;
      a.dgr = dGR[dir] + (size_t)st * g.B * g.GH;
      a.dh_dir = dh_dir[dir] + (size_t)(st & 1) * g.BH;
    }
    step(p);
  }
  if (dhx) {
    StepBwd p{};
    p.B = g.B;
    p.H = g.H;
    for (int dir = 0; dir < g.D; ++dir) {
      CellBwd& a = p.d[dir];
      a.dhx = dhx + (size_t)(l * g.D + dir) * g.BH;
      a.dh_a = dh_dir[dir];
      a.R = w + offsets(g, l * g.D + dir).R;
      a.dgr_next = dGR[dir];
    }
    step(p);
  }
  if (dcx && MODE == RNN_LSTM)
    for (int dir = 0; dir < g.D; ++dir)
      hipLaunchKernelGGL(rnn_init_kernel, dim3(nblocks(g.BH)), dim3(256), 0, s, dc[dir],
                         dcx + (size_t)(l * g.D + dir) * g.BH, g.BH);
  }
  const Scratch sc = scratch_of(g, ws);
  Offsets os[2];
  const float *hps[2], *gws[2], *grs[2];
  // gradients of the layer input: where they are small and neither is cut into slices, both directions' in a launch and one that adds them (of the pass
  // 0.69 to 1.01; above it is level, us as it is / in one launch: 2873 columns of 512 inputs 1595 / 1596, 4641 of 40 and 1280 1373 / 1381, 4876 of 512
  // 396 / 388, 2220 of 1024 226 / 219)
  int pair = -1;
  if (g.D == 2 && TB * inl <= 512 * 1024 && gemm32_ws_bytes(0, (int)inl, (int)TB, (int)g.GH) == 0) {
    pair = gemm32_pair(0, w + offsets(g, l * 2).W, w + offsets(g, l * 2 + 1).W, dGW[0], dGW[1], gin, tmp, (int)inl, (int)TB, (int)g.GH, nullptr, nullptr,
                       nullptr, 0, s);
    if (pair > 0) return pair;
    if (pair == 0) hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(TB * inl)), dim3(256), 0, s, gin, tmp, 1, gin, TB * inl);
  }
  for (int dir = 0; dir < g.D; ++dir) {
    const int pl = l * g.D + dir;
    const Offsets o = offsets(g, pl);
    os[dir] = o, hps[dir] = res + (size_t)pl * r.per_pl + r.hp, gws[dir] = dGW[dir], grs[dir] = dGR[dir];
    // gradient of the layer input, the second direction's added to the first's
    if (pair == 0) continue;
    int rc = dir == 0 ? -1 : gemm32(0, w + o.W, dGW[dir], gin, (int)inl, (int)TB, (int)g.GH, nullptr, sc.p, sc.bytes, s, gin);
    if (rc > 0) return rc;
    if (rc < 0) {
      float* gdst = dir == 0 ? gin : tmp;
      if ((rc = mm(w + o.W, dGW[dir], gdst, inl, TB, g.GH, 0, 0, nullptr, s, sc))) return rc;
      if (dir)
        hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(TB * inl)), dim3(256), 0, s, gin, tmp, 1, gin, TB * inl);
    }
  }
  if (const int rc = weight_gradients(g, g.D, os, in, inl, hps, gws, grs, dw, ws, s)) return rc;
  return check_launch("rnn_bwd");
}

}  // namespace
}  // namespace flhip

using namespace flhip;

extern "C" uint64_t flhip_rnn_sequence_launches(void) { return g_seq_launches.load(std::memory_order_relaxed); }

extern "C" size_t flhip_rnn_param_count(const flhip_rnn_desc* d) {
  RnnGeom g;
  return make_geom(d, &g) == FLHIP_OK ? g.nparams : 0;
}
extern "C" size_t flhip_rnn_reserve_bytes(const flhip_rnn_desc* d) {
  RnnGeom g;
  return make_geom(d, &g) == FLHIP_OK ? reserve_layout(g).total * sizeof(float) : 0;
}
extern "C" size_t flhip_rnn_workspace_bytes(const flhip_rnn_desc* d) {
  RnnGeom g;
  return make_geom(d, &g) == FLHIP_OK ? workspace_bytes(g) : 0;
}

extern "C" int flhip_rnn_fwd(const flhip_rnn_desc* d, const void* x, const void* hx, const void* cx,
                             const void* w, void* y, void* hy, void* cy, void* reserve,
                             size_t reserve_bytes, void* ws, size_t ws_bytes, void* stream) {
  RnnGeom g;
  const int rc0 = make_geom(d, &g);
  if (rc0 != FLHIP_OK) return rc0;
  FLHIP_REQUIRE(x && w && y && hy, "rnn_fwd: null argument");
  FLHIP_REQUIRE(reserve && reserve_bytes >= flhip_rnn_reserve_bytes(d), "rnn_fwd: reserve buffer too small");
  FLHIP_REQUIRE(ws && ws_bytes >= base_bytes(g), "rnn_fwd: workspace too small");
  hipStream_t s = as_stream(stream);
  const Reserve r = reserve_layout(g);
  float* res = static_cast<float*>(reserve);
  const float* wf = static_cast<const float*>(w);
  const size_t act = (size_t)g.T * g.B * g.D * g.H;
  if (stack_units(g)) {
    const bool captured = !seq_uncaptured(s);
    auto stack = [&](auto fn) {
      return fn(g, static_cast<const float*>(x), wf, static_cast<const float*>(hx), static_cast<const float*>(cx), static_cast<float*>(y),
                static_cast<float*>(hy), static_cast<float*>(cy), res, static_cast<float*>(ws), captured, s);
    };
    const int rc = g.mode == RNN_TANH ? stack(forward_stack<RNN_TANH>) : g.mode == RNN_LSTM ? stack(forward_stack<RNN_LSTM>) : stack(forward_stack<RNN_GRU>);
    if (rc != FLHIP_DECLINED) return rc;
  }
  bool seq = seq_applies(g, false, s) && ws_bytes >= seq_end(g, false) * sizeof(float);
  for (int l = 0; l < g.L; ++l) {
    const float* in = l == 0 ? static_cast<const float*>(x) : res + r.acts + (size_t)(l - 1) * act;
    float* out = l == g.L - 1 ? static_cast<float*>(y) : res + r.acts + (size_t)l * act;
    const size_t inl = l == 0 ? g.I : (size_t)g.D * g.H;
    int rc = FLHIP_DECLINED;
    if (seq || fused_applies(g)) {
      auto args = [&](auto fn) {
        return fn(g, l, in, inl, wf, static_cast<const float*>(hx), static_cast<const float*>(cx), out,
                  static_cast<float*>(hy), static_cast<float*>(cy), res, static_cast<float*>(ws), seq, s);
      };
      switch (g.mode) {
        case RNN_RELU: rc = args(forward_layer_fused<RNN_RELU>); break;
        case RNN_TANH: rc = args(forward_layer_fused<RNN_TANH>); break;
        case RNN_LSTM: rc = args(forward_layer_fused<RNN_LSTM>); break;
        default: rc = args(forward_layer_fused<RNN_GRU>);
      }
      if (rc != FLHIP_OK && rc != FLHIP_DECLINED) return rc;
    }
    if (rc == FLHIP_DECLINED) {
      for (int dir = 0; dir < g.D; ++dir) {
        const int pl = l * g.D + dir;
        auto args = [&](auto fn) {
          return fn(g, pl, in, inl, wf, static_cast<const float*>(hx), static_cast<const float*>(cx), out,
                    static_cast<float*>(hy), static_cast<float*>(cy), res, static_cast<float*>(ws), s);
        };
        switch (g.mode) {
          case RNN_RELU: rc = args(forward_pl<RNN_RELU>); break;
          case RNN_TANH: rc = args(forward_pl<RNN_TANH>); break;
          case RNN_LSTM: rc = args(forward_pl<RNN_LSTM>); break;
          default: rc = args(forward_pl<RNN_GRU>);
        }
        if (rc != FLHIP_OK) return rc;
      }
    }
    // what the next layer reads (and the backward pass reads again as that layer's input); the
    // layer's own recurrence and hy / cy used the states kept beside it in the reserve buffer
    if (g.dropout > 0.f && l + 1 < g.L)
      hipLaunchKernelGGL(rnn_dropout_kernel, dim3(nblocks(act)), dim3(256), 0, s, out, act, g.seed_lo, g.seed_hi,
                         (uint32_t)l, g.dropout, 1.0f / (1.0f - g.dropout));
  }
  return check_launch("rnn_fwd");
}

extern "C" int flhip_rnn_bwd(const flhip_rnn_desc* d, const void* x, const void* w, const void* dy,
                             const void* dhy, const void* dcy, const void* reserve,
                             size_t reserve_bytes, void* dx, void* dhx, void* dcx, void* dw, void* ws,
                             size_t ws_bytes, void* stream) {
  RnnGeom g;
  const int rc0 = make_geom(d, &g);
  if (rc0 != FLHIP_OK) return rc0;
  FLHIP_REQUIRE(x && w && dx && dw, "rnn_bwd: null argument");
  FLHIP_REQUIRE(reserve && reserve_bytes >= flhip_rnn_reserve_bytes(d),
                "rnn_bwd: needs the reserve buffer of the forward pass");
  FLHIP_REQUIRE(ws && ws_bytes >= base_bytes(g), "rnn_bwd: workspace too small");
  hipStream_t s = as_stream(stream);
  const Reserve r = reserve_layout(g);
  const float* res = static_cast<const float*>(reserve);
  const float* wf = static_cast<const float*>(w);
  float* wsf = static_cast<float*>(ws);
  const size_t TB = (size_t)g.T * g.B, act = TB * g.D * g.H, inmax = widest_input(g);
  float* goutbuf = wsf + 2 * TB * g.GH;
  float* ginbuf = goutbuf + act;
  const float* gout = static_cast<const float*>(dy);   // gradient of the top layer's output (may be null)
  bool seq = seq_applies(g, true, s) && ws_bytes >= seq_end(g, true) * sizeof(float);
  for (int l = g.L - 1; l >= 0; --l) {
    const float* in = l == 0 ? static_cast<const float*>(x) : res + r.acts + (size_t)(l - 1) * act;
    const size_t inl = l == 0 ? g.I : (size_t)g.D * g.H;
    float* gin = l == 0 ? static_cast<float*>(dx) : ginbuf;
    int rc = FLHIP_DECLINED;
    if (seq || fused_applies(g)) {
      auto args = [&](auto fn) {
        return fn(g, l, in, inl, wf, gout, static_cast<const float*>(dhy), static_cast<const float*>(dcy), gin,
                  static_cast<float*>(dhx), static_cast<float*>(dcx), static_cast<float*>(dw), res, wsf, seq, s);
      };
      switch (g.mode) {
        case RNN_RELU: rc = args(backward_layer_fused<RNN_RELU>); break;
        case RNN_TANH: rc = args(backward_layer_fused<RNN_TANH>); break;
        case RNN_LSTM: rc = args(backward_layer_fused<RNN_LSTM>); break;
        default: rc = args(backward_layer_fused<RNN_GRU>);
      }
      if (rc != FLHIP_OK && rc != FLHIP_DECLINED) return rc;
    }
    if (rc == FLHIP_DECLINED) {
      for (int dir = 0; dir < g.D; ++dir) {
        const int pl = l * g.D + dir;
        auto args = [&](auto fn) {
          return fn(g, pl, in, inl, wf, gout, static_cast<const float*>(dhy), static_cast<const float*>(dcy),
                    gin, dir == 0, static_cast<float*>(dhx), static_cast<float*>(dcx), static_cast<float*>(dw),
                    res, wsf, s);
        };
        switch (g.mode) {
          case RNN_RELU: rc = args(backward_pl<RNN_RELU>); break;
          case RNN_TANH: rc = args(backward_pl<RNN_TANH>); break;
          case RNN_LSTM: rc = args(backward_pl<RNN_LSTM>); break;
          default: rc = args(backward_pl<RNN_GRU>);
        }
        if (rc != FLHIP_OK) return rc;
      }
    }
    if (l > 0) {
      // the gradient of this layer's input is the gradient of the output of the layer below
      hipLaunchKernelGGL(rnn_add2_kernel, dim3(nblocks(TB * inl)), dim3(256), 0, s, ginbuf, (const float*)nullptr, 0,
                         goutbuf, TB * inl);
      gout = goutbuf;
      if (g.dropout > 0.f)
        hipLaunchKernelGGL(rnn_dropout_kernel, dim3(nblocks(act)), dim3(256), 0, s, goutbuf, act, g.seed_lo, g.seed_hi,
                           (uint32_t)(l - 1), g.dropout, 1.0f / (1.0f - g.dropout));
    }
  }
  (void)inmax;
  return FLHIP_OK;
}
