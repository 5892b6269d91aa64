// Operations along contiguous rows: log-softmax and its gradient, the gradient of the categorical cross-entropy, and layer
// norm over the leading dimensions with its scale and shift, forward and backward.
//
// All are bound by memory: what each cannot do without is every tensor once.  A row is therefore read once into registers
// (raw 16-byte pieces, whatever the element type) and everything follows from there: one wave to a row of at most 64 NP
// pieces (four rows to a workgroup), one workgroup of 256 to a longer one; NP pieces per thread, 1 .. 8.  Rows need not start
// on 16-byte boundaries (9998 classes in bf16: every other row is 4 bytes off): the elements before the first and
// behind the last whole piece of a row are handled one per thread.
#include <algorithm>

#include "common.h"

namespace flhip {
namespace {

template <typename T> struct Piece { static constexpr int N = 16 / (int)sizeof(T); };

// element e of a raw piece, and a raw piece of elements
template <typename T>
__device__ __forceinline__ void unpack(const uintx4_t& r, float (&v)[Piece<T>::N]) {
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(r[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (std::is_same<T, f16_t>::value) {
        v[2 * i] = f16lo(r[i]); v[2 * i + 1] = f16hi(r[i]);
      } else {
        v[2 * i] = __uint_as_float(r[i] << 16); v[2 * i + 1] = __uint_as_float(r[i] & 0xffff0000u);
      }
    }
  }
}
template <typename T>
__device__ __forceinline__ uintx4_t packed(const float (&v)[Piece<T>::N]) {
  uintx4_t r;
  if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __float_as_uint(v[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      r[i] = std::is_same<T, f16_t>::value ? pack_f16(v[2 * i], v[2 * i + 1]) : pack_bf16(v[2 * i], v[2 * i + 1]);
  }
  return r;
}

// The split of a row of n elements: `head` single ones, `body` whole pieces, single ones again.  The single elements
// (fewer than two pieces together) belong to the threads 0 .. in order.
template <typename T>
struct RowSplit {
  int head, body, singles;
  __device__ __forceinline__ RowSplit(const T* row, int n) {
    constexpr int N = Piece<T>::N;
    head = (int)((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / (int)sizeof(T);
    if (head > n) head = n;
    body = (n - head) / N;
    singles = n - body * N;
  }
  // element index of single i
  __device__ __forceinline__ int at(int i) const { return i < head ? i : i + body * Piece<T>::N; }
};

template <int THREADS>
__device__ __forceinline__ float row_sum(float v, float* smem) {
  if constexpr (THREADS == 64) return wave_sum(v);
  else return block_sum<THREADS / 64>(v, smem);
}
template <int THREADS>
__device__ __forceinline__ float row_max(float v, float* smem) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o, 64));
  if constexpr (THREADS > 64) {
    __syncthreads();
    if ((threadIdx.x & 63) == 0) smem[threadIdx.x >> 6] = v;
    __syncthreads();
    v = smem[0];
#pragma unroll
    for (int i = 1; i < THREADS / 64; ++i) v = fmaxf(v, smem[i]);
  }
  return v;
}

// ---- log-softmax over rows (Functions.cpp:1044-1070) --------------------------------------------------------------------
// 4000 rows of 9998 in bf16 (160 MB): 137 -> 29 us (before: one wave to a row, element by element, three times over).
template <typename T, int THREADS, int NP>
__global__ void __launch_bounds__(THREADS == 64 ? 256 : THREADS) logsoftmax_rows_fwd(const T* __restrict__ x, T* __restrict__ y, int n, int rows) {
  constexpr int N = Piece<T>::N;
  __shared__ float smem[8];
  const int row = THREADS == 64 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  const int t = THREADS == 64 ? threadIdx.x & 63 : threadIdx.x;
  if (THREADS == 64 && row >= rows) return;
  const T* xr = x + (size_t)row * n;
  T* yr = y + (size_t)row * n;
  const RowSplit<T> sp(xr, n);
  const uintx4_t* xb = reinterpret_cast<const uintx4_t*>(xr + sp.head);
  uintx4_t r[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) r[i] = xb[t + i * THREADS];
  const bool has1 = t < sp.singles;
  const float one = has1 ? ld(xr, sp.at(t)) : -INFINITY;
  float mx = one;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      float v[N];
      unpack<T>(r[i], v);
#pragma unroll
      for (int e = 0; e < N; ++e) mx = fmaxf(mx, v[e]);
    }
  mx = row_max<THREADS>(mx, smem);
  float s = has1 ? expf(one - mx) : 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      float v[N];
      unpack<T>(r[i], v);
#pragma unroll
      for (int e = 0; e < N; ++e) s += expf(v[e] - mx);
    }
  s = row_sum<THREADS>(s, smem);
  const float lse = logf(s) + mx;
  uintx4_t* yb = reinterpret_cast<uintx4_t*>(yr + sp.head);
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      float v[N];
      unpack<T>(r[i], v);
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] -= lse;
      yb[t + i * THREADS] = packed<T>(v);
    }
  if (has1) st(yr, sp.at(t), one - lse);
}

// dx = dy - exp(y) * sum of dy: 4000 rows of 9998 in bf16 (240 MB): 113 -> 44 us.  Rows of more than 16 KB have 512 threads: 8 pieces
// of both operands in each of 256 do not fit the registers (8032 rows of 4917 in fp32 219 us, one wave to a row 130; 8760 of 5127
// 258 -> 99 with 512 threads)
template <typename T, int THREADS, int NP>
__global__ void __launch_bounds__(THREADS == 64 ? 256 : THREADS)
logsoftmax_rows_bwd(const T* __restrict__ dy, const T* __restrict__ y, T* __restrict__ dx, int n, int rows) {
  constexpr int N = Piece<T>::N;
  __shared__ float smem[8];
  const int row = THREADS == 64 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  const int t = THREADS == 64 ? threadIdx.x & 63 : threadIdx.x;
  if (THREADS == 64 && row >= rows) return;
  const size_t o = (size_t)row * n;
  const RowSplit<T> sp(dy + o, n);
  const uintx4_t* gb = reinterpret_cast<const uintx4_t*>(dy + o + sp.head);
  const uintx4_t* yb = reinterpret_cast<const uintx4_t*>(y + o + sp.head);
  uintx4_t g[NP], p[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      g[i] = gb[t + i * THREADS];
      p[i] = yb[t + i * THREADS];
    }
  const bool has1 = t < sp.singles;
  const float g1 = has1 ? ld(dy + o, sp.at(t)) : 0.f, y1 = has1 ? ld(y + o, sp.at(t)) : 0.f;
  float s = g1;
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      float v[N];
      unpack<T>(g[i], v);
#pragma unroll
      for (int e = 0; e < N; ++e) s += v[e];
    }
  s = row_sum<THREADS>(s, smem);
  uintx4_t* xb = reinterpret_cast<uintx4_t*>(dx + o + sp.head);
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (t + i * THREADS < sp.body) {
      float v[N], q[N];
      unpack<T>(g[i], v);
      unpack<T>(p[i], q);
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] -= expf(q[e]) * s;
      xb[t + i * THREADS] = packed<T>(v);
    }
  if (has1) st(dx + o, sp.at(t), g1 - expf(y1) * s);
}

// ---- gradient of the categorical cross-entropy (Functions.cpp:1128-1150) ----------------------------------------------
// dx[c, col] = -(g_col) where c == target[col] and the column counts, else 0; g_col = grad[0] / count (mean), grad[0] (sum)
// or grad[col] (none).  A store stream of one row per workgroup: 4000 x 9998 in bf16 (80 MB): 35 -> 13 us.
template <typename T>
__global__ void __launch_bounds__(256)
cce_rows_bwd(const float* __restrict__ grad, const int32_t* __restrict__ target, const float* __restrict__ stats,
             T* __restrict__ dx, int n, int rows, int reduction, int ignore) {
  constexpr int N = Piece<T>::N;
  for (int row = blockIdx.x; row < rows; row += gridDim.x) {
    const int tg = target[row];
    const float g = tg == ignore ? 0.f : -(reduction == 0 ? grad[row] : reduction == 1 ? grad[0] / stats[1] : grad[0]);
    T* xr = dx + (size_t)row * n;
    const RowSplit<T> sp(xr, n);
    uintx4_t* xb = reinterpret_cast<uintx4_t*>(xr + sp.head);
    for (int i = threadIdx.x; i < sp.body; i += 256) {
      float v[N];
      const int c0 = sp.head + i * N;
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] = c0 + e == tg ? g : 0.f;
      xb[i] = packed<T>(v);
    }
    if ((int)threadIdx.x < sp.singles) {
      const int c = sp.at(threadIdx.x);
      st(xr, c, c == tg ? g : 0.f);
    }
  }
}

// ---- layer norm over rows, with scale and shift (nn/modules/LayerNorm.cpp:42-131) --------------------------------------
// y = w * (x - mean) / sqrt(var + eps) + b, statistics per row; w, b per element of the row (or one each), fp32, rounded to
// the storage type first as the composed form has it.  Composed of a batch norm and a broadcast the forward pass moved
// every element five times and the backward pass eight, the sums for dw and db with a stride of a row between lanes:
// 4000 rows of 2000 in bf16: forward 21 + 20 -> 11 us, backward 155 + 5 + 25 -> 20 + 6 us.
template <typename T>
__device__ __forceinline__ float as_stored(float v) {
  T t[1];
  st(t, 0, v);
  return ld(t, 0);
}

// A thread has the same N elements at col + i * THREADS * N in every row, and keeps their scales and shifts in registers from
// row to row (fetched again for every row they are most of the loads: 35 us for those 4000 rows of 2000).  N is a piece of 16
// bytes where the rows are of whole pieces on 16-byte boundaries, or else one: neighbouring threads then read neighbouring
// elements wherever a row, of x or of y, starts (10000 rows of 2001 in bf16: 78 -> 27 us against pieces with single elements around
// them and parameters per row; composed 57).
template <typename T, int N>
struct Elements {                  // N elements of T as they are held
  typename std::conditional<N == 1, float, uintx4_t>::type raw;
  __device__ __forceinline__ void load(const T* p) {
    if constexpr (N == 1) raw = ld(p, 0);
    else raw = *reinterpret_cast<const uintx4_t*>(p);
  }
  __device__ __forceinline__ void get(float (&v)[N]) const {
    if constexpr (N == 1) v[0] = raw;
    else unpack<T>(raw, v);
  }
  static __device__ __forceinline__ void store(T* p, const float (&v)[N]) {
    if constexpr (N == 1) st(p, 0, v[0]);
    else *reinterpret_cast<uintx4_t*>(p) = packed<T>(v);
  }
};
// their fp32 parameters
template <typename T, int N>
__device__ __forceinline__ void load_params(const float* p, int c, int n, int pstride, float (&v)[N]) {
  if constexpr (N == 1) {
    v[0] = c < n ? as_stored<T>(p[pstride * c]) : 0.f;
  } else {
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      float4 f = make_float4(0.f, 0.f, 0.f, 0.f);
      if (c < n) f = pstride ? *reinterpret_cast<const float4*>(p + c + e) : make_float4(p[0], p[0], p[0], p[0]);
      v[e] = as_stored<T>(f.x); v[e + 1] = as_stored<T>(f.y); v[e + 2] = as_stored<T>(f.z); v[e + 3] = as_stored<T>(f.w);
    }
  }
}

template <typename T, int THREADS, int NP, int N>
__global__ void __launch_bounds__(THREADS == 64 ? 256 : THREADS)
layernorm_rows_fwd(const T* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, T* __restrict__ y,
                   float* __restrict__ mean, float* __restrict__ invstd, int n, int rows, int pstride, float eps) {
  constexpr int RPB = THREADS == 64 ? 4 : 1;
  __shared__ float smem[16];
  const int t = THREADS == 64 ? threadIdx.x & 63 : threadIdx.x;
  auto col = [&](int i) { return (t + i * THREADS) * N; };
  float wv[NP][N], bv[NP][N];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    load_params<T>(w, col(i), n, pstride, wv[i]);
    load_params<T>(b, col(i), n, pstride, bv[i]);
  }
  for (int row = blockIdx.x * RPB + (THREADS == 64 ? threadIdx.x >> 6 : 0); row < rows; row += gridDim.x * RPB) {
    const T* xr = x + (size_t)row * n;
    T* yr = y + (size_t)row * n;
    Elements<T, N> r[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n) r[i].load(xr + col(i));
    float s = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n) {
        float v[N];
        r[i].get(v);
#pragma unroll
        for (int e = 0; e < N; ++e) s += v[e];
      }
    const float m = row_sum<THREADS>(s, smem) / (float)n;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n) {
        float v[N];
        r[i].get(v);
#pragma unroll
        for (int e = 0; e < N; ++e) q += (v[e] - m) * (v[e] - m);
      }
    const float is = 1.f / sqrtf(row_sum<THREADS>(q, smem) / (float)n + eps);
    if (t == 0) {
      mean[row] = m;
      invstd[row] = is;
    }
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n) {
        float v[N];
        r[i].get(v);
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = wv[i][e] * ((v[e] - m) * is) + bv[i][e];
        Elements<T, N>::store(yr + col(i), v);
      }
  }
}

// Rows that are not of whole pieces, with one scale and shift: pieces on 16-byte boundaries and single elements around them, as
// the log-softmax takes them, since there are no parameters per element to fetch (8558 rows of 2113 in f16: 44 us element by
// element, 21 so; x and y have to start alike).
template <typename T, int THREADS, int NP>
__global__ void __launch_bounds__(256)
layernorm_ragged_fwd(const T* __restrict__ x, const float* __restrict__ w, const float* __restrict__ b, T* __restrict__ y,
                     float* __restrict__ mean, float* __restrict__ invstd, int n, int rows, float eps) {
  constexpr int N = Piece<T>::N, RPB = 256 / THREADS;
  __shared__ float smem[4];
  const int t = THREADS == 64 ? threadIdx.x & 63 : threadIdx.x;
  const float we = as_stored<T>(w[0]), be = as_stored<T>(b[0]);
  for (int row = blockIdx.x * RPB + (THREADS == 64 ? threadIdx.x >> 6 : 0); row < rows; row += gridDim.x * RPB) {
    const T* xr = x + (size_t)row * n;
    T* yr = y + (size_t)row * n;
    const RowSplit<T> sp(xr, n);
    const uintx4_t* xb = reinterpret_cast<const uintx4_t*>(xr + sp.head);
    uintx4_t r[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (t + i * THREADS < sp.body) r[i] = xb[t + i * THREADS];
    const bool has1 = t < sp.singles;
    const float one = has1 ? ld(xr, sp.at(t)) : 0.f;
    float s = one;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (t + i * THREADS < sp.body) {
        float v[N];
        unpack<T>(r[i], v);
#pragma unroll
        for (int e = 0; e < N; ++e) s += v[e];
      }
    const float m = row_sum<THREADS>(s, smem) / (float)n;
    float q = has1 ? (one - m) * (one - m) : 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (t + i * THREADS < sp.body) {
        float v[N];
        unpack<T>(r[i], v);
#pragma unroll
        for (int e = 0; e < N; ++e) q += (v[e] - m) * (v[e] - m);
      }
    const float is = 1.f / sqrtf(row_sum<THREADS>(q, smem) / (float)n + eps);
    if (t == 0) {
      mean[row] = m;
      invstd[row] = is;
    }
    uintx4_t* yb = reinterpret_cast<uintx4_t*>(yr + sp.head);
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (t + i * THREADS < sp.body) {
        float v[N];
        unpack<T>(r[i], v);
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = we * ((v[e] - m) * is) + be;
        yb[t + i * THREADS] = packed<T>(v);
      }
    if (has1) st(yr, sp.at(t), we * ((one - m) * is) + be);
  }
}

// dx = invstd * (g - mean(g) - xhat * mean(g * xhat)), g = w * dy, and over slice blockIdx.x of the rows the sums of
// dy * xhat and dy per element of the row: part[slice][2][n].  A thread has the same elements in every row, as above, and
// keeps their sums from row to row.  A row of one wave takes no barrier, and the four waves of a workgroup each have a row in
// flight.  (100000 rows in bf16, before, a workgroup to every row and runs of 8 elements per thread: 29 elements 359 -> 31 us, 100
// elements 429 -> 53, 256 elements 190 -> 51, 257 elements 433 -> 104; composed 168, 482, 1194 and 790.)
template <typename T, int THREADS, int NP, int N>
__global__ void __launch_bounds__(256)
layernorm_rows_bwd(const T* __restrict__ dy, const T* __restrict__ x, const float* __restrict__ w,
                   const float* __restrict__ mean, const float* __restrict__ invstd, T* __restrict__ dx,
                   float* __restrict__ part, int n, int rows, int rps, int pstride) {
  constexpr int RPB = 256 / THREADS;
  __shared__ float smem[8];
  const int wave = threadIdx.x >> 6, t = THREADS == 64 ? threadIdx.x & 63 : threadIdx.x;
  const int r0 = blockIdx.x * rps, r1 = min(rows, r0 + rps);
  auto col = [&](int i) { return (t + i * THREADS) * N; };
  float sw[NP][N], sb[NP][N], wv[NP][N];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    load_params<T>(w, col(i), n, pstride, wv[i]);
#pragma unroll
    for (int e = 0; e < N; ++e) sw[i][e] = sb[i][e] = 0.f;
  }
  for (int row = r0 + (THREADS == 64 ? wave : 0); row < r1; row += RPB) {
    const size_t o = (size_t)row * n;
    Elements<T, N> rg[NP] = {}, rx[NP] = {};
    float g[NP][N], xh[NP][N];
    const float m = mean[row], is = invstd[row];
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n) {
        rg[i].load(dy + o + col(i));
        rx[i].load(x + o + col(i));
      }
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < NP; ++i) {             // (elements that do not exist are zeros)
      rg[i].get(g[i]);
      rx[i].get(xh[i]);
#pragma unroll
      for (int e = 0; e < N; ++e) {
        if (col(i) < n) xh[i][e] = (xh[i][e] - m) * is;
        sw[i][e] += g[i][e] * xh[i][e];
        sb[i][e] += g[i][e];
        g[i][e] *= wv[i][e];
        s1 += g[i][e];
        s2 += g[i][e] * xh[i][e];
      }
    }
    if constexpr (THREADS == 64) {
      s1 = wave_sum(s1);
      s2 = wave_sum(s2);
    } else {
      block_sum2<4>(s1, s2, smem);
    }
    s1 /= (float)n;
    s2 /= (float)n;
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      float v[N];
#pragma unroll
      for (int e = 0; e < N; ++e) v[e] = is * (g[i][e] - s1 - xh[i][e] * s2);
      if (col(i) < n) Elements<T, N>::store(dx + o + col(i), v);
    }
  }
  float* out = part + (size_t)blockIdx.x * 2 * n;
  if constexpr (THREADS == 64) {               // the four waves' sums meet in LDS, added in wave order
    __shared__ float comb[4][64 * NP * N];
#pragma unroll
    for (int which = 0; which < 2; ++which) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < NP; ++i)
#pragma unroll
        for (int e = 0; e < N; ++e) comb[wave][col(i) + e] = which ? sb[i][e] : sw[i][e];
      __syncthreads();
      for (int c = threadIdx.x; c < n; c += 256) out[which * n + c] = comb[0][c] + comb[1][c] + comb[2][c] + comb[3][c];
    }
  } else {
#pragma unroll
    for (int i = 0; i < NP; ++i)
      if (col(i) < n)
#pragma unroll
        for (int e = 0; e < N; ++e) {
          out[col(i) + e] = sw[i][e];
          out[n + col(i) + e] = sb[i][e];
        }
  }
}

// dw[c], db[c] = sums over the slices of part[slice][2][n]: a workgroup adds 64 columns, its 16 waves every 16th slice
__global__ void __launch_bounds__(1024)
layernorm_fold(const float* __restrict__ part, float* __restrict__ dw, float* __restrict__ db, int n, int slices) {
  __shared__ float red[16][65];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = blockIdx.x * 64 + lane;      // of 2 n
  float s = 0.f;
  if (c < 2 * n)
#pragma unroll 4
    for (int k = wave; k < slices; k += 16) s += part[(size_t)k * 2 * n + c];
  red[wave][lane] = s;
  __syncthreads();
  if (wave == 0 && c < 2 * n) {
#pragma unroll
    for (int k = 1; k < 16; ++k) s += red[k][lane];
    if (c < n) dw[c] = s;
    else db[c - n] = s;
  }
}
// one parameter element for the whole row: the sums over its columns (16 waves: with four, a row of 5000 columns takes 20 rounds
// of loads one after the other)
__global__ void __launch_bounds__(1024)
layernorm_fold_scalar(const float* __restrict__ cols, float* __restrict__ dw, float* __restrict__ db, int n) {
  __shared__ float smem[32];
  float a = 0.f, b = 0.f;
#pragma unroll 4
  for (int i = threadIdx.x; i < n; i += 1024) {
    a += cols[i];
    b += cols[n + i];
  }
  block_sum2<16>(a, b, smem);
  if (threadIdx.x == 0) {
    dw[0] = a;
    db[0] = b;
  }
}

// f(threads tag, pieces tag) for rows of n elements; false: too long for registers
template <typename T, typename F>
bool by_row(int n, F&& f) {
  const int pieces = (n + Piece<T>::N - 1) / Piece<T>::N;
  using std::integral_constant;
  integral_constant<int, 64> wave;
  integral_constant<int, 256> wg;
  integral_constant<int, 1> n1;
  integral_constant<int, 2> n2;
  integral_constant<int, 4> n4;
  if (pieces <= 64) f(wave, n1);
  else if (pieces <= 128) f(wave, n2);
  else if (pieces <= 256) f(wg, n1);
  else if (pieces <= 512) f(wg, n2);
  else if (pieces <= 1024) f(wg, n4);
  else if (pieces <= 2048) f(integral_constant<int, 512>{}, n4);
  else return false;
  return true;
}

// the same with the elements of a row (at most 8192) dealt out one by one
template <typename F>
void by_element(int n, F&& f) {
  using std::integral_constant;
  integral_constant<int, 64> wave;
  integral_constant<int, 256> wg;
  if (n <= 64) f(wave, integral_constant<int, 1>{});
  else if (n <= 128) f(wave, integral_constant<int, 2>{});
  else if (n <= 256) f(wave, integral_constant<int, 4>{});
  else if (n <= 512) f(wave, integral_constant<int, 8>{});
  else if (n <= 1024) f(wave, integral_constant<int, 16>{});
  else if (n <= 2048) f(wg, integral_constant<int, 8>{});
  else if (n <= 4096) f(wg, integral_constant<int, 16>{});
  else f(wg, integral_constant<int, 32>{});
}

bool same_offset(const void* a, const void* b, const void* c = nullptr) {
  const uintptr_t x = reinterpret_cast<uintptr_t>(a) & 15;
  return x == (reinterpret_cast<uintptr_t>(b) & 15) && (!c || x == (reinterpret_cast<uintptr_t>(c) & 15));
}

// slices of the rows for the backward pass: about two workgroups per compute unit.  A workgroup goes through its rows one after the
// other (four at a time, where a wave has a row of its own), so few long rows get one each: with four to a workgroup, 5 rows of 6590
// in f16 took 46 us, 12 of 6803 42 (composed 17 and 18); with one each, 4 rows of 6789 13 and 22 of 6897 14 (composed 20 and 21).
// More rows have more partial sums for the fold to read: 843 of 8104 in bf16 27 us with four to a workgroup, 35 with 512 workgroups
int ln_slices(int n, int rows) { return std::max(n > 1024 ? std::min(rows, 128) : 1, std::min(512, rows / 4)); }

}  // namespace

// Rows of less than 320 bytes leave most of a wave's lanes without a piece, and the single elements around the pieces cost
// more than they save: a lane per element is faster then (100000 rows, us by elements / by pieces: bf16 forward 29 elements 20.7 / 33.0,
// 128 31.5 / 32.5, 192 43.1 / 32.8, backward 16.4 / 31.8, 24.4 / 27.5, 33.4 / 27.8; fp32 forward 29 elements 22.0 / 25.3, 64 23.7 /
// 25.1, 100 33.3 / 25.5, backward 17.7 / 22.5, 19.8 / 19.5, 27.1 / 21.3).  Backward the line lies at 352 bytes, and at 400 where rows are
// not whole pieces (152202 rows of 182 in f16 48.9 / 55.2, 14592 6.5 / 8.5, 8518 of 178 in bf16 5.1 / 5.7; but 105143 of 176 33.9 / 30.1,
// 45584 of 219 in f16 21.8 / 20.3).
bool short_row(int n, int dtype, bool bwd) {
  const int bytes = n * (int)dtype_size(dtype);
  return bytes < (!bwd ? 320 : bytes % 16 ? 400 : 352);
}

// -> false where the row does not fit (the caller's element-wise kernels take it)
bool rows_logsoftmax_fwd(const void* x, void* y, int n, int rows, int dtype, hipStream_t s) {
  if (short_row(n, dtype, false) || !same_offset(x, y)) return false;
  return by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    return by_row<T>(n, [&](auto th, auto np) {
      const dim3 grid((unsigned)(th.value == 64 ? (rows + 3) / 4 : rows));
      hipLaunchKernelGGL((logsoftmax_rows_fwd<T, th.value, np.value>), grid, dim3(std::max(256, th.value)), 0, s, (const T*)x, (T*)y, n, rows);
    });
  });
}

bool rows_logsoftmax_bwd(const void* dy, const void* y, void* dx, int n, int rows, int dtype, hipStream_t s) {
  if (short_row(n, dtype, true) || !same_offset(dy, y, dx)) return false;
  return by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    return by_row<T>(n, [&](auto th, auto np) {
      const dim3 grid((unsigned)(th.value == 64 ? (rows + 3) / 4 : rows));
      hipLaunchKernelGGL((logsoftmax_rows_bwd<T, th.value, np.value>), grid, dim3(std::max(256, th.value)), 0, s, (const T*)dy, (const T*)y, (T*)dx,
                         n, rows);
    });
  });
}

// Rows of fewer than 384 elements leave most of a workgroup idle: an element per thread is faster (100000 rows in bf16, us by
// elements / here: 29 classes 10.0 / 31.5, 128 16.0 / 31.4, 256 27.3 / 33.0, 400 38.1 / 34.1; 1000000 rows of 21: 30 / 303)
bool rows_cce_bwd(const float* grad, const int32_t* target, const float* stats, void* dx, int n, int rows, int reduction,
                  int ignore, int dtype, hipStream_t s) {
  if (n < 384) return false;
  by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    hipLaunchKernelGGL((cce_rows_bwd<T>), dim3((unsigned)std::min(rows, 16384)), dim3(256), 0, s, grad, target, stats, (T*)dx, n,
                       rows, reduction, ignore);
  });
  return true;
}

}  // namespace flhip

using namespace flhip;

extern "C" int flhip_layernorm_applies(int64_t n, int64_t rows, int dtype) {
  if (n <= 0 || rows <= 0 || rows > 1 << 30 || !dtype_ok(dtype)) return 0;      // (a grid's stride past the last row stays an int)
  // a row of one element has nothing to sum: with many of them the general kernels are faster (forward / backward in f16, 123245
  // rows: 11 / 19 us there, 23 / 35 here; 59588: 10.5 / 15.7, 13.2 / 21.4; 33092: backward 14.3, 15.8)
  if (n == 1 && rows > (1 << 14)) return 0;
  return n <= 1024 * 16 / (int64_t)dtype_size(dtype);      // four pieces per thread (the backward pass's registers)
}

extern "C" int flhip_layernorm_fwd(const void* x, const float* w, const float* b, void* y, float* mean, float* invstd,
                                   int64_t n, int64_t rows, int scalar_params, double epsilon, int dtype, void* stream) {
  FLHIP_REQUIRE(x && w && b && y && mean && invstd, "layernorm: null argument");
  FLHIP_REQUIRE(dtype_ok(dtype), "layernorm: unknown dtype");
  FLHIP_REQUIRE(flhip_layernorm_applies(n, rows, dtype), "layernorm: row length not supported");
  by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    const bool whole = n % Piece<T>::N == 0 && ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(y) |
                                                 reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(b)) & 15) == 0;
    auto go = [&](auto th, auto np, auto ne) {
      // up to eight workgroups for each compute unit (with four, 10000 rows of 2001 in bf16 take 42 us instead of 27)
      const int64_t blocks = std::min<int64_t>(th.value == 64 ? (rows + 3) / 4 : rows, th.value == 1024 ? 512 : 2048);
      hipLaunchKernelGGL((layernorm_rows_fwd<T, th.value, np.value, ne.value>), dim3((unsigned)blocks), dim3(std::max(256, th.value)), 0,
                         as_stream(stream), (const T*)x, w, b, (T*)y, mean, invstd, (int)n, (int)rows, scalar_params ? 0 : 1,
                         (float)epsilon);
    };
    // 1024 threads to a row that 256 would hold with 32 elements, scales and shifts each: registers for three such rows on a compute
    // unit hide too little (3261 rows of 6147 in f16: 85 us, composed 63; with 1024 threads 3405 rows of 6463 54, composed 70)
    if (whole) by_row<T>((int)n, [&](auto th, auto np) {
      if constexpr (th.value <= 256) go(th, np, std::integral_constant<int, Piece<T>::N>{});      // (no longer ones apply)
    });
    else if (scalar_params && n >= 256 && same_offset(x, y)) by_row<T>((int)n, [&](auto th, auto np) {
      if constexpr (th.value <= 256)
        hipLaunchKernelGGL((layernorm_ragged_fwd<T, th.value, np.value>),
                           dim3((unsigned)std::min<int64_t>(th.value == 64 ? (rows + 3) / 4 : rows, 2048)), dim3(256), 0, as_stream(stream),
                           (const T*)x, w, b, (T*)y, mean, invstd, (int)n, (int)rows, (float)epsilon);
    });
    else if (n > 4096) go(std::integral_constant<int, 1024>{}, std::integral_constant<int, 8>{}, std::integral_constant<int, 1>{});
    else by_element((int)n, [&](auto th, auto np) { go(th, np, std::integral_constant<int, 1>{}); });
  });
  return check_launch("layernorm_fwd");
}

extern "C" size_t flhip_layernorm_bwd_workspace_bytes(int64_t n, int64_t rows, int dtype) {
  if (!flhip_layernorm_applies(n, rows, dtype)) return 0;
  return (size_t)(ln_slices((int)n, (int)rows) + 1) * 2 * (size_t)n * sizeof(float);
}

extern "C" int flhip_layernorm_bwd(const void* dy, const void* x, const float* w, const float* mean, const float* invstd,
                                   void* dx, float* dw, float* db, int64_t n, int64_t rows, int scalar_params, int dtype,
                                   void* ws, size_t ws_bytes, void* stream) {
  FLHIP_REQUIRE(dy && x && w && mean && invstd && dx && dw && db, "layernorm_bwd: null argument");
  FLHIP_REQUIRE(dtype_ok(dtype), "layernorm_bwd: unknown dtype");
  FLHIP_REQUIRE(flhip_layernorm_applies(n, rows, dtype), "layernorm_bwd: row length not supported");
  FLHIP_REQUIRE(ws && ws_bytes >= flhip_layernorm_bwd_workspace_bytes(n, rows, dtype), "layernorm_bwd: workspace too small");
  hipStream_t s = as_stream(stream);
  const int want = ln_slices((int)n, (int)rows), rps = (int)((rows + want - 1) / want), slices = (int)((rows + rps - 1) / rps);
  float* part = static_cast<float*>(ws);
  by_dtype(dtype, [&](auto* t_) {
    using T = FLHIP_T_OF(t_);
    const bool whole = n % Piece<T>::N == 0 && ((reinterpret_cast<uintptr_t>(dy) | reinterpret_cast<uintptr_t>(x) |
                                                 reinterpret_cast<uintptr_t>(dx) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
    auto go = [&](auto th, auto np, auto ne) {
      hipLaunchKernelGGL((layernorm_rows_bwd<T, th.value, np.value, ne.value>), dim3((unsigned)slices), dim3(256), 0, s, (const T*)dy,
                         (const T*)x, w, mean, invstd, (T*)dx, part, (int)n, (int)rows, rps, scalar_params ? 0 : 1);
    };
    if (whole) by_row<T>((int)n, [&](auto th, auto np) {
      if constexpr (th.value <= 256) go(th, np, std::integral_constant<int, Piece<T>::N>{});      // (no longer ones apply)
    });
    else by_element((int)n, [&](auto th, auto np) { go(th, np, std::integral_constant<int, 1>{}); });
  });
  if (const int rc = check_launch("layernorm_bwd")) return rc;
  float* cols = part + (size_t)slices * 2 * n;
  hipLaunchKernelGGL(layernorm_fold, dim3((unsigned)((2 * n + 63) / 64)), dim3(1024), 0, s, part, scalar_params ? cols : dw,
                     scalar_params ? cols + n : db, (int)n, slices);
  if (scalar_params) hipLaunchKernelGGL(layernorm_fold_scalar, dim3(1), dim3(1024), 0, s, cols, dw, db, (int)n);
  return check_launch("layernorm_bwd (sums)");
}
