// What the two kernels for fp32 matrix products share.
#pragma once
#include <stddef.h>
#include <hip/hip_runtime.h>

namespace flhip {

constexpr int G32_KC = 16;          // contraction indexes per stage

struct Gemm32 {
  int M, N, K;
  int mtiles, ntiles;
  int nstages, sps;            // stages of the contraction, stages per slice
  unsigned a_bytes, b_bytes;
  size_t slice;                // elements between the partial results of consecutive slices
  // 1x1 windows, whose positions are rows of A and C (modes 0 and 2) or the contraction (mode 1): positions of an image, of the source's
  // image, of a result row, and the source's step per result row and column
  int P, SP, OW, rowstep, colstep, slices;
  // the second of two products of one shape in a launch (gemm32_pair): blockIdx.z = 1
  const float *A2, *B2, *bias2;
  float* C2;
};

// consecutive workgroups go to the eight dies in turn: each die takes one run of tiles, and within a run the tiles of
// a column block follow each other, so that a die's cache holds what its workgroups share
__device__ __forceinline__ int gemm32_tile_of(int wg, int tiles) {
  const int per = tiles >> 3, rem = tiles & 7, die = wg & 7;
  return die * per + (die < rem ? die : rem) + (wg >> 3);
}

// gemm_f32_split.hip: mode and tile tm x tn (128 x 128, 128 x 64 or 64 x 128); -1 where the tile has no kernel
int gemm32_split(int mode, int tm, int tn, int slices, const Gemm32& p, const float* A, const float* B, const float* bias,
                 const float* addend, float* C, hipStream_t s);
// the same with A, C (mode 1: A, B) in planes of one image after the other
int gemm32_split_planes(int mode, int tm, int tn, int slices, const Gemm32& p, const float* A, const float* B, const float* bias,
                        const float* addend, float* C, hipStream_t s);

}  // namespace flhip
