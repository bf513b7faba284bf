// Pieces that the deformable grad-input kernels of dk_deform_fast.hip (a lane owns an output pixel) and of
// dk_deform_lanes.hip (a lane owns a pair of channels) share: the bound on |out_grad| their fixed-point sums are
// scaled by, and the rounding onto the sums' grid.
#pragma once

#include "dk_common.h"

namespace dk {

constexpr int kAbsParts = 512;  // workgroups of absmax_kernel = words the consumers reduce

// The maximum of absmax_kernel's words, for every thread of the workgroup (two barriers).
__device__ __forceinline__ float block_absmax(const unsigned* __restrict__ parts) {
  __shared__ unsigned s_max;
  if (threadIdx.x == 0) s_max = 0u;
  __syncthreads();
  unsigned m = 0u;
  for (int i = threadIdx.x; i < kAbsParts; i += blockDim.x) m = max(m, parts[i]);
  for (int s = 32; s > 0; s >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, s));
  if ((threadIdx.x & 63) == 0) atomicMax(&s_max, m);
  __syncthreads();
  return __uint_as_float(s_max);
}

// The fixed-point sums need a finite bound gmax * wmax[c] on a term.  With an infinity or a NaN in
// out_grad (gmax is then that value: the maximum is taken on bit patterns) or in a channel's filter
// there is none, and the conversions to integers would turn such terms into zeros or wrapped numbers:
// the workgroup then writes NaN to the planes it owns instead (all of grad_input for a non-finite
// out_grad).  The reference's float atomics carry a non-finite term to the elements it touches;
// what a caller tests -- any non-finite value in the gradient, as loss scaling does -- gives the
// same answer.  Uniform over the workgroup; must be called by all its threads after wmax is visible.
template <typename T>
__device__ __forceinline__ bool write_nan_if_unbounded(float gmax, const float* wmax, int nch, T* planes0, size_t step,
                                                       int plane) {
  bool bounded = true;
  for (int j = 0; j < nch; ++j) bounded = bounded && (fabsf(gmax * wmax[j]) < __builtin_inff());  // false for NaN
  if (bounded) return false;
  for (int j = 0; j < nch; ++j)
    for (int e = threadIdx.x; e < plane; e += blockDim.x) dk::st(planes0 + (size_t)j * step + e, __builtin_nanf(""));
  return true;
}

// A result element that is not read again by the operator: non-temporal for 4-byte elements (a wave writes whole
// lines), the plain store for 2-byte ones (as partial lines they reach memory one by one).
__device__ __forceinline__ void st_stream(float* p, float v) { __builtin_nontemporal_store(v, p); }
template <typename T>
__device__ __forceinline__ void st_stream(T* p, float v) { dk::st(p, v); }

// Two channels share a 64-bit sum while at most 2^kPairHead samples touch one input element: a term is then
// rounded on a grid of 2^-(31 - kPairHead) = 2^-24 of the largest possible term or finer.  (3 x 3 taps at stride 1
// put 36 samples on an element on average and about 65 on the fullest element of a large plane.)
constexpr int kPairHead = 7;

// Grad input with the lanes along the channels, in bands of rows (dk_deform_lanes.hip): 64 consecutive output pixels are walked
// once for every band that their samples read, with wide offsets nearly all of them.  Whether that form takes a call is
// therefore read off the offsets, on the device: it does while its units meet at most `most` bands in all; the form with a
// pixel per lane is launched behind it and takes the others.  (Not per image: with a few images each the two would run one after
// the other on a chip that is half empty, N=24 C=64 64 x 64 116 -> 216 us.)
struct BandWalk {
  int2* unit_rows;  // [image][ceil(output pixels / 64)]: least and largest image row that a unit's samples read
  unsigned* met;    // bands that all units meet, written by deform_tile_rows_kernel; null: the bands, if there are any, take the call
  unsigned most;
  int rows;         // image rows of a band; 0: no bands
};
__device__ __forceinline__ bool bands_take(const BandWalk& walk) { return *walk.met <= walk.most; }

// All gradients but the input's from one pass over the samples (dk_deform_tile.hip): a tile of 64 output pixels is walked once
// for every window of the input that its samples read, with wide offsets four times and more.  As above the offsets
// decide, on the device: deform_tile_boxes_kernel leaves the windows of all tiles in `words` words, and beyond `most` in all the
// kernels of the separate gradients, launched behind, take the call.  (Those read one word, 1 where the call is theirs.)
struct TileChoice {
  const unsigned* windows;  // null: no choice
  int words;
  unsigned most;
};
__device__ __forceinline__ bool tiles_take(const TileChoice& c) {
  unsigned sum = 0u;
  for (int i = threadIdx.x & 63; i < c.words; i += 64) sum += c.windows[i];
  for (int s = 32; s > 0; s >>= 1) sum += (unsigned)__shfl_xor((int)sum, s);
  return (unsigned)__builtin_amdgcn_readfirstlane((int)sum) <= c.most;
}

// A reduction left to the caller: `parts` partial sums of `count` elements each, to be added up in order into `out`
template <typename T>
struct ReduceJob {
  const float* partial;
  int parts;
  long count;
  T* out;
};

// floor(v + 0.5) as a signed 32-bit integer, one instruction
__device__ __forceinline__ int round_half_up(float v) {
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

}  // namespace dk
