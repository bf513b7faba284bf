// The 3 x 3 offset convolution of the layers (padding 1, dilation 1, stride 1 or 2, up to 18 outputs) on few images:
// forward, input gradient and weight gradient on the vector unit, one launch each and no packed weights.
//
// What bounds these calls is latency: one image of 192 channels on 28 x 28 is 25 M multiply-adds, a microsecond of the
// chip, but the matrix-instruction kernels (dk_offset_conv16.hip) take a launch to pack the weights, a tile of 448 pixels
// per workgroup and a launch to add their parts, and the framework's convolution transposes twice around its kernel and
// takes 40 us of host time per call.  A lane owns a pixel (of the flattened batch, so that 7 x 7 planes leave no lanes
// over) and multiplies its nine inputs with the weights of all outputs, read from LDS at one address per wave.
// Arithmetic: fp32 products and sums for every tensor type, no split operands.
#include <algorithm>

#include "dk_common.h"
#include "dk_kernels.h"

namespace dk {
namespace {

constexpr int kDcOut = 18;    // outputs of a layer with one rotation group
constexpr int kDcTaps = 9;

struct DirectConv {
  int batch, cin, cout, h, w, oh, ow, stride;
};

// The nine inputs of an output pixel as byte offsets from the plane's start (kOutOfRange: in the padding).
template <typename T>
__device__ __forceinline__ void tap_offsets(const DirectConv& g, int y, int x, unsigned image_off, unsigned (&off)[kDcTaps]) {
#pragma unroll
  for (int t = 0; t < kDcTaps; ++t) {
    const int iy = y * g.stride + t / 3 - 1, ix = x * g.stride + t % 3 - 1;
    off[t] = iy >= 0 && iy < g.h && ix >= 0 && ix < g.w ? (image_off + iy * g.w + ix) * (unsigned)sizeof(T) : kOutOfRange;
  }
}

// One channel's weights of OB outputs from `o0` on, [tap][output] in LDS (rows of OBP floats); a lane fetches PER of them.
template <typename T, int OB, int PER>
__device__ __forceinline__ void load_weights(const DirectConv& g, const T* __restrict__ weight, int o0, int c, int lane, float (&v)[PER]) {
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i, o = o0 + e / kDcTaps;
    v[i] = e < OB * kDcTaps && o < g.cout && c < g.cin ? ld(weight + ((long)o * g.cin + c) * kDcTaps + e % kDcTaps) : 0.f;
  }
}
template <int OB, int OBP, int PER>
__device__ __forceinline__ void store_weights(float* lds, int lane, const float (&v)[PER]) {
#pragma unroll
  for (int i = 0; i < PER; ++i) {
    const int e = lane + 64 * i;
    if (e < OB * kDcTaps) lds[(e % kDcTaps) * OBP + e / kDcTaps] = v[i];
  }
}

// Forward.  A workgroup owns 64 * PX output pixels and OB outputs; its WAVES waves take every WAVES-th channel each, and
// their sums are added in wave order.  What bounds it is the CU's LDS pipe, which delivers every weight to 64 lanes: with
// (OB, WAVES, PX) = (18, 8, 2) a read of four weights feeds eight products.  Few pixels: (6, 16, 1) and (2, 16, 1), the input
// read three and nine times, from L2, so that the work reaches more CUs.
template <typename T, int OB, int WAVES, int PX>
__global__ __launch_bounds__(64 * WAVES) void direct_conv_forward_kernel(DirectConv g, const T* __restrict__ x, const T* __restrict__ weight,
                                                                         const T* __restrict__ bias, T* __restrict__ out) {
  constexpr int OBP = OB <= 2 ? OB : (OB + 3) / 4 * 4, PER = (OB * kDcTaps + 63) / 64, PIX = 64 * PX;
  __shared__ __align__(16) float wl[WAVES][kDcTaps * OBP];
  __shared__ float part[WAVES][OB][PIX];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int plane = g.oh * g.ow, total = g.batch * plane, o0 = blockIdx.y * OB;
  const int in_plane = g.h * g.w;
  unsigned off[PX][kDcTaps];
#pragma unroll
  for (int j = 0; j < PX; ++j) {
    const int pix = min((int)blockIdx.x * PIX + j * 64 + lane, total - 1);
    const int n = pix / plane, p = pix - n * plane;
    tap_offsets<T>(g, p / g.ow, p % g.ow, (unsigned)n * g.cin * in_plane, off[j]);
  }
  const rsrc_t rs = plane_rsrc(x, g.batch * g.cin * in_plane);
  float acc[PX][OB];
#pragma unroll
  for (int j = 0; j < PX; ++j)
#pragma unroll
    for (int o = 0; o < OB; ++o) acc[j][o] = 0.f;
  float wv[PER], xv[PX][kDcTaps];
  auto fetch = [&](int c) {
    load_weights<T, OB, PER>(g, weight, o0, c, lane, wv);
    const int so = min(c, g.cin - 1) * in_plane * (int)sizeof(T);
#pragma unroll
    for (int j = 0; j < PX; ++j)
#pragma unroll
      for (int t = 0; t < kDcTaps; ++t) xv[j][t] = buf_ld2(rs, off[j][t], so, static_cast<const T*>(nullptr));
  };
  fetch(wave);
  for (int c = wave; c < g.cin; c += WAVES) {
    store_weights<OB, OBP, PER>(wl[wave], lane, wv);
    float cur[PX][kDcTaps];
#pragma unroll
    for (int j = 0; j < PX; ++j)
#pragma unroll
      for (int t = 0; t < kDcTaps; ++t) cur[j][t] = xv[j][t];
    fetch(c + WAVES);
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int t = 0; t < kDcTaps; ++t) {
      float w[OBP];
#pragma unroll
      for (int o = 0; o < OBP; ++o) w[o] = wl[wave][t * OBP + o];
#pragma unroll
      for (int j = 0; j < PX; ++j)
#pragma unroll
        for (int o = 0; o < OB; ++o) acc[j][o] = fmaf(cur[j][t], w[o], acc[j][o]);
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int j = 0; j < PX; ++j)
#pragma unroll
    for (int o = 0; o < OB; ++o) part[wave][o][j * 64 + lane] = acc[j][o];
  __syncthreads();
  for (int e = threadIdx.x; e < OB * PIX; e += 64 * WAVES) {
    const int o = o0 + e / PIX, q = blockIdx.x * PIX + e % PIX;
    if (o >= g.cout || q >= total) continue;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) s += part[k][e / PIX][e % PIX];
    const int m = q / plane;
    st(out + ((long)m * g.cout + o) * plane + (q - m * plane), s + ld(bias + o));
  }
}

// Input gradient.  A lane owns PX input pixels, a wave CH channels: per tap the 18 output gradients that touch a pixel
// through it are multiplied with each channel's weights.  Nothing is added across waves.
template <typename T, int CH, int PX>
__global__ __launch_bounds__(256) void direct_conv_backward_input_kernel(DirectConv g, const T* __restrict__ gout,
                                                                         const T* __restrict__ weight, T* __restrict__ gin) {
  constexpr int OBP = 20, PER = 3;
  __shared__ __align__(16) float wl[4][CH][kDcTaps * OBP];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int in_plane = g.h * g.w, plane = g.oh * g.ow, total = g.batch * in_plane;
  const rsrc_t rs = plane_rsrc(gout, g.batch * g.cout * plane);
  const int c0 = (blockIdx.y * 4 + wave) * CH;
#pragma unroll
  for (int k = 0; k < CH; ++k) {
    float wv[PER];
    load_weights<T, kDcOut, PER>(g, weight, 0, c0 + k, lane, wv);
    store_weights<kDcOut, OBP, PER>(wl[wave][k], lane, wv);
  }
  __builtin_amdgcn_wave_barrier();
  float acc[PX][CH];
  int n[PX], q[PX];
#pragma unroll
  for (int j = 0; j < PX; ++j) {
    const int pix = min((int)(blockIdx.x * PX + j) * 64 + lane, total - 1);
    n[j] = pix / in_plane, q[j] = pix - n[j] * in_plane;
#pragma unroll
    for (int k = 0; k < CH; ++k) acc[j][k] = 0.f;
  }
#pragma unroll 1
  for (int t = 0; t < kDcTaps; ++t) {
    float gv[PX][kDcOut];
#pragma unroll
    for (int j = 0; j < PX; ++j) {
      // output pixel (oy, ox) with oy * stride + t / 3 - 1 == y
      const int sy = q[j] / g.w + 1 - t / 3, sx = q[j] % g.w + 1 - t % 3;
      const int oy = sy / g.stride, ox = sx / g.stride;
      const bool hit = sy >= 0 && sx >= 0 && oy * g.stride == sy && ox * g.stride == sx && oy < g.oh && ox < g.ow;
      const unsigned off = hit ? ((unsigned)n[j] * g.cout * plane + oy * g.ow + ox) * (unsigned)sizeof(T) : kOutOfRange;
#pragma unroll
      for (int o = 0; o < kDcOut; ++o)
        gv[j][o] = buf_ld2(rs, o < g.cout ? off : kOutOfRange, min(o, g.cout - 1) * plane * (int)sizeof(T), static_cast<const T*>(nullptr));
    }
#pragma unroll
    for (int k = 0; k < CH; ++k) {
      float w[OBP], s[PX];  // a tap's sum by itself: one chain over all 162 products rounds twice as far
#pragma unroll
      for (int o = 0; o < OBP; ++o) w[o] = wl[wave][k][t * OBP + o];
#pragma unroll
      for (int j = 0; j < PX; ++j) {
        s[j] = 0.f;
#pragma unroll
        for (int o = 0; o < kDcOut; ++o) s[j] = fmaf(gv[j][o], w[o], s[j]);
        acc[j][k] += s[j];
      }
    }
  }
#pragma unroll
  for (int j = 0; j < PX; ++j)
    if ((int)(blockIdx.x * PX + j) * 64 + lane < total)
#pragma unroll
      for (int k = 0; k < CH; ++k)
        if (c0 + k < g.cin) st(gin + ((long)n[j] * g.cin + c0 + k) * in_plane + q[j], acc[j][k]);
}

// Weight gradient.  A workgroup owns one input channel and ROWS tap rows; its waves take every WAVES-th group of 64 output
// pixels, a lane keeps the ROWS x 3 x 18 products' sums of its pixels.  The sums are added over the lanes by DPP steps
// (wave_sum) and over the waves, through LDS, in order: no atomics, the same result every time.
template <typename T, int ROWS, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void direct_conv_backward_weight_kernel(DirectConv g, const T* __restrict__ gout,
                                                                                 const T* __restrict__ x, T* __restrict__ gweight) {
  constexpr int NV = ROWS * 3 * kDcOut;
  __shared__ float sums[WAVES][NV];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = blockIdx.x, row0 = blockIdx.y * ROWS;
  const int in_plane = g.h * g.w, plane = g.oh * g.ow, total = g.batch * plane;
  const rsrc_t rx = plane_rsrc(x, g.batch * g.cin * in_plane), rg = plane_rsrc(gout, g.batch * g.cout * plane);
  float acc[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) acc[i] = 0.f;
  for (int base = wave * 64; base < total; base += WAVES * 64) {
    const int pix = base + lane;
    const bool live = pix < total;
    const int n = live ? pix / plane : 0, p = pix - n * plane, y = p / g.ow, xc = p % g.ow;
    float xv[ROWS * 3], gv[kDcOut];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        const int iy = y * g.stride + row0 + r - 1, ix = xc * g.stride + k - 1;
        const bool hit = live && iy >= 0 && iy < g.h && ix >= 0 && ix < g.w;
        xv[r * 3 + k] = buf_ld(rx, hit ? (((unsigned)n * g.cin + c) * in_plane + iy * g.w + ix) * (unsigned)sizeof(T) : kOutOfRange,
                               static_cast<const T*>(nullptr));
      }
    const unsigned go = live ? ((unsigned)n * g.cout * plane + p) * (unsigned)sizeof(T) : kOutOfRange;
#pragma unroll
    for (int o = 0; o < kDcOut; ++o)
      gv[o] = buf_ld2(rg, go, min(o, g.cout - 1) * plane * (int)sizeof(T), static_cast<const T*>(nullptr));
#pragma unroll
    for (int t = 0; t < ROWS * 3; ++t)
#pragma unroll
      for (int o = 0; o < kDcOut; ++o) acc[t * kDcOut + o] = fmaf(xv[t], gv[o], acc[t * kDcOut + o]);
  }
#pragma unroll
  for (int i = 0; i < NV; ++i) {
    const float s = wave_sum(acc[i]);
    if (lane == (i & 63)) sums[wave][i] = s;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < NV; i += 64 * WAVES) {
    const int t = i / kDcOut, o = i % kDcOut;
    if (o >= g.cout) continue;
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < WAVES; ++k) s += sums[k][i];
    st(gweight + ((long)o * g.cin + c) * kDcTaps + (row0 + t / 3) * 3 + t % 3, s);
  }
}

DirectConv geometry(int batch, int cin, int cout, int h, int w, int stride) {
  return DirectConv{batch, cin, cout, h, w, (h - 1) / stride + 1, (w - 1) / stride + 1, stride};
}

}  // namespace

// 32-bit byte offsets into the tensors, below the out-of-range marker; the input gradient's grid has 16 channels per row at least
bool offset_conv_direct_supported(int batch, int cin, int cout, int h, int w) {
  return cout <= kDcOut && batch >= 1 && cin <= 16 * 65535 && (long)batch * std::max(cin, cout) * h * w * 4 < (1L << 30);
}

template <typename T>
void offset_conv_direct_forward(int batch, int cin, int cout, int h, int w, int stride, const T* x, const T* weight, const T* bias, T* out,
                                hipStream_t stream) {
  const DirectConv g = geometry(batch, cin, cout, h, w, stride);
  const int pixels = batch * g.oh * g.ow, tiles = ceil_div(pixels, 64);
  // as many outputs per workgroup as leave about one workgroup per CU.  The operator's call on 192 x 28 x 28, one image (13
  // tiles): 12.9 us with two outputs per workgroup, 14.8 with six, 31 - 39 on the framework's convolution
  if (tiles <= 32)
    direct_conv_forward_kernel<T, 2, 16, 1><<<dim3(tiles, ceil_div(cout, 2)), 1024, 0, stream>>>(g, x, weight, bias, out);
  else if (tiles <= 128)
    direct_conv_forward_kernel<T, 6, 16, 1><<<dim3(tiles, ceil_div(cout, 6)), 1024, 0, stream>>>(g, x, weight, bias, out);
  else
    direct_conv_forward_kernel<T, 18, 8, 2><<<dim3(ceil_div(pixels, 128), 1), 512, 0, stream>>>(g, x, weight, bias, out);
}

template <typename T>
void offset_conv_direct_backward_input(int batch, int cin, int cout, int h, int w, int stride, const T* gout, const T* weight, T* gin,
                                       hipStream_t stream) {
  const DirectConv g = geometry(batch, cin, cout, h, w, stride);
  const int tiles = ceil_div(batch * h * w, 64);
  if ((long)tiles * ceil_div(cin, 8) < 2048)
    direct_conv_backward_input_kernel<T, 4, 1><<<dim3(tiles, ceil_div(cin, 16)), 256, 0, stream>>>(g, gout, weight, gin);
  else
    direct_conv_backward_input_kernel<T, 8, 2><<<dim3(ceil_div(tiles, 2), ceil_div(cin, 32)), 256, 0, stream>>>(g, gout, weight, gin);
}

template <typename T>
void offset_conv_direct_backward_weight(int batch, int cin, int cout, int h, int w, int stride, const T* gout, const T* x, T* gweight,
                                        hipStream_t stream) {
  const DirectConv g = geometry(batch, cin, cout, h, w, stride);
  if (cin < 256)
    direct_conv_backward_weight_kernel<T, 1, 16><<<dim3(cin, 3), 1024, 0, stream>>>(g, gout, x, gweight);
  else
    direct_conv_backward_weight_kernel<T, 3, 8><<<dim3(cin, 1), 512, 0, stream>>>(g, gout, x, gweight);
}

#define DK_INSTANTIATE(T)                                                                                                             \
  template void offset_conv_direct_forward<T>(int, int, int, int, int, int, const T*, const T*, const T*, T*, hipStream_t);          \
  template void offset_conv_direct_backward_input<T>(int, int, int, int, int, int, const T*, const T*, T*, hipStream_t);             \
  template void offset_conv_direct_backward_weight<T>(int, int, int, int, int, int, const T*, const T*, T*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
