// The kernels of a GlobalDeformKernel2d layer for one batch (reference modules/deform_kernel.py:68-101): the pooled
// input, the linear layer that turns it into one set of kernel-space offsets per image, the clamp of the coordinates and
// the sampling of the scope weights -- and their gradients.  The framework's operators for this (mean, linear, add,
// clamp, reshape and their backward: about twenty launches on tensors of a few KB besides one pass over the input each
// way) cost a host several times what the device needs; here it is two launches forward and, besides the sampler's own
// two gradients, one backward.  The input's share of the pooled gradient is a constant per plane, which the input
// gradient of the per-image convolution adds as it writes (dk_image_conv.hip) instead of two passes over the tensor.
// N=128 C=256 28x28 scope 5x5, float16, forward and backward of the layer: 590 us (host bound; 190 us of kernels) with the
// framework's operators, 115 us, all of it kernels, with these.
#include <algorithm>

#include "dk_kernels.h"
#include "dk_nd.h"

namespace dk {

namespace {

constexpr int kGlobalMaxTaps = 64;
constexpr int kGlobalMaxChannels = 8192;  // a row of the pooled input sits in LDS

template <typename T>
__device__ __forceinline__ float rounded(float v) {  // v as the tensor type holds it
  T t;
  st(&t, v);
  return ld(&t);
}

// pooled[plane] = mean of the plane.  A wave takes PP planes at a time, 16-byte loads where WIDE (planes of whole,
// aligned 16-byte groups); 103 MB of float16 input in 28 x 28 planes: bound by memory.
template <typename T, int PP, bool WIDE>
__global__ __launch_bounds__(256) void plane_mean_kernel(const T* __restrict__ x, T* __restrict__ pooled, int planes, int hw) {
  constexpr int V = WIDE ? 16 / (int)sizeof(T) : 1;
  struct alignas(V * sizeof(T)) Vec {
    T e[V];
  };
  const int lane = threadIdx.x & 63, p0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * PP;
  if (p0 >= planes) return;
  const int nv = hw / V;
  float sum[PP];
#pragma unroll
  for (int k = 0; k < PP; ++k) sum[k] = 0.f;
  constexpr int U = 8 / PP;  // groups of a plane in flight besides the planes
  for (int v0 = lane; v0 < nv; v0 += 64 * U) {
    Vec q[PP][U];
#pragma unroll
    for (int k = 0; k < PP; ++k) {
      const Vec* row = reinterpret_cast<const Vec*>(x + (size_t)min(p0 + k, planes - 1) * hw);
#pragma unroll
      for (int u = 0; u < U; ++u) q[k][u] = row[min(v0 + 64 * u, nv - 1)];
    }
#pragma unroll
    for (int k = 0; k < PP; ++k)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        float part = 0.f;
#pragma unroll
        for (int e = 0; e < V; ++e) part += ld(&q[k][u].e[e]);
        sum[k] += v0 + 64 * u < nv ? part : 0.f;
      }
  }
#pragma unroll
  for (int k = 0; k < PP; ++k) {
    const float total = wave_sum(sum[k]);
    if (lane == k && p0 + k < planes) st(pooled + p0 + k, total / (float)hw);
  }
}

struct GlobalGeo {
  int batch, channel, taps, k_w, scope_h, scope_w, hw;
  float centre_h, centre_w, limit;  // limit: every coordinate is clamped to [0, scope_h - 1] (:83)
};

// Coordinates and sampled kernels of image blockIdx.x (channels of split blockIdx.y): fc(pooled) + undeformed tap position
// (:76-83), each step rounded to the tensor type as the layer-by-layer form does; coord keeps the values before the
// clamp (whose gradient needs them).  kernels[image * taps + tap][channel].
template <typename T>
__global__ __launch_bounds__(256) void global_kernels_kernel(GlobalGeo g, const T* __restrict__ pooled,
                                                             const T* __restrict__ fc_w, const T* __restrict__ fc_b,
                                                             const T* __restrict__ weight, T* __restrict__ coord,
                                                             T* __restrict__ clamped, T* __restrict__ kernels, int per_split) {
  extern __shared__ float row[];  // [channel]
  __shared__ float at[2 * kGlobalMaxTaps];
  const int n = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c = threadIdx.x; c < g.channel; c += 256) row[c] = ld(pooled + (size_t)n * g.channel + c);
  __syncthreads();
  for (int j = wave; j < 2 * g.taps; j += 4) {
    const T* w = fc_w + (size_t)j * g.channel;
    float acc = 0.f;
    for (int c = lane; c < g.channel; c += 64) acc = fmaf(row[c], ld(w + c), acc);
    const float fc = rounded<T>(wave_sum(acc) + ld(fc_b + j));
    const int t = j >> 1;
    const float raw = rounded<T>(fc + ((j & 1) ? g.centre_w + float(t % g.k_w) : g.centre_h + float(t / g.k_w)));
    const float lim = raw < 0.f ? 0.f : raw > g.limit ? g.limit : raw;
    if (lane == 0) {
      at[j] = rounded<T>(lim);
      if (blockIdx.y == 0) {
        st(coord + (size_t)n * 2 * g.taps + j, raw);
        st(clamped + (size_t)n * 2 * g.taps + j, lim);
      }
    }
  }
  __syncthreads();
  const int c0 = blockIdx.y * per_split, nc = min(per_split, g.channel - c0);
  const int plane = g.scope_h * g.scope_w;
  int t = threadIdx.x / nc, c = threadIdx.x - t * nc;
  const int dt = 256 / nc, dc = 256 - dt * nc;
  while (t < g.taps) {
    const float h = at[2 * t], w = at[2 * t + 1];
    float v = 0.f;
    if (h > -1.f && w > -1.f && h < float(g.scope_h) && w < float(g.scope_w)) {
      const int h0 = (int)floorf(h), w0 = (int)floorf(w);
      const float lh = h - floorf(h), lw = w - floorf(w);
      const T* f = weight + (size_t)(c0 + c) * plane;
      const bool in_h0 = h0 >= 0, in_h1 = h0 + 1 < g.scope_h, in_w0 = w0 >= 0, in_w1 = w0 + 1 < g.scope_w;
      if (in_h0 && in_w0) v += (1.f - lh) * (1.f - lw) * ld(f + h0 * g.scope_w + w0);
      if (in_h0 && in_w1) v += (1.f - lh) * lw * ld(f + h0 * g.scope_w + w0 + 1);
      if (in_h1 && in_w0) v += lh * (1.f - lw) * ld(f + (h0 + 1) * g.scope_w + w0);
      if (in_h1 && in_w1) v += lh * lw * ld(f + (h0 + 1) * g.scope_w + w0 + 1);
    }
    st(kernels + ((size_t)n * g.taps + t) * g.channel + c0 + c, v);
    t += dt;
    c += dc;
    if (c >= nc) {
      c -= nc;
      ++t;
    }
  }
}

// Gradients of the linear layer and of the pooled input from the coordinates' (zero where the clamp was active, as
// torch.clamp's is): each of the first `pool_blocks` workgroups computes pooled_grad[n][c] = sum_j gcoord[n][j] W[j][c] /
// (H W) of an image, the others the weight gradient of 64 channels and up to kFcRows rows each (column `channel` stands for the bias:
// its pooled input is 1), every sum over the images in a fixed order.
// Bound by the latency of a few loads: the operands of a step are all asked for before the first is used (one by one, in
// the order of the sums, the kernel took 37 us at N=128 C=256).
constexpr int kFcRows = 18, kFcSlices = 16, kFcImages = 128;
template <typename T>
__global__ __launch_bounds__(64 * kFcSlices) void global_fc_grad_kernel(GlobalGeo g, const T* __restrict__ gcoord,
                                                                       const T* __restrict__ coord,
                                                                       const T* __restrict__ pooled,
                                                                       const T* __restrict__ fc_w, T* __restrict__ gfc_w,
                                                                       T* __restrict__ gfc_b, float* __restrict__ gpooled,
                                                                       int pool_blocks) {
  const int rows = 2 * g.taps;
  __shared__ float gc[kFcImages][kFcRows];  // the coordinates' gradients behind the clamp
  __shared__ float part[kFcSlices][kFcRows][64];
  auto stage = [&](int n0, int images, int j0) {
    for (int e = threadIdx.x; e < images * kFcRows; e += 64 * kFcSlices) {
      const int n = n0 + e / kFcRows, j = j0 + e % kFcRows;
      const size_t at = (size_t)n * rows + min(j, rows - 1);
      const float raw = ld(coord + at), v = ld(gcoord + at);
      gc[e / kFcRows][e % kFcRows] = j < rows && raw >= 0.f && raw <= g.limit ? v : 0.f;
    }
  };
  if ((int)blockIdx.x < pool_blocks) {
    const int n = blockIdx.x;
    for (int c0 = 0; c0 < g.channel; c0 += 64 * kFcSlices) {
      const int c = min(c0 + (int)threadIdx.x, g.channel - 1);
      float acc = 0.f;
      for (int j0 = 0; j0 < rows; j0 += kFcRows) {
        __syncthreads();
        stage(n, 1, j0);
        float w[kFcRows];
#pragma unroll
        for (int j = 0; j < kFcRows; ++j) w[j] = ld(fc_w + (size_t)min(j0 + j, rows - 1) * g.channel + c);
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kFcRows; ++j) acc = fmaf(gc[0][j], w[j], acc);
      }
      if (c0 + (int)threadIdx.x < g.channel) gpooled[(size_t)n * g.channel + c] = acc / (float)g.hw;
    }
    return;
  }
  const int ctiles = ceil_div(g.channel + 1, 64), b = blockIdx.x - pool_blocks;
  const int lane = threadIdx.x & 63, slice = threadIdx.x >> 6;
  const int c = b % ctiles * 64 + lane, j0 = b / ctiles * kFcRows;
  float acc[kFcRows];
#pragma unroll
  for (int j = 0; j < kFcRows; ++j) acc[j] = 0.f;
  for (int n0 = 0; n0 < g.batch; n0 += kFcImages) {
    const int images = min(kFcImages, g.batch - n0);
    __syncthreads();
    stage(n0, images, j0);
    float x[kFcImages / kFcSlices];
#pragma unroll
    for (int i = 0; i < kFcImages / kFcSlices; ++i)
      x[i] = ld(pooled + (size_t)min(n0 + slice + i * kFcSlices, g.batch - 1) * g.channel + min(c, g.channel - 1));
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kFcImages / kFcSlices; ++i) {
      const int n = slice + i * kFcSlices;
      if (n >= images) break;
      const float v = c < g.channel ? x[i] : 1.f;
#pragma unroll
      for (int j = 0; j < kFcRows; ++j) acc[j] = fmaf(gc[n][j], v, acc[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < kFcRows; ++j) part[slice][j][lane] = acc[j];
  __syncthreads();
  for (int j = slice; j < kFcRows; j += kFcSlices) {
    if (j0 + j >= rows || c > g.channel) continue;
    float total = 0.f;
#pragma unroll
    for (int s = 0; s < kFcSlices; ++s) total += part[s][j][lane];
    if (c < g.channel) {
      if (gfc_w) st(gfc_w + (size_t)(j0 + j) * g.channel + c, total);
    } else if (gfc_b) {
      st(gfc_b + j0 + j, total);
    }
  }
}

GlobalGeo global_geo(const Geo& g) {
  return GlobalGeo{g.batch, g.channel, g.k_h * g.k_w, g.k_w, g.scope_h, g.scope_w, g.in_h * g.in_w,
                   (float)g.centre_h, (float)g.centre_w, (float)(g.scope_h - 1)};
}

// the sampler's call: batch * taps points on `channel` grids of scope_h x scope_w
dk_nd_desc sampler_desc(const Geo& g, int dtype) {
  dk_nd_desc d{};
  d.batch = (int64_t)g.batch * g.k_h * g.k_w;
  d.channel = g.channel;
  d.dims = 2;
  d.shape[0] = g.scope_h;
  d.shape[1] = g.scope_w;
  d.dtype = dtype;
  return d;
}

size_t round256(size_t n) { return (n + 255) / 256 * 256; }

}  // namespace

bool global_kernels_supported(const Geo& g, int dtype) {
  const long planes = (long)g.batch * g.channel;
  return dtype != DK_F64 && g.groups == 1 && (long)g.k_h * g.k_w <= kGlobalMaxTaps && g.channel <= kGlobalMaxChannels &&
         planes * g.k_h * g.k_w < (1L << 31) && (long)g.in_h * g.in_w < (1L << 30) &&
         (long)g.channel * g.scope_h * g.scope_w < (1L << 31);
}

template <typename T>
void global_kernels_forward(const Geo& geo, const T* x, const T* fc_w, const T* fc_b, const T* weight, T* pooled, T* coord,
                            T* clamped, T* kernels, hipStream_t stream) {
  const GlobalGeo g = global_geo(geo);
  const int planes = g.batch * g.channel;
  const bool wide = (size_t)g.hw * sizeof(T) % 16 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0;
  const int nv = wide ? (int)(g.hw * sizeof(T) / 16) : g.hw;
  // four planes per wave while a plane is a few loads of the wave and the waves are plenty
  const bool four = nv <= 256 && planes >= 4096;
  const unsigned grid = (unsigned)((planes + (four ? 15 : 3)) / (four ? 16 : 4));
  if (four && wide) plane_mean_kernel<T, 4, true><<<grid, 256, 0, stream>>>(x, pooled, planes, g.hw);
  else if (four) plane_mean_kernel<T, 4, false><<<grid, 256, 0, stream>>>(x, pooled, planes, g.hw);
  else if (wide) plane_mean_kernel<T, 1, true><<<grid, 256, 0, stream>>>(x, pooled, planes, g.hw);
  else plane_mean_kernel<T, 1, false><<<grid, 256, 0, stream>>>(x, pooled, planes, g.hw);
  // channel splits: enough workgroups for the chip, each with at least 64 channels
  const int want = std::max(1, std::min(ceil_div(g.channel, 64), ceil_div(512, g.batch)));
  const int per = ceil_div(g.channel, want);
  global_kernels_kernel<T><<<dim3((unsigned)g.batch, (unsigned)ceil_div(g.channel, per)), 256, (size_t)g.channel * sizeof(float), stream>>>(
      g, pooled, fc_w, fc_b, weight, coord, clamped, kernels, per);
}

size_t global_kernels_backward_workspace(const Geo& g, int dtype) {
  const dk_nd_desc d = sampler_desc(g, dtype);
  const size_t gcoord = round256((size_t)d.batch * 2 * sizeof(float));
  return gcoord + std::max(nd_grad_data_workspace(d), nd_data_cl_workspace(d));
}

template <typename T>
void global_kernels_backward(const Geo& geo, int dtype, const T* gkernels, const T* pooled, const T* coord,
                             const T* clamped, const T* weight, const T* fc_w, T* gweight, T* gfc_w, T* gfc_b,
                             float* gpooled, void* ws, hipStream_t stream) {
  const GlobalGeo g = global_geo(geo);
  const dk_nd_desc d = sampler_desc(geo, dtype);
  T* gcoord = static_cast<T*>(ws);
  void* nd_ws = static_cast<char*>(ws) + round256((size_t)d.batch * 2 * sizeof(float));
  if (gweight) nd_grad_data<T>(d, gkernels, clamped, gweight, nd_ws, nullptr, stream);
  if (!gfc_w && !gfc_b && !gpooled) return;
  nd_grad_coord<T>(d, gkernels, weight, clamped, gcoord, nd_ws, nullptr, stream);
  constexpr int kThreads = 64 * kFcSlices;
  const int pool_blocks = gpooled ? g.batch : 0;
  const int fc_blocks = gfc_w || gfc_b ? ceil_div(g.channel + 1, 64) * ceil_div(2 * g.taps, kFcRows) : 0;
  global_fc_grad_kernel<T><<<(unsigned)(pool_blocks + fc_blocks), kThreads, 0, stream>>>(g, gcoord, coord, pooled, fc_w, gfc_w, gfc_b,
                                                                                 gpooled, pool_blocks);
}

#define DK_INSTANTIATE(T)                                                                                             \
  template void global_kernels_forward<T>(const Geo&, const T*, const T*, const T*, const T*, T*, T*, T*, T*, hipStream_t); \
  template void global_kernels_backward<T>(const Geo&, int, const T*, const T*, const T*, const T*, const T*, const T*, T*, \
                                           T*, T*, float*, void*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
