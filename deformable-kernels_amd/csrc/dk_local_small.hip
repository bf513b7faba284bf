// The gradients of the local operator on small layers in one launch: 3 x 3 taps, scopes 3 x 3 / 4 x 4 / 5 x 5 / 7 x 7,
// float32 / float16 / bfloat16 tensors, planar or channels-last, any stride, padding, dilation and group count.
//
// What bounds a small layer is launches: the tuned kernels take three to five of them (grad filter and grad rotation add
// their partial sums in kernels of their own), 3.4 us of host time each, and each is a chain of ramps and load latencies of
// 8 - 14 us on an idle chip.  Here the workgroups of one grid take one of three roles, so that the chains run side by side,
// and what a role adds up is added inside a workgroup, in a fixed order, through LDS: no workspace, no second launch.
//   grad input     64 input pixels, a share of the channels: a wave walks channels, a lane gathers its pixel's taps
//   grad rotation  64 output pixels: 16 waves share the channels, their sums are added in wave order
//   grad filter    one channel: 16 waves share the pixels; a lane keeps a sum per scope cell, dense hat weights
// fp32 arithmetic for every type (reference kernels: K.cu:577-702, 836-999, 1285-1408).  What the reference skips -- a tap
// outside the image, off the stride's grid or outside the scope, a cell that a tap does not read -- takes nothing from a value
// that is not finite.  Registers: 1024 threads leave 128 of them; nothing spills.
#include <algorithm>

#include "dk_common.h"
#include "dk_kernels.h"
#include "dk_scope_table.h"

namespace dk {
namespace {

constexpr int kSmWaves = 16, kSmTaps = 9;

// Element strides of image, channel and plane position of the three tensors
struct SmallStrides {
  int xn, xc, xp, on, oc, op, rn, rc, rp;
};
struct SmallRoles {
  int input_tiles, input_splits;  // tiles of 64 input pixels, all groups; shares of the channels
  int rotation_tiles;             // tiles of 64 output pixels, all groups
  int filter_channels;            // channels (0: that gradient is not wanted)
};

// The scope table of one channel, staged by the wave that uses it: lane m writes block m.
template <typename T, int S>
struct WaveTable {
  using Tb = WideTable<S, S>;
  unsigned off[4];
  float v[4];
  __device__ __forceinline__ void init(int lane) {
    const int i = lane / Tb::RS - 1, k = lane % Tb::RS - 1;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int ii = i + (q >> 1), kk = k + (q & 1);
      off[q] = lane < Tb::BLOCKS && ii >= 0 && ii < S && kk >= 0 && kk < S ? (unsigned)(ii * S + kk) * (unsigned)sizeof(T) : kOutOfRange;
    }
  }
  __device__ __forceinline__ void load(rsrc_t rf, int c) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] = buf_ld2(rf, off[q], c * S * S * (int)sizeof(T), static_cast<const T*>(nullptr));
  }
  __device__ __forceinline__ void store(float* tbl, int lane) const {
    if (lane < Tb::BLOCKS)
      *reinterpret_cast<float4*>(tbl + Tb::slot(lane) * 4) = make_float4(v[0], v[1] - v[0], v[2] - v[0], (v[3] - v[1]) - (v[2] - v[0]));
  }
};

// A tap's descriptor; one that contributes nothing (`in` false: not `ok`, or outside the scope) points at a block of zeros
// behind the table.  (The table's own block (-1, -1), which make_lite_tap takes for it, holds cell (0, 0) in its last entry:
// a weight that is not finite there would reach every such tap.)
template <int S>
__device__ __forceinline__ LiteTap small_tap(float h, float w, bool ok, bool& in) {
  in = ok && h > -1.f && w > -1.f && h < float(S) && w < float(S);
  LiteTap t = make_lite_tap<S, S>(h, w, in);
  t.cell = in ? t.cell : WideTable<S, S>::SIZE;
  return t;
}

template <typename T, int S>
__global__ __launch_bounds__(64 * kSmWaves) void local_small_backward_kernel(Geo g, SmallStrides st, SmallRoles roles, const T* __restrict__ gout,
                                                                             const T* __restrict__ x, const T* __restrict__ rot,
                                                                             const T* __restrict__ filter, T* __restrict__ gin,
                                                                             T* __restrict__ grot, T* __restrict__ gfilter) {
  using Tb = WideTable<S, S>;
  constexpr int CELLS = S * S, PARTS = kSmTaps * 64 > CELLS ? kSmTaps * 64 : CELLS;
  __shared__ __align__(16) float tables[kSmWaves][Tb::SIZE + 4];  // and the block of zeros
  __shared__ float part[kSmWaves][PARTS];
  constexpr const T* tag = nullptr;
  constexpr unsigned E = sizeof(T);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int in_plane = g.in_h * g.in_w, out_plane = g.out_h * g.out_w, cpg = g.channel / g.groups;
  const rsrc_t rg = plane_rsrc(gout, g.batch * g.channel * out_plane), rx = plane_rsrc(x, g.batch * g.channel * in_plane);
  const rsrc_t rr = plane_rsrc(rot, g.batch * g.groups * 2 * kSmTaps * out_plane), rf = plane_rsrc(filter, g.channel * CELLS);
  int b = blockIdx.x;
  if (lane < 4) tables[wave][Tb::SIZE + lane] = 0.f;

  if (b < roles.input_tiles * roles.input_splits) {
    const int split = b % roles.input_splits, tile = b / roles.input_splits;
    const int per_group = roles.input_tiles / g.groups, grp = tile / per_group;
    const int pix = (tile - grp * per_group) * 64 + lane;
    const bool live = pix < g.batch * in_plane;
    const int n = live ? pix / in_plane : 0, q = live ? pix - n * in_plane : 0, y = q / g.in_w, xc = q - y * g.in_w;
    LiteTap tap[kSmTaps];
    unsigned off[kSmTaps];
#pragma unroll
    for (int t = 0; t < kSmTaps; ++t) {
      // the output pixel whose tap t reads this input pixel
      const int ny = y + g.pad_h - t / 3 * g.dil_h, nx = xc + g.pad_w - t % 3 * g.dil_w;
      const int oy = ny / g.stride_h, ox = nx / g.stride_w;
      const bool hit = live && ny >= 0 && nx >= 0 && oy * g.stride_h == ny && ox * g.stride_w == nx && oy < g.out_h && ox < g.out_w;
      const int p = hit ? oy * g.out_w + ox : 0;
      const unsigned ro = hit ? (unsigned)(n * st.rn + (grp * 18 + 2 * t) * st.rc + p * st.rp) * E : kOutOfRange;
      const float h = scope_coord<float>(g, t / 3, buf_ld2(rr, ro, 0, tag), g.centre_h);
      const float w = scope_coord<float>(g, t % 3, buf_ld2(rr, ro, st.rc * (int)E, tag), g.centre_w);
      bool in;
      tap[t] = small_tap<S>(h, w, hit, in);
      off[t] = hit ? (unsigned)(n * st.on + p * st.op) * E : kOutOfRange;
    }
    WaveTable<T, S> table;
    table.init(lane);
    float gv[kSmTaps];
    auto fetch = [&](int j) {
      const int c = grp + g.groups * min(j, cpg - 1);
      table.load(rf, c);
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) gv[t] = buf_ld2(rg, off[t], c * st.oc * (int)E, tag);
    };
    const int step = kSmWaves * roles.input_splits;
    int j = split * kSmWaves + wave;
    if (j < cpg) fetch(j);
    for (; j < cpg; j += step) {
      table.store(tables[wave], lane);
      float cur[kSmTaps];
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) cur[t] = gv[t];
      fetch(j + step);
      __builtin_amdgcn_wave_barrier();
      float acc = 0.f;
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t)
        acc = fmaf(cur[t], lite_weight(tap[t], *reinterpret_cast<const float4*>(&tables[wave][tap[t].cell])), acc);
      __builtin_amdgcn_wave_barrier();
      if (live) dk::st(gin + n * st.xn + (grp + g.groups * j) * st.xc + q * st.xp, acc);
    }
    return;
  }
  b -= roles.input_tiles * roles.input_splits;

  if (b < roles.rotation_tiles) {
    const int per_group = roles.rotation_tiles / g.groups, grp = b / per_group, pix0 = (b - grp * per_group) * 64;
    const int total = g.batch * out_plane;
    const bool live = pix0 + lane < total;
    const int n = live ? (pix0 + lane) / out_plane : 0, p = live ? pix0 + lane - n * out_plane : 0, oh = p / g.out_w, ow = p - oh * g.out_w;
    LiteTap tap[kSmTaps];
    unsigned off[kSmTaps], open = 0;  // bits 2 t + dir of `open`: the tap reads image and scope, and the offset is not clamped
#pragma unroll
    for (int t = 0; t < kSmTaps; ++t) {
      const unsigned ro = live ? (unsigned)(n * st.rn + (grp * 18 + 2 * t) * st.rc + p * st.rp) * E : kOutOfRange;
      bool oh_open, ow_open;
      const float h = scope_coord<float>(g, t / 3, buf_ld2(rr, ro, 0, tag), g.centre_h, &oh_open);
      const float w = scope_coord<float>(g, t % 3, buf_ld2(rr, ro, st.rc * (int)E, tag), g.centre_w, &ow_open);
      const int iy = oh * g.stride_h - g.pad_h + t / 3 * g.dil_h, ix = ow * g.stride_w - g.pad_w + t % 3 * g.dil_w;
      const bool hit = live && iy >= 0 && iy < g.in_h && ix >= 0 && ix < g.in_w;
      bool in;
      tap[t] = small_tap<S>(h, w, hit, in);
      open |= (in && oh_open ? 1u : 0u) << (2 * t) | (in && ow_open ? 2u : 0u) << (2 * t);
      off[t] = hit ? (unsigned)(n * st.xn + (iy * g.in_w + ix) * st.xp) * E : kOutOfRange;
    }
    const unsigned goff = live ? (unsigned)(n * st.on + p * st.op) * E : kOutOfRange;
    WaveTable<T, S> table;
    table.init(lane);
    float xv[kSmTaps], gv = 0.f;
    auto fetch = [&](int j) {
      const int c = grp + g.groups * min(j, cpg - 1);
      table.load(rf, c);
      gv = buf_ld2(rg, goff, c * st.oc * (int)E, tag);
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) xv[t] = buf_ld2(rx, off[t], c * st.xc * (int)E, tag);
    };
    float sb[kSmTaps], sc[kSmTaps], sd[kSmTaps];
#pragma unroll
    for (int t = 0; t < kSmTaps; ++t) sb[t] = sc[t] = sd[t] = 0.f;
    if (wave < cpg) fetch(wave);
    for (int j = wave; j < cpg; j += kSmWaves) {
      table.store(tables[wave], lane);
      float cur[kSmTaps];
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) cur[t] = xv[t] * gv;
      fetch(j + kSmWaves);
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) {
        const float4 w = lds_read4(&tables[wave][tap[t].cell]);
        sb[t] = fmaf(cur[t], w.y, sb[t]);
        sc[t] = fmaf(cur[t], w.z, sc[t]);
        sd[t] = fmaf(cur[t], w.w, sd[t]);
      }
      __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int dir = 0; dir < 2; ++dir) {
      if (dir) __syncthreads();
#pragma unroll
      for (int t = 0; t < kSmTaps; ++t) {
        const float d = dir ? fmaf(tap[t].lh, sd[t], sb[t]) : fmaf(tap[t].lw, sd[t], sc[t]);
        part[wave][t * 64 + lane] = open >> (2 * t + dir) & 1u ? d : 0.f;
      }
      __syncthreads();
      if (threadIdx.x < kSmTaps * 64) {
        const int t = threadIdx.x >> 6, at = pix0 + lane;
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < kSmWaves; ++k) s += part[k][t * 64 + lane];
        if (at < total) dk::st(grot + n * st.rn + (grp * 18 + 2 * t + dir) * st.rc + p * st.rp, s);
      }
    }
    return;
  }
  b -= roles.rotation_tiles;

  const int c = b, grp = c % g.groups, total = g.batch * out_plane;
  float acc[CELLS], z = 0.f;  // z: NaN where a product is not finite
#pragma unroll
  for (int i = 0; i < CELLS; ++i) acc[i] = 0.f;
  for (int base = wave * 64; base < total; base += kSmWaves * 64) {
    const bool live = base + lane < total;
    const int n = live ? (base + lane) / out_plane : 0, p = live ? base + lane - n * out_plane : 0, oh = p / g.out_w, ow = p - oh * g.out_w;
    const float gv = buf_ld2(rg, live ? (unsigned)(n * st.on + p * st.op) * E : kOutOfRange, c * st.oc * (int)E, tag);
    float xv[kSmTaps], rh[kSmTaps], rw[kSmTaps];
#pragma unroll
    for (int t = 0; t < kSmTaps; ++t) {
      const int iy = oh * g.stride_h - g.pad_h + t / 3 * g.dil_h, ix = ow * g.stride_w - g.pad_w + t % 3 * g.dil_w;
      const bool hit = live && iy >= 0 && iy < g.in_h && ix >= 0 && ix < g.in_w;
      xv[t] = buf_ld2(rx, hit ? (unsigned)(n * st.xn + (iy * g.in_w + ix) * st.xp) * E : kOutOfRange, c * st.xc * (int)E, tag);
      const unsigned ro = live ? (unsigned)(n * st.rn + (grp * 18 + 2 * t) * st.rc + p * st.rp) * E : kOutOfRange;
      rh[t] = buf_ld2(rr, ro, 0, tag), rw[t] = buf_ld2(rr, ro, st.rc * (int)E, tag);
    }
#pragma unroll
    for (int t = 0; t < kSmTaps; ++t) {
      const float h = scope_coord<float>(g, t / 3, rh[t], g.centre_h), w = scope_coord<float>(g, t % 3, rw[t], g.centre_w);
      const float v = xv[t] * gv;
      z = fmaf(v, 0.f, z);
      float hw[S];
#pragma unroll
      for (int k = 0; k < S; ++k) hw[k] = fmaxf(0.f, 1.f - fabsf(w - (float)k));
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const float a = v * fmaxf(0.f, 1.f - fabsf(h - (float)i));
#pragma unroll
        for (int k = 0; k < S; ++k) acc[i * S + k] = fmaf(a, hw[k], acc[i * S + k]);
      }
    }
  }
  if (__any(z != 0.f)) {
    // a product that is not finite must not meet the zero hats of the cells that its tap does not read (K.cu:85-114), nor the zero
    // read for a tap outside the image: the wave's pixels once more, a tap and its own cells at a time
#pragma unroll
    for (int i = 0; i < CELLS; ++i) acc[i] = 0.f;
    for (int base = wave * 64; base < total; base += kSmWaves * 64)
#pragma unroll 1
    for (int t = 0; t < kSmTaps; ++t) {
      const int q = base + lane;
      const bool live = q < total;
      const int n = live ? q / out_plane : 0, p = live ? q - n * out_plane : 0, oh = p / g.out_w, ow = p - oh * g.out_w;
      const int iy = oh * g.stride_h - g.pad_h + t / 3 * g.dil_h, ix = ow * g.stride_w - g.pad_w + t % 3 * g.dil_w;
      const bool hit = live && iy >= 0 && iy < g.in_h && ix >= 0 && ix < g.in_w;
      const float v = buf_ld2(rg, live ? (unsigned)(n * st.on + p * st.op) * E : kOutOfRange, c * st.oc * (int)E, tag) *
                      buf_ld2(rx, hit ? (unsigned)(n * st.xn + (iy * g.in_w + ix) * st.xp) * E : kOutOfRange, c * st.xc * (int)E, tag);
      const unsigned ro = live ? (unsigned)(n * st.rn + (grp * 18 + 2 * t) * st.rc + p * st.rp) * E : kOutOfRange;
      const float h = scope_coord<float>(g, t / 3, buf_ld2(rr, ro, 0, tag), g.centre_h);
      const float w = scope_coord<float>(g, t % 3, buf_ld2(rr, ro, st.rc * (int)E, tag), g.centre_w);
      const bool in = hit && h > -1.f && w > -1.f && h < float(S) && w < float(S);
      const int i0 = in ? (int)floorf(h) : 0, k0 = in ? (int)floorf(w) : 0;
#pragma unroll
      for (int i = 0; i < S; ++i) {
        const float a = v * (1.f - fabsf(h - (float)i));
#pragma unroll
        for (int k = 0; k < S; ++k)
          acc[i * S + k] += in && (unsigned)(i - i0) < 2u && (unsigned)(k - k0) < 2u ? a * (1.f - fabsf(w - (float)k)) : 0.f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < CELLS; ++i) {
    const float s = wave_sum(acc[i]);
    if (lane == 0) part[wave][i] = s;
  }
  __syncthreads();
  if (threadIdx.x < CELLS) {
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < kSmWaves; ++k) s += part[k][threadIdx.x];
    dk::st(gfilter + c * CELLS + threadIdx.x, s);
  }
}

SmallRoles small_roles(const Geo& g, bool input, bool rotation, bool filter) {
  SmallRoles roles{};
  if (input) {
    roles.input_tiles = g.groups * ceil_div(g.batch * g.in_h * g.in_w, 64);
    // two channels per wave at least, about a workgroup per CU
    roles.input_splits = std::max(1, std::min(ceil_div(g.channel / g.groups, 2 * kSmWaves), 256 / roles.input_tiles));
  }
  if (rotation) roles.rotation_tiles = g.groups * ceil_div(g.batch * g.out_h * g.out_w, 64);
  if (filter) roles.filter_channels = g.channel;
  return roles;
}
int small_blocks(const SmallRoles& r) { return r.input_tiles * r.input_splits + r.rotation_tiles + r.filter_channels; }
}  // namespace

// At most 2048 output pixels and 256 channels per group: a wave of the grad filter then has two groups of pixels, one of the
// grad rotation at most 16 channels in a row.  All gradients, us on the GPU alone, one launch / the larger layers' kernels, whose
// four or five launches also take 14 - 20 us of host time more: 2 x 32 x 28^2 float32 12.1 / 33.3, 10 x 96 x 14^2 18.3 / 37.2, 2 x 256 x
// 32^2 37.4 / 45.7, 2 x 128 x 56^2 stride 2 26.0 / 39.3; beyond: 3 x 912 x 14^2 (57 channels in a row) and 100 x 200 x 7^2 (4900 pixels)
// a third slower.  Several groups multiply the input's and rotation's workgroups: up to 850 of all roles (a CU holds one at a
// time) 2 x 512 x 32^2 in two groups 47 / 59, 28^2 in eight 30 / 36; more: 28^2 in sixteen (928) bfloat16 35 / 33, 2 x 512 x 32^2 in eight
// (1024) 50 / 45, 2 x 256 x 32^2 in sixteen (1280) 48 / 31.
// Channels-last: a channel's lanes read elements that are far apart, so where the larger layers' kernels run on the matrix
// cores (one group, channels in eights) they are level at 32 channels: 2 x 16 x 32^2 18.7 / 19.1, 32 channels 22.8 / 21.0 (float32 at stride 2, whose
// input gradient is a launch of its own, 16 channels 22.6 / 20.7, 32 channels 27.6 / 22.4), 64 channels 32.5 / 25.1, 128 channels 51 / 32; scope 7,
// 128 channels, 51 / 55, 192 channels of 28^2 69 / 65.  Elsewhere: 2 x 33 x 32^2 20 / 48, 132 channels 39 / 57, 2 x 64 x 32^2 in two groups 26 / 378.
bool local_small_backward_supported(const Geo& g, bool channels_last, bool float32) {
  if (test_switches() != 0 || g.k_h != 3 || g.k_w != 3 || g.scope_h != g.scope_w || g.batch <= 0) return false;
  if (g.scope_h != 3 && g.scope_h != 4 && g.scope_h != 5 && g.scope_h != 7) return false;
  if ((long)g.batch * g.out_h * g.out_w > 2048 || (long)g.batch * g.in_h * g.in_w > 16384) return false;
  if (g.channel / g.groups > 256 || g.groups > 16) return false;
  if (!channels_last) return small_blocks(small_roles(g, true, true, true)) <= 850;
  if (g.groups > 1 || g.channel % 8 != 0) return true;
  const bool apart = float32 && (g.stride_h > 1 || g.stride_w > 1);
  return g.channel <= (g.scope_h == 7 ? 128 : apart ? 16 : 32);
}

template <typename T>
void local_small_backward(const Geo& g, bool channels_last, const T* gout, const T* x, const T* rot, const T* filter, T* gin, T* grot,
                          T* gfilter, hipStream_t stream) {
  const int pi = g.in_h * g.in_w, po = g.out_h * g.out_w, cr = 18 * g.groups;
  const SmallStrides st = channels_last ? SmallStrides{pi * g.channel, 1, g.channel, po * g.channel, 1, g.channel, po * cr, 1, cr}
                                        : SmallStrides{pi * g.channel, pi, 1, po * g.channel, po, 1, po * cr, po, 1};
  const SmallRoles roles = small_roles(g, gin, grot, gfilter);
  const int blocks = small_blocks(roles);
  if (blocks == 0) return;
#define DK_LAUNCH(S) local_small_backward_kernel<T, S><<<blocks, 64 * kSmWaves, 0, stream>>>(g, st, roles, gout, x, rot, filter, gin, grot, gfilter)
  if (g.scope_h == 3) DK_LAUNCH(3);
  else if (g.scope_h == 4) DK_LAUNCH(4);
  else if (g.scope_h == 5) DK_LAUNCH(5);
  else DK_LAUNCH(7);
#undef DK_LAUNCH
}

#define DK_INSTANTIATE(T) \
  template void local_small_backward<T>(const Geo&, bool, const T*, const T*, const T*, const T*, T*, T*, T*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
