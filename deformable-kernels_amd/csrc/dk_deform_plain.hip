// Deformable forward and grad offset without kernel-space offsets (rotation == NULL: DeformKernelConv2d, DeformConv2d).
//
// Reference kernels covered (K.cu =
// deformable_kernels/ops/deform_kernel/csrc/filter_sample_depthwise_cuda_kernel.cu): forward, K.cu:433-528, and grad
// offset, K.cu:1147-1243, where every kernel-space offset is zero.
//
// Each tap then reads the scope tile at one place for all pixels, so a channel has nine weights and no table: what
// dk_deform_fast.hip reads per sample and channel at an address of its own (16 bytes of LDS) is one broadcast read per
// tap and group of channels.  The rest is as there -- a lane owns an output pixel, zero-padded input planes double
// buffered in LDS, interleaved 16 bytes to a position -- except that 16-bit planes stay 16-bit, eight channels to a
// position, and their corners enter the multiply-adds as stored (v_fma_mix_f32 for float16).
// What bounds it now is the vector unit: five (forward) and eight (grad offset) instructions per sample and channel.
// us, with the tables / here: forward and grad offset of N=64 C=192 28x28 float16 90 / 38 and 111 / 45, float32 85 / 46 and
// 94 / 52; C=144 56x56 float32 179 / 143 and 215 / 169; N=128 C=960 7x7 float16 150 / 28 and 188 / 40 (a chunk of channels
// per wave there: the tables' kernel fills 49 of 256 lanes).
#include <algorithm>
#include <type_traits>

#include "dk_common.h"
#include "dk_kernels.h"

namespace dk {

namespace {

constexpr int K9 = 9;
constexpr int kPlPos = 16;          // bytes of a position of the interleaved planes
constexpr int kPlThreads = 1024;    // most threads of a workgroup
constexpr long kPlLds = 150 * 1024;

// Four channels of float32 or eight of a 16-bit type
template <typename T>
constexpr int kPlCh = kPlPos / (int)sizeof(T);

template <typename T>
__device__ __forceinline__ float element(const uint4& v, int c) {
  const unsigned w[4] = {v.x, v.y, v.z, v.w};
  if constexpr (sizeof(T) == 4) {
    return __uint_as_float(w[c]);
  } else {
    const unsigned h = w[c >> 1];
    if constexpr (std::is_same<T, __half>::value)
      return static_cast<float>(__builtin_bit_cast(_Float16, (unsigned short)(c & 1 ? h >> 16 : h & 0xffffu)));
    else
      return __uint_as_float(c & 1 ? h & 0xffff0000u : h << 16);
  }
}
// element c of a minus element c of b
template <typename T>
__device__ __forceinline__ float difference(const uint4& a, const uint4& b, int c) {
  if constexpr (std::is_same<T, __half>::value) {
    const unsigned wa[4] = {a.x, a.y, a.z, a.w}, wb[4] = {b.x, b.y, b.z, b.w};
    float r;  // a * 1 - b on the elements as stored, one instruction for both conversions and the subtraction
    if (c & 1)
      asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,1] op_sel_hi:[1,0,1]" : "=v"(r) : "v"(wa[c >> 1]), "v"(wb[c >> 1]));
    else
      asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[0,0,0] op_sel_hi:[1,0,1]" : "=v"(r) : "v"(wa[c >> 1]), "v"(wb[c >> 1]));
    return r;
  } else {
    return element<T>(a, c) - element<T>(b, c);
  }
}

// kPlCh<T> planes on their way to LDS: element e of the planes for e = thread, thread + block, ...
template <typename T, int PASSES>
struct PlainStage {
  static constexpr int CH = kPlCh<T>;
  unsigned v[CH][PASSES];
  __device__ __forceinline__ void load(const T* plane0, size_t step, int live, int in_plane) {
    const rsrc_t r = plane_rsrc(plane0, (int)((live - 1) * step) + in_plane);
    const int bytes = (int)(step * sizeof(T));
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      const int e = threadIdx.x + k * blockDim.x;
      const unsigned o = e < in_plane ? (unsigned)e * (unsigned)sizeof(T) : kOutOfRange;
#pragma unroll
      for (int c = 0; c < CH; ++c) {
        // (the scalar part stays inside the buffer; a channel past the last one reads as zeros)
        const int s = min(c, live - 1) * bytes;
        const unsigned at = c < live ? o : kOutOfRange;
        if constexpr (sizeof(T) == 4)
          v[c][k] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)at, s, 0);
        else
          v[c][k] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)at, s, 0);
      }
    }
  }
  __device__ __forceinline__ void store(char* planes, const int (&dst)[PASSES]) const {
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (dst[k] < 0) continue;
      uint4 q;
      if constexpr (sizeof(T) == 4)
        q = make_uint4(v[0][k], v[1][k], v[2][k], v[3][k]);
      else
        q = make_uint4(v[0][k] | v[1][k] << 16, v[2][k] | v[3][k] << 16, v[4][k] | v[5][k] << 16, v[6][k] | v[7][k] << 16);
      *reinterpret_cast<uint4*>(planes + dst[k]) = q;
    }
  }
};

// One workgroup per (pixel tile, channel chunk, image, group), a lane per pixel of the tile, the chunk's channels kPlCh<T>
// at a time.  GRAD: grad offset, partial[group][chunk][image][18][pixel] in fp32; else the forward.
// A weight that is not finite must not meet the zeros that stand for a tap outside the image (the reference skips such
// taps): a chunk that holds one masks the weights of those taps.
// Registers: 1024 threads leave 128 of them.  Instances that spill, bytes per lane for two, three and four staging passes (they
// hold the next channels' planes): grad offset bfloat16 36, 100, 144; float16 0, 12, 80; float32 0, 0, 16; forward bfloat16
// in four passes 8.
template <typename T, int PASSES, bool GRAD>
__global__ __launch_bounds__(kPlThreads) void deform_plain_kernel(
    Geo g, const T* __restrict__ gout, const T* __restrict__ x, const T* __restrict__ off, const T* __restrict__ filter,
    T* __restrict__ out, float* __restrict__ partial, int tiles, int chunks, int ch_per_block) {
  constexpr int CH = kPlCh<T>;
  extern __shared__ __align__(16) char pl_lds[];
  const int H = g.in_h, W = g.in_w, RS = W + 2;
  const int plane_bytes = (H + 2) * RS * kPlPos;
  float* wts = reinterpret_cast<float*>(pl_lds + 2 * plane_bytes);  // [channels / CH][K9][CH]

  const int cpg = g.channel / g.groups;
  const int out_plane = g.out_h * g.out_w, in_plane = H * W;
  const int total = tiles * chunks * g.batch * g.groups;
  const int lb = logical_block(total);
  if (lb >= total) return;
  const int tile = lb % tiles, chunk = lb / tiles % chunks;
  const int n = lb / tiles / chunks / g.groups, grp = lb / tiles / chunks % g.groups;
  const int j0 = chunk * ch_per_block, nch = min(ch_per_block, cpg - j0), steps = ceil_div(nch, CH);

  for (int e = threadIdx.x; e < 2 * plane_bytes / 16; e += blockDim.x) reinterpret_cast<uint4*>(pl_lds)[e] = make_uint4(0u, 0u, 0u, 0u);
  // weight of tap t and channel j: the scope tile read bilinearly at the tap's own place (K.cu:51-83, 338-341)
  bool finite = true;
  for (int e = threadIdx.x; e < steps * K9 * CH; e += blockDim.x) {
    const int j = e / (K9 * CH) * CH + e % CH, t = e / CH % K9;
    const float h = scope_coord<float>(g, t / 3, 0.f, g.centre_h), w = scope_coord<float>(g, t % 3, 0.f, g.centre_w);
    const bool in = j < nch && h > -1.f && w > -1.f && h < float(g.scope_h) && w < float(g.scope_w);
    const int i = (int)floorf(h), k = (int)floorf(w);
    const float lh = h - float(i), lw = w - float(k);
    const T* f = filter + (size_t)(grp + g.groups * (j0 + min(j, nch - 1))) * (g.scope_h * g.scope_w);
    auto at = [&](int a, int b) { return in && a >= 0 && a < g.scope_h && b >= 0 && b < g.scope_w ? ld(f + a * g.scope_w + b) : 0.f; };
    const float tl = at(i, k), tr = at(i, k + 1), bl = at(i + 1, k), br = at(i + 1, k + 1);
    const float v = fmaf(lh, fmaf(lw, (br - tr) - (bl - tl), bl - tl), fmaf(lw, tr - tl, tl));
    wts[e] = in ? v : 0.f;
    finite = finite && fabsf(v) < __builtin_inff();
  }

  const int p = tile * (int)blockDim.x + threadIdx.x;
  const bool live = p < out_plane;
  // where tap t of the lane's pixel samples the image (K.cu:486-499): tap position plus the learned offset
  const rsrc_t roff = plane_rsrc(off + (size_t)n * (K9 * 2) * out_plane, K9 * 2 * out_plane);
  const int pc = live ? p : 0, oh = pc / g.out_w, ow = pc % g.out_w;
  auto sample = [&](int t, float& h, float& w) {
    const unsigned o = live ? (unsigned)((2 * t) * out_plane + pc) * (unsigned)sizeof(T) : kOutOfRange;
    h = float(oh * g.stride_h - g.pad_h + t / 3 * g.dil_h) + buf_ld(roff, o, off);
    w = float(ow * g.stride_w - g.pad_w + t % 3 * g.dil_w) + buf_ld(roff, o + (unsigned)out_plane * (unsigned)sizeof(T), off);
    return live && (h > -1.f) && (w > -1.f) && (h < float(H)) && (w < float(W));
  };
  // byte offset of the sample's top-left corner; a tap outside the image: the last column of the top padding row, whose
  // four corners -- that position, the next row's first and last, the one after's first -- are all padding
  int at[K9];
  float lh[GRAD ? 1 : K9], lw[GRAD ? 1 : K9];
  unsigned hits = 0u;
#pragma unroll
  for (int t = 0; t < K9; ++t) {
    float h, w;
    const bool hit = sample(t, h, w);
    const float hf = floorf(h), wf = floorf(w);
    at[t] = hit ? ((static_cast<int>(hf) + 1) * RS + static_cast<int>(wf) + 1) * kPlPos : (W + 1) * kPlPos;
    if constexpr (!GRAD) lh[t] = hit ? h - hf : 0.f, lw[t] = hit ? w - wf : 0.f;
    hits |= hit ? 1u << t : 0u;
  }
  int dst[PASSES];
#pragma unroll
  for (int k = 0; k < PASSES; ++k) {
    const int e = threadIdx.x + k * blockDim.x;
    dst[k] = e < in_plane ? ((e / W + 1) * RS + e % W + 1) * kPlPos : -1;
  }

  const size_t chan0 = (size_t)n * g.channel + grp + (size_t)g.groups * j0;
  const size_t x_step = (size_t)g.groups * in_plane, o_step = (size_t)g.groups * out_plane;
  const T* xp = x + chan0 * in_plane;
  const unsigned ooff = live ? (unsigned)p * (unsigned)sizeof(T) : kOutOfRange;
  // sums of g * w * {bottom - top, right - left, the difference of the two}, which give both slopes
  float sh[GRAD ? K9 : 1], sw[GRAD ? K9 : 1], sx[GRAD ? K9 : 1];
  if constexpr (GRAD) {
#pragma unroll
    for (int t = 0; t < K9; ++t) sh[t] = sw[t] = sx[t] = 0.f;
  }

  PlainStage<T, PASSES> stage;
  stage.load(xp, x_step, min(nch, CH), in_plane);
  const bool masked = __syncthreads_or(!finite);  // (and the zero fill is done)
  stage.store(pl_lds, dst);
  __syncthreads();
  const unsigned row_bytes = (unsigned)RS * kPlPos;

  auto step_of = [&](auto mask_tag, int s) {
    constexpr bool MASK = decltype(mask_tag)::value;
    const char* planes = pl_lds + (s & 1) * plane_bytes;
    const float* wt = wts + s * (K9 * CH);
    const int live_ch = min(CH, nch - s * CH);
    float io[CH];  // the result, or the output gradient
    const T* op = (GRAD ? gout : out) + (chan0 + (size_t)(s * CH) * g.groups) * out_plane;
    const rsrc_t ro = plane_rsrc(op, (int)((live_ch - 1) * o_step) + out_plane);
#pragma unroll
    for (int c = 0; c < CH; ++c) {
      io[c] = 0.f;
      if constexpr (GRAD) {
        const unsigned oc = c < live_ch ? ooff : kOutOfRange;
        io[c] = buf_ld2(ro, oc, min(c, live_ch - 1) * (int)(o_step * sizeof(T)), gout);
      }
    }
#pragma unroll
    for (int t = 0; t < K9; ++t) {
      const char* c0 = planes + at[t];
      const char* c1 = c0 + row_bytes;
      const uint4 a = *reinterpret_cast<const uint4*>(c0), b = *reinterpret_cast<const uint4*>(c0 + kPlPos);
      const uint4 c = *reinterpret_cast<const uint4*>(c1), d = *reinterpret_cast<const uint4*>(c1 + kPlPos);
      float w[CH];
#pragma unroll
      for (int q = 0; q < CH; q += 4) {
        const float4 v = *reinterpret_cast<const float4*>(wt + t * CH + q);
        w[q] = v.x, w[q + 1] = v.y, w[q + 2] = v.z, w[q + 3] = v.w;
      }
      if constexpr (MASK) {
#pragma unroll
        for (int q = 0; q < CH; ++q) w[q] = hits >> t & 1u ? w[q] : 0.f;
      }
      if constexpr (GRAD) {
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const float gw = io[q] * w[q];
          const float down = difference<T>(c, a, q), right = difference<T>(b, a, q);
          const float cross = difference<T>(d, c, q) - right;
          sh[t] = fmaf(gw, down, sh[t]);
          sw[t] = fmaf(gw, right, sw[t]);
          sx[t] = fmaf(gw, cross, sx[t]);
        }
        asm volatile("" : "+v"(sh[t]), "+v"(sw[t]), "+v"(sx[t])::"memory");
      } else {
        float fh = lh[t], fw = lw[t];
        asm volatile("" : "+v"(fh), "+v"(fw));  // (four products per tap, or the compiler keeps all 36)
        const float d11 = fh * fw, d10 = fh - d11, d01 = fw - d11, d00 = (1.f - fh) - d01;  // K.cu:197-226
#pragma unroll
        for (int q = 0; q < CH; ++q)
          io[q] = fmaf(fmaf(element<T>(d, q), d11, fmaf(element<T>(c, q), d10,
                            fmaf(element<T>(b, q), d01, element<T>(a, q) * d00))), w[q], io[q]);
        // (a tap's sums are complete here, or the compiler reads every tap's corners first)
#pragma unroll
        for (int q = 0; q < CH; ++q) asm volatile("" : "+v"(io[q])::"memory");
      }
      __builtin_amdgcn_sched_barrier(0);  // (a tap's 64 bytes of corners at a time)
    }
    if constexpr (!GRAD) {
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (c < live_ch) buf_st(plane_rsrc(op + (size_t)c * o_step, out_plane), ooff, io[c], out);
    }
  };
  for (int s = 0; s < steps; ++s) {
    const bool more = s + 1 < steps;
    if (more) stage.load(xp + (size_t)((s + 1) * CH) * x_step, x_step, min(CH, nch - (s + 1) * CH), in_plane);
    if (masked)
      step_of(std::true_type{}, s);
    else
      step_of(std::false_type{}, s);
    if (more) stage.store(pl_lds + ((s + 1) & 1) * plane_bytes, dst);
    __syncthreads();
  }

  if constexpr (GRAD) {
    if (live) {
      float* base = partial + ((((size_t)grp * chunks + chunk) * g.batch + (size_t)n) * (K9 * 2)) * out_plane + p;
#pragma unroll
      for (int t = 0; t < K9; ++t) {
        float h, w;  // (read again: eighteen registers fewer in the loop)
        const bool hit = sample(t, h, w);
        base[(size_t)(2 * t) * out_plane] = hit ? fmaf(w - floorf(w), sx[t], sh[t]) : 0.f;
        base[(size_t)(2 * t + 1) * out_plane] = hit ? fmaf(h - floorf(h), sx[t], sw[t]) : 0.f;
      }
    }
  }
}

struct PlainPlan {
  bool ok;
  int tiles, chunks, per, block, passes;
  size_t lds;
};

// Launch shape; ok where two buffers of padded planes and a chunk's weights fit a CU's LDS and the plane is staged in at
// most four passes.  Tiles of equal numbers of waves: up to eight per workgroup where two workgroups' planes fit a CU
// (one stages while the other computes), else up to sixteen.  Channels in chunks that give about fourteen waves per
// CU, of at least two steps.
template <typename T>
PlainPlan plain_plan(const Geo& g) {
  PlainPlan m{};
  m.ok = false;
  if (path_disabled(kNoDeformFast) || path_disabled(kNoDeformPlain) || g.k_h != 3 || g.k_w != 3) return m;
  constexpr int CH = kPlCh<T>;
  const long in_plane = (long)g.in_h * g.in_w, out_plane = (long)g.out_h * g.out_w;
  if (in_plane > 8192 || out_plane > (1L << 24) || CH * (long)g.groups * std::max(in_plane, out_plane) * (long)sizeof(T) >= (1L << 31)) return m;
  if (g.scope_h != g.scope_w || g.scope_h < 3 || g.scope_h > 5) return m;  // as dk_deform_fast.hip's
  const int cpg = g.channel / g.groups;
  const long planes = 2L * (g.in_h + 2) * (g.in_w + 2) * kPlPos;
  const int waves = (int)((out_plane + 63) / 64), most = planes <= 70 * 1024 ? 8 : 16;
  m.tiles = ceil_div(waves, most);
  m.block = ceil_div(waves, m.tiles) * 64;
  m.passes = (int)((in_plane + m.block - 1) / m.block);
  if (m.passes > 4) {  // a small output plane of a large input plane: threads that only stage
    m.block = (int)std::min<long>(kPlThreads, (in_plane + 255) / 256 * 64);
    m.tiles = (int)((out_plane + m.block - 1) / m.block);
    m.passes = (int)((in_plane + m.block - 1) / m.block);
    if (m.passes > 4) return m;
  }
  const long base = std::max(1L, (long)m.tiles * g.batch * g.groups);  // batch may be 0
  const long room = (kPlLds - planes) / (K9 * (long)sizeof(float)) / CH * CH;
  if (room < CH) return m;
  const long waves_all = base * ceil_div(waves, m.tiles);
  const int want = (int)std::min<long>(std::max(1L, (14 * 256 + waves_all - 1) / waves_all), std::max(1, cpg / (2 * CH)));
  m.per = (int)std::min<long>(room, ceil_div(ceil_div(cpg, want), CH) * CH);
  m.chunks = ceil_div(cpg, m.per);
  m.lds = (size_t)(planes + (long)m.per * K9 * 4);
  if ((long)m.chunks * base >= (1L << 31) - 8) return m;
  m.ok = true;
  return m;
}

template <typename T, bool GRAD>
bool launch_plain(const Geo& g, const PlainPlan& m, const T* gout, const T* x, const T* off, const T* filter, T* out,
                  float* partial, hipStream_t stream) {
  auto kernel = m.passes == 1 ? deform_plain_kernel<T, 1, GRAD> : m.passes == 2 ? deform_plain_kernel<T, 2, GRAD>
              : m.passes == 3 ? deform_plain_kernel<T, 3, GRAD> : deform_plain_kernel<T, 4, GRAD>;
  if (!allow_max_dynamic_lds(reinterpret_cast<const void*>(kernel))) return false;
  kernel<<<(unsigned)xcd_grid_size((long)m.tiles * m.chunks * g.batch * g.groups), m.block, m.lds, stream>>>(
      g, gout, x, off, filter, out, partial, m.tiles, m.chunks, m.per);
  return true;
}

}  // namespace

template <typename T>
bool plain_deform_forward(const Geo& g, const T* x, const T* off, const T* filter, T* out, hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g);
  return m.ok && launch_plain<T, false>(g, m, static_cast<const T*>(nullptr), x, off, filter, out, nullptr, stream);
}

// (whether the call comes with a rotation tensor is not known to a workspace query, nor its element type: the most that
// either needs)
size_t plain_deform_grad_offset_workspace(const Geo& g) {
  const PlainPlan a = plain_plan<float>(g), b = plain_plan<__half>(g);
  const int chunks = std::max(a.ok ? a.chunks : 0, b.ok ? b.chunks : 0);
  return (size_t)chunks * g.groups * g.batch * 18 * g.out_h * g.out_w * sizeof(float);
}

template <typename T>
bool plain_deform_grad_offset(const Geo& g, const T* gout, const T* x, const T* off, const T* filter, T* goff, float* ws,
                              hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g);
  // (eight 16-bit channels in four passes take registers that the sums need, and spill: at stride 2 slower than the kernel with the
  // tables, bfloat16 N=64 C=512 28x28 57 against 53 us; at stride 1, 56x56, still 140 against 209)
  if (sizeof(T) == 2 && m.passes == 4 && 2L * g.out_h * g.out_w < (long)g.in_h * g.in_w) return false;
  if (!m.ok || !launch_plain<T, true>(g, m, gout, x, off, filter, static_cast<T*>(nullptr), ws, stream)) return false;
  launch_reduce_partials<float, T>(ws, m.chunks * g.groups, (long)g.batch * 18 * g.out_h * g.out_w, goff, stream);
  return true;
}

#define DK_INSTANTIATE(T)                                                                                          \
  template bool plain_deform_forward<T>(const Geo&, const T*, const T*, const T*, T*, hipStream_t);                 \
  template bool plain_deform_grad_offset<T>(const Geo&, const T*, const T*, const T*, const T*, T*, float*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
