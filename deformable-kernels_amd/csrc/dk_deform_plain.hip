// Deformable forward, grad offset and grad filter without kernel-space offsets (rotation == NULL: DeformKernelConv2d,
// DeformConv2d).
//
// Reference kernels covered (K.cu =
// deformable_kernels/ops/deform_kernel/csrc/filter_sample_depthwise_cuda_kernel.cu): forward, K.cu:433-528, grad filter,
// K.cu:926-1018, and grad offset, K.cu:1147-1243, where every kernel-space offset is zero.
//
// Each tap then reads the scope tile at one place for all pixels, so a channel has nine weights and no table: what
// dk_deform_fast.hip reads per sample and channel at an address of its own (16 bytes of LDS) is one broadcast read per
// tap and group of channels.  The rest is as there -- a lane owns an output pixel, zero-padded input planes double
// buffered in LDS, interleaved 16 bytes to a position -- except that 16-bit planes stay 16-bit, eight channels to a
// position, and their corners enter the multiply-adds as stored (v_fma_mix_f32 for float16).
// What bounds it now is the vector unit: five (forward) and eight (grad offset) instructions per sample and channel.
// us, with the tables / here: forward and grad offset of N=64 C=192 28x28 float16 90 / 38 and 111 / 45, float32 85 / 46 and
// 94 / 52; C=144 56x56 float32 179 / 143 and 215 / 169; N=128 C=960 7x7 float16 150 / 28 and 188 / 40 (a chunk of channels
// per wave there: the tables' kernel fills 49 of 256 lanes).  Grad offset and grad filter, in two passes with the filter's on the
// matrix cores / in one here: N=64 C=192 28x28 float32 138 / 77, float16 132 / 76; C=144 56x56 float32 487 / 210, float16
// 869 / 229; C=512 28x28 at stride 2 float32 105 / 66, bfloat16 110 / 83; N=64 C=960 7x7 79 / 44.
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

// kPlCh<T> planes on their way to LDS, or HALVES = 2: half of them at a time; element e of the planes for
// e = thread, thread + block, ...
template <typename T, int PASSES, int HALVES>
struct PlainStage {
  static constexpr int CH = kPlCh<T> / HALVES;
  unsigned v[CH][PASSES];
  __device__ __forceinline__ void load(const T* plane0, size_t step, int live, int in_plane, int half = 0) {
    const rsrc_t r = plane_rsrc(plane0, (int)((live - 1) * step) + in_plane);
    const int bytes = (int)(step * sizeof(T));
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      const int e = threadIdx.x + k * blockDim.x;
      const unsigned o = e < in_plane ? (unsigned)e * (unsigned)sizeof(T) : kOutOfRange;
#pragma unroll
      for (int i = 0; i < CH; ++i) {
        // (the scalar part stays inside the buffer; a channel past the last one reads as zeros)
        const int c = half * CH + i, s = min(c, live - 1) * bytes;
        const unsigned at = c < live ? o : kOutOfRange;
        if constexpr (sizeof(T) == 4)
          v[i][k] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)at, s, 0);
        else
          v[i][k] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)at, s, 0);
      }
    }
  }
  __device__ __forceinline__ void store(char* planes, const int (&dst)[PASSES], int half = 0) const {
#pragma unroll
    for (int k = 0; k < PASSES; ++k) {
      if (dst[k] < 0) continue;
      unsigned q[4 / HALVES];
#pragma unroll
      for (int i = 0; i < 4 / HALVES; ++i) {
        if constexpr (sizeof(T) == 4)
          q[i] = v[i][k];
        else
          q[i] = v[2 * i][k] | v[2 * i + 1][k] << 16;
      }
      if constexpr (HALVES == 1)
        *reinterpret_cast<uint4*>(planes + dst[k]) = make_uint4(q[0], q[1], q[2], q[3]);
      else
        *reinterpret_cast<uint2*>(planes + dst[k] + half * (kPlPos / 2)) = make_uint2(q[0], q[1]);
    }
  }
};

// The sums of v[0 .. CH - 1] over the wave, of channel q in the lanes q * (64 / CH) and on.  Exchanging halves, each step
// leaves half the registers: 17 instructions for eight channels (14 and three), where a sum by itself takes six.
template <int CH>
__device__ __forceinline__ float wave_sums(const float (&v)[CH]) {
  auto add = [](unsigned a, unsigned b) { return __builtin_bit_cast(unsigned, __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b)); };
  auto dpp_add = [&](unsigned a, auto ctrl) {
    return add(a, (unsigned)__builtin_amdgcn_update_dpp(0, (int)a, decltype(ctrl)::value, 0xf, 0xf, true));
  };
  unsigned h[CH / 2];
#pragma unroll
  for (int q = 0; q < CH / 2; ++q) {  // lanes 32 .. 63 go on with channels CH / 2 .. CH - 1
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, v[q]), __builtin_bit_cast(unsigned, v[q + CH / 2]), false, false);
    h[q] = add(r[0], r[1]);
  }
  unsigned k[CH / 4];
#pragma unroll
  for (int q = 0; q < CH / 4; ++q) {
    const auto r = __builtin_amdgcn_permlane16_swap(h[q], h[q + CH / 4], false, false);
    k[q] = add(r[0], r[1]);
  }
  unsigned s;
  if constexpr (CH == 8) {
    const bool up = threadIdx.x & 8;
    const unsigned keep = up ? k[1] : k[0], give = up ? k[0] : k[1];
    s = add(keep, (unsigned)__builtin_amdgcn_update_dpp(0, (int)give, 0x128 /* row_ror:8 */, 0xf, 0xf, true));
  } else {
    s = dpp_add(k[0], std::integral_constant<int, 0x128>{});
  }
  s = dpp_add(s, std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  s = dpp_add(s, std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  s = dpp_add(s, std::integral_constant<int, 0x141>{});  // row_half_mirror
  return __builtin_bit_cast(float, s);
}

// What a pass over the samples forms.  Without kernel-space offsets a tap's place in the scope tile is the same for all
// pixels, so the filter's gradient needs nine sums per channel, G_t[c] = sum over the pixels of out_grad * sample
// (plain_filter_cells_kernel spreads them over the cells), and not the products with a hat function per sample and cell.
enum PlainMode { kPlForward, kPlOffset, kPlFilter, kPlBoth };

// One workgroup per (pixel tile, channel chunk, image, group), a lane per pixel of the tile, the chunk's channels kPlCh<T>
// at a time.  Grad offset: partial[group][chunk][image][18][pixel] in fp32.  Grad filter: taps[image][tile][channel][9] in
// fp32, summed over a wave's lanes per step (wave_sums), then over the waves in their order.  kPlBoth forms the two from
// one read of the corners.
// A weight that is not finite must not meet the zeros that stand for a tap outside the image (the reference skips such
// taps): a chunk that holds one masks the weights of those taps.
// Registers: 1024 threads leave 128 of them.  Instances that spill, bytes per lane for one to four staging passes (they hold
// the next channels' planes): both gradients float16 0, 0, 48, 84, bfloat16 0, 8, 56, 96; grad offset alone bfloat16 0, 36,
// 24, 60, float32 in four passes 16; forward bfloat16 in four passes 20.
template <typename T, int PASSES, PlainMode MODE>
__global__ __launch_bounds__(kPlThreads) void deform_plain_kernel(
    Geo g, const T* __restrict__ gout, const T* __restrict__ x, const T* __restrict__ off, const T* __restrict__ filter,
    T* __restrict__ out, float* __restrict__ partial, float* __restrict__ taps, int tiles, int chunks, int ch_per_block) {
  constexpr int CH = kPlCh<T>;
  constexpr bool GRAD = MODE != kPlForward, OFFSET = MODE == kPlOffset || MODE == kPlBoth, FILTER = MODE == kPlFilter || MODE == kPlBoth;
  constexpr bool PLACE = MODE != kPlOffset;  // lh and lw are needed per channel
  extern __shared__ __align__(16) char pl_lds[];
  const int H = g.in_h, W = g.in_w, RS = W + 2;
  const int plane_bytes = (H + 2) * RS * kPlPos;
  float* wts = reinterpret_cast<float*>(pl_lds + 2 * plane_bytes);  // [channels / CH][K9][CH]
  float* red = wts + ch_per_block * K9;                             // FILTER: the same per wave

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
  for (int e = threadIdx.x; MODE != kPlFilter && e < steps * K9 * CH; e += blockDim.x) {
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
  float lh[PLACE ? K9 : 1], lw[PLACE ? K9 : 1];
  unsigned hits = 0u;
#pragma unroll
  for (int t = 0; t < K9; ++t) {
    float h, w;
    const bool hit = sample(t, h, w);
    const float hf = floorf(h), wf = floorf(w);
    at[t] = hit ? ((static_cast<int>(hf) + 1) * RS + static_cast<int>(wf) + 1) * kPlPos : (W + 1) * kPlPos;
    if constexpr (PLACE) lh[t] = hit ? h - hf : 0.f, lw[t] = hit ? w - wf : 0.f;
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
  // sums of g * w * {bottom - top, right - left, the difference of the two}, which give both slopes; kPlBoth, which has the
  // sample's place at hand: of the slopes themselves (nine registers fewer)
  float sh[OFFSET ? K9 : 1], sw[OFFSET ? K9 : 1], sx[OFFSET ? K9 : 1];
  if constexpr (OFFSET) {
#pragma unroll
    for (int t = 0; t < K9; ++t) sh[t] = sw[t] = sx[t] = 0.f;
  }

  // (kPlBoth: the next step's planes by halves, eight registers fewer; the second half is asked for in mid-step)
  // (and grad offset alone where eight 16-bit planes take 24 or 32 registers)
  constexpr int HALVES = MODE == kPlBoth || (MODE == kPlOffset && CH == 8 && PASSES > 2) ? 2 : 1;
  PlainStage<T, PASSES, HALVES> stage;
  stage.load(xp, x_step, min(nch, CH), in_plane);
  const bool masked = __syncthreads_or(!finite);  // (and the zero fill is done)
  stage.store(pl_lds, dst);
  if constexpr (HALVES == 2) {
    stage.load(xp, x_step, min(nch, CH), in_plane, 1);
    stage.store(pl_lds, dst, 1);
  }
  __syncthreads();
  const unsigned row_bytes = (unsigned)RS * kPlPos;

  auto load_io = [&](float (&io)[CH], int s) {  // the step's output gradients
    const int live_ch = min(CH, nch - s * CH);
    const rsrc_t ro = plane_rsrc(gout + (chan0 + (size_t)(s * CH) * g.groups) * out_plane, (int)((live_ch - 1) * o_step) + out_plane);
#pragma unroll
    for (int c = 0; c < CH; ++c)
      io[c] = buf_ld2(ro, c < live_ch ? ooff : kOutOfRange, min(c, live_ch - 1) * (int)(o_step * sizeof(T)), gout);
  };
  // (grad offset alone loads its output gradients here into an array of its own: through the caller's array the bfloat16 instances of
  // one and two passes are scheduled 8 - 15 % slower, N=128 C=576 14x14 68 -> 78 us, N=128 C=192 28x28 80 -> 88)
  auto step_of = [&](auto mask_tag, int s, float (&outer)[CH]) {
    float own[CH];
    if constexpr (MODE == kPlOffset) load_io(own, s);
    float (&io)[CH] = *(MODE == kPlOffset ? &own : &outer);
    constexpr bool MASK = decltype(mask_tag)::value;  // a tap outside the image may meet a weight or a gradient that is not finite
    const char* planes = pl_lds + (s & 1) * plane_bytes;
    const float* wt = wts + s * (K9 * CH);
    float* sums = red + (threadIdx.x >> 6) * (ch_per_block * K9) + s * (K9 * CH) + (threadIdx.x & 63) / (64 / CH);
#pragma unroll
    for (int t = 0; t < K9; ++t) {
      if constexpr (HALVES == 2) {
        if (t == K9 / 2 && s + 1 < steps) {
          stage.store(pl_lds + ((s + 1) & 1) * plane_bytes, dst);
          stage.load(xp + (size_t)((s + 1) * CH) * x_step, x_step, min(CH, nch - (s + 1) * CH), in_plane, 1);
        }
      }
      const char* c0 = planes + at[t];
      const char* c1 = c0 + row_bytes;
      const uint4 a = *reinterpret_cast<const uint4*>(c0), b = *reinterpret_cast<const uint4*>(c0 + kPlPos);
      const uint4 c = *reinterpret_cast<const uint4*>(c1), d = *reinterpret_cast<const uint4*>(c1 + kPlPos);
      float w[CH];
      if constexpr (MODE != kPlFilter) {
#pragma unroll
        for (int q = 0; q < CH; q += 4) {
          const float4 v = *reinterpret_cast<const float4*>(wt + t * CH + q);
          w[q] = v.x, w[q + 1] = v.y, w[q + 2] = v.z, w[q + 3] = v.w;
        }
      }
      const bool skip = MASK && !(hits >> t & 1u);
      if constexpr (MASK && MODE != kPlFilter) {
#pragma unroll
        for (int q = 0; q < CH; ++q) w[q] = skip ? 0.f : w[q];
      }
      if constexpr (MODE == kPlOffset) {
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const float gw = io[q] * w[q];
          const float down = difference<T>(c, a, q), right = difference<T>(b, a, q);
          const float cross = difference<T>(d, c, q) - right;
          sh[t] = fmaf(gw, down, sh[t]);
          sw[t] = fmaf(gw, right, sw[t]);
          sx[t] = fmaf(gw, cross, sx[t]);
          // (a channel at a time, or the differences of all eight stay alive)
          if constexpr (std::is_same<T, __half>::value) asm volatile("" : "+v"(sh[t]), "+v"(sw[t]), "+v"(sx[t]));
        }
        asm volatile("" : "+v"(sh[t]), "+v"(sw[t]), "+v"(sx[t])::"memory");
      } else if constexpr (MODE == kPlBoth) {
        float v[CH];
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const float gw = io[q] * w[q];
          const float down = difference<T>(c, a, q), right = difference<T>(b, a, q);
          const float cross = difference<T>(d, c, q) - right;
          const float slope_h = fmaf(lw[t], cross, down), slope_w = fmaf(lh[t], cross, right);
          sh[t] = fmaf(gw, slope_h, sh[t]);
          sw[t] = fmaf(gw, slope_w, sw[t]);
          v[q] = io[q] * fmaf(lh[t], slope_h, fmaf(lw[t], right, element<T>(a, q)));
          if constexpr (MASK) v[q] = skip ? 0.f : v[q];
          asm volatile("" : "+v"(v[q]), "+v"(sh[t]), "+v"(sw[t]));  // (as above)
        }
        const float sum = wave_sums<CH>(v);
        if ((threadIdx.x & (64 / CH - 1)) == 0) sums[t * CH] = sum;
        asm volatile("" : "+v"(sh[t]), "+v"(sw[t])::"memory");
      } else {
        float fh = lh[t], fw = lw[t];
        asm volatile("" : "+v"(fh), "+v"(fw));  // (four products per tap, or the compiler keeps all 36)
        const float d11 = fh * fw, d10 = fh - d11, d01 = fw - d11, d00 = (1.f - fh) - d01;  // K.cu:197-226
        float v[CH];
#pragma unroll
        for (int q = 0; q < CH; ++q) {
          const float at_q = fmaf(element<T>(d, q), d11, fmaf(element<T>(c, q), d10,
                                  fmaf(element<T>(b, q), d01, element<T>(a, q) * d00)));
          if constexpr (FILTER)
            v[q] = skip ? 0.f : io[q] * at_q;
          else
            io[q] = fmaf(at_q, w[q], io[q]);
        }
        if constexpr (FILTER) {
          const float sum = wave_sums<CH>(v);
          if ((threadIdx.x & (64 / CH - 1)) == 0) sums[t * CH] = sum;
          asm volatile("" ::: "memory");
        } else {
          // (a tap's sums are complete here, or the compiler reads every tap's corners first)
#pragma unroll
          for (int q = 0; q < CH; ++q) asm volatile("" : "+v"(io[q])::"memory");
        }
      }
      __builtin_amdgcn_sched_barrier(0);  // (a tap's 64 bytes of corners at a time)
    }
    if constexpr (!GRAD) {
      const int live_ch = min(CH, nch - s * CH);
      T* op = out + (chan0 + (size_t)(s * CH) * g.groups) * out_plane;
#pragma unroll
      for (int c = 0; c < CH; ++c)
        if (c < live_ch) buf_st(plane_rsrc(op + (size_t)c * o_step, out_plane), ooff, io[c], out);
    }
  };
  for (int s = 0; s < steps; ++s) {
    const bool more = s + 1 < steps;
    if (more) stage.load(xp + (size_t)((s + 1) * CH) * x_step, x_step, min(CH, nch - (s + 1) * CH), in_plane);
    float io[CH];  // the result, or the output gradient
    bool mask = masked;
    if constexpr (FILTER) {
      load_io(io, s);
      float z = 0.f;  // NaN where one of them is not finite
#pragma unroll
      for (int c = 0; c < CH; ++c) z = fmaf(io[c], 0.f, z);
      mask = masked || __any(z != 0.f);
    } else if constexpr (!GRAD) {
#pragma unroll
      for (int c = 0; c < CH; ++c) io[c] = 0.f;
    }
    if (mask)
      step_of(std::true_type{}, s, io);
    else
      step_of(std::false_type{}, s, io);
    if (more) stage.store(pl_lds + ((s + 1) & 1) * plane_bytes, dst, HALVES - 1);
    __syncthreads();
  }

  if constexpr (OFFSET) {
    if (live) {
      float* base = partial + ((((size_t)grp * chunks + chunk) * g.batch + (size_t)n) * (K9 * 2)) * out_plane + p;
#pragma unroll
      for (int t = 0; t < K9; ++t) {
        if constexpr (MODE == kPlBoth) {
          const bool hit = hits >> t & 1u;
          base[(size_t)(2 * t) * out_plane] = hit ? sh[t] : 0.f;
          base[(size_t)(2 * t + 1) * out_plane] = hit ? sw[t] : 0.f;
        } else {
          float h, w;  // (read again: eighteen registers fewer in the loop)
          const bool hit = sample(t, h, w);
          base[(size_t)(2 * t) * out_plane] = hit ? fmaf(w - floorf(w), sx[t], sh[t]) : 0.f;
          base[(size_t)(2 * t + 1) * out_plane] = hit ? fmaf(h - floorf(h), sx[t], sw[t]) : 0.f;
        }
      }
    }
  }
  if constexpr (FILTER) {  // (the loop ends with a barrier)
    float* dst = taps + ((size_t)n * tiles + tile) * g.channel * K9;
    for (int e = threadIdx.x; e < nch * K9; e += blockDim.x) {
      const int j = e / K9, t = e % K9;
      const float* src = red + (j / CH * K9 + t) * CH + j % CH;
      float v = 0.f;
      for (int w = 0; w < (int)(blockDim.x >> 6); ++w) v += src[w * (ch_per_block * K9)];
      dst[(grp + g.groups * (j0 + j)) * K9 + t] = v;
    }
  }
}

// Filter gradient from the taps' sums: taps[row][channel][9], rows summed in order; a cell receives each tap that reads it
// times the tap's bilinear weight of it (K.cu:85-145).  A workgroup per kCellCh channels; kCellSlices threads share a
// column's rows.  N=64 C=192 28x28 (128 rows of 1728 sums): 4.7 us, with seven threads to a column 8.4.
constexpr int kCellCh = 4, kCellSlices = 28, kCellBlock = 1024;
template <typename T>
__global__ __launch_bounds__(kCellBlock) void plain_filter_cells_kernel(Geo g, const float* __restrict__ taps, int rows, T* __restrict__ gfilter) {
  constexpr int COLS = kCellCh * K9;
  __shared__ float part[kCellSlices][COLS];
  const int c0 = blockIdx.x * kCellCh, cols = min(kCellCh, g.channel - c0) * K9;
  const int slice = threadIdx.x / COLS, col = threadIdx.x % COLS;
  if (slice < kCellSlices && col < cols) {
    const float* src = taps + (size_t)c0 * K9 + col;
    const size_t pitch = (size_t)g.channel * K9;
    float v = 0.f;
#pragma unroll 4
    for (int r = slice; r < rows; r += kCellSlices) v += src[(size_t)r * pitch];
    part[slice][col] = v;
  }
  __syncthreads();
  if (threadIdx.x < cols) {
    float v = 0.f;
    for (int s = 0; s < kCellSlices; ++s) v += part[s][threadIdx.x];
    part[0][threadIdx.x] = v;
  }
  __syncthreads();
  const int cells = g.scope_h * g.scope_w;
  for (int e = threadIdx.x; e < cols / K9 * cells; e += blockDim.x) {
    const int a = e % cells / g.scope_w, b = e % cells % g.scope_w;
    float v = 0.f;
    for (int t = 0; t < K9; ++t) {
      const float h = scope_coord<float>(g, t / 3, 0.f, g.centre_h), w = scope_coord<float>(g, t % 3, 0.f, g.centre_w);
      if (!(h > -1.f && w > -1.f && h < float(g.scope_h) && w < float(g.scope_w))) continue;
      const int i = (int)floorf(h), k = (int)floorf(w);
      if ((a != i && a != i + 1) || (b != k && b != k + 1)) continue;
      const float lh = h - float(i), lw = w - float(k);
      v = fmaf((a == i ? 1.f - lh : lh) * (b == k ? 1.f - lw : lw), part[0][e / cells * K9 + t], v);
    }
    st(gfilter + (size_t)c0 * cells + e, v);
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
PlainPlan plain_plan(const Geo& g, PlainMode mode) {
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
  // floats of LDS per channel and tap: the weight and, of the filter's gradient, a sum per wave
  const int words = mode == kPlFilter || mode == kPlBoth ? 1 + m.block / 64 : 1;
  const long room = (kPlLds - planes) / (K9 * (long)sizeof(float) * words) / CH * CH;
  if (room < CH) return m;
  const long waves_all = base * ceil_div(waves, m.tiles);
  const int want = (int)std::min<long>(std::max(1L, (14 * 256 + waves_all - 1) / waves_all), std::max(1, cpg / (2 * CH)));
  m.per = (int)std::min<long>(room, ceil_div(ceil_div(cpg, want), CH) * CH);
  m.chunks = ceil_div(cpg, m.per);
  m.lds = (size_t)(planes + (long)m.per * K9 * 4 * words);
  if ((long)m.chunks * base >= (1L << 31) - 8) return m;
  m.ok = true;
  return m;
}

template <typename T, PlainMode MODE>
bool launch_plain(const Geo& g, const PlainPlan& m, const T* gout, const T* x, const T* off, const T* filter, T* out,
                  float* partial, float* taps, hipStream_t stream) {
  auto kernel = m.passes == 1 ? deform_plain_kernel<T, 1, MODE> : m.passes == 2 ? deform_plain_kernel<T, 2, MODE>
              : m.passes == 3 ? deform_plain_kernel<T, 3, MODE> : deform_plain_kernel<T, 4, MODE>;
  if (!allow_max_dynamic_lds(reinterpret_cast<const void*>(kernel))) return false;
  kernel<<<(unsigned)xcd_grid_size((long)m.tiles * m.chunks * g.batch * g.groups), m.block, m.lds, stream>>>(
      g, gout, x, off, filter, out, partial, taps, m.tiles, m.chunks, m.per);
  return true;
}

// The most bytes that the offsets' partial sums and the taps' take in either element size (which a workspace query for a
// geometry does not know, nor whether the call comes with a rotation tensor)
size_t offset_bytes(const Geo& g, PlainMode mode) {
  const PlainPlan a = plain_plan<float>(g, mode), b = plain_plan<__half>(g, mode);
  const int chunks = std::max(a.ok ? a.chunks : 0, b.ok ? b.chunks : 0);
  return (size_t)chunks * g.groups * g.batch * 18 * g.out_h * g.out_w * sizeof(float);
}
size_t taps_bytes(const Geo& g, PlainMode mode) {
  const PlainPlan a = plain_plan<float>(g, mode), b = plain_plan<__half>(g, mode);
  const int tiles = std::max(a.ok ? a.tiles : 0, b.ok ? b.tiles : 0);
  return (size_t)g.batch * tiles * g.channel * K9 * sizeof(float);
}

template <typename T>
void launch_cells(const Geo& g, const PlainPlan& m, const float* taps, T* gfilter, hipStream_t stream) {
  plain_filter_cells_kernel<T><<<ceil_div(g.channel, kCellCh), kCellBlock, 0, stream>>>(g, taps, g.batch * m.tiles, gfilter);
}

// (eight 16-bit channels in four passes take registers that the sums need: grad offset alone at stride 2 slower than the
// kernel with the tables, bfloat16 N=64 C=512 28x28 57 against 53 us; at stride 1, 56x56, 140 against 209)
template <typename T>
bool offset_spills(const Geo& g, const PlainPlan& m) {
  return sizeof(T) == 2 && m.passes == 4 && 2L * g.out_h * g.out_w < (long)g.in_h * g.in_w;
}

}  // namespace

template <typename T>
bool plain_deform_forward(const Geo& g, const T* x, const T* off, const T* filter, T* out, hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g, kPlForward);
  return m.ok && launch_plain<T, kPlForward>(g, m, static_cast<const T*>(nullptr), x, off, filter, out, nullptr, nullptr, stream);
}

size_t plain_deform_grad_offset_workspace(const Geo& g) { return offset_bytes(g, kPlOffset); }

template <typename T>
bool plain_deform_grad_offset(const Geo& g, const T* gout, const T* x, const T* off, const T* filter, T* goff, float* ws,
                              hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g, kPlOffset);
  if (!m.ok || offset_spills<T>(g, m)) return false;
  if (!launch_plain<T, kPlOffset>(g, m, gout, x, off, filter, static_cast<T*>(nullptr), ws, nullptr, stream)) return false;
  launch_reduce_partials<float, T>(ws, m.chunks * g.groups, (long)g.batch * 18 * g.out_h * g.out_w, goff, stream);
  return true;
}

size_t plain_deform_grad_filter_workspace(const Geo& g) { return taps_bytes(g, kPlFilter); }

template <typename T>
bool plain_deform_grad_filter(const Geo& g, const T* gout, const T* x, const T* off, T* gfilter, float* ws, hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g, kPlFilter);
  if (!m.ok || !launch_plain<T, kPlFilter>(g, m, gout, x, off, static_cast<const T*>(nullptr), static_cast<T*>(nullptr), nullptr, ws, stream))
    return false;
  launch_cells<T>(g, m, ws, gfilter, stream);
  return true;
}

size_t plain_deform_grad_offset_filter_workspace(const Geo& g) { return offset_bytes(g, kPlBoth) + taps_bytes(g, kPlBoth); }

template <typename T>
bool plain_deform_grad_offset_filter(const Geo& g, const T* gout, const T* x, const T* off, const T* filter, T* goff,
                                     T* gfilter, float* ws, hipStream_t stream) {
  const PlainPlan m = plain_plan<T>(g, kPlBoth);
  if (!m.ok) return false;
  float* taps = ws + (size_t)m.chunks * g.groups * g.batch * 18 * g.out_h * g.out_w;
  if (!launch_plain<T, kPlBoth>(g, m, gout, x, off, filter, static_cast<T*>(nullptr), ws, taps, stream)) return false;
  launch_reduce_partials<float, T>(ws, m.chunks * g.groups, (long)g.batch * 18 * g.out_h * g.out_w, goff, stream);
  launch_cells<T>(g, m, taps, gfilter, stream);
  return true;
}

#define DK_INSTANTIATE(T)                                                                                          \
  template bool plain_deform_forward<T>(const Geo&, const T*, const T*, const T*, T*, hipStream_t);                 \
  template bool plain_deform_grad_offset<T>(const Geo&, const T*, const T*, const T*, const T*, T*, float*, hipStream_t); \
  template bool plain_deform_grad_filter<T>(const Geo&, const T*, const T*, const T*, T*, float*, hipStream_t);      \
  template bool plain_deform_grad_offset_filter<T>(const Geo&, const T*, const T*, const T*, const T*, T*, T*, float*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
