// Deformable grad input with the lanes along the CHANNELS (dk_deform_fast.hip holds the forms with a pixel per lane).
//
// Reference kernel covered (K.cu =
// deformable_kernels/ops/deform_kernel/csrc/filter_sample_depthwise_cuda_kernel.cu): grad input, K.cu:704-795.
//
// What bounds the scatter with a pixel per lane is LDS: 36 fixed-point adds per output pixel and channel pair, whose
// targets are spread over the plane, and a 64-bit LDS add of a wave then takes 6.3 ns of the CU's LDS pipe (measured,
// 16 waves per CU; bank conflicts); where 16 consecutive lanes add to 16 consecutive 64-bit words it takes 3.0 ns.  So here an input position holds the sums of 32 channels side by side, 16 pairs of signed 32-bit sums in
// 64-bit words (b * 2^32 + a, as in deform_grad_input_kernel), and a row of 16 lanes adds one sample of all 32
// channels: lane n owns channels 2 n and 2 n + 1, the wave's four rows take four pixels at a time.  What depends on
// (pixel, tap) only -- the target, the scope cell, the corner weights -- is computed once per sample by one of the
// row's lanes and reaches the others as a DPP operand (row_newbcast) of the arithmetic that uses it.  The scope
// tables are laid out the same way, [cell][channel], so that their 16-byte reads are free of bank conflicts too.
// That leaves the kernel bound by vector instructions (31 per sample of 32 channels and four pixels; LDS busy a third of
// the time).  N=64 C=192 28x28, stride 1: 156 us with a pixel per lane, 108 here (float32), 151 and 101 (float16).
#include <algorithm>
#include <type_traits>

#include "dk_deform.h"
#include "dk_kernels.h"

namespace dk {

namespace {

constexpr int kLnBlock = 1024, kLnWaves = kLnBlock / 64;
constexpr int kLnCh = 32, kLnPairs = kLnCh / 2;  // channels of a workgroup, a pair per lane of a row
constexpr int kLnPix = 16;                       // output pixels of a wave's unit: four per row of lanes
// 64-bit words per position: the pairs, and one more so that positions next to each other start on different banks
// (the read-back of a pair walks the positions, lane by lane); it holds the number of samples added to the position
constexpr int kLnPitch = kLnPairs + 1;
constexpr int kLnLds = 160 * 1024 - 512;  // dynamic LDS: the kernel's static arrays come out of the same 160 KB

// The value that lane K of the 16-lane row holds
template <int K>
__device__ __forceinline__ int row_lane(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xf, 0xf, true);
}
template <int K>
__device__ __forceinline__ float row_lane(float v) {
  return __builtin_bit_cast(float, row_lane<K>(__builtin_bit_cast(int, v)));
}

// c + (the value of a that lane K of the row holds) * b, rounded once.  (A DPP operand must not have been written by the
// two vector instructions in front: a is written once per unit of work, far ahead.)
template <int K>
__device__ __forceinline__ double fma_row_lane(double a, double b, double c) {
  asm("v_fmac_f64_dpp %0, %1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf" : "+v"(c) : "v"(a), "v"(b), "n"(K));
  return c;
}
// 1.5 * 2^52: what a double of that size has in its low mantissa bits is a rounded integer; and with 2^31 more the low
// word of it is the integer plus kBias
constexpr double kMagic = 6755399441055744.0, kMagicBias = kMagic + 2147483648.0;
constexpr unsigned long long kBias = 1ull << 31;

template <int... I, typename F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for(std::make_integer_sequence<int, N>{}, f);
}

// Four consecutive elements as stored, by one wide load where `wide` says that every group of four is aligned
template <typename T>
__device__ __forceinline__ auto load4(rsrc_t r, unsigned off, bool wide, const T* tag) {
  using V = decltype(raw_ld4(r, off, tag));
  if (wide) return raw_ld4(r, off, tag);
  unsigned e[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if constexpr (sizeof(T) == 4)
      e[i] = __builtin_amdgcn_raw_buffer_load_b32(r, (int)(off + 4u * i), 0, 0);
    else
      e[i] = __builtin_amdgcn_raw_buffer_load_b16(r, (int)(off + 2u * i), 0, 0);
  }
  if constexpr (sizeof(T) == 4)
    return V{e[0], e[1], e[2], e[3]};
  else
    return V{e[0] | (e[1] << 16), e[2] | (e[3] << 16)};
}

// LDS positions: the zero-padded plane; of a band: its rows, one more (the last row's right padding), the two spare ones
__host__ __device__ __forceinline__ int lanes_positions(int rows, int w, bool band) {
  return band ? rows * (w + 1) + 3 : (rows + 2) * (w + 1) + 1;
}

// ---------------------------------------------------------------------------
// One workgroup per (image, group, 32 channels); its LDS holds the whole zero-padded plane.  A unit of work is 16 output pixels x one row of
// three taps: 12 samples for each of the wave's four rows of lanes, the waves take units in turn and load the next
// unit's operands before they work on the present one.
// The sums are exact on their grid and independent of the order of the additions; scale, grid and the fallback for
// inputs with more than 2^kPairHead samples on one element are those of deform_grad_input_kernel.
// ---------------------------------------------------------------------------
// PLAIN: no kernel-space offsets (rot is null).  A tap then reads the scope tile at one place for all pixels: nine weights
// per channel, a lane's two of each tap of its unit in registers, instead of two table reads and six multiply-adds per
// sample (N=64 C=192 28x28 float16: 99 -> 82 us).
// BAND: planes whose sums do not fit LDS for 32 channels.  A workgroup owns `band_rows` image rows of its 32 channels and
// walks the units whose samples touch them (BandWalk, dk_deform.h, which also says in which calls); a corner pair in another band's row is added to two spare positions instead, uncounted.  A band of 19
// rows of a 56 x 56 plane meets 61 % of the samples of the 31 - 36 rows it walks; N=64 C=144 56x56 float32, all kernels of
// the gradient: 428 us with eight channels per workgroup and a pixel per lane (deform_grad_input_tiled_kernel, whose
// descriptors alone take 100 vector instructions per sample and eight channels), 342 here; without a rotation tensor 417 and
// 276, bfloat16 N=32 262 and 185.
template <typename T, int SH, int SW, bool PLAIN, bool BAND>
__global__ __launch_bounds__(kLnBlock) void deform_grad_input_lanes_kernel(
    Geo g, const T* __restrict__ gout, const T* __restrict__ off, const T* __restrict__ rot,
    const T* __restrict__ filter, T* __restrict__ gin, const unsigned* __restrict__ gmax_bits, unsigned inv_out_w,
    unsigned inv_in_w, int wide, BandWalk by_bands, const int2* __restrict__ unit_rows) {
  constexpr int CELLS = (SH + 1) * (SW + 1);
  extern __shared__ __align__(16) unsigned long long sums[];  // [positions][kLnPitch], then the tables
  const int H = g.in_h, W = g.in_w, RS = W + 1;               // one padding column between two rows serves both
  const int band_rows = by_bands.rows;
  const int npos = lanes_positions(BAND ? band_rows : H, W, BAND);
  float4* tbl = reinterpret_cast<float4*>(sums + ((npos * kLnPitch + 1) & ~1));  // [CELLS][2][kLnPairs]
  __shared__ float wmax[kLnCh];
  __shared__ unsigned wave_most[kLnWaves];
  __shared__ float unscale32[kLnCh];

  const int cpg = g.channel / g.groups;
  const int out_plane = g.out_h * g.out_w, in_plane = H * W;
  const int bands = BAND ? ceil_div(H, band_rows) : 1;
  const int chunks = ceil_div(cpg, kLnCh), total = bands * chunks * g.batch * g.groups;
  const int lb = logical_block(total);
  if (lb >= total) return;
  const int chunk = lb % chunks, band = lb / chunks % bands, z = lb / chunks / bands;
  // image rows r_lo .. r_hi - 1 are this workgroup's; image row r sits in LDS row r + row0
  const int r_lo = band * band_rows, r_hi = BAND ? min(H, r_lo + band_rows) : H;
  const int row0 = BAND ? -r_lo : 1;
  const int spare = BAND ? band_rows * RS + 1 : 0;  // position of what is no sample of these rows (not BAND: the padding row on top)
  const int n = z / g.groups, grp = z % g.groups;
  if (BAND && by_bands.met && !bands_take(by_bands)) return;
  const int j0 = chunk * kLnCh, nch = min(kLnCh, cpg - j0);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pair = lane & 15, kg = lane >> 4;  // channel pair and row of lanes
  const int si = lane & 3, sc = (lane & 15) >> 2;  // the sample a lane describes: pixel kg * 4 + si, tap column sc (< 3)

  for (int e = threadIdx.x; e < npos * kLnPitch; e += kLnBlock) sums[e] = 0ull;
  // tables: cell (i, k) of the zero-padded scope tile, {tl, tr - tl, bl - tl, br - tr - bl + tl} per channel
  for (int e = threadIdx.x; PLAIN && e < 9 * kLnCh; e += kLnBlock) {  // [tap][channel]
    const int t = e / kLnCh, ch = e % kLnCh;
    const float h = scope_coord<float>(g, t / 3, 0.f, g.centre_h), w = scope_coord<float>(g, t % 3, 0.f, g.centre_w);
    const bool in = ch < nch && h > -1.f && w > -1.f && h < float(SH) && w < float(SW);
    const int i = (int)floorf(h), k = (int)floorf(w);
    const float lh = h - float(i), lw = w - float(k);
    const T* f = filter + (size_t)(grp + g.groups * (j0 + min(ch, nch - 1))) * (SH * SW);
    auto at = [&](int a, int b) { return in && a >= 0 && a < SH && b >= 0 && b < SW ? ld(f + a * SW + b) : 0.f; };
    const float tl = at(i, k), tr = at(i, k + 1), bl = at(i + 1, k), br = at(i + 1, k + 1);
    reinterpret_cast<float*>(tbl)[e] = fmaf(lh, fmaf(lw, (br - tr) - (bl - tl), bl - tl), fmaf(lw, tr - tl, tl));
  }
  for (int e = threadIdx.x; !PLAIN && e < CELLS * kLnCh; e += kLnBlock) {
    const int cell = e / kLnCh, odd = e / kLnPairs & 1, ch = (e % kLnPairs) * 2 + odd;
    const int i = cell / (SW + 1) - 1, k = cell % (SW + 1) - 1;
    const T* f = filter + (size_t)(grp + g.groups * (j0 + min(ch, nch - 1))) * (SH * SW);
    auto at = [&](int a, int b) { return ch < nch && a >= 0 && a < SH && b >= 0 && b < SW ? ld(f + a * SW + b) : 0.f; };
    const float tl = at(i, k), tr = at(i, k + 1), bl = at(i + 1, k), br = at(i + 1, k + 1);
    tbl[e] = make_float4(tl, tr - tl, bl - tl, (br - tr) - (bl - tl));
  }
  if (threadIdx.x < kLnCh) {
    const T* f = filter + (size_t)(grp + g.groups * (j0 + min((int)threadIdx.x, nch - 1))) * (SH * SW);
    unsigned m = 0u;  // on bit patterns, so that a NaN is not dropped
    for (int e = 0; e < SH * SW; ++e) m = max(m, __float_as_uint(ld(f + e)) & 0x7fffffffu);
    wmax[threadIdx.x] = __uint_as_float(m);
  }
  const float gmax = block_absmax(gmax_bits);  // (its barriers make sums, tbl and wmax visible)
  const size_t chan0 = (size_t)n * g.channel + grp + (size_t)g.groups * j0;
  const T* gp = gout + chan0 * out_plane;
  T* ip = gin + chan0 * in_plane;
  const size_t i_step = (size_t)g.groups * in_plane;
  if (write_nan_if_unbounded(gmax, wmax, nch, ip, i_step, in_plane)) return;  // (BAND: every band writes the same)

  const rsrc_t ro = plane_rsrc(off + (size_t)n * 18 * out_plane, 18 * out_plane);
  const rsrc_t rr = rot ? plane_rsrc(rot + (size_t)(n * g.groups + grp) * 18 * out_plane, 18 * out_plane) : plane_rsrc(rot, 0);
  const unsigned step = (unsigned)out_plane * (unsigned)sizeof(T);
  const float fH = float(H), fW = float(W);

  // image position of tap (f_h, f_w) of pixel p with offsets (dh, dw) (K.cu:486-500)
  auto image_pos = [&](int p, int f_h, int f_w, float dh, float dw, float& h, float& w) {
    const int oh = (int)__umulhi((unsigned)p, inv_out_w), ow = p - oh * g.out_w;
    h = float(oh * g.stride_h - g.pad_h + f_h * g.dil_h) + dh;
    w = float(ow * g.stride_w - g.pad_w + f_w * g.dil_w) + dw;
    return p < out_plane && h > -1.f && w > -1.f && h < fH && w < fW;
  };

  auto touches = [&](int p) {  // whether samples of the 64 output pixels that p is one of read rows of this band
    const int2 rows = unit_rows[(size_t)n * ceil_div(out_plane, 64) + (p >> 6)];
    return rows.x < r_hi && rows.y >= r_lo;
  };

  // The number of samples added to each position, kept beside its sums, and the largest, M.
  unsigned most = 1u;
  {
    unsigned* count = reinterpret_cast<unsigned*>(sums + kLnPairs);
    constexpr int CP = 2 * kLnPitch;  // words between two positions' counts
    for (int p0 = wave * 64; p0 < out_plane; p0 += kLnBlock) {
      if (BAND && !touches(p0)) continue;
      const int p = p0 + lane;
      float dh[9], dw[9];
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        const unsigned o = p < out_plane ? (unsigned)(2 * t * out_plane + p) * (unsigned)sizeof(T) : kOutOfRange;
        dh[t] = buf_ld(ro, o, off);
        dw[t] = buf_ld(ro, o + step, off);
      }
#pragma unroll
      for (int t = 0; t < 9; ++t) {
        float h, w;
        if (!image_pos(p, t / 3, t % 3, dh[t], dw[t], h, w)) continue;
        const int top = (int)floorf(h), at = ((top + row0) * RS + (int)floorf(w) + 1) * CP;
        if (!BAND || (top >= r_lo && top < r_hi)) {
          atomicAdd(count + at, 1u);
          atomicAdd(count + at + CP, 1u);
        }
        if (!BAND || (top + 1 >= r_lo && top + 1 < r_hi)) {
          atomicAdd(count + at + RS * CP, 1u);
          atomicAdd(count + at + RS * CP + CP, 1u);
        }
      }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < npos; e += kLnBlock) most = max(most, count[e * CP]);
    for (int s = 32; s > 0; s >>= 1) most = max(most, (unsigned)__shfl_xor((int)most, s));
    if (lane == 0) wave_most[wave] = most;
    __syncthreads();
    for (int w = 0; w < kLnWaves; ++w) most = max(most, wave_most[w]);
  }
  const int head = most <= 1u ? 0 : 32 - __builtin_clz(most - 1u);  // ceil(log2(most))
  const bool paired = head <= kPairHead;
  if (threadIdx.x < kLnCh) {
    int e;
    (void)frexpf(gmax * wmax[threadIdx.x], &e);
    unscale32[threadIdx.x] = ldexpf(1.f, -min(max(30 - head - e, -100), 100));  // (read behind the barrier after the walk)
  }

  const rsrc_t rg = plane_rsrc(gp, ((nch - 1) * g.groups + 1) * out_plane);
  unsigned g_off[2];
  int expo[2];  // a term of channel c is below gmax * wmax[c] < 2^expo
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const int ch = 2 * pair + c;
    g_off[c] = ch < nch ? (unsigned)(ch * g.groups * out_plane + 4 * kg) * (unsigned)sizeof(T) : kOutOfRange;
    (void)frexpf(gmax * wmax[ch], &expo[c]);
  }
  const int units = ceil_div(out_plane, kLnPix) * 3;
  using Vec = decltype(raw_ld4(rg, 0u, gout));
  struct Raw {
    float dh, dw, rh, rw;
    Vec g0, g1;
  };
  auto load_unit = [&](int u) {
    Raw r;
    const int p0 = u / 3 * kLnPix, p = p0 + 4 * kg + si, t = u % 3 * 3 + sc;
    const unsigned o = sc < 3 && p < out_plane && u < units ? (unsigned)(2 * t * out_plane + p) * (unsigned)sizeof(T) : kOutOfRange;
    r.dh = buf_ld(ro, o, off);
    r.dw = buf_ld(ro, o + step, off);
    if constexpr (!PLAIN) {
      r.rh = buf_ld(rr, o, rot);
      r.rw = buf_ld(rr, o + step, rot);
    }
    const unsigned po = (unsigned)p0 * (unsigned)sizeof(T);
    r.g0 = load4(rg, g_off[0] + po, wide, gout);
    r.g1 = load4(rg, g_off[1] + po, wide, gout);
    return r;
  };

  // One walk over the output plane.  PAIR: both channels of the lane's pair, 32-bit terms; else its channel `c` alone on
  // a grid of 2^-44 of the largest possible term.
  auto walk = [&](auto pair_tag, int c) {
    constexpr bool PAIR = decltype(pair_tag)::value;
    float scale[2];
#pragma unroll
    for (int k = 0; k < 2; ++k)
      scale[k] = 2 * pair + k < nch ? ldexpf(1.f, min(max(30 - head - expo[k], -100), 100)) : 0.f;
    const double dscale = ldexp(1.0, 44 - (c ? expo[1] : expo[0]));
    const int lane8 = pair * 8, lane16 = pair * 16;
    auto next_unit = [&](int u) {
      if constexpr (BAND)
        while (u < units && !touches(u / 3 * kLnPix)) u += kLnWaves;
      return u;
    };
    int next = next_unit(wave);
    Raw nxt = load_unit(next);
    while (next < units) {
      const int u = next;
      const Raw cur = nxt;
      next = next_unit(u + kLnWaves);
      nxt = load_unit(next);
      const int p0 = u / 3 * kLnPix, f_h = u % 3;
      // the sample this lane describes
      float h, w;
      const bool hit = image_pos(p0 + 4 * kg + si, f_h, sc, cur.dh, cur.dw, h, w);
      const float sh = PLAIN ? 0.f : scope_coord<float>(g, f_h, cur.rh, g.centre_h);
      const float sw = PLAIN ? 0.f : scope_coord<float>(g, sc, cur.rw, g.centre_w);
      // a sample outside the scope band is added with weight zero: it is counted
      const float hf = floorf(h), wf = floorf(w);
      const int itop = (int)hf;
      const bool in_top = !BAND || (itop >= r_lo && itop < r_hi), in_bot = !BAND || (itop + 1 >= r_lo && itop + 1 < r_hi);
      const bool on = sc < 3 && hit && (in_top || in_bot), in = on && sh > -1.f && sw > -1.f && sh < float(SH) && sw < float(SW);
      const float shf = floorf(sh), swf = floorf(sw);
      const float lh = on ? h - hf : 0.f, lw = on ? w - wf : 0.f;
      const float hh = on ? 1.f - lh : 0.f, hw = 1.f - lw;
      const float d00 = hh * hw, d01 = hh * lw, d10 = lh * hw, d11 = lh * lw;  // K.cu:776-789
      double e00 = d00, e01 = d01, e10 = d10, e11 = d11;
      asm volatile("s_nop 1" : "+v"(e00), "+v"(e01), "+v"(e10), "+v"(e11));  // (see fma_row_lane)
      const float slh = in ? sh - shf : 0.f, slw = in ? sw - swf : 0.f;
      const int cell = in ? (((int)shf + 1) * (SW + 1) + (int)swf + 1) * (kLnCh * 16) : 0;
      const int at = ((itop + row0) * RS + (int)wf + 1) * (kLnPitch * 8);
      const int top = on && in_top ? at : spare * (kLnPitch * 8), bot = on && in_bot ? at + RS * (kLnPitch * 8) : spare * (kLnPitch * 8);
      const unsigned long long any = __ballot(on);
      if (any == 0ull) continue;
      float2 wt[3];  // PLAIN: the weights of the unit's taps
      if constexpr (PLAIN) {
#pragma unroll
        for (int c3 = 0; c3 < 3; ++c3) wt[c3] = reinterpret_cast<const float2*>(tbl)[(f_h * 3 + c3) * kLnPairs + pair];
      }
      float g0[4], g1[4];
      raw_cvt4(cur.g0, g0, gout);
      raw_cvt4(cur.g1, g1, gout);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if constexpr (PAIR) {
          g0[i] *= scale[0];
          g1[i] *= scale[1];
        } else {
          g0[i] = c ? g1[i] : g0[i];
        }
      }
      static_for<12>([&](auto s_tag) {
        constexpr int S = decltype(s_tag)::value, I = S & 3;
        if (!(any >> S & 0x0001000100010001ull)) return;  // none of the four rows' samples adds anything here
        float ma, mb;
        if constexpr (PLAIN) {
          ma = g0[I] * (PAIR || !c ? wt[S >> 2].x : wt[S >> 2].y);
          mb = PAIR ? g1[I] * wt[S >> 2].y : 0.f;
        } else {
          const char* q = reinterpret_cast<const char*>(tbl) + (row_lane<S>(cell) + lane16);
          const float4 qa = *reinterpret_cast<const float4*>(q), qb = *reinterpret_cast<const float4*>(q + kLnPairs * 16);
          const float fh = row_lane<S>(slh), fw = row_lane<S>(slw);
          ma = g0[I] * fmaf(fh, fmaf(fw, (PAIR || !c ? qa : qb).w, (PAIR || !c ? qa : qb).z),
                            fmaf(fw, (PAIR || !c ? qa : qb).y, (PAIR || !c ? qa : qb).x));
          mb = PAIR ? g1[I] * fmaf(fh, fmaf(fw, qb.w, qb.z), fmaf(fw, qb.y, qb.x)) : 0.f;
        }
        const double ma_d = ma;
        auto add = [&](int addr, float cw, double cwd) {
          unsigned long long* target = reinterpret_cast<unsigned long long*>(reinterpret_cast<char*>(sums) + addr);
          if constexpr (PAIR) {
            // two signed 32-bit fixed-point terms in one 64-bit add, b * 2^32 + a + kBias: "add a constant in double"
            // rounds a's product and makes its word positive, so that no borrow has to be taken from b's
            const unsigned long long a = (unsigned long long)__double_as_longlong(fma_row_lane<S>(cwd, ma_d, kMagicBias));
            const int ib = round_half_up(row_lane<S>(cw) * mb);
            atomicAdd(target, ((unsigned long long)(unsigned)ib << 32) | (unsigned long long)(unsigned)a);
          } else {
            // "add 1.5 * 2^52 in double": the low mantissa bits of the sum are the rounded integer
            const double d = fma((double)(row_lane<S>(cw) * ma), dscale, kMagic);
            atomicAdd(target, (unsigned long long)__double_as_longlong(d) - 0x4338000000000000ull);
          }
        };
        const int a0 = row_lane<S>(top) + lane8;
        add(a0, d00, e00);
        add(a0 + kLnPitch * 8, d01, e01);
        const int a1 = row_lane<S>(bot) + lane8;
        add(a1, d10, e10);
        add(a1 + kLnPitch * 8, d11, e11);
      });
    }
  };

  // Write the planes of the walk's channels and clear the sums: the lanes of a wave take pixels, for one pair after
  // another.
  auto read_back = [&](auto pair_tag, int c, bool clear) {
    constexpr bool PAIR = decltype(pair_tag)::value;
    const int own = (r_hi - r_lo) * W;
    for (int e0 = wave * 64; e0 < own; e0 += kLnBlock) {
      const int e = e0 + lane;
      if (e >= own) continue;
      const int r = (int)__umulhi((unsigned)e, inv_in_w);
      unsigned long long* cell = sums + ((r + (BAND ? 0 : 1)) * RS + (e - r * W) + 1) * kLnPitch;
      const unsigned long long bias = cell[kLnPairs] * kBias;
      T* dst = ip + r_lo * W + e;
      for (int q = 0; 2 * q < nch; ++q) {
        const unsigned long long v = cell[q];
        if constexpr (PAIR) {
          const unsigned long long w = v - bias;
          const int lo = (int)(unsigned)w, hi = (int)(unsigned)(w >> 32) + (lo < 0 ? 1 : 0);
          st_stream(dst + (size_t)(2 * q) * i_step, (float)lo * unscale32[2 * q]);
          if (2 * q + 1 < nch) st_stream(dst + (size_t)(2 * q + 1) * i_step, (float)hi * unscale32[2 * q + 1]);
        } else {
          int ea;
          (void)frexpf(gmax * wmax[2 * q + c], &ea);
          if (2 * q + c < nch) st_stream(dst + (size_t)(2 * q + c) * i_step, (float)((double)(long long)v * ldexp(1.0, ea - 44)));
          if (clear) cell[q] = 0ull;
        }
      }
    }
  };

  if (paired) {
    walk(std::true_type{}, 0);
    __syncthreads();
    read_back(std::true_type{}, 0, false);
    return;
  }
  // many samples on one element: one channel per sum
  for (int c = 0; c < 2; ++c) {
    walk(std::false_type{}, c);
    __syncthreads();
    read_back(std::false_type{}, c, true);
    __syncthreads();
  }
}

constexpr int kLnBandRows = 12;

struct LanesPlan {
  bool ok, band;
  int rows;  // image rows of a workgroup
  size_t lds;
  long blocks;
};

// Where this form applies and is the faster one.  It wants output planes that amortise a workgroup's fixed costs (tables,
// clearing and reading back 118 KB of sums at 28 x 28) and enough workgroups for the chip, as it has no more than one per
// 32 channels (us here / with a pixel per lane, float32): N=64 C=192 28x28 108 / 156, C=144 100 / 134, C=96 20x20
// 31 / 42, N=32 C=100 24x24 (128 workgroups) 39 / 53, N=128 C=384 14x14 107 / 117; but N=64 C=24 28x28 (64 workgroups)
// 48 / 31, N=64 C=512 28x28 to 14x14 (stride 2) 92 / 91, N=64 C=960 7x7 79 / 73.
template <int SH, int SW>
LanesPlan lanes_plan(const Geo& g) {
  LanesPlan m{};
  m.ok = false;
  if (path_disabled(kNoDeformFast) || path_disabled(kNoDeformLanes)) return m;
  const long plane = (long)g.out_h * g.out_w, in_plane = (long)g.in_h * g.in_w, cpg = g.channel / g.groups;
  // 32-bit byte offsets inside a chunk's planes, and products of a pixel and a width below 2^32 (the divisions)
  if (plane > 16384 || in_plane > 16384 || plane * g.groups * kLnCh * 4 >= (1L << 31) || g.in_w < 2 || g.out_w < 2) return m;
  const long tables = (long)(SH + 1) * (SW + 1) * kLnCh * 16 + 16;
  const long fit = (kLnLds - tables) / (kLnPitch * 8);  // positions
  m.rows = g.in_h;
  if (lanes_positions(g.in_h, g.in_w, false) > fit) {
    // bands of equal height.  Every band walks the rows its samples can come from: with fewer than kLnBandRows rows the
    // walk is mostly over samples of other bands (us here / with a pixel per lane, offsets ~ N(0, 2^2): N=64 C=96 40 x 40
    // 130 / 149, N=24 C=64 64 x 64 101 / 113, N=16 80 x 80 (12 rows) 106 / 113; 75 x 101 float16 (10 rows) 135 / 118).
    // Wide offsets: band_limit
    const int most = (int)std::max(0L, (fit - 3) / (g.in_w + 1));
    if (most < 1) return m;
    m.rows = ceil_div(g.in_h, ceil_div(g.in_h, most));
    m.band = true;
    if (path_disabled(kNoDeformWindow)) return m;
  }
  const int bands = m.band ? ceil_div(g.in_h, m.rows) : 1;
  m.lds = (size_t)((long)lanes_positions(m.rows, g.in_w, m.band) * kLnPitch * 8 + tables);
  m.blocks = (cpg + kLnCh - 1) / kLnCh * g.batch * g.groups * bands;
  if (m.blocks >= (1L << 31) - 8) return m;
  m.ok = path_disabled(kForceDeformLanes) || (plane >= 192 && in_plane <= 2 * plane && m.blocks >= 128 && cpg > kLnCh / 2 &&
                                              (!m.band || m.rows >= kLnBandRows));
  return m;
}

// Bands that a unit of 64 pixels meets on average, in sixteenths, up to which the bands are the faster form.  float32, us in
// bands / with a pixel per lane at so many, offsets ~ N(0, 2^2 .. 10^2), with a rotation tensor: N=64 C=96 40 x 40 (two bands) 1.51: 136 / 143,
// 1.78: 145 / 139; N=64 C=144 56 x 56 (three) 1.72: 360 / 403, 2.15: 405 / 390, 2.73: 468 / 373; N=24 C=64 64 x 64 (four) 1.95:
// 113 / 116, 2.45: 130 / 114; N=16 C=64 80 x 80 (seven) 2.08: 108 / 115, 2.49: 121 / 119, 4.9: 187 / 127.  Without one: 56 x 56 2.73: 378 /
// 376; 64 x 64 2.45: 108 / 116, 3.4: 127 / 111; 80 x 80 3.25: 118 / 121, 4.9: 152 / 127; two bands are never slower.  The launches of
// the form that finds nothing to do take 5 - 9 us (56 x 56: 340 -> 343 in bands, 390 -> 396 beside them).
int band_limit(bool plain, int bands) {
  if (plain) return bands <= 4 ? 43 : 50;
  return bands == 2 ? 25 : bands <= 4 ? 32 : 36;
}

template <typename T, int SH, int SW>
bool run_lanes_grad_input(const Geo& g, const T* gout, const T* off, const T* rot, const T* filter, T* gin,
                          const unsigned* gmax, BandWalk walk, hipStream_t stream) {
  const LanesPlan m = lanes_plan<SH, SW>(g);
  if (!m.ok) return false;
  const int wide = g.out_h * g.out_w % 4 == 0 && reinterpret_cast<uintptr_t>(gout) % (4 * sizeof(T)) == 0;
  auto inverse = [](int w) { return (unsigned)(((1ull << 32) + w - 1) / w); };
  const bool plain = !rot && !path_disabled(kNoDeformPlain);
  auto kernel = m.band ? plain ? deform_grad_input_lanes_kernel<T, SH, SW, true, true> : deform_grad_input_lanes_kernel<T, SH, SW, false, true>
                       : plain ? deform_grad_input_lanes_kernel<T, SH, SW, true, false> : deform_grad_input_lanes_kernel<T, SH, SW, false, false>;
  if (!allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kLnLds)) return false;
  walk.rows = m.rows;
  kernel<<<(unsigned)xcd_grid_size(m.blocks), kLnBlock, m.lds, stream>>>(g, gout, off, rot, filter, gin, gmax,
                                                                         inverse(g.out_w), inverse(g.in_w), wide, walk, walk.unit_rows);
  return true;
}

}  // namespace

#define DK_LANES_SCOPE(G, CALL)                                   \
  if ((G).scope_h == 4 && (G).scope_w == 4) return CALL(4, 4);    \
  if ((G).scope_h == 3 && (G).scope_w == 3) return CALL(3, 3);    \
  if ((G).scope_h == 5 && (G).scope_w == 5) return CALL(5, 5);

bool lanes_deform_grad_input_applies(const Geo& g) {
  if (g.k_h != 3 || g.k_w != 3) return false;
#define CALL(SH, SW) lanes_plan<SH, SW>(g).ok
  DK_LANES_SCOPE(g, CALL)
#undef CALL
  return false;
}

BandWalk lanes_band_walk(const Geo& g, bool rotation) {
  auto walk = [&](const LanesPlan& m) {
    BandWalk w{};
    if (!m.ok || !m.band) return w;
    const int bands = ceil_div(g.in_h, m.rows), limit = band_limit(!rotation && !path_disabled(kNoDeformPlain), bands);
    w.rows = m.rows;
    w.most = path_disabled(kForceDeformLanes) || 16 * bands <= limit ? ~0u : (unsigned)((long)g.batch * ceil_div(g.out_h * g.out_w, 64) * limit / 16);
    return w;
  };
#define CALL(SH, SW) walk(lanes_plan<SH, SW>(g))
  DK_LANES_SCOPE(g, CALL)
#undef CALL
  return BandWalk{};
}

template <typename T>
bool lanes_deform_grad_input(const Geo& g, const T* gout, const T* off, const T* rot, const T* filter, T* gin,
                             const unsigned* gmax, const BandWalk& walk, hipStream_t stream) {
#define CALL(SH, SW) run_lanes_grad_input<T, SH, SW>(g, gout, off, rot, filter, gin, gmax, walk, stream)
  DK_LANES_SCOPE(g, CALL)
#undef CALL
  return false;
}

#define DK_INSTANTIATE(T)                                                                                         \
  template bool lanes_deform_grad_input<T>(const Geo&, const T*, const T*, const T*, const T*, T*, const unsigned*, \
                                           const BandWalk&, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
