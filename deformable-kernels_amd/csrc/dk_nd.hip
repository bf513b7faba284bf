// N-d linear sample: out[b, c] = multilinear(data[c], coord[b]), zero outside.
//
// ND.cu = deformable_kernels/ops/deform_kernel/csrc/nd_linear_sample_cuda_kernel.cu
//   nd_linear ND.cu:45-88, nd_linear_backward_data ND.cu:90-131,
//   nd_linear_backward_coord ND.cu:133-177; kernels ND.cu:183-287.
//
// Two main paths.
//  * Channel-last path (1..3 sampling dimensions, enough work to pay for a transpose):
//    `data` [C, P] is first copied to [P, C] in the caller's workspace, so the C values of
//    one corner are contiguous.  A wave takes 64 points: with lane <-> point it derives each
//    point's 2^n corner offsets and weights once, then walks its points with lane <-> channel,
//    broadcasting the point's corners by readlane; every corner read and every output row
//    is one contiguous run.  The reference maps adjacent threads to adjacent channels whose
//    data lie a whole volume apart (ND.cu:197-199).
//  * Direct path (any dimension count, small problems): one lane per (point, channel).
// The coordinate gradient is reduced over channels inside the kernel instead of
// materialising the reference's [B, n, C] intermediate (ND.cu:281-286 and the caller's sum).

#include "dk_kernels.h"
#include "dk_nd.h"

namespace dk {

namespace {

constexpr int kBlock = 256;
constexpr int kClMaxDims = 3;
constexpr int kClCorners = 1 << kClMaxDims;

struct NdGeo {
  long batch;
  int channel;
  int dims;  // kernels with a template parameter ND > 0 set it to that, see DK_ND_BY_ANY_DIMS
  long prod_shape;
  int shape[DK_ND_MAX_DIMS];
};

// ---------------------------------------------------------------------------
// per-point corner bookkeeping shared by both paths
// ---------------------------------------------------------------------------
template <typename CT>
struct NdPoint {
  int low[DK_ND_MAX_DIMS];
  CT frac[DK_ND_MAX_DIMS];
  bool inside;  // false: some x <= -1 or x >= s, the whole sample is zero (ND.cu:47-53)
};

template <typename T, typename CT>
__device__ __forceinline__ NdPoint<CT> load_point(const NdGeo& g, const T* coord_b) {
  NdPoint<CT> p;
  p.inside = true;
#pragma unroll
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) {
    if (d < g.dims) {
      const CT x = ld(coord_b + d);
      const CT xf = floor(x);
      const bool in = x > CT(-1) && x < CT(g.shape[d]);
      if (!in) p.inside = false;
      p.low[d] = in ? (int)xf : 0;
      p.frac[d] = x - xf;
    } else {
      p.low[d] = 0;
      p.frac[d] = CT(0);
    }
  }
  return p;
}

// Offset and weight of corner `i` (bit d selects low/high in dimension d, ND.cu:67);
// `skip_dim` >= 0 replaces that dimension's weight by -1 / +1 (ND.cu:161,165).
// Returns false where the reference breaks out of the corner.
template <typename CT>
__device__ __forceinline__ bool corner(const NdGeo& g, const NdPoint<CT>& p, unsigned i,
                                       int skip_dim, long& offset, CT& weight) {
  offset = 0;
  weight = CT(1);
#pragma unroll
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) {
    if (d < g.dims) {
      const int s = g.shape[d];
      offset *= s;
      const unsigned hi = (i >> d) & 1u;
      if (hi == 0 && p.low[d] >= 0) {
        offset += p.low[d];
        weight *= (d == skip_dim) ? CT(-1) : CT(1) - p.frac[d];
      } else if (hi == 1 && p.low[d] + 1 <= s - 1) {
        offset += p.low[d] + 1;
        weight *= (d == skip_dim) ? CT(1) : p.frac[d];
      } else {
        return false;
      }
    }
  }
  return true;
}

// ---------------------------------------------------------------------------
// direct path
// ---------------------------------------------------------------------------
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_forward_kernel(NdGeo g, const T* __restrict__ data,
                                                            const T* __restrict__ coord,
                                                            T* __restrict__ out, long total) {
  if constexpr (ND > 0) g.dims = ND;
  using CT = compute_t<T>;
  for (long id = (long)blockIdx.x * kBlock + threadIdx.x; id < total; id += (long)gridDim.x * kBlock) {
    const int c = (int)(id % g.channel);
    const long b = id / g.channel;
    const NdPoint<CT> p = load_point<T, CT>(g, coord + b * g.dims);
    CT val = 0;
    if (p.inside) {
      const T* dc = data + (size_t)c * g.prod_shape;
      for (unsigned i = 0; i < (1u << g.dims); ++i) {
        long o;
        CT w;
        if (corner<CT>(g, p, i, -1, o, w)) val += w * ld(dc + o);
      }
    }
    st(out + id, val);
  }
}

// scatter with hardware float atomics into a zeroed buffer laid out [C][P] (cl = false) or
// [P][C] (cl = true)
template <typename T, typename CT, bool CL, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_data_kernel(NdGeo g, const T* __restrict__ gout,
                                                              const T* __restrict__ coord,
                                                              CT* __restrict__ gdata, long total) {
  if constexpr (ND > 0) g.dims = ND;
  for (long id = (long)blockIdx.x * kBlock + threadIdx.x; id < total; id += (long)gridDim.x * kBlock) {
    const int c = (int)(id % g.channel);
    const long b = id / g.channel;
    const NdPoint<CT> p = load_point<T, CT>(g, coord + b * g.dims);
    if (!p.inside) continue;
    const CT go = ld(gout + id);
    for (unsigned i = 0; i < (1u << g.dims); ++i) {
      long o;
      CT w;
      if (corner<CT>(g, p, i, -1, o, w))
        atomicAdd(CL ? gdata + (size_t)o * g.channel + c : gdata + (size_t)c * g.prod_shape + o, w * go);
    }
  }
}

// one wave per point, lanes over channels, shuffle reduction
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_coord_kernel(NdGeo g, const T* __restrict__ gout,
                                                               const T* __restrict__ data,
                                                               const T* __restrict__ coord,
                                                               T* __restrict__ gcoord) {
  if constexpr (ND > 0) g.dims = ND;
  using CT = compute_t<T>;
  const int lane = threadIdx.x & 63;
  const long waves = (long)gridDim.x * (kBlock / 64);
  for (long b = (long)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6); b < g.batch; b += waves) {
    const NdPoint<CT> p = load_point<T, CT>(g, coord + b * g.dims);
    CT acc[DK_ND_MAX_DIMS];
#pragma unroll
    for (int d = 0; d < DK_ND_MAX_DIMS; ++d) acc[d] = CT(0);
    if (p.inside) {
      for (int c = lane; c < g.channel; c += 64) {
        const CT go = ld(gout + b * g.channel + c);
        const T* dc = data + (size_t)c * g.prod_shape;
        for (unsigned i = 0; i < (1u << g.dims); ++i) {
          // a corner exists for every differentiated dimension or for none
          long o;
          CT w;
          if (!corner<CT>(g, p, i, -1, o, w)) continue;
          const CT dv = go * ld(dc + o);
#pragma unroll
          for (int d = 0; d < DK_ND_MAX_DIMS; ++d) {
            if (d < g.dims) {
              long o2;
              CT w2;
              corner<CT>(g, p, i, d, o2, w2);
              acc[d] += dv * w2;
            }
          }
        }
      }
    }
#pragma unroll
    for (int d = 0; d < DK_ND_MAX_DIMS; ++d) {
      if (d < g.dims) {
        CT v = acc[d];
        for (int sft = 32; sft > 0; sft >>= 1) v += __shfl_xor(v, sft, 64);
        if (lane == 0) st(gcoord + b * g.dims + d, v);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// channel-last path
// ---------------------------------------------------------------------------

// in [rows][cols] -> out [cols][rows], converting A -> B; 32 x 32 tiles through LDS.  zero != nullptr: as many floats, cleared
// beside it (a launch less).  One workgroup per tile, numbered along the columns first: in a two-dimensional grid a volume of more
// than 2.1 million cells passes the 65535 workgroups of its second dimension.
template <typename A, typename B>
__global__ __launch_bounds__(256) void nd_transpose_kernel(const A* __restrict__ in, B* __restrict__ out, float* __restrict__ zero,
                                                           long rows, long cols, unsigned col_tiles) {
  __shared__ float tile[32][33];
  const long r0 = (long)(blockIdx.x / col_tiles) * 32, c0 = (long)(blockIdx.x % col_tiles) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
  for (int k = 0; k < 32; k += 8) {
    const long r = r0 + ty + k, c = c0 + tx;
    tile[ty + k][tx] = (r < rows && c < cols) ? static_cast<float>(ld(in + r * cols + c)) : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 32; k += 8) {
    const long c = c0 + ty + k, r = r0 + tx;
    if (r < rows && c < cols) {
      st(out + c * rows + r, tile[tx][ty + k]);
      if (zero) zero[c * rows + r] = 0.f;
    }
  }
}

// Corner offsets (in units of C elements of the channel-last copy) and weights of one
// point, padded to kClCorners; absent corners get weight 0 at offset 0.
struct ClCorners {
  int off[kClCorners];
  float w[kClCorners];
  unsigned present;  // bit i: corner i lies inside the volume (its weight may still be 0)
};

template <typename T>
__device__ __forceinline__ ClCorners cl_corners(const NdGeo& g, const T* coord, long b, bool valid) {
  ClCorners cc;
  cc.present = 0u;
  NdPoint<float> p;
  p.inside = false;
  if (valid) p = load_point<T, float>(g, coord + b * g.dims);
#pragma unroll
  for (int i = 0; i < kClCorners; ++i) {
    long o = 0;
    float w = 0.f;
    const bool ok = valid && p.inside && i < (1 << g.dims) && corner<float>(g, p, (unsigned)i, -1, o, w);
    cc.off[i] = ok ? (int)o : 0;
    cc.w[i] = ok ? w : 0.f;
    cc.present |= ok ? (1u << i) : 0u;
  }
  return cc;
}

// forward: a wave owns `ppw` (a power of two <= 64) consecutive points and walks them four at a
// time so that the corner reads of four points are in flight together
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_forward_cl_kernel(NdGeo g, const T* __restrict__ data_cl,
                                                               const T* __restrict__ coord,
                                                               T* __restrict__ out, int ppw) {
  g.dims = ND;
  const int lane = threadIdx.x & 63;
  const long wave0 = ((long)blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * ppw;
  if (wave0 >= g.batch) return;
  const int npts = (int)min((long)ppw, g.batch - wave0);
  const ClCorners mine = cl_corners<T>(g, coord, wave0 + lane, lane < npts);
  const int ncorner = 1 << g.dims;
  constexpr int PU = 4;
  for (int q0 = 0; q0 < npts; q0 += PU) {
    int off[PU][kClCorners];
    float w[PU][kClCorners];
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const int q = min(q0 + u, npts - 1);
#pragma unroll
      for (int i = 0; i < kClCorners; ++i) {
        off[u][i] = __builtin_amdgcn_readlane(mine.off[i], q);
        w[u][i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.w[i]), q));
      }
    }
    for (int c = lane; c < g.channel; c += 64) {
      float v[PU][kClCorners];
#pragma unroll
      for (int u = 0; u < PU; ++u)
#pragma unroll
        for (int i = 0; i < kClCorners; ++i)
          v[u][i] = i < ncorner ? ld(data_cl + (size_t)off[u][i] * g.channel + c) : 0.f;
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        float acc = 0.f;
#pragma unroll
        for (int i = 0; i < kClCorners; ++i) acc += w[u][i] * v[u][i];
        if (q0 + u < npts) st(out + (wave0 + q0 + u) * g.channel + c, acc);
      }
    }
  }
}

// grad coord: same walk; per point the lanes' partial gradients are reduced by shuffles
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_coord_cl_kernel(NdGeo g, const T* __restrict__ gout,
                                                                  const T* __restrict__ data_cl,
                                                                  const T* __restrict__ coord,
                                                                  T* __restrict__ gcoord, int ppw) {
  g.dims = ND;
  const int lane = threadIdx.x & 63;
  const long wave0 = ((long)blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * ppw;
  if (wave0 >= g.batch) return;
  const int npts = (int)min((long)ppw, g.batch - wave0);
  const bool valid = lane < npts;
  const ClCorners mine = cl_corners<T>(g, coord, wave0 + lane, valid);
  const int ncorner = 1 << g.dims;
  // s[i] of point q lands in lane q: sum over channels of gout * data at corner i
  float s[kClCorners];
#pragma unroll
  for (int i = 0; i < kClCorners; ++i) s[i] = 0.f;
  for (int q = 0; q < npts; ++q) {
    int off[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) off[i] = __builtin_amdgcn_readlane(mine.off[i], q);
    float part[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) part[i] = 0.f;
    const T* grow = gout + (wave0 + q) * g.channel;
    for (int c = lane; c < g.channel; c += 64) {
      const float go = ld(grow + c);
#pragma unroll
      for (int i = 0; i < kClCorners; ++i)
        if (i < ncorner) part[i] += go * ld(data_cl + (size_t)off[i] * g.channel + c);
    }
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) {
      if (i < ncorner) {
        const float v = wave_sum(part[i]);
        if (lane == q) s[i] = v;
      }
    }
  }
  if (!valid) return;
  // lane <-> point again: apply the derivative weights (ND.cu:161,165) to the corner sums
  const NdPoint<float> p = load_point<T, float>(g, coord + (wave0 + lane) * g.dims);
#pragma unroll
  for (int d = 0; d < kClMaxDims; ++d) {
    if (d < g.dims) {
      float gd = 0.f;
      if (p.inside) {
#pragma unroll
        for (int i = 0; i < kClCorners; ++i) {
          long o;
          float w;
          if (i < ncorner && corner<float>(g, p, (unsigned)i, d, o, w)) gd += s[i] * w;
        }
      }
      st(gcoord + (wave0 + lane) * g.dims + d, gd);
    }
  }
}

// grad data: scatter into the zeroed channel-last fp32 image; one 64-channel run per atomic
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_data_cl_kernel(NdGeo g, const T* __restrict__ gout,
                                                                 const T* __restrict__ coord,
                                                                 float* __restrict__ gdata_cl, int ppw) {
  g.dims = ND;
  const int lane = threadIdx.x & 63;
  const long wave0 = ((long)blockIdx.x * (kBlock / 64) + __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6)) * ppw;
  if (wave0 >= g.batch) return;
  const int npts = (int)min((long)ppw, g.batch - wave0);
  const ClCorners mine = cl_corners<T>(g, coord, wave0 + lane, lane < npts);
  const int ncorner = 1 << g.dims;
  for (int q = 0; q < npts; ++q) {
    int off[kClCorners];
    float w[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) {
      off[i] = __builtin_amdgcn_readlane(mine.off[i], q);
      w[i] = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, mine.w[i]), q));
    }
    const T* grow = gout + (wave0 + q) * g.channel;
    for (int c = lane; c < g.channel; c += 64) {
      const float go = ld(grow + c);
#pragma unroll
      for (int i = 0; i < kClCorners; ++i)
        if (i < ncorner && w[i] != 0.f) atomicAdd(gdata_cl + (size_t)off[i] * g.channel + c, w[i] * go);
    }
  }
}

// ---------------------------------------------------------------------------
// few points on a tiny volume (GlobalDeformKernel2d: 9 points per image on a 5 x 5 scope, hundreds of
// channels).  The forward takes the direct kernel above (one launch, the volume stays in cache);
// grad data and grad coord are one launch each here instead of fill + atomics + transpose /
// transpose + kernel.  These calls are bound by the latency of their few dependent loads, so both
// kernels know the number of dimensions at compile time (no branches between the loads) and issue
// every load of a stage before the first use.
//
// grad data: a small dense product on the matrix cores (below; scattering into sums instead --
// LDS or global float atomics on 25 x 256 sums that each receive 184 additions -- took 75-100 us).
// grad coord: one wave per point, lanes over channels; the volume is read where it lies.
// ---------------------------------------------------------------------------
constexpr int kSmallMaxCells = 64;

// The point's low corner and fractions for NDIM dimensions (load_point above, without its loop over
// DK_ND_MAX_DIMS); b is clamped by the caller.
template <typename T, int NDIM>
__device__ __forceinline__ NdPoint<float> small_point(const NdGeo& g, const T* coord_b) {
  float x[NDIM];
#pragma unroll
  for (int d = 0; d < NDIM; ++d) x[d] = ld(coord_b + d);
  NdPoint<float> p;
  p.inside = true;
#pragma unroll
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) {
    p.low[d] = 0;
    p.frac[d] = 0.f;
  }
#pragma unroll
  for (int d = 0; d < NDIM; ++d) {
    const float xf = floorf(x[d]);
    const bool in = x[d] > -1.f && x[d] < (float)g.shape[d];
    if (!in) p.inside = false;
    p.low[d] = in ? (int)xf : 0;
    p.frac[d] = x[d] - xf;
  }
  return p;
}

// grad data as a small dense product on the matrix cores: gdata[c][cell] = sum_b gout[b][c] * W[b][cell],
// W[b][.] being the point's 2^n corner weights spread over a row of zeros.  A workgroup of 16 waves owns
// 16 channels.  Per chunk of points it writes W into LDS (row = point, 16 cells per column tile), then
// each wave multiplies its share of the chunk's points, four at a time, with
// v_mfma_f32_16x16x4_f32 (M = channels, N = cells, K = points; fp32 products and sums).  The waves'
// 16 x 16 tiles are added in wave order at the end: no atomics, a fixed order of additions.
typedef float nd_f4 __attribute__((ext_vector_type(4)));
constexpr int kSmallTileMax = 4;                 // column tiles of 16 cells: volumes of up to 64 cells
constexpr int kSmallWBytes = 144 * 1024;         // LDS for W

template <typename T, int NDIM, int NT>
__global__ __launch_bounds__(1024) void nd_small_grad_data_kernel(NdGeo g, const T* __restrict__ gout,
                                                                   const T* __restrict__ coord,
                                                                   T* __restrict__ gdata, int chunk_points) {
  constexpr int NC = 1 << NDIM;
  constexpr int ROW = NT * 16;  // floats of a row of W
  extern __shared__ __align__(16) unsigned char small_lds[];
  float* W = reinterpret_cast<float*>(small_lds);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int c = min(blockIdx.x * 16 + (lane & 15), g.channel - 1);  // lanes past the last channel repeat it; not stored
  nd_f4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = nd_f4{0.f, 0.f, 0.f, 0.f};

  for (long chunk0 = 0; chunk0 < g.batch; chunk0 += chunk_points) {
    const int npts = (int)min((long)chunk_points, g.batch - chunk0);
    const int rows = (npts + 63) & ~63;  // whole 4-point steps for every wave; the extra rows stay zero
    // this thread's points of the chunk (loads first), then W = 0, then the corners' weights
    NdPoint<float> p[2];
    bool has[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int q = threadIdx.x + 1024 * r;
      has[r] = q < npts;
      p[r] = small_point<T, NDIM>(g, coord + min(chunk0 + q, g.batch - 1) * NDIM);
    }
    __syncthreads();  // the previous chunk's products have read W
    for (int i = threadIdx.x; i < rows * ROW / 4; i += 1024) reinterpret_cast<nd_f4*>(W)[i] = nd_f4{0.f, 0.f, 0.f, 0.f};
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      if (has[r] && p[r].inside) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
          long o;
          float w;
          if (corner<float>(g, p[r], (unsigned)i, -1, o, w)) W[(threadIdx.x + 1024 * r) * ROW + (int)o] = w;
        }
      }
    }
    __syncthreads();
    // wave w: rows [w * share, (w + 1) * share), share a multiple of 4
    const int share = rows / 16;
    const int r0 = wave * share;
    for (int s0 = 0; s0 < share; s0 += 32) {  // eight 4-point steps at a time, their out_grad loads first
      T raw[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int row = r0 + s0 + 4 * k + (lane >> 4);
        raw[k] = gout[min(chunk0 + row, g.batch - 1) * g.channel + c];
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        if (s0 + 4 * k < share) {  // uniform over the wave
          const int row = r0 + s0 + 4 * k + (lane >> 4);
          // rows past the chunk's points re-read the last point's out_grad: they are zeroed by a select, not by
          // their zero row of W (0 * Inf would put a NaN into every cell of the channel)
          const float a = row < npts ? ld(&raw[k]) : 0.f;
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, W[row * ROW + t * 16 + (lane & 15)], acc[t], 0, 0, 0);
        }
      }
    }
  }
  __syncthreads();
  // the waves' tiles through LDS (W's space), added in wave order
  float* red = W;  // [16 waves][NT][16 channels][16 cells]
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) red[((wave * NT + t) * 16 + 4 * (lane >> 4) + i) * 16 + (lane & 15)] = acc[t][i];
  __syncthreads();
  const int cells = (int)g.prod_shape;
  for (int i = threadIdx.x; i < NT * 256; i += 1024) {
    const int t = i >> 8, m = (i >> 4) & 15, n = i & 15;
    float v = 0.f;
    for (int w = 0; w < 16; ++w) v += red[((w * NT + t) * 16 + m) * 16 + n];
    const int co = blockIdx.x * 16 + m, cell = t * 16 + n;
    if (co < g.channel && cell < cells) st(gdata + (size_t)co * g.prod_shape + cell, v);
  }
}

template <typename T, int NDIM>
__global__ __launch_bounds__(kBlock) void nd_small_grad_coord_kernel(NdGeo g, const T* __restrict__ gout,
                                                                     const T* __restrict__ data,
                                                                     const T* __restrict__ coord,
                                                                     T* __restrict__ gcoord) {
  constexpr int NC = 1 << NDIM;
  const int lane = threadIdx.x & 63;
  const long b = (long)blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
  if (b >= g.batch) return;
  const NdPoint<float> p = small_point<T, NDIM>(g, coord + b * NDIM);
  int off[NC];
  float dw[NDIM][NC];  // derivative weights (ND.cu:161,165); 0 for a corner outside the volume
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    long o = 0;
    float w = 0.f;
    const bool ok = p.inside && corner<float>(g, p, (unsigned)i, -1, o, w);
    off[i] = ok ? (int)o : 0;
#pragma unroll
    for (int d = 0; d < NDIM; ++d) {
      long o2;
      float w2 = 0.f;
      const bool ok2 = ok && corner<float>(g, p, (unsigned)i, d, o2, w2);
      dw[d][i] = ok2 ? w2 : 0.f;
    }
  }
  float part[NC];
#pragma unroll
  for (int i = 0; i < NC; ++i) part[i] = 0.f;
  const T* grow = gout + b * g.channel;
  for (int c0 = 0; c0 < g.channel; c0 += 256) {
    // four 64-channel tiles at a time, loads first (channels past the end repeat the last one with a zero out_grad)
    T graw[4], draw[4][NC];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const int c = min(c0 + 64 * t + lane, g.channel - 1);
      graw[t] = grow[c];
#pragma unroll
      for (int i = 0; i < NC; ++i) draw[t][i] = data[(size_t)c * g.prod_shape + off[i]];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const float go = c0 + 64 * t + lane < g.channel ? ld(&graw[t]) : 0.f;
#pragma unroll
      for (int i = 0; i < NC; ++i) part[i] += go * ld(&draw[t][i]);
    }
  }
  float gd[NDIM];
#pragma unroll
  for (int d = 0; d < NDIM; ++d) gd[d] = 0.f;
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const float v = wave_sum(part[i]);
#pragma unroll
    for (int d = 0; d < NDIM; ++d) gd[d] += v * dw[d][i];
  }
  if (lane == 0) {
#pragma unroll
    for (int d = 0; d < NDIM; ++d) st(gcoord + b * NDIM + d, gd[d]);
  }
}

// ---------------------------------------------------------------------------
// channel-last path of narrow rows: a wave holds 64 >> lg points, 1 << lg lanes of each along the channels (the least power
// of two that holds them, at most 64), and every lane derives its point's corners itself.  (One channel: the volume as it lies.)
// ---------------------------------------------------------------------------
template <int ND>
struct RowCorners {
  static constexpr int N = 1 << ND;
  int off[N];  // cells; 0 for an absent corner
  float w[N];  // 0 for an absent corner
  unsigned present;
};

template <typename T, int ND>
__device__ __forceinline__ RowCorners<ND> row_corners(const NdGeo& g, const T* coord_b, bool valid, NdPoint<float>& p) {
  p = small_point<T, ND>(g, coord_b);
  RowCorners<ND> r;
  r.present = 0u;
#pragma unroll
  for (int i = 0; i < RowCorners<ND>::N; ++i) {
    long o = 0;
    float w = 0.f;
    const bool ok = valid && p.inside && corner<float>(g, p, (unsigned)i, -1, o, w);
    r.off[i] = ok ? (int)o : 0;
    r.w[i] = ok ? w : 0.f;
    r.present |= ok ? 1u << i : 0u;
  }
  return r;
}

// Sum over aligned groups of 1 << lg lanes, for every lane
__device__ __forceinline__ float group_sum(float v, int lg) {
  auto add = [&](auto ctrl) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  if (lg > 0) add(std::integral_constant<int, 0xb1>{});   // quad_perm: the neighbour
  if (lg > 1) add(std::integral_constant<int, 0x4e>{});   // quad_perm: the other pair
  if (lg > 2) add(std::integral_constant<int, 0x141>{});  // row_half_mirror: the other four
  if (lg > 3) add(std::integral_constant<int, 0x140>{});  // row_mirror: the other eight
  if (lg > 4) v += __shfl_xor(v, 16, 64);
  if (lg > 5) v += __shfl_xor(v, 32, 64);
  return v;
}

template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_forward_rows_kernel(NdGeo g, const T* __restrict__ data_cl,
                                                                 const T* __restrict__ coord, T* __restrict__ out, int lg) {
  g.dims = ND;
  const long b = (long)blockIdx.x * (kBlock >> lg) + (threadIdx.x >> lg);
  if (b >= g.batch) return;
  NdPoint<float> p;
  const RowCorners<ND> r = row_corners<T, ND>(g, coord + b * ND, true, p);
  for (int c = threadIdx.x & ((1 << lg) - 1); c < g.channel; c += 1 << lg) {
    T raw[RowCorners<ND>::N];
#pragma unroll
    for (int i = 0; i < RowCorners<ND>::N; ++i) raw[i] = data_cl[(size_t)r.off[i] * g.channel + c];
    float acc = 0.f;
#pragma unroll
    for (int i = 0; i < RowCorners<ND>::N; ++i) acc += r.w[i] * (r.present >> i & 1u ? (float)ld(&raw[i]) : 0.f);
    st(out + b * g.channel + c, acc);
  }
}

template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_coord_rows_kernel(NdGeo g, const T* __restrict__ gout,
                                                                    const T* __restrict__ data_cl,
                                                                    const T* __restrict__ coord, T* __restrict__ gcoord, int lg) {
  constexpr int N = RowCorners<ND>::N;
  g.dims = ND;
  const long at = (long)blockIdx.x * (kBlock >> lg) + (threadIdx.x >> lg);
  const long b = min(at, g.batch - 1);  // (no lane leaves before the sum over its group)
  NdPoint<float> p;
  const RowCorners<ND> r = row_corners<T, ND>(g, coord + b * ND, true, p);
  float s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = 0.f;
  const int lane = threadIdx.x & ((1 << lg) - 1);
  for (int c = lane; c < g.channel; c += 1 << lg) {
    T raw[N];
    const T graw = gout[b * g.channel + c];
#pragma unroll
    for (int i = 0; i < N; ++i) raw[i] = data_cl[(size_t)r.off[i] * g.channel + c];
    const float go = ld(&graw);
#pragma unroll
    for (int i = 0; i < N; ++i) s[i] += r.present >> i & 1u ? go * ld(&raw[i]) : 0.f;
  }
  float gd[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) {
    gd[d] = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      long o;
      float w;
      if ((r.present >> i & 1u) && corner<float>(g, p, (unsigned)i, d, o, w)) gd[d] += s[i] * w;  // ND.cu:161,165
    }
    gd[d] = group_sum(gd[d], lg);
  }
  if (lane == 0 && at < g.batch)
#pragma unroll
    for (int d = 0; d < ND; ++d) st(gcoord + b * ND + d, gd[d]);
}

// grad data with the sums in LDS: a workgroup takes a share of the points, a slice of the channels and, of volumes that do
// not fit for one channel, a range of the cells, and holds the sums [cell][pitch] of that; they leave planar, one copy per
// share, and are added up in order.  Where points meet in cells, float atomics on memory take the additions one by one.  The
// sums are doubles: an LDS add of a wave takes 5 - 9 ns of the CU in double, 81 in float (the same addresses, 16 waves).
template <typename T, int ND>
__global__ __launch_bounds__(1024) void nd_grad_data_lds_kernel(NdGeo g, const T* __restrict__ gout, const T* __restrict__ coord,
                                                                float* __restrict__ partial, int lg, int slice_ch, int pitch,
                                                                int slices, int range, int ranges, long share) {
  constexpr int N = RowCorners<ND>::N, PU = 4;  // points of a lane in flight
  extern __shared__ __align__(16) unsigned char nd_lds_sums[];
  double* img = reinterpret_cast<double*>(nd_lds_sums);
  g.dims = ND;
  const int cells = (int)g.prod_shape;
  const int slice = blockIdx.x % slices, from = blockIdx.x / slices % ranges * range, part = blockIdx.x / slices / ranges;
  const int own = min(range, cells - from);
  const int c0 = slice * slice_ch, nc = min(slice_ch, g.channel - c0);
  for (int e = threadIdx.x; e < own * pitch; e += 1024) img[e] = 0.0;
  __syncthreads();
  const int lane = threadIdx.x & ((1 << lg) - 1), points = 1024 >> lg;
  const long b1 = min(g.batch, (part + 1) * share);
  for (long b0 = part * share + (threadIdx.x >> lg); b0 < b1; b0 += PU * points) {
    T x[PU][ND], graw[PU];
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const long b = min(b0 + u * points, b1 - 1);
#pragma unroll
      for (int d = 0; d < ND; ++d) x[u][d] = coord[b * ND + d];
      graw[u] = gout[b * g.channel + c0 + min(lane, nc - 1)];
    }
#pragma unroll
    for (int u = 0; u < PU; ++u) {
      const long b = b0 + u * points;
      if (b >= b1) break;
      NdPoint<float> p;
      const RowCorners<ND> r = row_corners<T, ND>(g, x[u], true, p);
      for (int c = lane; c < nc; c += 1 << lg) {
        const float go = c == lane ? ld(&graw[u]) : ld(gout + b * g.channel + c0 + c);
#pragma unroll
        for (int i = 0; i < N; ++i) {
          const int at = r.off[i] - from;
          if ((r.present >> i & 1u) && (unsigned)at < (unsigned)own) atomicAdd(img + at * pitch + c, (double)(r.w[i] * go));
        }
      }
    }
  }
  __syncthreads();
  for (int c = 0; c < nc; ++c) {
    float* out = partial + ((size_t)part * g.channel + c0 + c) * cells + from;
    for (int e = threadIdx.x; e < own; e += 1024) out[e] = (float)img[e * pitch + c];
  }
}

// ---------------------------------------------------------------------------
// binned channel-last path: many points per cell of the volume
//
// With more points than cells, points that fall into the same cell read (forward, grad coord)
// or update (grad data) the same 2^n corner rows.  The points are therefore sorted by cell
// first -- a radix sort of (key, point index) pairs (radix_*_kernel below), the key being the cell's low corner,
// (low[d] + 1) over extents shape[d] + 1, plus one last bin for the points outside the volume;
// a radix sort rather than a counting sort with atomics because the points of a real workload
// may all sit in a handful of cells -- and a wave walks 64
// consecutive points of the sorted order, lanes over channels: the corner rows stay in
// registers while the cell does not change (forward, grad coord), and the input gradient of a
// cell's corners is summed in registers and leaves as one atomic per corner and channel when the
// cell changes (grad data).  Results go to / come from each point's original row.
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ int point_bin(const NdGeo& g, const T* coord_b, int nbins) {
  const NdPoint<float> p = load_point<T, float>(g, coord_b);
  if (!p.inside) return nbins - 1;
  int key = 0;
#pragma unroll
  for (int d = 0; d < kClMaxDims; ++d)
    if (d < g.dims) key = key * (g.shape[d] + 1) + p.low[d] + 1;
  return key;
}

// What a wave of the binned kernels knows about its 64 sorted points: lane q holds point q.  An XCD walks one contiguous
// eighth of the sorted points, so that the corner rows of neighbouring cells are read into one L2 (2^20 points of a 32^3 volume of 64
// channels, 8 MB: forward 137 -> 131 us a call).
template <typename T>
struct BinnedWave {
  int npts, id, key;
  ClCorners cc;
  // the wave's `sub`-th chunk of 64 points when a wave walks `per_wave` consecutive chunks
  __device__ __forceinline__ bool init(const NdGeo& g, const T* coord, const int* order, int nbins,
                                       int per_wave = 1, int sub = 0) {
    const int lane = threadIdx.x & 63;
    // (the same for the wave's lanes, which the compiler does not see: loops and row addresses would be per lane)
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const long wave0 = (((long)logical_block((int)gridDim.x) * (kBlock / 64) + wave) * per_wave + sub) * 64;
    if (wave0 >= g.batch) return false;
    npts = (int)min(64L, g.batch - wave0);
    const bool valid = lane < npts;
    id = valid ? order[wave0 + lane] : 0;
    cc = cl_corners<T>(g, coord, id, valid);
    key = valid ? point_bin<T>(g, coord + (long)id * g.dims, nbins) : -1;
    return true;
  }
  __device__ __forceinline__ int key_of(int q) const { return __builtin_amdgcn_readlane(key, q); }
  __device__ __forceinline__ long id_of(int q) const { return __builtin_amdgcn_readlane(id, q); }
  __device__ __forceinline__ int off_of(int i, int q) const { return __builtin_amdgcn_readlane(cc.off[i], q); }
  __device__ __forceinline__ float w_of(int i, int q) const {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, cc.w[i]), q));
  }
};

// Makes the corner rows just loaded count as used here, so that the wait for them sits in the
// (rare) cell-change branch.  Otherwise the compiler waits for every outstanding memory operation
// at the first use after the branch, for every point, and that includes the point's own store.
__device__ __forceinline__ void settle(float (&v)[kClCorners]) {
  asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7]));
}

template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_forward_binned_kernel(NdGeo g, const T* __restrict__ data_cl,
                                                                   const T* __restrict__ coord,
                                                                   const int* __restrict__ order, int nbins,
                                                                   T* __restrict__ out) {
  g.dims = ND;
  BinnedWave<T> wv;
  if (!wv.init(g, coord, order, nbins)) return;
  const int lane = threadIdx.x & 63, ncorner = 1 << g.dims;
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    const int c = c0 + lane;
    const bool cin = c < g.channel;
    float v[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) v[i] = 0.f;
    int cur = -2;
    for (int q = 0; q < wv.npts; ++q) {
      const int key = wv.key_of(q);
      if (key != cur) {  // wave-uniform: a new cell, fetch its corner rows
        cur = key;
#pragma unroll
        for (int i = 0; i < kClCorners; ++i)
          v[i] = (cin && i < ncorner) ? ld(data_cl + (size_t)wv.off_of(i, q) * g.channel + c) : 0.f;
        settle(v);
      }
      float acc = 0.f;
#pragma unroll
      for (int i = 0; i < kClCorners; ++i) acc += wv.w_of(i, q) * v[i];
      if (cin) st(out + wv.id_of(q) * g.channel + c, acc);
    }
  }
}

template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_data_binned_kernel(NdGeo g, const T* __restrict__ gout,
                                                                     const T* __restrict__ coord,
                                                                     const int* __restrict__ order, int nbins,
                                                                     float* __restrict__ gdata_cl, int per_wave) {
  g.dims = ND;
  const int lane = threadIdx.x & 63, ncorner = 1 << g.dims;
  constexpr int PU = 8;  // output-gradient rows in flight
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    const int c = c0 + lane;
    const bool cin = c < g.channel;
    float acc[kClCorners];
    int at[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) acc[i] = 0.f, at[i] = 0;
    int cur = -2;
#define DK_FLUSH()                                                                             \
  _Pragma("unroll") for (int i = 0; i < kClCorners; ++i) if (cin && i < ncorner && acc[i] != 0.f) \
      atomicAdd(gdata_cl + (size_t)at[i] * g.channel + c, acc[i])
    // the sums of a cell stay in registers across the wave's chunks: when thousands of points
    // share a cell, fewer waves send fewer atomics to the same rows
    for (int sub = 0; sub < per_wave; ++sub) {
      BinnedWave<T> wv;
      if (!wv.init(g, coord, order, nbins, per_wave, sub)) break;
      for (int q0 = 0; q0 < wv.npts; q0 += PU) {
        float go[PU];
#pragma unroll
        for (int u = 0; u < PU; ++u)
          go[u] = (cin && q0 + u < wv.npts) ? ld(gout + wv.id_of(min(q0 + u, wv.npts - 1)) * g.channel + c) : 0.f;
#pragma unroll
        for (int u = 0; u < PU; ++u) {
          const int q = q0 + u;
          if (q < wv.npts) {
            const int key = wv.key_of(q);
            if (key != cur) {  // wave-uniform: the sums of the finished cell leave
              cur = key;
              int nat[kClCorners];
              float nacc[kClCorners];
#pragma unroll
              for (int i = 0; i < kClCorners; ++i) nacc[i] = 0.f, nat[i] = wv.off_of(i, q);
              // The next cell in key order is mostly the neighbour along the last dimension, whose
              // low-side rows are this cell's high-side rows: those sums stay in registers (rows are
              // matched by their offsets, so any other successor just flushes everything).  Atomics
              // on the volume are what bounds this kernel; this halves them.
#define DK_CARRY(HB)                                                                            \
  _Pragma("unroll") for (int i = 0; i < kClCorners; ++i) {                                      \
    if ((i & (HB)) && i < 2 * (HB)) {                                                           \
      if (at[i] == nat[i - (HB)]) {                                                             \
        nacc[i - (HB)] = acc[i];                                                                \
        acc[i] = 0.f;                                                                           \
      }                                                                                         \
    }                                                                                           \
  }
              if (g.dims == 3) {
                DK_CARRY(4)
              } else if (g.dims == 2) {
                DK_CARRY(2)
              } else {
                DK_CARRY(1)
              }
#undef DK_CARRY
              DK_FLUSH();
#pragma unroll
              for (int i = 0; i < kClCorners; ++i) acc[i] = nacc[i], at[i] = nat[i];
            }
#pragma unroll
            for (int i = 0; i < kClCorners; ++i) acc[i] += wv.w_of(i, q) * go[u];
          }
        }
      }
    }
    DK_FLUSH();
#undef DK_FLUSH
  }
}

// grad coord on the sorted points.  Per cell the eight corner rows are turned into the
// coefficients of the multilinear polynomial,
//   value = c0 + c1 f0 + c2 f1 + c3 f2 + c4 f0 f1 + c5 f0 f2 + c6 f1 f2 + c7 f0 f1 f2
// (f = fractional position; absent corners and absent dimensions enter as zeros, which is what
// skipping them amounts to), so that a point's three partial derivatives cost nine fused
// multiply-adds per channel instead of eight corner products, and three wave reductions
// instead of eight.
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_coord_binned_kernel(NdGeo g, const T* __restrict__ gout,
                                                                      const T* __restrict__ data_cl,
                                                                      const T* __restrict__ coord,
                                                                      const int* __restrict__ order, int nbins,
                                                                      T* __restrict__ gcoord) {
  g.dims = ND;
  BinnedWave<T> wv;
  if (!wv.init(g, coord, order, nbins)) return;
  const int lane = threadIdx.x & 63;
  const bool valid = lane < wv.npts;
  // lane <-> point: fractional position and its pairwise products
  NdPoint<float> p;
  p.inside = false;
#pragma unroll
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) p.frac[d] = 0.f, p.low[d] = 0;
  if (valid) p = load_point<T, float>(g, coord + (long)wv.id * g.dims);
  const float f0 = p.frac[0], f1 = p.frac[1], f2 = p.frac[2];
  const float f01 = f0 * f1, f02 = f0 * f2, f12 = f1 * f2;
  auto uni = [](float v, int q) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), q));
  };
  constexpr int PU = 4;
  float gd0 = 0.f, gd1 = 0.f, gd2 = 0.f;  // of point q, in lane q
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    const int c = c0 + lane;
    const bool cin = c < g.channel;
    float k1 = 0.f, k2 = 0.f, k3 = 0.f, k4 = 0.f, k5 = 0.f, k6 = 0.f, k7 = 0.f;
    int cur = -2;
    for (int q0 = 0; q0 < wv.npts; q0 += PU) {
      float go[PU];
#pragma unroll
      for (int u = 0; u < PU; ++u)
        go[u] = (cin && q0 + u < wv.npts) ? ld(gout + wv.id_of(min(q0 + u, wv.npts - 1)) * g.channel + c) : 0.f;
#pragma unroll
      for (int u = 0; u < PU; ++u) {
        const int q = q0 + u;
        if (q < wv.npts) {
          const int key = wv.key_of(q);
          if (key != cur) {
            cur = key;
            float v[kClCorners];
            const unsigned present = (unsigned)__builtin_amdgcn_readlane((int)wv.cc.present, q);
#pragma unroll
            for (int i = 0; i < kClCorners; ++i)
              v[i] = (cin && (present >> i & 1u)) ? ld(data_cl + (size_t)wv.off_of(i, q) * g.channel + c) : 0.f;
            settle(v);
            // corner index: bit d = high side of dimension d
            k1 = v[1] - v[0];
            k2 = v[2] - v[0];
            k3 = v[4] - v[0];
            k4 = (v[3] - v[2]) - k1;
            k5 = (v[5] - v[4]) - k1;
            k6 = (v[6] - v[4]) - k2;
            k7 = ((v[7] - v[6]) - (v[5] - v[4])) - k4;
          }
          const float u0 = uni(f0, q), u1 = uni(f1, q), u2 = uni(f2, q);
          const float u01 = uni(f01, q), u02 = uni(f02, q), u12 = uni(f12, q);
          const float d0 = fmaf(k7, u12, fmaf(k5, u2, fmaf(k4, u1, k1)));
          const float d1 = fmaf(k7, u02, fmaf(k6, u2, fmaf(k4, u0, k2)));
          const float d2 = fmaf(k7, u01, fmaf(k6, u1, fmaf(k5, u0, k3)));
          const float t0 = wave_sum(go[u] * d0);
          if (lane == q) gd0 += t0;
          if (g.dims > 1) {
            const float t1 = wave_sum(go[u] * d1);
            if (lane == q) gd1 += t1;
          }
          if (g.dims > 2) {
            const float t2 = wave_sum(go[u] * d2);
            if (lane == q) gd2 += t2;
          }
        }
      }
    }
  }
  if (!valid) return;
  const float gd[3] = {gd0, gd1, gd2};
#pragma unroll
  for (int d = 0; d < kClMaxDims; ++d)
    if (d < g.dims) st(gcoord + (long)wv.id * g.dims + d, p.inside ? gd[d] : 0.f);
}

// Orders LDS writes of a wave before the reads of its other lanes (a wave owns its LDS slice).
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

typedef float nd4 __attribute__((ext_vector_type(4)));

// Sum over the 16 lanes of a row, in each of them
__device__ __forceinline__ float row_sum(float v) {
  auto add = [&](auto ctrl) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xf, 0xf, true));
  };
  add(std::integral_constant<int, 0xB1>{});   // quad_perm [1,0,3,2]
  add(std::integral_constant<int, 0x4E>{});   // quad_perm [2,3,0,1]
  add(std::integral_constant<int, 0x141>{});  // row_half_mirror
  add(std::integral_constant<int, 0x140>{});  // row_mirror
  return v;
}

// grad coord on the sorted points with the sums over the channels on the matrix cores (fp32,
// channel count a multiple of 64).  With the polynomial coefficients k1 .. k7 of a cell (see
// nd_grad_coord_binned_kernel) a point's derivatives are
//   d0 = S1 + f1 S4 + f2 S5 + f1 f2 S7,  d1 = S2 + f0 S4 + f2 S6 + f0 f2 S7,
//   d2 = S3 + f0 S5 + f1 S6 + f0 f1 S7,       S_m = sum_c gout[c] * k_m[c],
// and the S_m of 16 points of one cell are a 16 x 64 by 64 x 16 product: v_mfma_f32_16x16x4_f32 with
// lane l supplying gout[point l % 16][channel 16 (l / 16) + step] and k_{l % 16}[the same channel]
// over 16 steps (step 4 j + i takes channel 16 j + 4 (l / 16) + i of the block, the same for both operands, so that
// the four lanes of a point read 64 contiguous bytes of its row with each of their four 16-byte loads; the
// coefficients go through the wave's LDS slice).  The three wave reductions per point and channel
// block of the VALU kernel (75 VALU instructions per point) become one MFMA per point.
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 4))) void nd_grad_coord_mfma_kernel(NdGeo g, const float* __restrict__ gout,
                                                                    const float* __restrict__ data_cl,
                                                                    const float* __restrict__ coord,
                                                                    const int* __restrict__ order, int nbins,
                                                                    float* __restrict__ gcoord) {
  g.dims = ND;
  __shared__ __align__(16) float s_coef[kBlock / 64][8][64];  // [wave][m][channel of the block]
  __shared__ __align__(16) float s_sum[kBlock / 64][16][16];  // [wave][point of the batch][m]
  BinnedWave<float> wv;
  if (!wv.init(g, coord, order, nbins)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float(*coef)[64] = s_coef[wave];
  float(*sums)[16] = s_sum[wave];
  const bool valid = lane < wv.npts;
  NdPoint<float> p;
  p.inside = false;
#pragma unroll
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) p.frac[d] = 0.f, p.low[d] = 0;
  if (valid) p = load_point<float, float>(g, coord + (long)wv.id * g.dims);
  const float f0 = p.frac[0], f1 = p.frac[1], f2 = p.frac[2];
  const float f01 = f0 * f1, f02 = f0 * f2, f12 = f1 * f2;
  const int pr = lane & 15, kg = lane >> 4;  // MFMA row (point of the batch / coefficient index), K group
  float gd0 = 0.f, gd1 = 0.f, gd2 = 0.f;     // of point q, in lane q

  int qs = 0;
  while (qs < wv.npts) {
    // the run of points in the cell of point qs: the keys are sorted
    const int key = wv.key_of(qs);
    const int qe = qs + (int)__popcll(__ballot(wv.key == key));
    const unsigned present = (unsigned)__builtin_amdgcn_readlane((int)wv.cc.present, qs);
    nd4 acc[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) acc[b] = nd4{0.f, 0.f, 0.f, 0.f};
    for (int c0 = 0; c0 < g.channel; c0 += 64) {
      // this lane's 16 channels of its point in batch b: issued two batches ahead of their MFMAs,
      // the first two before the cell's corner rows, so that the two latencies overlap (two buffers in turn:
      // with four the kernel takes 168 registers and a SIMD holds three waves of it; this is four)
      float av[2][16];
#define DK_ND_LOAD_A(b)                                                                          \
  if (qs + 16 * (b) < qe) {                                                                      \
    const int q_ = qs + 16 * (b) + pr;                                                           \
    const bool on_ = q_ < qe;                                                                    \
    const long id_ = __shfl(wv.id, on_ ? q_ : qs);                                               \
    const float4* rowp_ = reinterpret_cast<const float4*>(gout + id_ * g.channel + c0 + 4 * kg); \
    _Pragma("unroll") for (int j = 0; j < 4; ++j) {                                              \
      const float4 t_ = rowp_[4 * j];  /* the four lanes of a point: 64 contiguous bytes */      \
      av[(b) & 1][4 * j] = on_ ? t_.x : 0.f;                                                     \
      av[(b) & 1][4 * j + 1] = on_ ? t_.y : 0.f;                                                 \
      av[(b) & 1][4 * j + 2] = on_ ? t_.z : 0.f;                                                 \
      av[(b) & 1][4 * j + 3] = on_ ? t_.w : 0.f;                                                 \
    }                                                                                            \
  }
#define DK_ND_MFMA(b)                                                                            \
  if (qs + 16 * (b) < qe) {                                                                      \
    _Pragma("unroll") for (int s_ = 0; s_ < 16; ++s_)                                            \
      acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(av[(b) & 1][s_], bv[s_], acc[b], 0, 0, 0);   \
  }
      DK_ND_LOAD_A(0)
      DK_ND_LOAD_A(1)
      {
        float v[kClCorners];
#pragma unroll
        for (int i = 0; i < kClCorners; ++i)
          v[i] = (present >> i & 1u) ? data_cl[(size_t)wv.off_of(i, qs) * g.channel + c0 + lane] : 0.f;
        // corner index: bit d = high side of dimension d
        const float k1 = v[1] - v[0], k2 = v[2] - v[0], k3 = v[4] - v[0];
        const float k4 = (v[3] - v[2]) - k1, k5 = (v[5] - v[4]) - k1, k6 = (v[6] - v[4]) - k2;
        const float k7 = ((v[7] - v[6]) - (v[5] - v[4])) - k4;
        wave_lds_sync();  // the previous block's coefficient reads are done
        coef[1][lane] = k1;
        coef[2][lane] = k2;
        coef[3][lane] = k3;
        coef[4][lane] = k4;
        coef[5][lane] = k5;
        coef[6][lane] = k6;
        coef[7][lane] = k7;
        wave_lds_sync();
      }
      float bv[16];
      {
        const bool row = pr >= 1 && pr < 8;  // rows 0 and 8 .. 15 of the coefficient matrix are zero
        const float4* src = reinterpret_cast<const float4*>(&coef[row ? pr : 1][4 * kg]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float4 t = src[4 * j];
          bv[4 * j] = row ? t.x : 0.f;
          bv[4 * j + 1] = row ? t.y : 0.f;
          bv[4 * j + 2] = row ? t.z : 0.f;
          bv[4 * j + 3] = row ? t.w : 0.f;
        }
      }
      DK_ND_MFMA(0)
      DK_ND_LOAD_A(2)
      DK_ND_MFMA(1)
      DK_ND_LOAD_A(3)
      DK_ND_MFMA(2)
      DK_ND_MFMA(3)
#undef DK_ND_LOAD_A
#undef DK_ND_MFMA
    }
    // D[point 4 (l / 16) + r][m = l % 16] in register r of lane l: through LDS to the points' lanes
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      if (qs + 16 * b < qe) {
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < 4; ++r) sums[4 * kg + r][pr] = acc[b][r];
        wave_lds_sync();
        const int mine = lane - (qs + 16 * b);
        if (mine >= 0 && mine < 16 && lane < qe) {
          const float4 lo4 = *reinterpret_cast<const float4*>(&sums[mine][0]);
          const float4 hi4 = *reinterpret_cast<const float4*>(&sums[mine][4]);
          const float S1 = lo4.y, S2 = lo4.z, S3 = lo4.w, S4 = hi4.x, S5 = hi4.y, S6 = hi4.z, S7 = hi4.w;
          gd0 += fmaf(f12, S7, fmaf(f2, S5, fmaf(f1, S4, S1)));
          gd1 += fmaf(f02, S7, fmaf(f2, S6, fmaf(f0, S4, S2)));
          gd2 += fmaf(f01, S7, fmaf(f1, S6, fmaf(f0, S5, S3)));
        }
      }
    }
    qs = qe;
  }
  if (!valid) return;
  const float gd[3] = {gd0, gd1, gd2};
#pragma unroll
  for (int d = 0; d < kClMaxDims; ++d)
    if (d < g.dims) gcoord[(long)wv.id * g.dims + d] = p.inside ? gd[d] : 0.f;
}

// grad data on the sorted points on the matrix cores (fp32, channel count a multiple of 64): the
// sums of a cell's corner rows over the points of a run are a product
//   D[corner][channel] = sum_p w_corner(p) * gout[p][channel],
// done 16 points at a time by v_mfma_f32_16x16x4_f32: lane l supplies w_{l % 16}(point 4 step + l / 16)
// (from the wave's LDS copy of its points' corner weights; rows 8 .. 15 are zero) and the four
// channels 4 (l % 16) .. + 3 of that point's gout row (one 16-byte load; the 16 lanes of a point read
// its 256-byte row), one MFMA per channel of the quad.  The VALU kernel spends its time on the
// per-point broadcasts (v_readlane of eight weights, key and row index per point).
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_grad_data_mfma_kernel(NdGeo g, const float* __restrict__ gout,
                                                                   const float* __restrict__ coord,
                                                                   const int* __restrict__ order, int nbins,
                                                                   float* __restrict__ gdata_cl, int per_wave) {
  g.dims = ND;
  __shared__ __align__(16) float s_w[kBlock / 64][64][kClCorners];  // [wave][point][corner]
  __shared__ __align__(16) float s_d[kBlock / 64][kClCorners][64];  // [wave][corner][channel]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pr = lane & 15, kg = lane >> 4, ncorner = 1 << g.dims;
  float(*wl)[kClCorners] = s_w[wave];
  float(*dl)[64] = s_d[wave];
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    nd4 acc[4];
#pragma unroll
    for (int cb = 0; cb < 4; ++cb) acc[cb] = nd4{0.f, 0.f, 0.f, 0.f};
    int at[kClCorners];
#pragma unroll
    for (int i = 0; i < kClCorners; ++i) at[i] = 0;
    int cur = -2;
    // D[corner 4 (l / 16) + r][channel 4 (l % 16) + cb] sits in acc[cb][r] of lane l: through LDS to
    // one lane per channel, which sends the corner rows' sums
#define DK_FLUSH()                                                                                   \
  if (cur != -2) {                                                                                   \
    wave_lds_sync();                                                                                 \
    if (kg < 2) {                                                                                    \
      _Pragma("unroll") for (int r = 0; r < 4; ++r)                                                  \
        *reinterpret_cast<float4*>(&dl[4 * kg + r][4 * pr]) = make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]); \
    }                                                                                                \
    wave_lds_sync();                                                                                 \
    _Pragma("unroll") for (int i = 0; i < kClCorners; ++i) {                                         \
      if (i < ncorner) {                                                                             \
        const float v_ = dl[i][lane];                                                                \
        if (v_ != 0.f) atomicAdd(gdata_cl + (size_t)at[i] * g.channel + c0 + lane, v_);              \
      }                                                                                              \
    }                                                                                                \
  }
    // the sums of a cell stay in registers across the wave's chunks: when thousands of points
    // share a cell, fewer waves send fewer atomics to the same rows
    for (int sub = 0; sub < per_wave; ++sub) {
      BinnedWave<float> wv;
      if (!wv.init(g, coord, order, nbins, per_wave, sub)) break;
      wave_lds_sync();  // the previous chunk's weight reads are done
      *reinterpret_cast<float4*>(&wl[lane][0]) = make_float4(wv.cc.w[0], wv.cc.w[1], wv.cc.w[2], wv.cc.w[3]);
      *reinterpret_cast<float4*>(&wl[lane][4]) = make_float4(wv.cc.w[4], wv.cc.w[5], wv.cc.w[6], wv.cc.w[7]);
      wave_lds_sync();
      int qs = 0;
      while (qs < wv.npts) {
        const int key = wv.key_of(qs);
        const int qe = qs + (int)__popcll(__ballot(wv.key == key));  // the keys are sorted
        if (key != cur) {
          DK_FLUSH();
          cur = key;
#pragma unroll
          for (int i = 0; i < kClCorners; ++i) at[i] = wv.off_of(i, qs);
#pragma unroll
          for (int cb = 0; cb < 4; ++cb) acc[cb] = nd4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
          if (qs + 16 * b < qe) {  // wave-uniform
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              const int q = qs + 16 * b + 4 * s + kg;
              const bool on = q < qe;
              const int qc = on ? q : qs;
              const long id = __shfl(wv.id, qc);
              const float4 t = *reinterpret_cast<const float4*>(gout + id * g.channel + c0 + 4 * pr);
              const float a = (on && pr < kClCorners) ? wl[qc][pr & (kClCorners - 1)] : 0.f;
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.x, acc[0], 0, 0, 0);
              acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.y, acc[1], 0, 0, 0);
              acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.z, acc[2], 0, 0, 0);
              acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.w, acc[3], 0, 0, 0);
            }
          }
        }
        qs = qe;
      }
    }
    DK_FLUSH();
#undef DK_FLUSH
  }
}

// Both gradients on the sorted points from one read of gout, whose 256-byte rows in the points' original order are most
// of what either kernel above moves (fp32, channel count a multiple of 64).  Grad data as in nd_grad_data_mfma_kernel; grad
// coord takes the operand that the products need, four channels of a point per lane: the lane multiplies them with its
// channels' seven coefficients (28 multiply-adds), forms the three derivatives of its share and a DPP sum over the 16
// lanes of the point completes them.  What bounds it is the chain of a wave from one cell to the next: the rows of the next 16
// points and the corner rows of the next cell (a channel per lane; the coefficients take their four-channel form through
// LDS) are asked for before the present ones are worked off, always the same number of loads, so that a wait counts
// down to the older ones: 2^20 points x 64 channels of a 32^3 volume 161 us, 195 with loads by need and a cell's rows when
// it begins (the two kernels above: 114 + 95).  Four waves per SIMD hold the grid of one round; 76 bytes per lane of set-up spill
// for that.  A point outside the grid takes part in nothing.
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 4))) void nd_backward_mfma_kernel(
    NdGeo g, const float* __restrict__ gout, const float* __restrict__ data_cl, const float* __restrict__ coord,
    const int* __restrict__ order, int nbins, float* __restrict__ gdata_cl, float* __restrict__ gcoord, int per_wave) {
  g.dims = ND;
  constexpr int NC = 1 << ND;
  constexpr int KS = ND == 3 ? 7 : ND == 2 ? 3 : 1;                 // coefficients besides the constant one
  __shared__ __align__(16) float s_w[kBlock / 64][64][kClCorners];  // [wave][point][corner]
  __shared__ float4 s_p[kBlock / 64][64];                           // [wave][point]: fractions, then derivatives; the point's row
  __shared__ __align__(16) float s_d[kBlock / 64][kClCorners][64];  // [wave][corner][channel], or the coefficients [m][channel]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pr = lane & 15, kg = lane >> 4;
  float(*wl)[kClCorners] = s_w[wave];
  float4* pl = s_p[wave];
  float(*dl)[64] = s_d[wave];
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    nd4 acc[4], k[KS];  // the cell's sums (corner 4 kg + r of channel 4 pr + cb in acc[cb][r]) and coefficients
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = nd4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KS; ++i) k[i] = nd4{0.f, 0.f, 0.f, 0.f};
    int at[NC];
    unsigned present = 0u;  // corners of the cell that lie on the grid
#pragma unroll
    for (int i = 0; i < NC; ++i) at[i] = 0;
    int cur = -2;
    auto flush = [&] {
      if (!present) return;
      wave_lds_sync();
      if (4 * kg < NC) {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          *reinterpret_cast<float4*>(&dl[4 * kg + r][4 * pr]) = make_float4(acc[0][r], acc[1][r], acc[2][r], acc[3][r]);
      }
      wave_lds_sync();
#pragma unroll
      for (int i = 0; i < NC; ++i) {
        if (present >> i & 1u) {
          const float v = dl[i][lane];
          if (v != 0.f) atomicAdd(gdata_cl + (size_t)at[i] * g.channel + c0 + lane, v);
        }
      }
    };
    for (int sub = 0; sub < per_wave; ++sub) {
      BinnedWave<float> wv;
      if (!wv.init(g, coord, order, nbins, per_wave, sub)) break;
      const bool valid = lane < wv.npts;
      NdPoint<float> p;
      p.inside = false;
#pragma unroll
      for (int d = 0; d < DK_ND_MAX_DIMS; ++d) p.frac[d] = 0.f, p.low[d] = 0;
      if (valid) p = load_point<float, float>(g, coord + (long)wv.id * g.dims);
      wave_lds_sync();  // the previous chunk's reads are done
      *reinterpret_cast<float4*>(&wl[lane][0]) = make_float4(wv.cc.w[0], wv.cc.w[1], wv.cc.w[2], wv.cc.w[3]);
      *reinterpret_cast<float4*>(&wl[lane][4]) = make_float4(wv.cc.w[4], wv.cc.w[5], wv.cc.w[6], wv.cc.w[7]);
      pl[lane] = make_float4(p.frac[0], p.frac[1], p.frac[2], __int_as_float(wv.id));
      wave_lds_sync();
      auto run_end = [&](int q) {  // the keys are sorted
        return q < wv.npts ? q + (int)__popcll(__ballot(wv.key == wv.key_of(q))) : q;
      };
      // a lane's channels of the points q0 + kg, + 4, + 8, + 12 of the run that ends in front of qe
      float4 nxt[4];
      auto load = [&](int q0, int qe) {
        const int last = min(q0, wv.npts - 1);
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int q = q0 + 4 * s + kg;
          const long id = __float_as_int(pl[q < qe ? q : last].w);
          nxt[s] = *reinterpret_cast<const float4*>(gout + id * g.channel + c0 + 4 * pr);
        }
      };
      // the corner rows of point q's cell, channel c0 + lane (row 0 for a corner off the grid)
      float v[NC];
      int row[NC];
      unsigned on_grid = 0u;
      auto load_cell = [&](int q) {
        const int from = min(q, wv.npts - 1);
        on_grid = (unsigned)__builtin_amdgcn_readlane((int)wv.cc.present, from);
#pragma unroll
        for (int i = 0; i < NC; ++i) row[i] = wv.off_of(i, from);
#pragma unroll
        for (int i = 0; i < NC; ++i) v[i] = data_cl[(size_t)row[i] * g.channel + c0 + lane];
      };
      int q0 = 0, qe = run_end(0);
      bool start = true;  // of a run
      load_cell(q0);
      load(q0, qe);
      while (q0 < wv.npts) {
        float4 now[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) now[s] = nxt[s];
        if (start) {
          const int key = wv.key_of(q0);
          if (key != cur) {
            flush();
            cur = key;
            present = on_grid;
#pragma unroll
            for (int i = 0; i < NC; ++i) at[i] = row[i], v[i] = on_grid >> i & 1u ? v[i] : 0.f;
#pragma unroll
            for (int cb = 0; cb < 4; ++cb) acc[cb] = nd4{0.f, 0.f, 0.f, 0.f};
            // corner index: bit d = high side of dimension d (the coefficients of nd_grad_coord_binned_kernel)
            wave_lds_sync();
            const float k1 = v[1] - v[0];
            dl[0][lane] = k1;
            if constexpr (ND > 1) {
              const float k2 = v[2] - v[0], k4 = (v[3] - v[2]) - k1;
              dl[1][lane] = k2;
              dl[2][lane] = k4;
              if constexpr (ND > 2) {
                dl[3][lane] = v[4] - v[0];
                dl[4][lane] = (v[5] - v[4]) - k1;
                dl[5][lane] = (v[6] - v[4]) - k2;
                dl[6][lane] = ((v[7] - v[6]) - (v[5] - v[4])) - k4;
              }
            }
            wave_lds_sync();
#pragma unroll
            for (int i = 0; i < KS; ++i) k[i] = *reinterpret_cast<const nd4*>(&dl[i][4 * pr]);
          }
          load_cell(qe);
        }
        const int n0 = q0 + 16 < qe ? q0 + 16 : qe, ne = n0 < qe ? qe : run_end(n0);
        load(n0, ne);
        if (present) {
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            if (q0 + 4 * s < qe) {  // wave-uniform
              const int q = q0 + 4 * s + kg;
              const bool on = q < qe;
              const float4 t = now[s], f = pl[on ? q : q0];
              const float a = (on && pr < kClCorners) ? wl[q & 63][pr & (kClCorners - 1)] : 0.f;
              acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.x, acc[0], 0, 0, 0);
              acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.y, acc[1], 0, 0, 0);
              acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.z, acc[2], 0, 0, 0);
              acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, t.w, acc[3], 0, 0, 0);
              float S[KS];  // of k1, k2, k4, k3, k5, k6, k7
#pragma unroll
              for (int m = 0; m < KS; ++m) S[m] = fmaf(t.w, k[m][3], fmaf(t.z, k[m][2], fmaf(t.y, k[m][1], t.x * k[m][0])));
              float d[3] = {S[0], 0.f, 0.f};
              if constexpr (ND == 2) d[0] = fmaf(f.y, S[2], S[0]), d[1] = fmaf(f.x, S[2], S[1]);
              if constexpr (ND == 3) {
                d[0] = fmaf(f.y * f.z, S[6], fmaf(f.z, S[4], fmaf(f.y, S[2], S[0])));
                d[1] = fmaf(f.x * f.z, S[6], fmaf(f.z, S[5], fmaf(f.x, S[2], S[1])));
                d[2] = fmaf(f.x * f.y, S[6], fmaf(f.y, S[5], fmaf(f.x, S[4], S[3])));
              }
#pragma unroll
              for (int i = 0; i < ND; ++i) d[i] = row_sum(d[i]);
              if (on && pr == 0) *reinterpret_cast<float3*>(&pl[q]) = make_float3(d[0], d[1], d[2]);
            }
          }
        }
        start = n0 == qe;
        q0 = n0, qe = ne;
      }
      wave_lds_sync();
      if (valid) {
        const float4 r = pl[lane];
        const float d[3] = {r.x, r.y, r.z};
#pragma unroll
        for (int i = 0; i < ND; ++i) {
          float* to = gcoord + (long)wv.id * ND + i;
          *to = (c0 ? *to : 0.f) + (p.inside ? d[i] : 0.f);
        }
      }
    }
    flush();
  }
}

// forward on the sorted points on the matrix cores (fp32, channel count a multiple of 64): for the
// points of a cell run,
//   out[p][channel] = sum_corner w_corner(p) * row_corner[channel],
// 16 points at a time: lane l supplies w_{4 step + l / 16}(point l % 16) (from the wave's LDS copy of
// its points' corner weights) and the channels 4 (l % 16) .. + 3 of corner row 4 step + l / 16 (one
// 16-byte load per run), two steps of v_mfma_f32_16x16x4_f32 per channel of the quad; the results
// leave as 16-byte stores, the 16 lanes of a point writing its 256-byte row.
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void nd_forward_mfma_kernel(NdGeo g, const float* __restrict__ data_cl,
                                                                 const float* __restrict__ coord,
                                                                 const int* __restrict__ order, int nbins,
                                                                 float* __restrict__ out) {
  g.dims = ND;
  __shared__ __align__(16) float s_w[kBlock / 64][64][kClCorners];  // [wave][point][corner]
  BinnedWave<float> wv;
  if (!wv.init(g, coord, order, nbins)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int pr = lane & 15, kg = lane >> 4;
  float(*wl)[kClCorners] = s_w[wave];
  *reinterpret_cast<float4*>(&wl[lane][0]) = make_float4(wv.cc.w[0], wv.cc.w[1], wv.cc.w[2], wv.cc.w[3]);
  *reinterpret_cast<float4*>(&wl[lane][4]) = make_float4(wv.cc.w[4], wv.cc.w[5], wv.cc.w[6], wv.cc.w[7]);
  wave_lds_sync();
  for (int c0 = 0; c0 < g.channel; c0 += 64) {
    int qs = 0;
    while (qs < wv.npts) {
      const int key = wv.key_of(qs);
      const int qe = qs + (int)__popcll(__ballot(wv.key == key));  // the keys are sorted
      const unsigned present = (unsigned)__builtin_amdgcn_readlane((int)wv.cc.present, qs);
      float4 bq[2];
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const int o0 = wv.off_of(4 * s, qs), o1 = wv.off_of(4 * s + 1, qs), o2 = wv.off_of(4 * s + 2, qs),
                  o3 = wv.off_of(4 * s + 3, qs);
        const int o = kg == 0 ? o0 : kg == 1 ? o1 : kg == 2 ? o2 : o3;
        const bool on = present >> (4 * s + kg) & 1u;
        const float4 t = *reinterpret_cast<const float4*>(data_cl + (size_t)(on ? o : 0) * g.channel + c0 + 4 * pr);
        bq[s] = on ? t : make_float4(0.f, 0.f, 0.f, 0.f);
      }
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        if (qs + 16 * b < qe) {  // wave-uniform
          const int q = qs + 16 * b + pr;
          const bool onp = q < qe;
          const int qc = onp ? q : qs;
          nd4 acc[4];
#pragma unroll
          for (int cb = 0; cb < 4; ++cb) acc[cb] = nd4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int s = 0; s < 2; ++s) {
            const float a = onp ? wl[qc][4 * s + kg] : 0.f;
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[s].x, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[s].y, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[s].z, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[s].w, acc[3], 0, 0, 0);
          }
          // D[point 4 (l / 16) + r][channel 4 (l % 16) + cb] in acc[cb][r] of lane l
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int qo = qs + 16 * b + 4 * kg + r;
            const long id = __shfl(wv.id, qo < qe ? qo : qs);
            if (qo < qe)
              // non-temporal: the 256-byte rows are not read again, and written with the default policy they push
              // the volume out of L2 (config 5: forward 159 -> 150 us)
              __builtin_nontemporal_store(nd4{acc[0][r], acc[1][r], acc[2][r], acc[3][r]},
                                          reinterpret_cast<nd4*>(out + id * g.channel + c0 + 4 * pr));
          }
        }
      }
      qs = qe;
    }
  }
}

template <typename CT>
__global__ void nd_fill_zero_kernel(CT* p, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    p[i] = CT(0);
}
template <typename CT, typename T>
__global__ void nd_convert_kernel(const CT* __restrict__ a, T* __restrict__ out, long n) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    st(out + i, a[i]);
}

// ---------------------------------------------------------------------------
// Sort of the (cell key, point) pairs: a least-significant-digit radix sort in two passes of at
// most 9 bits (the keys have at most 18), each pass three kernels that launch nothing but
// themselves (so the sorted path can be captured into a graph).  What bounds it is the launches, 4 - 13 us each: the keys are formed
// with the first count, the tile sums added up in the scatter, grad data's image cleared by the transpose beside it (2^20 points
// of 64 x 32^3, forward and gradients: 306 us a pass with launches of their own, 297 without; tiles of 2048 keys instead of 4096, two
// waves per SIMD of 2^20 points, 293):
//   radix_keys_kernel (first pass), radix_count_kernel    a workgroup counts the digits of its tile of 2048 keys (LDS atomics) into
//                         table[digit][workgroup];
//   radix_scan_*_kernel   exclusive prefix sum of the table in (digit, workgroup) order (per tile of
//                         4096 entries, then over the tile sums -- those of up to 64 tiles in the scatter):
//                         where each workgroup's keys of each digit start in the output;
//   radix_scatter_kernel  stable scatter.  A wave owns 512 consecutive keys of the tile, 8 rounds
//                         of 64; the four waves' starts per digit follow from their counts; within
//                         a round a lane's rank among the lanes with its digit comes from nine
//                         ballots, and the first of them advances the wave's LDS counter.
// ---------------------------------------------------------------------------
constexpr int kSortTile = 2048, kSortWaveKeys = kSortTile / (kBlock / 64), kSortRounds = kSortWaveKeys / 64;
constexpr int kSortMaxDigits = 512;

template <typename KeyOf>
__device__ __forceinline__ void count_digits(KeyOf key_of, long n, int shift, int digits, int nblocks, unsigned* __restrict__ table) {
  __shared__ unsigned h[kSortMaxDigits];
  for (int d = threadIdx.x; d < digits; d += kBlock) h[d] = 0u;
  __syncthreads();
  const long base = (long)blockIdx.x * kSortTile + threadIdx.x;
  unsigned key[kSortTile / kBlock];
#pragma unroll
  for (int r = 0; r < kSortTile / kBlock; ++r) key[r] = key_of(min(base + r * kBlock, n - 1));
#pragma unroll
  for (int r = 0; r < kSortTile / kBlock; ++r)
    if (base + r * kBlock < n) atomicAdd(&h[(key[r] >> shift) & (unsigned)(digits - 1)], 1u);
  __syncthreads();
  for (int d = threadIdx.x; d < digits; d += kBlock) table[(size_t)d * nblocks + blockIdx.x] = h[d];
}
__global__ __launch_bounds__(kBlock) void radix_count_kernel(const unsigned* __restrict__ keys, long n, int shift,
                                                             int digits, int nblocks, unsigned* __restrict__ table) {
  count_digits([&](long i) { return keys[i]; }, n, shift, digits, nblocks, table);
}
// The first pass's, which forms the keys from the coordinates and leaves them for the scatter (a thread past the end writes
// the last point's key once more).
template <typename T, int ND>
__global__ __launch_bounds__(kBlock) void radix_keys_kernel(NdGeo g, const T* __restrict__ coord, int nbins, unsigned* __restrict__ keys,
                                                            int digits, int nblocks, unsigned* __restrict__ table) {
  g.dims = ND;
  count_digits([&](long i) { return keys[i] = (unsigned)point_bin<T>(g, coord + i * ND, nbins); }, g.batch, 0, digits, nblocks, table);
}

// Exclusive prefix sum of 1024 values, one per thread of the workgroup; `total` receives their sum.
__device__ __forceinline__ unsigned block_exclusive_scan(unsigned v, unsigned* wave_sum /* [16] LDS */, unsigned& total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  unsigned incl = v;
#pragma unroll
  for (int step = 1; step < 64; step <<= 1) {
    const unsigned up = (unsigned)__shfl_up((int)incl, step);
    if (lane >= step) incl += up;
  }
  __syncthreads();  // the previous use of wave_sum is over
  if (lane == 63) wave_sum[wave] = incl;
  __syncthreads();
  unsigned before = 0u, all = 0u;
#pragma unroll
  for (int w = 0; w < 16; ++w) {
    const unsigned t = wave_sum[w];
    before += w < wave ? t : 0u;
    all += t;
  }
  total = all;
  return before + incl - v;
}

// in place, per tile of 4096 entries (a thread owns four consecutive ones); sums[tile] = the tile's sum
constexpr int kScanTile = 4096;
__global__ __launch_bounds__(1024) void radix_scan_tiles_kernel(unsigned* __restrict__ table, int total,
                                                               unsigned* __restrict__ sums) {
  __shared__ unsigned wave_sum[16];
  const int i0 = blockIdx.x * kScanTile + 4 * (int)threadIdx.x;
  unsigned v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = i0 + k < total ? table[i0 + k] : 0u;
  unsigned all;
  unsigned run = block_exclusive_scan(v[0] + v[1] + v[2] + v[3], wave_sum, all);
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (i0 + k < total) table[i0 + k] = run;
    run += v[k];
  }
  if (threadIdx.x == 0) sums[blockIdx.x] = all;
}
// exclusive prefix sum of the tile sums, in place: one workgroup walks them 1024 at a time (more than kScanInScatter tiles)
__global__ __launch_bounds__(1024) void radix_scan_sums_kernel(unsigned* __restrict__ sums, int count) {
  __shared__ unsigned wave_sum[16];
  unsigned carry = 0u;
  for (int base = 0; base < count; base += 1024) {
    const int i = base + (int)threadIdx.x;
    const unsigned v = i < count ? sums[i] : 0u;
    unsigned all;
    const unsigned excl = block_exclusive_scan(v, wave_sum, all);
    if (i < count) sums[i] = carry + excl;
    carry += all;
  }
}

// idx_in == nullptr: the points are still in their own order (index = position);
// keys_out == nullptr: the keys are not needed after this pass
// raw_tiles != 0: tile_start holds that many sums, not yet their prefix sums, which every workgroup's first wave then forms
// for itself (a lane per tile): a launch of one workgroup less
constexpr int kScanInScatter = 64;
__global__ __launch_bounds__(kBlock) void radix_scatter_kernel(const unsigned* __restrict__ keys,
                                                               const int* __restrict__ idx_in, long n, int shift,
                                                               int digits, int nblocks,
                                                               const unsigned* __restrict__ table,
                                                               const unsigned* __restrict__ tile_start, int raw_tiles,
                                                               unsigned* __restrict__ keys_out,
                                                               int* __restrict__ idx_out) {
  constexpr int kWaves = kBlock / 64;
  __shared__ unsigned h[kWaves][kSortMaxDigits];
  __shared__ unsigned starts[kScanInScatter];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (raw_tiles && wave == 0) {
    const unsigned own = lane < raw_tiles ? tile_start[lane] : 0u;
    unsigned incl = own;
#pragma unroll
    for (int step = 1; step < 64; step <<= 1) {
      const unsigned up = (unsigned)__shfl_up((int)incl, step);
      if (lane >= step) incl += up;
    }
    starts[lane] = incl - own;
  }
  for (int e = threadIdx.x; e < kWaves * kSortMaxDigits; e += kBlock) (&h[0][0])[e] = 0u;
  __syncthreads();
  const long base = (long)blockIdx.x * kSortTile + (long)wave * kSortWaveKeys;
  const unsigned mask = (unsigned)(digits - 1);
  unsigned key[kSortRounds];
  int idx[kSortRounds];
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const long i = base + r * 64 + lane;
    key[r] = i < n ? keys[i] : 0u;
    idx[r] = i < n ? (idx_in ? idx_in[i] : (int)i) : 0;
  }
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r)
    if (base + r * 64 + lane < n) atomicAdd(&h[wave][(key[r] >> shift) & mask], 1u);
  __syncthreads();
  // counts -> where each wave's keys of each digit start
  for (int d = threadIdx.x; d < digits; d += kBlock) {
    const size_t j = (size_t)d * nblocks + blockIdx.x;
    unsigned run = table[j] + (raw_tiles ? starts[j / kScanTile] : tile_start[j / kScanTile]);
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
      const unsigned c = h[w][d];
      h[w][d] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSortRounds; ++r) {
    const bool valid = base + r * 64 + lane < n;
    const unsigned d = (key[r] >> shift) & mask;
    // the lanes of this round with the same digit
    unsigned long long same = __ballot(valid);
    for (int b = 0; (1 << b) < digits; ++b) {
      const bool bit = (d >> b) & 1u;
      const unsigned long long set = __ballot(bit);
      same &= bit ? set : ~set;
    }
    if (valid) {
      const unsigned rank = (unsigned)__popcll(same & ((1ull << lane) - 1ull));
      const unsigned pos = h[wave][d] + rank;
      if (rank == 0u) h[wave][d] += (unsigned)__popcll(same);  // after every lane of the wave has read
      if (keys_out) keys_out[pos] = key[r];
      idx_out[pos] = idx[r];
    }
    wave_lds_sync();  // the next round reads the counters this round advanced
  }
}

// Launches with the number of sampling dimensions as the constant ND (DK_ND_BY_ANY_DIMS: 0 above three, g.dims says).  With
// the loops over the dimensions of a point's cell, corners and key unrolled over DK_ND_MAX_DIMS and a test in each, the
// corners alone are eight times eight of them per point.  us a call with g.dims / with the constant: 2^20 points x 64 channels
// of a 32^3 volume forward 151 / 137, grad coord 149 / 112, both gradients 228 / 199 (the kernel); 3 * 10^5 x 7 of 40^3, unsorted, grad
// coord 956 / 144; 20000 x 100 of 96 x 80 forward 26 / 16.
#define DK_ND_BY_DIMS(dims, ...)                        \
  do {                                                  \
    if ((dims) == 1) { constexpr int ND = 1; __VA_ARGS__; }      \
    else if ((dims) == 2) { constexpr int ND = 2; __VA_ARGS__; } \
    else { constexpr int ND = 3; __VA_ARGS__; }                  \
  } while (0)
#define DK_ND_BY_ANY_DIMS(dims, ...)                       \
  do {                                                     \
    if ((dims) <= 3) { DK_ND_BY_DIMS(dims, __VA_ARGS__); } \
    else { constexpr int ND = 0; __VA_ARGS__; }            \
  } while (0)

inline int grid_for(long total) {
  long b = (total + kBlock - 1) / kBlock;
  if (b > 1048576) b = 1048576;
  if (b < 1) b = 1;
  return (int)b;
}

NdGeo make_geo(const dk_nd_desc& d) {
  NdGeo g;
  g.batch = d.batch;
  g.channel = d.channel;
  g.dims = d.dims;
  g.prod_shape = 1;
  for (int i = 0; i < DK_ND_MAX_DIMS; ++i) {
    g.shape[i] = i < d.dims ? d.shape[i] : 1;
    if (i < d.dims) g.prod_shape *= d.shape[i];
  }
  return g;
}

size_t elem_size(int dtype) { return dtype == DK_F64 ? 8 : dtype == DK_F32 ? 4 : 2; }

// points per wave of the channel-last kernels: as many as keep at least ~8192 waves in the grid
int points_per_wave(const NdGeo& g) {
  int ppw = 64;
  while (ppw > 1 && g.batch / ppw < 8192) ppw >>= 1;
  return ppw;
}

// chunks of 64 sorted points per wave of the kernels that add to grad data: as many as keep about 16 waves per CU in the
// grid (a cell's sums stay with the wave over its chunks)
int chunks_per_wave(const NdGeo& g) {
  int per_wave = 1;
  while (per_wave < 8 && g.batch / (64L * per_wave * 2) >= 4096) per_wave *= 2;
  return per_wave;
}

template <typename A, typename B>
void transpose(const A* in, B* out, long rows, long cols, hipStream_t stream, float* zero = nullptr) {
  const unsigned col_tiles = (unsigned)((cols + 31) / 32);
  nd_transpose_kernel<A, B><<<col_tiles * (unsigned)((rows + 31) / 32), 256, 0, stream>>>(in, out, zero, rows, cols, col_tiles);
}

}  // namespace

static long nd_cells(const dk_nd_desc& d) {
  long cells = 1;
  for (int i = 0; i < d.dims; ++i) cells *= d.shape[i];
  return cells;
}

// Few points on a tiny volume: the direct kernels and the one-launch grad data (nd_small_grad_data_kernel).
bool nd_small(const dk_nd_desc& d) {
  if (d.dtype == DK_F64 || d.dims > kClMaxDims || path_disabled(kNoNdSmall)) return false;
  const long cells = nd_cells(d);
  if (cells > kSmallMaxCells || d.batch <= 0 || d.batch * d.channel > 1L << 20) return false;
  // A workgroup of the grad data walks over all points, in rows of 16 cells per tile: up to about 50 us of that, and 4096 points at
  // least; beyond, however few the channels, the sums of nd_grad_data_lds_kernel.  us a pass, here / there: 16 channels of 60
  // cells 5000 points 54 / 62 (six launches instead of three), 20000 188 / 62; 15 of 30 cells 8000 54 / 62, 16000 97 / 62; 15 of 7 x 7 4097 54 / 62, 8000
  // 88 / 63; 15 of 4^3 4097 63 / 62, 8000 109 / 63; 1 of 4^3 30000 377 / 64.
  return d.batch * (7 * ((cells + 15) / 16) + 5 * d.dims + 3) <= 200000 || path_disabled(kNoNdRows);
}

// The channel-last path pays for a transpose of `data`; it is taken for 1..3 dimensions in
// fp32 / fp16 / bf16 when there are enough (point, channel) pairs to amortise it.
//
// Below 16 channels the planar volume serves many calls faster: its cost goes with the corners that the points read and add to
// (corners x channels), the copies' with the volume.  us a pass, planar / here, float32, by channels:
//   copies of a volume larger than what is read of it: 61250 points x 3 of 1400 x 1400 83 / 154, 122500 x 3 148 / 173, 245000 x 3
//   278 / 213, 31250 x 3 of 100^3 78 / 102, 62500 x 3 138 / 122; 122500 x 2 of 1400 x 1400 115 / 161, 245000 x 2 212 / 196; 61250 x 8 177 / 172,
//   61250 x 12 258 / 235: corners x channels from 1.5 times the cells on;
//   little work, where the launches count (six instead of four): 8000 x 15 of 60 x 60 (480 k) 56 / 63, 8000 x 15 of 8^3 (960 k) 57 / 62,
//   65000 x 2 of 60 x 60 (520 k) 57 / 63, 16000 x 15 of 60 x 60 (960 k) 66 / 62, 65000 x 4 (1.0 M) 82 / 63;
//   additions of many points to the same cells, one by one: 16000 x 8 of 400 (80 corners a cell) 55 / 62, 32000 x 4 (160) 62 / 62,
//   32000 x 8 (160) 69 / 63, 16000 x 8 of 100 (320) 88 / 62, 130000 x 4 of 30 x 20 (870) 217 / 62.
// One channel is in this layout as it is and is never copied.
bool nd_use_channel_last(const dk_nd_desc& d) {
  if (d.dtype == DK_F64 || d.dims > kClMaxDims || nd_small(d)) return false;
  const long cells = nd_cells(d);
  // corner offsets are kept as 32-bit element counts, and a launch holds fewer than 2^32 threads: 2^24 tiles of the transposes
  if (cells > (1L << 29) - 32) return false;
  const bool rows = !path_disabled(kNoNdRows);
  if (rows && cells <= kSmallMaxCells && d.batch > 4096) return true;  // too many points for nd_small()
  if (d.batch * d.channel < 65536) return false;
  if (d.channel >= 16) return true;
  if (!rows) return false;
  const long corners = d.batch << d.dims, all = corners * d.channel;
  return d.channel == 1 || corners >= 200 * cells || (all >= 900000 && 2 * all >= 3 * cells);
}

// ... by way of copies of the volume
static bool nd_copies(const dk_nd_desc& d) { return d.channel > 1 && nd_use_channel_last(d); }

// The forward reads a corner where the gradients also add to it, so its copy needs more of them below 16 channels.  us, planar / copied:
// 61250 points x 3 of 1400 x 1400 14 / 41, 245000 x 3 (2.9 M corners times channels, 1.5 per cell) 49 / 51, 490000 x 3 89 / 60, 125000 x 3 of 100^3 (3.0 M,
// 3 per cell) 40 / 37; 250000 x 2 (4 per cell) 39 / 42, 500000 x 2 73 / 53; 31250 x 8 of 50^3 (2.0 M) 16 / 18, 62500 x 8 24 / 18.
static bool nd_forward_channel_last(const dk_nd_desc& d) {
  if (!nd_use_channel_last(d) || !nd_copies(d) || d.channel >= 16) return nd_use_channel_last(d);
  const long all = (d.batch << d.dims) * d.channel;
  return all >= 2500000 && 2 * all >= 5 * nd_cells(d);
}

namespace {

// log2 of a point's lanes in the kernels of narrow rows, or -1 where a wave per point serves the call.  Up to 32 channels, us
// a wave per point / narrow rows, forward and grad coord: 19023 points x 22 channels of 29 x 6 x 25 bfloat16 15.5 / 6.2 and
// 12.0 / 8.8; but 60000 x 40 of 40 x 30 float32 13.9 / 13.0 and 12.6 / 21.4.  Below 16 channels, against a lane per (point,
// channel) on the planar volume: 568761 x 14 of 70 x 78 float16 102 / 27 and 164 / 46, and 4.5 for the transposes.
int row_lanes(const NdGeo& g) {
  if (path_disabled(kNoNdRows) || g.channel > 32) return -1;
  int lg = 0;
  while (1 << lg < g.channel && lg < 6) ++lg;
  return lg;
}

// launch(points' geometry, first point, workgroups) over runs of at most 2^31 lanes: a launch holds fewer than 2^32 threads.  (A
// loop over the points in the kernels takes 7 % of their time: 16 channels of 20 x 30, 300000 points 70 -> 75 us a pass.)
template <typename F>
void row_launches(const NdGeo& g, int lg, F&& launch) {
  NdGeo part = g;
  for (long b0 = 0; b0 < g.batch; b0 += part.batch) {
    part.batch = std::min(g.batch - b0, 1L << (31 - lg));
    launch(part, b0, (unsigned)((part.batch + (kBlock >> lg) - 1) / (kBlock >> lg)));
  }
}

struct LdsSums {
  int slices, channels, pitch, lg;  // slices == 0: not this way
  int range, ranges;                // cells of a workgroup
  long share;                       // points of a workgroup
  int parts;
  size_t lds;
};

LdsSums lds_sums(const dk_nd_desc& d) {
  LdsSums m{};
  if (!nd_use_channel_last(d) || path_disabled(kNoNdRows)) return m;
  const long cells = nd_cells(d);
  const long adds = d.batch << d.dims;  // of a channel
  // How many additions a sum must receive, and how often the points may be walked over.  Float atomics on memory take a row of 16
  // channels and more at once, fewer mostly one by one.  us a pass with the atomics / the sums in LDS: 60000 points x 40
  // channels of 40 x 30 float32 (200 additions, 8 slices) 76 / 58; 19023 x 22 of 29 x 6 x 25 (35) 51 / 66; 10^5 x 10 of 30^3 (30,
  // 20 slices of cells and channels) 108 / 67; 2^20 x 3 of 40^3 (131, 12) 564 / 168; 568761 x 14 of 70 x 78 float16 (416, 5)
  // 1842 / 129; 128941 x 11 of 6 x 12 bfloat16 (7164, 1) 1540 / 42.
  const bool narrow = d.channel < 16;
  if (adds < (narrow ? 4 : 64) * cells) return m;
  auto pitch_of = [](long c) { return c | 1; };
  const long all = kMaxDynamicLds / 8, half = 78 * 1024 / 8;  // sums of a workgroup that has its CU alone, and of one that shares it
  long c = d.channel;
  m.range = (int)cells;
  if (cells * pitch_of(c) > half) {
    c = std::min<long>(all / cells, d.channel);
    if (c % 2 == 0) --c;
    if (c < 1) {
      c = 1;
      m.range = (int)((cells + (cells + all - 1) / all - 1) / ((cells + all - 1) / all));
    }
  }
  m.ranges = (int)((cells + m.range - 1) / m.range);
  m.slices = (int)((d.channel + c - 1) / c);
  if (m.slices * m.ranges > (narrow ? 32 : 16)) return LdsSums{};
  m.channels = (d.channel + m.slices - 1) / m.slices;
  m.pitch = (int)pitch_of(m.channels);
  m.lds = (size_t)m.range * m.pitch * 8;
  while (1 << m.lg < m.channels && m.lg < 6) ++m.lg;
  const long room = (m.lds <= 78 * 1024 ? 512 : 256) / (m.slices * m.ranges);
  const long parts = std::max(1L, std::min({room, adds / (2 * cells), (d.batch + 255) / 256}));
  m.share = (d.batch + parts - 1) / parts;
  m.parts = (int)((d.batch + m.share - 1) / m.share);
  return m;
}

}  // namespace

// Bins of the counting sort (cells of low corners plus the bin of outside points), or 0 when
// the binned kernels do not apply: they pay off with several points per cell.
int nd_bins(const dk_nd_desc& d) {
  if (!nd_use_channel_last(d) || d.channel < 16 || path_disabled(kNoNdBins)) return 0;
  // Where two slices of LDS hold the volume's sums, calls that do not run on the matrix cores go unsorted up to some number of
  // points: the sort costs 30 - 60 us, and the sorted kernels take less for each point.  us on the device, sorted / not:
  //   16 channels, a lane each: 10^3 float32 1.2 M points 437 / 348, 20 x 30 float16 352 / 199: never sorted;
  //   17 - 32 and more than 64, float32: 300 cells x 24 300 k 94 / 87, 600 k 138 / 141; 16 x 16 x 20 300 k 116 / 112, 600 k 176 / 194; 90 cells x 100 150 k
  //   111 / 104, 300 k 143 / 159; 8 x 7 x 160 150 k 186 / 157, 300 k 257 / 273; in three dimensions 7^3 x 24 150 k 134 / 118, 300 k 167 / 197, 4 x 4 x 5 x 100
  //   150 k 209 / 204, 300 k 265 / 354 (float16 the same); float16, whose sorted kernels convert more: 90 cells x 100 600 k 313 / 267, 70 x 250 300 k
  //   343 / 256, 16 x 16 x 28 600 k 212 / 206, 1.2 M 347 / 377, 5 x 5 x 100 600 k 367 / 369;
  //   33 - 64, a wave per point with lanes idle or one channel each: float32 200 x 40 150 k 78 / 80, 12 x 14 x 40 70 k 77 / 76, 5^3 x 40 70 k 103 / 116, 1.2 M
  //   478 / 985; float16 200 x 40 150 k 100 / 80, 300 k 116 / 118, 7 x 9 x 48 150 k 111 / 102, 300 k 136 / 166, 5^3 x 48 70 k 99 / 119.
  if (const LdsSums m = lds_sums(d); m.slices && m.slices * m.ranges <= 2 && !(d.dtype == DK_F32 && d.channel % 64 == 0)) {
    const bool half = d.dtype != DK_F32, idle = d.channel > 32 && d.channel <= 64;
    long most;
    if (d.channel == 16) most = std::numeric_limits<long>::max();
    else if (idle) most = half && d.dims < 3 ? 150000 : 0;
    else if (d.dims == 3) most = 160000;
    else if (half) most = d.dims == 1 ? std::numeric_limits<long>::max() : 520000;
    else most = 260000;
    if (d.batch <= most) return 0;
  }
  long bins = 1;
  for (int i = 0; i < d.dims; ++i) bins *= (long)d.shape[i] + 1;
  bins += 1;
  if (bins > 262144 || d.batch < 2 * bins || d.batch < 65536 || d.batch >= (1L << 30)) return 0;
  return (int)bins;
}

size_t round256(size_t n) { return (n + 255) / 256 * 256; }

namespace {

int key_bits(int bins) {
  int bits = 1;
  while ((1L << bits) < bins) ++bits;
  return bits;
}

}  // namespace

// bytes for the sort: keys, half-sorted keys, the sorted order of the points, the half-sorted order,
// and the (digit, workgroup) table of the radix passes with its tile sums
size_t nd_sort_workspace(const dk_nd_desc& d) {
  const int bins = nd_bins(d);
  if (!bins) return 0;
  const size_t n4 = round256((size_t)d.batch * sizeof(int));
  const size_t table = (size_t)kSortMaxDigits * ((d.batch + kSortTile - 1) / kSortTile);  // entries
  return 4 * n4 + round256((table + table / kScanTile + 1) * sizeof(unsigned));
}

size_t nd_forward_workspace(const dk_nd_desc& d) { return nd_forward_channel_last(d) ? nd_data_cl_workspace(d) : 0; }

size_t nd_data_cl_workspace(const dk_nd_desc& d) {
  if (!nd_copies(d)) return 0;
  size_t n = (size_t)d.channel;
  for (int i = 0; i < d.dims; ++i) n *= (size_t)d.shape[i];
  return round256(n * elem_size(d.dtype)) + nd_sort_workspace(d);
}

namespace {

// Sorts the points by cell into `order`, or, if that is null, into its place in `sort_ws` (laid out as nd_sort_workspace
// says).
template <typename T>
const int* sort_points(const NdGeo& g, const T* coord, int bins, void* sort_ws, hipStream_t stream, int* order = nullptr) {
  const size_t n4 = round256((size_t)g.batch * sizeof(int));
  char* base = static_cast<char*>(sort_ws);
  unsigned* keys = reinterpret_cast<unsigned*>(base);
  unsigned* keys_sorted = reinterpret_cast<unsigned*>(base + n4);
  if (!order) order = reinterpret_cast<int*>(base + 2 * n4);
  {
    // two radix passes of half the key bits each (one pass for keys of up to 9 bits)
    const int bits = key_bits(bins);
    const int lo_bits = bits <= 9 ? bits : (bits + 1) / 2, hi_bits = bits - lo_bits;
    const int nblocks = (int)((g.batch + kSortTile - 1) / kSortTile);
    int* half_order = reinterpret_cast<int*>(base + 3 * n4);
    unsigned* table = reinterpret_cast<unsigned*>(base + 4 * n4);
    unsigned* sums = table + (size_t)kSortMaxDigits * nblocks;
    auto pass = [&](const unsigned* k_in, const int* i_in, int shift, int nbits, unsigned* k_out, int* i_out) {
      const int digits = 1 << nbits, total = digits * nblocks, tiles = (total + kScanTile - 1) / kScanTile;
      if (shift == 0)
        DK_ND_BY_DIMS(g.dims, radix_keys_kernel<T, ND><<<nblocks, kBlock, 0, stream>>>(g, coord, bins, keys, digits, nblocks, table));
      else
        radix_count_kernel<<<nblocks, kBlock, 0, stream>>>(k_in, g.batch, shift, digits, nblocks, table);
      radix_scan_tiles_kernel<<<tiles, 1024, 0, stream>>>(table, total, sums);
      const bool raw = tiles <= kScanInScatter;
      if (!raw) radix_scan_sums_kernel<<<1, 1024, 0, stream>>>(sums, tiles);
      radix_scatter_kernel<<<nblocks, kBlock, 0, stream>>>(k_in, i_in, g.batch, shift, digits, nblocks, table, sums, raw ? tiles : 0, k_out, i_out);
    };
    if (hi_bits == 0) {
      pass(keys, nullptr, 0, lo_bits, nullptr, order);
    } else {
      pass(keys, nullptr, 0, lo_bits, keys_sorted, half_order);
      pass(keys_sorted, half_order, lo_bits, hi_bits, nullptr, order);
    }
  }
  return order;
}

size_t data_bytes(const dk_nd_desc& d) {
  size_t n = (size_t)d.channel;
  for (int i = 0; i < d.dims; ++i) n *= (size_t)d.shape[i];
  return n;
}

}  // namespace

template <typename T>
void nd_forward(const dk_nd_desc& d, const T* data, const T* coord, T* out, void* ws, const int* order,
                hipStream_t stream) {
  const NdGeo g = make_geo(d);
  if constexpr (!std::is_same<T, double>::value) {
    if (nd_forward_channel_last(d)) {
      const T* data_cl = data;
      if (nd_copies(d)) {
        data_cl = static_cast<T*>(ws);
        transpose<T, T>(data, static_cast<T*>(ws), g.channel, g.prod_shape, stream);
      }
      if (const int bins = nd_bins(d)) {
        if (!order) order = sort_points<T>(g, coord, bins, static_cast<char*>(ws) + round256(data_bytes(d) * sizeof(T)), stream);
        if constexpr (std::is_same<T, float>::value) {
          // rows of out are written as 16-byte vectors at multiples of 4 channels
          if (g.channel % 64 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0 && !path_disabled(kNoNdMfma)) {
            DK_ND_BY_DIMS(g.dims, nd_forward_mfma_kernel<T, ND><<<(unsigned)xcd_grid_size((g.batch + 255) / 256), kBlock, 0, stream>>>(g, data_cl, coord, order, bins, out));
            return;
          }
        }
        DK_ND_BY_DIMS(g.dims, nd_forward_binned_kernel<T, ND><<<(unsigned)xcd_grid_size((g.batch + 255) / 256), kBlock, 0, stream>>>(g, data_cl, coord, order, bins, out));
        return;
      }
      if (const int lg = row_lanes(g); lg >= 0) {
        row_launches(g, lg, [&](const NdGeo& part, long b0, unsigned grid) {
          DK_ND_BY_DIMS(g.dims, nd_forward_rows_kernel<T, ND><<<grid, kBlock, 0, stream>>>(part, data_cl, coord + b0 * g.dims, out + b0 * g.channel, lg));
        });
        return;
      }
      const int ppw = points_per_wave(g);
      const long waves = (g.batch + ppw - 1) / ppw;
      DK_ND_BY_DIMS(g.dims, nd_forward_cl_kernel<T, ND><<<(unsigned)((waves + 3) / 4), kBlock, 0, stream>>>(g, data_cl, coord, out, ppw));
      return;
    }
  }
  const long total = g.batch * g.channel;
  DK_ND_BY_ANY_DIMS(g.dims, nd_forward_kernel<T, ND><<<grid_for(total), kBlock, 0, stream>>>(g, data, coord, out, total));
}

size_t nd_grad_data_workspace(const dk_nd_desc& d) {
  if (nd_small(d)) return 0;
  size_t n = (size_t)d.channel;
  for (int i = 0; i < d.dims; ++i) n *= (size_t)d.shape[i];
  const size_t sums = (size_t)lds_sums(d).parts * n * sizeof(float);
  // fp32 channel-last accumulation image; or copies of the sums, without a sort
  if (nd_copies(d)) return std::max(round256(n * sizeof(float)) + nd_sort_workspace(d), sums);
  return std::max(d.dtype == DK_F16 || d.dtype == DK_BF16 ? n * sizeof(float) : 0, sums);
}

template <typename T>
void nd_grad_data(const dk_nd_desc& d, const T* gout, const T* coord, T* gdata, void* ws, const int* order,
                  hipStream_t stream) {
  using CT = compute_t<T>;
  const NdGeo g = make_geo(d);
  const long n_data = (long)g.channel * g.prod_shape;
  const long total = g.batch * g.channel;
  if constexpr (!std::is_same<T, double>::value) {
    if (nd_small(d)) {
      const int nt = ((int)g.prod_shape + 15) / 16;
      // points per chunk: rows of W that fit its LDS, a multiple of 64, at most two points per thread
      int chunk = kSmallWBytes / (nt * 16 * (int)sizeof(float)) / 64 * 64;
      if (chunk > 2048) chunk = 2048;
      const size_t lds = std::max<size_t>((size_t)std::min<long>(chunk, (g.batch + 63) / 64 * 64) * nt * 16 * sizeof(float),
                                          (size_t)16 * nt * 256 * sizeof(float));
      const unsigned grid = (unsigned)((g.channel + 15) / 16);
#define DK_ND_SMALL_GD(ND, NT)                                                                                                    \
  if (lds <= 64 * 1024 || allow_dynamic_lds(reinterpret_cast<const void*>(&nd_small_grad_data_kernel<T, ND, NT>), kSmallWBytes)) \
  nd_small_grad_data_kernel<T, ND, NT><<<grid, 1024, lds, stream>>>(g, gout, coord, gdata, chunk)
#define DK_ND_SMALL_GD_NT(ND)          \
  if (nt == 1) { DK_ND_SMALL_GD(ND, 1); } \
  else if (nt == 2) { DK_ND_SMALL_GD(ND, 2); } \
  else if (nt == 3) { DK_ND_SMALL_GD(ND, 3); } \
  else { DK_ND_SMALL_GD(ND, 4); }
      if (g.dims == 1) { DK_ND_SMALL_GD_NT(1) }
      else if (g.dims == 2) { DK_ND_SMALL_GD_NT(2) }
      else { DK_ND_SMALL_GD_NT(3) }
#undef DK_ND_SMALL_GD_NT
#undef DK_ND_SMALL_GD
      return;
    }
    if (const LdsSums m = lds_sums(d); m.slices && !nd_bins(d)) {
      float* partial = static_cast<float*>(ws);
      bool ok = true;
      DK_ND_BY_DIMS(g.dims, {
        auto kernel = nd_grad_data_lds_kernel<T, ND>;
        ok = m.lds <= 64 * 1024 || allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kMaxDynamicLds);
        if (ok) kernel<<<(unsigned)(m.slices * m.ranges * m.parts), 1024, m.lds, stream>>>(g, gout, coord, partial, m.lg, m.channels, m.pitch, m.slices, m.range, m.ranges, m.share);
      });
      if (ok) {
        launch_reduce_partials<float, T>(partial, m.parts, n_data, gdata, stream);
        return;
      }
    }
    if (nd_copies(d)) {
      float* acc = static_cast<float*>(ws);
      nd_fill_zero_kernel<float><<<grid_for(n_data), kBlock, 0, stream>>>(acc, n_data);
      if (const int bins = nd_bins(d)) {
        if (!order) order = sort_points<T>(g, coord, bins, static_cast<char*>(ws) + round256((size_t)n_data * sizeof(float)), stream);
        const int per_wave = chunks_per_wave(g);
        const long waves = (g.batch + 64L * per_wave - 1) / (64L * per_wave);
        bool on_matrix_cores = false;
        if constexpr (std::is_same<T, float>::value)
          // rows of gout are read as 16-byte vectors at multiples of 4 channels
          on_matrix_cores = g.channel % 64 == 0 && reinterpret_cast<uintptr_t>(gout) % 16 == 0 && !path_disabled(kNoNdMfma);
        if (on_matrix_cores) {
          if constexpr (std::is_same<T, float>::value)
            DK_ND_BY_DIMS(g.dims, nd_grad_data_mfma_kernel<T, ND><<<(unsigned)xcd_grid_size((waves + 3) / 4), kBlock, 0, stream>>>(g, gout, coord, order, bins, acc, per_wave));
        } else {
          DK_ND_BY_DIMS(g.dims, nd_grad_data_binned_kernel<T, ND><<<(unsigned)xcd_grid_size((waves + 3) / 4), kBlock, 0, stream>>>(g, gout, coord, order, bins, acc, per_wave));
        }
      } else {
        const int ppw = points_per_wave(g);
        const long waves = (g.batch + ppw - 1) / ppw;
        DK_ND_BY_DIMS(g.dims, nd_grad_data_cl_kernel<T, ND><<<(unsigned)((waves + 3) / 4), kBlock, 0, stream>>>(g, gout, coord, acc, ppw));
      }
      transpose<float, T>(acc, gdata, g.prod_shape, g.channel, stream);
      return;
    }
  }
  constexpr bool direct = sizeof(T) == sizeof(CT);
  CT* acc = direct ? reinterpret_cast<CT*>(gdata) : static_cast<CT*>(ws);
  nd_fill_zero_kernel<CT><<<grid_for(n_data), kBlock, 0, stream>>>(acc, n_data);
  if (total > 0)
    DK_ND_BY_ANY_DIMS(g.dims, nd_grad_data_kernel<T, CT, false, ND><<<grid_for(total), kBlock, 0, stream>>>(g, gout, coord, acc, total));
  if (!direct) nd_convert_kernel<CT, T><<<grid_for(n_data), kBlock, 0, stream>>>(acc, gdata, n_data);
}

template <typename T>
void nd_grad_coord(const dk_nd_desc& d, const T* gout, const T* data, const T* coord, T* gcoord,
                   void* ws, const int* order, hipStream_t stream) {
  const NdGeo g = make_geo(d);
  if constexpr (!std::is_same<T, double>::value) {
    if (nd_small(d)) {
      const unsigned grid = (unsigned)((g.batch + kBlock / 64 - 1) / (kBlock / 64));
      if (g.dims == 1) nd_small_grad_coord_kernel<T, 1><<<grid, kBlock, 0, stream>>>(g, gout, data, coord, gcoord);
      else if (g.dims == 2) nd_small_grad_coord_kernel<T, 2><<<grid, kBlock, 0, stream>>>(g, gout, data, coord, gcoord);
      else nd_small_grad_coord_kernel<T, 3><<<grid, kBlock, 0, stream>>>(g, gout, data, coord, gcoord);
      return;
    }
    if (nd_use_channel_last(d)) {
      const T* data_cl = data;
      if (nd_copies(d)) {
        data_cl = static_cast<T*>(ws);
        transpose<T, T>(data, static_cast<T*>(ws), g.channel, g.prod_shape, stream);
      }
      if (const int bins = nd_bins(d)) {
        if (!order) order = sort_points<T>(g, coord, bins, static_cast<char*>(ws) + round256(data_bytes(d) * sizeof(T)), stream);
        if constexpr (std::is_same<T, float>::value) {
          // rows of gout are read as 16-byte vectors at multiples of 16 channels
          if (g.channel % 64 == 0 && reinterpret_cast<uintptr_t>(gout) % 16 == 0 && !path_disabled(kNoNdMfma)) {
            DK_ND_BY_DIMS(g.dims, nd_grad_coord_mfma_kernel<T, ND><<<(unsigned)xcd_grid_size((g.batch + 255) / 256), kBlock, 0, stream>>>(g, gout, data_cl, coord, order, bins, gcoord));
            return;
          }
        }
        DK_ND_BY_DIMS(g.dims, nd_grad_coord_binned_kernel<T, ND><<<(unsigned)xcd_grid_size((g.batch + 255) / 256), kBlock, 0, stream>>>(g, gout, data_cl, coord, order, bins, gcoord));
        return;
      }
      if (const int lg = row_lanes(g); lg >= 0) {
        row_launches(g, lg, [&](const NdGeo& part, long b0, unsigned grid) {
          DK_ND_BY_DIMS(g.dims, nd_grad_coord_rows_kernel<T, ND><<<grid, kBlock, 0, stream>>>(part, gout + b0 * g.channel, data_cl, coord + b0 * g.dims,
                                                                                             gcoord + b0 * g.dims, lg));
        });
        return;
      }
      const int ppw = points_per_wave(g);
      const long waves = (g.batch + ppw - 1) / ppw;
      DK_ND_BY_DIMS(g.dims, nd_grad_coord_cl_kernel<T, ND><<<(unsigned)((waves + 3) / 4), kBlock, 0, stream>>>(g, gout, data_cl, coord, gcoord, ppw));
      return;
    }
  }
  long blocks = (g.batch + 3) / 4;
  if (blocks > 65536) blocks = 65536;
  DK_ND_BY_ANY_DIMS(g.dims, nd_grad_coord_kernel<T, ND><<<(int)blocks, kBlock, 0, stream>>>(g, gout, data, coord, gcoord));
}

namespace {
// Whether nd_backward_mfma_kernel serves the call (the rule of the two kernels that it takes the place of).
bool nd_one_pass(const dk_nd_desc& d) {
  return d.dtype == DK_F32 && d.channel % 64 == 0 && nd_bins(d) && !path_disabled(kNoNdMfma);
}
}  // namespace

size_t nd_backward_workspace(const dk_nd_desc& d) {
  const size_t apart = std::max(nd_grad_data_workspace(d), nd_data_cl_workspace(d));
  return nd_one_pass(d) ? std::max(apart, 2 * round256(data_bytes(d) * sizeof(float)) + nd_sort_workspace(d)) : apart;
}

template <typename T>
void nd_backward(const dk_nd_desc& d, const T* gout, const T* data, const T* coord, T* gdata, T* gcoord, void* ws,
                 const int* order, hipStream_t stream) {
  if constexpr (std::is_same<T, float>::value) {
    // rows of gout are read as 16-byte vectors at multiples of 4 channels
    if (nd_one_pass(d) && reinterpret_cast<uintptr_t>(gout) % 16 == 0) {
      const NdGeo g = make_geo(d);
      const long n_data = (long)g.channel * g.prod_shape;
      const size_t image = round256((size_t)n_data * sizeof(float));
      float *acc = static_cast<float*>(ws), *data_cl = reinterpret_cast<float*>(static_cast<char*>(ws) + image);
      const int bins = nd_bins(d), per_wave = chunks_per_wave(g);
      if (!order) order = sort_points<T>(g, coord, bins, static_cast<char*>(ws) + 2 * image, stream);
      transpose<T, T>(data, data_cl, g.channel, g.prod_shape, stream, acc);
      const long waves = (g.batch + 64L * per_wave - 1) / (64L * per_wave);
      DK_ND_BY_DIMS(g.dims, nd_backward_mfma_kernel<T, ND><<<(unsigned)xcd_grid_size((waves + 3) / 4), kBlock, 0, stream>>>(g, gout, data_cl, coord, order, bins, acc, gcoord, per_wave));
      transpose<float, T>(acc, gdata, g.prod_shape, g.channel, stream);
      return;
    }
  }
  // one after the other, sharing the workspace (stream order)
  nd_grad_data<T>(d, gout, coord, gdata, ws, order, stream);
  if (d.batch > 0) nd_grad_coord<T>(d, gout, data, coord, gcoord, ws, order, stream);
}

// The sorted order of the points alone, for a caller that issues several of the three calls on
// the same coordinates: `order` receives batch ints; ws as nd_sort_workspace() sizes it.
size_t nd_order_bytes(const dk_nd_desc& d) { return nd_bins(d) ? (size_t)d.batch * sizeof(int) : 0; }

template <typename T>
void nd_order(const dk_nd_desc& d, const T* coord, int* order, void* ws, hipStream_t stream) {
  const NdGeo g = make_geo(d);
  if constexpr (!std::is_same<T, double>::value) {
    if (const int bins = nd_bins(d)) {
      sort_points<T>(g, coord, bins, ws, stream, order);
    }
  }
}

#define DK_INSTANTIATE(T)                                                                             \
  template void nd_forward<T>(const dk_nd_desc&, const T*, const T*, T*, void*, const int*, hipStream_t);   \
  template void nd_grad_data<T>(const dk_nd_desc&, const T*, const T*, T*, void*, const int*, hipStream_t); \
  template void nd_grad_coord<T>(const dk_nd_desc&, const T*, const T*, const T*, T*, void*, const int*,    \
                                 hipStream_t);                                                         \
  template void nd_backward<T>(const dk_nd_desc&, const T*, const T*, const T*, T*, T*, void*, const int*, hipStream_t); \
  template void nd_order<T>(const dk_nd_desc&, const T*, int*, void*, hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(double)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
