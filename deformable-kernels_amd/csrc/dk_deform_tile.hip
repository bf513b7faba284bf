// Deformable coordinate gradients and filter gradient from one pass over the samples, lanes along the CHANNELS
// (dk_deform_fast.hip holds the forms that make them apart).
//
// Reference kernels covered (K.cu =
// deformable_kernels/ops/deform_kernel/csrc/filter_sample_depthwise_cuda_kernel.cu): grad filter K.cu:836-955, grad offset
// K.cu:1147-1243, grad rotation K.cu:1410-1508.
//
// All three gradients need every sample's value or its slopes, and reading the four corners is what they cost.  A row of 16
// lanes takes the 16 channels of a block at one output pixel, the wave's four rows four pixels, the workgroup's 16
// waves a tile of 8 x 8 pixels.  In that arrangement
//   * the corners of a sample are four runs of 64 bytes of LDS, whatever the offsets are;
//   * what depends on (pixel, tap) only is computed once, by lane `tap` of the pixel's row, and reaches the others as a DPP
//     operand (row_newbcast);
//   * the coordinates' gradients are sums over channels: a lane keeps those of its channels (36 registers) over all
//     blocks, and the row's lanes are added up once per tile;
//   * sample * out_grad is the right operand of the filter gradient's matrix product as it stands: gW[cell][c] = sum_k
//     A[cell][k] * P[k][c], k = (pixel, tap), by v_mfma_f32_16x16x4_f32 (deform_grad_filter_mfma_kernel has the layout).
// The window of the input that a tile reads -- a square, so its size follows the offsets and not the plane -- is staged per
// block of 16 channels as [position][channel], in two buffers, one barrier per block.  Samples spread over more than the
// window take several passes over neighbouring windows, each sample counted in the pass that holds its corners.
//
// N=64 C=144 56 x 56 float32: both coordinate gradients 323 us and the filter gradient 320 with a pixel per lane, 20 of reductions;
// 450 here and 6.  What bounds it is vector issue (24 instructions per tap and four pixels x 16 channels, and half as many again
// per block and tile): 62 % of the cycles; without the loads of the window it takes 49 us less, without the matrix
// instructions 22.  The DPP operands inside the multiply-adds (27 instructions per tap with moves: 563 -> 513 us) and the
// tiles' windows from a kernel in front (513 -> 453: two barriers and a round trip to memory less per tile) carry it.  With a rotation
// tensor the kernels take all 128 registers and keep 13 or 15 more in scratch, which are read once per tile; where a spill
// falls into the loop over the blocks it costs more than either.
#include <algorithm>
#include <type_traits>

#include "dk_deform.h"
#include "dk_kernels.h"

namespace dk {

namespace {

constexpr int kTlBlock = 1024, kTlWaves = kTlBlock / 64;
constexpr int kTlCh = 16;             // channels of a block
constexpr int kTlSide = 8;            // output pixels of a tile's side: four per wave
constexpr int kTlRows = 27, kTlCols = 27;  // window: 8 + 2 taps and offsets of 8 either way
constexpr int kTlPos = kTlRows * kTlCols;
constexpr int kTlSlots = kTlPos + kTlCols + 2;  // ... and zeros where a tap that contributes nothing reads its corners
constexpr int kTlStage = (kTlPos / 16 + kTlWaves) / kTlWaves;  // units of 16 positions that a wave stages
constexpr int kTlLds = 160 * 1024 - 512;
constexpr int kTlMostBlocks = 10;     // channel blocks of a workgroup: 2 KB of LDS each
static_assert(kTlStage * kTlWaves * 16 >= kTlPos && kTlSide * kTlSide == 4 * kTlWaves, "the window's units, the tile's pixels");

typedef float tl_f4 __attribute__((ext_vector_type(4)));

template <int K>
__device__ __forceinline__ int row_lane(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x150 + K, 0xf, 0xf, true);
}
template <int K>
__device__ __forceinline__ float row_lane(float v) {
  return __builtin_bit_cast(float, row_lane<K>(__builtin_bit_cast(int, v)));
}
// A sample and the scope's weight at it.  In: the corners (a, b; c, d); {wgt, w_w, w_h, wc}, the table's entry {value, difference along
// the columns, along the rows, difference of these}; the four fractions, in lane K of the row, as DPP operands.  Out: the slopes, each
// a difference of corners and its change across the cell (OWN: from the differences on either side, as sample_slopes; else one change
// for both), and the values, a corner and the slopes.
// A DPP operand must not have been written by the two vector instructions in front, and the compiler, which does not look into the
// asm, may place a register's copy or reload there.  The block's own first instructions, subtractions of corners, keep that distance,
// and it writes none of the four.  (s_nop 1 in front in their place: 2 % of the kernel's time.)
template <int K, bool ROT, bool OWN>
__device__ __forceinline__ void lerp_row(float lh, float lw, float fh, float fw, float a, float b, float c, float d, float wc, float& s_h,
                                         float& s_w, float& val, float& w_h, float& w_w, float& wgt) {
#define DK_SUB(D, A, B) "v_sub_f32 %[" D "], %[" A "], %[" B "]\n\t"
#define DK_FMAC_ROW(D, A, B) "v_fmac_f32_dpp %[" D "], %[" A "], %[" B "] row_newbcast:%[k] row_mask:0xf bank_mask:0xf\n\t"
#define DK_OWN DK_SUB("b", "d", "b") DK_SUB("c", "d", "c") DK_SUB("b", "b", "s_h")
#define DK_LERP_ROW(CHANGES, ACROSS, W_W)                                                                                           \
  asm(DK_SUB("s_w", "b", "a") DK_SUB("s_h", "c", "a") CHANGES DK_SUB("c", "c", "s_w")                                               \
      DK_FMAC_ROW("a", "lw", "s_w") DK_FMAC_ROW("wgt", "fw", "w_w") DK_FMAC_ROW("s_h", "lw", ACROSS) DK_FMAC_ROW("w_h", "fw", "wc") \
      DK_FMAC_ROW("s_w", "lh", "c") W_W DK_FMAC_ROW("a", "lh", "s_h") DK_FMAC_ROW("wgt", "fh", "w_h")                               \
      : [s_h] "=&v"(s_h), [s_w] "=&v"(s_w), [a] "+&v"(a), [b] "+&v"(b), [c] "+&v"(c), [w_h] "+&v"(w_h), [w_w] "+&v"(w_w),           \
        [wgt] "+&v"(wgt)                                                                                                            \
      : [lh] "v"(lh), [lw] "v"(lw), [fh] "v"(fh), [fw] "v"(fw), [d] "v"(d), [wc] "v"(wc), [k] "n"(K))
  // (without ROT w_w stays)
  if constexpr (ROT && OWN) DK_LERP_ROW(DK_OWN, "b", DK_FMAC_ROW("w_w", "fh", "wc"));
  else if constexpr (ROT) DK_LERP_ROW(DK_SUB("c", "d", "c"), "c", DK_FMAC_ROW("w_w", "fh", "wc"));
  else if constexpr (OWN) DK_LERP_ROW(DK_OWN, "b", "");
  else DK_LERP_ROW(DK_SUB("c", "d", "c"), "c", "");
#undef DK_LERP_ROW
#undef DK_OWN
#undef DK_FMAC_ROW
#undef DK_SUB
  val = a;
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// Sums of four values over the 16 lanes of a row: lane q holds that of value q % 4
__device__ __forceinline__ float row_sums(float a, float b, float c, float d, int q) {
  const bool odd = q & 1, high = q & 2;
  const float ab = (odd ? b : a) + dpp<0xB1>(odd ? a : b), cd = (odd ? d : c) + dpp<0xB1>(odd ? c : d);  // the neighbour
  float v = (high ? cd : ab) + dpp<0x4E>(high ? ab : cd);  // the other pair
  v += dpp<0x124>(v);                                      // row_ror:4, row_ror:8
  return v + dpp<0x128>(v);
}
// v[0] + ... + v[N - 1] in pairs: the rounding error of a chain grows with its length
template <int N>
__device__ __forceinline__ float tree_sum(float (&v)[N]) {
#pragma unroll
  for (int n = N / 2; n > 0; n /= 2)
#pragma unroll
    for (int i = 0; i < n; ++i) v[i] += v[i + n];
  return v[0];
}
template <int... I, typename F>
__device__ __forceinline__ void static_for(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for(std::make_integer_sequence<int, N>{}, f);
}
__device__ __forceinline__ float hat(float d) { return __builtin_amdgcn_fmed3f(1.f - fabsf(d), 0.f, 1.f); }

struct TilePlan {
  bool ok;
  bool boxed;              // the window depends on the offsets
  int tiles_x, tiles;      // of a plane
  int chunks, per_chunk;   // shares of the channel blocks, blocks of a share
  int wgs;                 // workgroups per (group, share), each with a run of tiles
  size_t lds;
};

__host__ __device__ __forceinline__ int tile_passes(int extent, int window) { return ceil_div(extent, window - 1); }

// boxes[image * tiles + tile] = {first row, rows, first column, columns} of the top-left corners, in the plane with one
// element of zeros around it, that the tile's samples read; windows[workgroup] = how many windows its tiles take.  A wave
// per tile.
template <typename T>
__global__ __launch_bounds__(256) void deform_tile_boxes_kernel(Geo g, const T* __restrict__ off, int4* __restrict__ boxes,
                                                                unsigned* __restrict__ windows, int tiles_x, int tiles) {
  __shared__ int wave_sum_[4];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int out_plane = g.out_h * g.out_w, all = g.batch * tiles;
  int sum = 0;
  for (int id = blockIdx.x * 4 + wave; id < all; id += gridDim.x * 4) {
    const int n = id / tiles, t = id - n * tiles;
    const int oh = t / tiles_x * kTlSide + lane / kTlSide, ow = t % tiles_x * kTlSide + lane % kTlSide;
    const bool live = oh < g.out_h && ow < g.out_w;
    const rsrc_t ro = plane_rsrc(off + (size_t)n * 18 * out_plane, 18 * out_plane);
    float dh[9], dw[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const unsigned o = live ? (unsigned)(2 * k * out_plane + oh * g.out_w + ow) * (unsigned)sizeof(T) : kOutOfRange;
      dh[k] = buf_ld(ro, o, off), dw[k] = buf_ld(ro, o + (unsigned)out_plane * (unsigned)sizeof(T), off);
    }
    int r_lo = 1 << 30, r_hi = -1, c_lo = 1 << 30, c_hi = -1;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const float h = float(oh - g.pad_h + k / 3) + dh[k], w = float(ow - g.pad_w + k % 3) + dw[k];
      if (live && h > -1.f && w > -1.f && h < float(g.in_h) && w < float(g.in_w)) {
        const int row = (int)floorf(h) + 1, col = (int)floorf(w) + 1;
        r_lo = min(r_lo, row), r_hi = max(r_hi, row), c_lo = min(c_lo, col), c_hi = max(c_hi, col);
      }
    }
    r_lo = wave_min(r_lo), r_hi = wave_max(r_hi), c_lo = wave_min(c_lo), c_hi = wave_max(c_hi);
    const int4 box = r_hi >= 0 ? make_int4(r_lo, r_hi - r_lo + 1, c_lo, c_hi - c_lo + 1) : make_int4(0, 1, 0, 1);
    if (lane == 0) boxes[id] = box;
    sum += tile_passes(box.y, kTlRows) * tile_passes(box.w, kTlCols);
  }
  if (lane == 0) wave_sum_[wave] = sum;
  __syncthreads();
  if (threadIdx.x == 0) windows[blockIdx.x] = (unsigned)(wave_sum_[0] + wave_sum_[1] + wave_sum_[2] + wave_sum_[3]);
}

// ROT: false: rotation is null (all zeros), and there is no gradient for it.  OWN: lerp_row.
template <typename T, int SH, int SW, bool ROT, bool OWN>
__global__ __launch_bounds__(kTlBlock, 1) void deform_grad_tile_kernel(
    Geo g, const T* __restrict__ gout, const T* __restrict__ x, const T* __restrict__ off, const T* __restrict__ rot,
    const T* __restrict__ filter, T* __restrict__ goff, T* __restrict__ grot, float* __restrict__ part_off,
    float* __restrict__ part_rot, float* __restrict__ part_filter, TilePlan plan, const int4* __restrict__ boxes, TileChoice choice,
    unsigned* __restrict__ left) {
  if (choice.windows) {
    const bool take = tiles_take(choice);
    if (blockIdx.x == 0 && threadIdx.x == 0) *left = take ? 0u : 1u;  // for the kernels behind, which read one word each
    if (!take) return;
  }
  constexpr int K9 = 9, TCELLS = (SH + 1) * (SW + 1), CELLS = SH * SW;
  extern __shared__ __align__(16) char lds[];
  char* planes = lds;                                                    // [2][kTlSlots][kTlCh] floats
  char* tbl = planes + 2 * kTlSlots * kTlCh * 4;                         // [2][TCELLS][kTlCh] float4
  float* red = reinterpret_cast<float*>(tbl + 2 * TCELLS * kTlCh * 16);  // [2][kTlWaves][256]
  float* fsum = red + 2 * kTlWaves * 256;                                // [per_chunk][256]
  float* wts = fsum + plan.per_chunk * 256;                              // [per_chunk][CELLS][kTlCh]

  const int H = g.in_h, W = g.in_w;
  const int cpg = g.channel / g.groups;
  const int out_plane = g.out_h * g.out_w, in_plane = H * W;
  const int total = plan.wgs * plan.chunks * g.groups;
  const int lb = logical_block(total);
  if (lb >= total) return;
  const int wg = lb % plan.wgs, chunk = lb / plan.wgs % plan.chunks, grp = lb / plan.wgs / plan.chunks;
  const int cb_lo = chunk * plan.per_chunk, nblk = min(plan.per_chunk, ceil_div(cpg, kTlCh) - cb_lo);
  const long all_tiles = (long)g.batch * plan.tiles;
  // The workgroups of an XCD (32 consecutive ones) walk their share of the tiles side by side, so that the windows of
  // neighbouring tiles are read into one L2.
  const int reg = wg / 32 * 32, reg_n = min(32, plan.wgs - reg);
  const int tile_lo = (int)(all_tiles * reg / plan.wgs) + wg - reg, tile_hi = (int)(all_tiles * (reg + reg_n) / plan.wgs);

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int q = lane & 15, kg = lane >> 4;           // channel of the block (tap, while descriptors are made); pixel
  const float ci = q < CELLS ? float(q / SW) : 64.f, cj = float(q % SW);  // rows of A past the last cell stay 0
  const int x_cs = g.groups * in_plane * (int)sizeof(T), g_cs = g.groups * out_plane * (int)sizeof(T);

  for (int e = threadIdx.x; e < 2 * (kTlSlots - kTlPos) * kTlCh; e += kTlBlock) {
    const int b = e / ((kTlSlots - kTlPos) * kTlCh), i = e % ((kTlSlots - kTlPos) * kTlCh);
    reinterpret_cast<float*>(planes)[(b * kTlSlots + kTlPos) * kTlCh + i] = 0.f;
  }
  for (int e = threadIdx.x; e < nblk * 256; e += kTlBlock) fsum[e] = 0.f;
  for (int e = threadIdx.x; e < nblk * CELLS * kTlCh; e += kTlBlock) {
    const int c = cb_lo * kTlCh + e / (CELLS * kTlCh) * kTlCh + e % kTlCh, cell = e / kTlCh % CELLS;
    wts[e] = c < cpg ? ld(filter + (size_t)(grp + g.groups * c) * CELLS + cell) : 0.f;
  }

  // output pixel of this lane in tile `id`
  struct Pixel {
    int n, top, left;  // image, and the tile's first pixel: the same for all lanes
    int at;            // this lane's pixel in the output plane, -1: none
  };
  // (what follows from the lane's number is worked out anew at every tile: kept, it takes registers from the sums)
  auto own = [&](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  auto pixel = [&](int id) {
    const int i = wave * 4 + own(kg), ty = i / kTlSide, tx = i % kTlSide;
    const int n = id / plan.tiles, t = id - n * plan.tiles;
    const int top = t / plan.tiles_x * kTlSide, left = t % plan.tiles_x * kTlSide;
    return Pixel{n, top, left, top + ty < g.out_h && left + tx < g.out_w ? (top + ty) * g.out_w + left + tx : -1};
  };
  struct Raw {
    float dh, dw, rh, rw;
  };
  auto load_raw = [&](const Pixel& p) {
    const rsrc_t ro = plane_rsrc(off + (size_t)p.n * 18 * out_plane, 18 * out_plane);
    const unsigned step = (unsigned)out_plane * (unsigned)sizeof(T);
    const unsigned o = p.at >= 0 && q < K9 ? (unsigned)(2 * q * out_plane + p.at) * (unsigned)sizeof(T) : kOutOfRange;
    Raw r{buf_ld(ro, o, off), buf_ld(ro, o + step, off), 0.f, 0.f};
    if constexpr (ROT) {
      const rsrc_t rr = plane_rsrc(rot + (size_t)(p.n * g.groups + grp) * 18 * out_plane, 18 * out_plane);
      r.rh = buf_ld(rr, o, rot), r.rw = buf_ld(rr, o + step, rot);
    }
    return r;
  };
  // what lane `tap` knows of its sample (K.cu:486-500 and 338-341)
  struct Tap {
    int at;  // top-left corner in the plane with one element of zeros around it, row * 2^16 + column; -1: no contribution
    float lh, lw, sh, sw;
  };
  auto describe = [&](const Pixel& p, const Raw& r) {
    Tap t;
    const int i = wave * 4 + own(kg), ty = i / kTlSide, tx = i % kTlSide, f = min(own(q), K9 - 1), f_h = f / 3, f_w = f % 3;
    const float h = float(p.top + ty - g.pad_h + f_h) + r.dh, w = float(p.left + tx - g.pad_w + f_w) + r.dw;
    const bool hit = p.at >= 0 && q < K9 && h > -1.f && w > -1.f && h < float(H) && w < float(W);
    const float hf = floorf(h), wf = floorf(w);
    t.at = hit ? ((int)hf + 1) << 16 | ((int)wf + 1) : -1;
    t.lh = hit ? h - hf : 0.f, t.lw = hit ? w - wf : 0.f;
    const float sh = scope_coord<float>(g, f_h, r.rh, g.centre_h), sw = scope_coord<float>(g, f_w, r.rw, g.centre_w);
    const bool in = hit && sh > -1.f && sw > -1.f && sh < float(SH) && sw < float(SW);
    t.sh = in ? sh : -2.f, t.sw = in ? sw : -2.f;
    return t;
  };
  // rows and columns of top-left corners, and how many windows they take
  struct Box {
    int row, rows, col, cols, passes_r, passes_c;
  };
  auto read_box = [&](int tile) {
    // without a table: the whole plane, which fits the window
    const int4 b = boxes ? boxes[tile] : make_int4(0, H + 1, 0, W + 1);
    return Box{b.x, b.y, b.z, b.w, tile_passes(b.y, kTlRows), tile_passes(b.w, kTlCols)};
  };

  // register stage of a (tile, pass, block): four channels of this lane's positions -- four consecutive lanes take the
  // sixteen channels of one position, so the stores to LDS are contiguous --, and out_grad at its pixel and channel
  float r_x[kTlStage][4], r_g;
  struct Window {
    int row, col, rows, cols;  // first position; rows and columns that samples of the pass read
  };
  auto window = [&](const Box& v, int pass) {
    const int row = v.row + pass / v.passes_c * (kTlRows - 1), col = v.col + pass % v.passes_c * (kTlCols - 1);
    return Window{row, col, min(v.row + v.rows - row + 1, kTlRows), min(v.col + v.cols - col + 1, kTlCols)};
  };
  unsigned x_off[kTlStage];  // byte offsets of this lane's positions and first channel in a block's planes
  auto aim = [&](const Window& w) {
    const int l = own(lane);
#pragma unroll
    for (int k = 0; k < kTlStage; ++k) {
      const int pos = (wave + kTlWaves * k) * 16 + (l >> 2);
      const int pr = pos / kTlCols, pc = pos % kTlCols, row = w.row + pr - 1, col = w.col + pc - 1;
      const bool ok = pr < w.rows && pc < w.cols && row >= 0 && row < H && col >= 0 && col < W;
      x_off[k] = ok ? (unsigned)((l & 3) * 4 * x_cs) + (unsigned)(row * W + col) * (unsigned)sizeof(T) : kOutOfRange;
    }
  };
  // block b's table, cell (i, k) of the zero-padded scope tile: {tl, tr - tl, bl - tl, br - tr - bl + tl} per channel
  auto make_table = [&](int b, char* dst) {
    if (threadIdx.x < TCELLS * kTlCh) {
      const int e = own((int)threadIdx.x), ch = e % kTlCh, i = e / kTlCh / (SW + 1) - 1, k = e / kTlCh % (SW + 1) - 1;
      float w[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const int ii = i + (c >> 1), kk = k + (c & 1);
        const float v = wts[(b * CELLS + min(max(ii, 0), SH - 1) * SW + min(max(kk, 0), SW - 1)) * kTlCh + ch];
        w[c] = ii >= 0 && ii < SH && kk >= 0 && kk < SW ? v : 0.f;
      }
      *reinterpret_cast<float4*>(dst + e * 16) = make_float4(w[0], w[1] - w[0], w[2] - w[0], (w[3] - w[1]) - (w[2] - w[0]));
    }
  };
  auto issue = [&](const Pixel& p, int rows, int cb) {
    const int last = min(kTlCh, cpg - cb * kTlCh) - 1;
    const size_t c0 = (size_t)p.n * g.channel + grp + (size_t)g.groups * (cb * kTlCh);
    // (a channel past the block's last one lies outside: it reads as zeros)
    const rsrc_t rx = plane_rsrc(x + c0 * in_plane, last * g.groups * in_plane + in_plane);
    const rsrc_t rg = plane_rsrc(gout + c0 * out_plane, last * g.groups * out_plane + out_plane);
#pragma unroll
    for (int k = 0; k < kTlStage; ++k)
      if ((wave + kTlWaves * k) * 16 < rows * kTlCols)  // uniform
#pragma unroll
        for (int c = 0; c < 4; ++c) r_x[k][c] = c <= last ? buf_ld2(rx, x_off[k], c * x_cs, x) : 0.f;
    r_g = buf_ld(rg, p.at >= 0 ? (unsigned)(q * g_cs) + (unsigned)p.at * (unsigned)sizeof(T) : kOutOfRange, gout);
  };

  // the waves' products of a block, added up in pairs by the threads that own them
  auto flush = [&](int b, int par) {
    if (threadIdx.x >= kTlBlock - 256) {  // (the first waves make the table)
      const int e = threadIdx.x - (kTlBlock - 256);
      float s[kTlWaves];
#pragma unroll
      for (int w = 0; w < kTlWaves; ++w) s[w] = red[par * kTlWaves * 256 + w * 256 + e];
      fsum[b * 256 + e] += tree_sum(s);
    }
  };

  int id = tile_lo;
  Pixel pix = pixel(id);
  Raw raw = load_raw(pix);
  Box box = read_box(id);
  __syncthreads();  // the weights are in place
  make_table(0, tbl);
  Window win = window(box, 0);
  aim(win);
  issue(pix, win.rows, cb_lo);

  int step = 0, flush_blk = -1;
  for (; id < tile_hi; id += reg_n) {
    const bool more = id + reg_n < tile_hi;
    const Tap tap = describe(pix, raw);
    float A[K9];
    static_for<K9>([&](auto t_tag) {
      constexpr int t = decltype(t_tag)::value;
      A[t] = hat(row_lane<t>(tap.sh) - ci) * hat(row_lane<t>(tap.sw) - cj);
    });
    const float shf = floorf(tap.sh), swf = floorf(tap.sw);
    const bool in = tap.sh > -1.f;
    const float d_fh = in ? tap.sh - shf : 0.f, d_fw = in ? tap.sw - swf : 0.f;
    const int d_cell = in ? (((int)shf + 1) * (SW + 1) + (int)swf + 1) * (kTlCh * 16) : 0;  // (cell (-1, -1): a weight of zero)
    float o_h[K9], o_w[K9], r_h[ROT ? K9 : 1], r_w[ROT ? K9 : 1];
#pragma unroll
    for (int t = 0; t < K9; ++t) o_h[t] = o_w[t] = 0.f;
#pragma unroll
    for (int t = 0; t < (ROT ? K9 : 1); ++t) r_h[t] = r_w[t] = 0.f;

    const int passes = box.passes_r * box.passes_c;
    for (int pass = 0; pass < passes; ++pass) {
      const int row = (tap.at >> 16) - win.row, col = (tap.at & 0xffff) - win.col;
      const bool here = tap.at >= 0 && row >= 0 && row < kTlRows - 1 && col >= 0 && col < kTlCols - 1;
      const int d_off = (here ? row * kTlCols + col : kTlPos) * (kTlCh * 4);
      for (int b = 0; b < nblk; ++b, ++step) {
        const int par = step & 1;
        char* pl = planes + par * kTlSlots * kTlCh * 4;
        char* tb = tbl + par * TCELLS * kTlCh * 16;
        const bool tile_ends = b + 1 == nblk && pass + 1 == passes;
#pragma unroll
        for (int k = 0; k < kTlStage; ++k) {
          const int unit = wave + kTlWaves * k;
          if (unit * 16 + (lane >> 2) < kTlPos)
            *reinterpret_cast<float4*>(pl + unit * 1024 + lane * 16) = make_float4(r_x[k][0], r_x[k][1], r_x[k][2], r_x[k][3]);
        }
        const float gv = r_g;
        __syncthreads();
        // the next step's loads
        Pixel p_next = pix;
        if (b + 1 == nblk) {
          if (pass + 1 < passes) {
            win = window(box, pass + 1);
            aim(win);
          } else if (more) {
            p_next = pixel(id + reg_n);
            box = read_box(id + reg_n);
            win = window(box, 0);
            aim(win);
          }
        }
        if (!tile_ends || more) {
          issue(p_next, win.rows, cb_lo + (b + 1 < nblk ? b + 1 : 0));
          make_table(b + 1 < nblk ? b + 1 : 0, tbl + (par ^ 1) * TCELLS * kTlCh * 16);
        }
        if (flush_blk >= 0) flush(flush_blk, par ^ 1);
        flush_blk = b;

        // (the descriptors look new in every block: else the compiler keeps what all 54 DPP operands select in registers)
        int off_ = d_off, cell_ = d_cell;
        float lh_ = tap.lh, lw_ = tap.lw, fh_ = d_fh, fw_ = d_fw;
        asm volatile("" : "+v"(off_), "+v"(cell_), "+v"(lh_), "+v"(lw_), "+v"(fh_), "+v"(fw_));
        const char* c_lane = pl + q * 4;
        const char* t_lane = tb + q * 16;
        tl_f4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
        // corners and table entry of tap t + 1 are read in front of tap t's arithmetic
        float cr[2][4];
        float4 wt[2];
        auto read = [&](auto t_tag) {
          constexpr int t = decltype(t_tag)::value;
          const char* c0 = c_lane + row_lane<t>(off_);
          cr[t & 1][0] = *reinterpret_cast<const float*>(c0);
          cr[t & 1][1] = *reinterpret_cast<const float*>(c0 + kTlCh * 4);
          cr[t & 1][2] = *reinterpret_cast<const float*>(c0 + kTlCols * kTlCh * 4);
          cr[t & 1][3] = *reinterpret_cast<const float*>(c0 + (kTlCols + 1) * kTlCh * 4);
          wt[t & 1] = *reinterpret_cast<const float4*>(t_lane + row_lane<t>(cell_));
        };
        read(std::integral_constant<int, 0>{});
        static_for<K9>([&](auto t_tag) {
          constexpr int t = decltype(t_tag)::value;
          if constexpr (t + 1 < K9) read(std::integral_constant<int, t + 1>{});
          __builtin_amdgcn_sched_barrier(0);
          const float ca = cr[t & 1][0], cb = cr[t & 1][1], cc = cr[t & 1][2], cd = cr[t & 1][3];
          const float4 f = wt[t & 1];
          float s_h, s_w, val, w_h = f.z, w_w = f.y, wgt = f.x;
          lerp_row<t, ROT, OWN>(lh_, lw_, fh_, fw_, ca, cb, cc, cd, f.w, s_h, s_w, val, w_h, w_w, wgt);
          const float ps = gv * val, gw = gv * wgt;
          o_h[t] = fmaf(gw, s_h, o_h[t]);
          o_w[t] = fmaf(gw, s_w, o_w[t]);
          if constexpr (ROT) {
            r_h[t] = fmaf(ps, w_h, r_h[t]);
            r_w[t] = fmaf(ps, w_w, r_w[t]);
          }
          if (t & 1)
            acc1 = __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], ps, acc1, 0, 0, 0);
          else
            acc0 = __builtin_amdgcn_mfma_f32_16x16x4f32(A[t], ps, acc0, 0, 0, 0);
          __builtin_amdgcn_sched_barrier(0);
        });
        *reinterpret_cast<tl_f4*>(red + par * kTlWaves * 256 + wave * 256 + lane * 4) = acc0 + acc1;
      }
    }

    const Pixel done = pix;
    if (more) {
      pix = pixel(id + reg_n);
      raw = load_raw(pix);
    }
    // the tile's coordinate gradients: lane q gets kind q % 4 of taps q / 4, 4 + q / 4, 8 + q / 4
    float v[3] = {0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < K9; ++t) {
      const float s = row_sums(o_h[t], o_w[t], ROT ? r_h[ROT ? t : 0] : 0.f, ROT ? r_w[ROT ? t : 0] : 0.f, q);
      v[t / 4] = q / 4 == t % 4 ? s : v[t / 4];
    }
    const bool of_rot = q & 2;
    if (done.at >= 0 && (ROT || !of_rot)) {
      const size_t img18 = (size_t)18 * out_plane;
      const size_t img = of_rot ? (size_t)done.n * g.groups + grp : (size_t)done.n;
      float* part = of_rot ? part_rot : part_off;
      if (part)
        part += (of_rot ? (size_t)chunk * g.batch * g.groups + img : ((size_t)grp * plan.chunks + chunk) * g.batch + img) * img18 + done.at;
      T* full = (of_rot ? grot : goff) + img * img18 + done.at;
#pragma unroll
      for (int j = 0; j < 3; ++j) {
        const int t = 4 * j + q / 4;
        if (t < K9) {
          const size_t at = (size_t)(2 * t + (q & 1)) * out_plane;
          float r = v[j];
          if (of_rot && g.clip_mode != kClipNone) {  // a clamped offset has no gradient
            bool open;
            scope_coord<float>(g, q & 1 ? t % 3 : t / 3, ld(rot + img * img18 + done.at + at), q & 1 ? g.centre_w : g.centre_h, &open);
            r = open ? r : 0.f;
          }
          if (part) part[at] = r;
          else st(full + at, r);
        }
      }
    }
  }
  __syncthreads();
  flush(flush_blk, (step - 1) & 1);
  // entry e of a block: D[cell = 4 * (l / 16) + r][channel l % 16] with l = e / 4, r = e % 4 (register r of lane l); every
  // thread writes what it added up
  if (threadIdx.x >= kTlBlock - 256) {
    const int e = threadIdx.x - (kTlBlock - 256), l = e / 4, cell = 4 * (l / 16) + e % 4;
    for (int b = 0; b < nblk; ++b) {
      const int c = (cb_lo + b) * kTlCh + l % 16;
      if (cell < CELLS && c < cpg)
        part_filter[((size_t)wg * g.channel + grp + (size_t)g.groups * c) * CELLS + cell] = fsum[b * 256 + e];
    }
  }
}

// The reductions of the form that took the call, in one launch: each takes its turn over the whole grid.  Many elements (the
// coordinates'): one or four per thread, several parts in flight; few (the filter's, whose parts are many): 16 per workgroup,
// every 64th part per row of 16 threads.
template <typename T>
struct ReduceJobs {
  ReduceJob<T> tile[3], wide[3];
};
constexpr long kTlManyElements = 32768;
template <typename T>
__global__ __launch_bounds__(1024) void deform_reduce_jobs_kernel(ReduceJobs<T> jobs, TileChoice choice) {
  constexpr int PU = 8;
  __shared__ float rows[16][16];
  const bool wide = choice.windows && !tiles_take(choice);
  const int e = threadIdx.x & 15, row = threadIdx.x >> 4;
  for (int k = 0; k < 3; ++k) {
    const ReduceJob<T> j = wide ? jobs.wide[k] : jobs.tile[k];
    if (j.count >= kTlManyElements && j.count % 4 == 0 && reinterpret_cast<size_t>(j.partial) % 16 == 0) {
      for (long at = ((long)blockIdx.x * 1024 + threadIdx.x) * 4; at < j.count; at += (long)gridDim.x * 4096) {
        tl_f4 s = {0.f, 0.f, 0.f, 0.f};
        for (int p0 = 0; p0 < j.parts; p0 += PU / 2) {
          tl_f4 p[PU / 2];
#pragma unroll
          for (int i = 0; i < PU / 2; ++i)
            p[i] = p0 + i < j.parts ? *reinterpret_cast<const tl_f4*>(j.partial + (size_t)(p0 + i) * j.count + at) : tl_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int i = 0; i < PU / 2; ++i) s += p[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) st(j.out + at + i, s[i]);
      }
      continue;
    }
    if (j.count >= kTlManyElements) {
      for (long at = (long)blockIdx.x * 1024 + threadIdx.x; at < j.count; at += (long)gridDim.x * 1024) {
        float s = 0.f;
        for (int p0 = 0; p0 < j.parts; p0 += PU) {
          float p[PU];
#pragma unroll
          for (int i = 0; i < PU; ++i) p[i] = p0 + i < j.parts ? j.partial[(size_t)(p0 + i) * j.count + at] : 0.f;
#pragma unroll
          for (int i = 0; i < PU; ++i) s += p[i];
        }
        st(j.out + at, s);
      }
      continue;
    }
    for (long i = blockIdx.x; i < (j.count + 15) / 16; i += gridDim.x) {
      const long at = i * 16 + e;
      float s = 0.f;
      if (at < j.count) {
#pragma unroll 4
        for (int p = row; p < j.parts; p += 64) s += j.partial[(size_t)p * j.count + at];
      }
      // 64 rows in pairs: the four of a wave, then the waves'
      s += __shfl_xor(s, 16);
      s += __shfl_xor(s, 32);
      __syncthreads();
      if (row % 4 == 0) rows[row / 4][e] = s;
      __syncthreads();
      if (row == 0 && at < j.count) {
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) v[r] = rows[r][e];
        st(j.out + at, tree_sum(v));
      }
    }
  }
}

TilePlan tile_plan(const Geo& g, bool rotation) {
  TilePlan m{};
  if (path_disabled(kNoDeformFast) || path_disabled(kNoDeformMfma) || path_disabled(kNoDeformWindow)) return m;
  if (g.k_h != 3 || g.k_w != 3 || g.stride_h != 1 || g.stride_w != 1 || g.dil_h != 1 || g.dil_w != 1) return m;
  if (!(g.scope_h == 4 && g.scope_w == 4) && !(g.scope_h == 3 && g.scope_w == 3)) return m;
  const long out_plane = (long)g.out_h * g.out_w, in_plane = (long)g.in_h * g.in_w;
  // 32-bit byte offsets in the 18 offset planes, and in a block's planes of 16 channels
  if (g.in_h >= 1 << 15 || g.in_w >= 1 << 16) return m;  // Tap::at: row and column of a corner, up to the sides, in one word
  if (18 * out_plane * 4 >= (1L << 31) || 16L * g.groups * std::max(out_plane, in_plane) * 4 >= (1L << 31)) return m;
  if ((long)g.channel * g.scope_h * g.scope_w * 4 >= (1L << 31)) return m;
  const int cpg = g.channel / g.groups, nblk = ceil_div(cpg, kTlCh);
  m.tiles_x = ceil_div(g.out_w, kTlSide);
  m.tiles = m.tiles_x * ceil_div(g.out_h, kTlSide);
  const long tiles = (long)g.batch * m.tiles;
  if (tiles == 0 || tiles >= (1L << 30)) return m;
  // one workgroup per CU; the channel blocks are shared out where the tiles are too few
  const long spread = std::max(1L, 256 / std::max(1L, tiles * g.groups));
  const int want = (int)std::max<long>(ceil_div(nblk, kTlMostBlocks), std::min<long>(nblk, spread));
  m.per_chunk = ceil_div(nblk, want);
  m.chunks = ceil_div(nblk, m.per_chunk);
  m.wgs = (int)std::max(1L, std::min<long>(tiles, 256 / ((long)m.chunks * g.groups)));
  m.lds = (size_t)2 * kTlSlots * kTlCh * 4 + (size_t)2 * (g.scope_h + 1) * (g.scope_w + 1) * kTlCh * 16 +
          (size_t)2 * kTlWaves * 1024 + (size_t)m.per_chunk * (1024 + g.scope_h * g.scope_w * kTlCh * 4);
  if (m.lds > (size_t)kTlLds) return m;
  // Where it is the faster form; us, all three gradients, separate kernels / this one, offsets ~ N(0, 2^2).  Planes that the
  // separate kernels take in windows or in one workgroup per CU: everywhere but with mostly empty blocks: float32 N=64 C=144
  // 56 x 56 632 / 440, N=4 90 / 56, N=1 C=118 46 / 33, N=21 C=32 101 / 78, N=32 C=32 112 x 112 391 / 290, N=16 C=17 120 x 70 146 / 118, float16
  // N=32 C=144 56 x 56 495 / 305; C=8 49 / 53, C=4 46 / 50.
  if (cpg <= kTlCh / 2) return m;
  m.boxed = g.in_h + 2 > kTlRows || g.in_w + 2 > kTlCols;
  // Planes that they take whole in three workgroups per CU: few tiles that fill their pixels and channels, on planes that fit the
  // window whatever the offsets: N=115 C=193 7 x 7 90 / 36, N=16 C=384 14 x 14 55 / 35, N=2 C=600 14 x 14 bfloat16 35 / 24; but
  // N=128 C=384 14 x 14 156 / 225, N=100 C=12 30 x 12 bfloat16 36 / 47, N=64 C=192 28 x 28 190 / 215.
  if (rotation && deform_small_plane(g)) {
    const bool filled = (double)out_plane * cpg >= 0.6 * (double)(m.tiles * kTlSide * kTlSide) * (nblk * kTlCh);
    if (m.boxed || tiles * g.groups * nblk > 8 * 256 || !filled) return m;
  }
  m.ok = true;
  return m;
}

// Workspace: the tiles' boxes, the windows of the workgroups that made them and the word that says whose the call is; then the
// partial sums, of the offset, rotation and filter gradient or, if the choice falls on the separate kernels, theirs.
constexpr int kTlBoxGrid = 256;
struct TileWorkspace {
  size_t boxes, off, rot, filter;  // bytes; floats
};
TileWorkspace tile_workspace(const Geo& g, const TilePlan& m) {
  const size_t img = (size_t)18 * g.out_h * g.out_w * g.batch;
  TileWorkspace w;
  w.boxes = m.boxed ? ((size_t)g.batch * m.tiles * sizeof(int4) + (kTlBoxGrid + 1) * sizeof(unsigned) + 255) / 256 * 256 : 0;
  w.off = m.chunks * g.groups > 1 ? (size_t)m.chunks * g.groups * img : 0;
  w.rot = m.chunks > 1 ? (size_t)m.chunks * g.groups * img : 0;
  w.filter = (size_t)m.wgs * g.channel * g.scope_h * g.scope_w;
  return w;
}

template <typename T, int SH, int SW>
bool run_tile(const Geo& g, const TilePlan& m, const T* gout, const T* x, const T* off, const T* rot, const T* filter, T* goff,
              T* grot, T* gfilter, float* ws0, hipStream_t stream) {
  const TileWorkspace w = tile_workspace(g, m);
  int4* boxes = m.boxed ? reinterpret_cast<int4*>(ws0) : nullptr;
  float* ws = ws0 + w.boxes / sizeof(float);
  float *p_off = w.off ? ws : nullptr, *p_rot = w.rot && rot ? ws + w.off : nullptr, *p_filter = ws + w.off + w.rot;
  // One change for both slopes is 3 % of the kernel's time; with few channels the longer sums of the separate kernels do not make up for its
  // rounding: offset gradient's error against float64 in 10^-8, separate kernels / one change / each its own: 16 channels 10.4 / 10.6 / 10.4,
  // 48 11.02 / 11.06 / 10.81, 64 11.3 / 11.0, 144 17.7 / 11.8.
  const bool own = g.channel / g.groups < 64;
  auto kernel = rot ? (own ? deform_grad_tile_kernel<T, SH, SW, true, true> : deform_grad_tile_kernel<T, SH, SW, true, false>)
                    : (own ? deform_grad_tile_kernel<T, SH, SW, false, true> : deform_grad_tile_kernel<T, SH, SW, false, false>);
  if (!allow_dynamic_lds(reinterpret_cast<const void*>(kernel), kTlLds)) return false;
  TileChoice choice{}, behind{};
  unsigned* left = nullptr;
  if (m.boxed) {
    unsigned* windows = reinterpret_cast<unsigned*>(boxes + (size_t)g.batch * m.tiles);
    deform_tile_boxes_kernel<T><<<kTlBoxGrid, 256, 0, stream>>>(g, off, boxes, windows, m.tiles_x, m.tiles);
    // Windows per tile, in sixteenths, up to which this is the faster form: N=64 C=144 56 x 56 float32, offsets ~ N(0, s^2),
    // windows per tile, separate kernels / this one: s = 2 1.0: 632 / 440; s = 3 1.3: 780 / 545; s = 4 2.5: 909 / 1060; with a few
    // tiles per workgroup the slowest one counts: N=4 s = 3 105 / 131.  Where it does not take the call its launches cost 2 - 20 us,
    // where it does theirs 10.
    const int limit = (long)g.batch * m.tiles >= 4L * m.wgs ? 25 : 17;
    if (wide_deform_grads_workspace(g, rot != nullptr)) choice = {windows, kTlBoxGrid, (unsigned)((long)g.batch * m.tiles * limit / 16)};
    left = windows + kTlBoxGrid;
    if (choice.windows) behind = {left, 1, 0u};
  }
  kernel<<<(unsigned)xcd_grid_size((long)m.wgs * m.chunks * g.groups), kTlBlock, m.lds, stream>>>(
      g, gout, x, off, rot, filter, goff, grot, p_off, p_rot, p_filter, m, boxes, choice, left);
  const long img = (long)18 * g.out_h * g.out_w * g.batch;
  ReduceJobs<T> jobs{};
  if (p_off) jobs.tile[0] = {p_off, m.chunks * g.groups, img, goff};
  if (p_rot) jobs.tile[1] = {p_rot, m.chunks, img * g.groups, grot};
  jobs.tile[2] = {p_filter, m.wgs, (long)g.channel * SH * SW, gfilter};
  if (choice.windows && !wide_deform_grads<T>(g, gout, x, off, rot, filter, goff, grot, gfilter, ws, behind, jobs.wide, stream)) return false;
  long most = 0;  // elements, a thread each; of the filter's, a workgroup for 16
  for (const ReduceJob<T>* j : {&jobs.tile[0], &jobs.tile[1], &jobs.wide[0], &jobs.wide[1]}) most = std::max(most, j->count);
  const long grid = std::max(ceil_div((int)std::min(most, 1L << 30), 1024), ceil_div(g.channel * SH * SW, 16));
  deform_reduce_jobs_kernel<T><<<(unsigned)std::min(1024L, grid), 1024, 0, stream>>>(jobs, behind);
  return true;
}

}  // namespace

size_t tile_deform_grads_workspace(const Geo& g, bool rotation) {
  const TilePlan m = tile_plan(g, rotation);
  if (!m.ok) return 0;
  const TileWorkspace w = tile_workspace(g, m);
  return w.boxes + std::max((w.off + w.rot + w.filter) * sizeof(float), m.boxed ? wide_deform_grads_workspace(g, rotation) : 0);
}

template <typename T>
bool tile_deform_grads(const Geo& g, const T* gout, const T* x, const T* off, const T* rot, const T* filter, T* goff, T* grot,
                       T* gfilter, float* ws, hipStream_t stream) {
  const TilePlan m = tile_plan(g, rot != nullptr);
  if (!m.ok) return false;
  if (g.scope_h == 4) return run_tile<T, 4, 4>(g, m, gout, x, off, rot, filter, goff, grot, gfilter, ws, stream);
  return run_tile<T, 3, 3>(g, m, gout, x, off, rot, filter, goff, grot, gfilter, ws, stream);
}

#define DK_INSTANTIATE(T)                                                                                              \
  template bool tile_deform_grads<T>(const Geo&, const T*, const T*, const T*, const T*, const T*, T*, T*, T*, float*, \
                                     hipStream_t);
DK_INSTANTIATE(float)
DK_INSTANTIATE(__half)
DK_INSTANTIATE(bf16_t)
#undef DK_INSTANTIATE

}  // namespace dk
