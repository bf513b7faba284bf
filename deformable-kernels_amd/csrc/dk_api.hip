// C ABI of libdk_hip.so (declared in include/dk_hip.h): argument validation,
// geometry derivation and dispatch to the tuned or the generic kernels.
// Each entry point names the reference pybind function it stands in for
// (K.cpp = deformable_kernels/ops/deform_kernel/csrc/filter_sample_depthwise_cuda.cpp,
//  ND.cpp = .../csrc/nd_linear_sample_cuda.cpp).
#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <initializer_list>
#include <mutex>
#include <type_traits>
#include <utility>
#include <vector>

#include "dk_kernels.h"
#include "dk_nd.h"

using namespace dk;

namespace dk {

namespace {
constexpr unsigned kSwitchesUnread = 0x80000000u;
std::atomic<unsigned> g_switches{kSwitchesUnread};

unsigned switches_from_environment() {
  static const struct { const char* name; unsigned bit; } vars[] = {
      {"DK_NO_ROWS", kNoRows}, {"DK_NO_MFMA", kNoMfma}, {"DK_NO_MFMA_S2", kNoMfmaS2},
      {"DK_NO_S2_QUADS", kNoS2Quads}, {"DK_NO_DEFORM_FAST", kNoDeformFast}, {"DK_NO_DEFORM_CH", kNoDeformCh},
      {"DK_NO_DEFORM_CH_BIG", kNoDeformChBig}, {"DK_NO_DEFORM_MFMA", kNoDeformMfma},
      {"DK_NO_ND_BINS", kNoNdBins}, {"DK_NO_ND_MFMA", kNoNdMfma}, {"DK_NO_GATHER_MFMA", kNoGatherMfma},
      {"DK_NO_FILTER_SPLIT", kNoFilterSplit}, {"DK_NO_IMAGE_FLAT", kNoImageFlat},
      {"DK_NO_ND_SMALL", kNoNdSmall}, {"DK_NO_ND_ROWS", kNoNdRows}, {"DK_NO_NHWC_MFMA", kNoNhwcMfma},
      {"DK_FORCE_GATHER_MFMA", kForceGatherMfma}, {"DK_NO_PIXEL_LANES", kNoPixelLanes},
      {"DK_FORCE_PIXEL_LANES", kForcePixelLanes}, {"DK_NO_OFFSET_PAIRS", kNoOffsetPairs}, {"DK_NO_OFFSET_WGRAD16", kNoOffsetWgrad16}, {"DK_NO_DEFORM_WINDOW", kNoDeformWindow}, {"DK_FORCE_WIN2", kForceWin2}, {"DK_NO_NHWC_STAGED", kNoNhwcStaged}, {"DK_FORCE_NHWC_GATHER_MFMA", kForceNhwcGatherMfma}, {"DK_NO_IMAGE_PACKED", kNoImagePacked}, {"DK_NO_DEFORM_LANES", kNoDeformLanes}, {"DK_FORCE_DEFORM_LANES", kForceDeformLanes}, {"DK_NO_DEFORM_PLAIN", kNoDeformPlain}, {"DK_NO_SMALL_BACKWARD", kNoSmallBackward}};
  // a production process ignores these variables: they count only next to DK_ENABLE_TEST_SWITCHES=1
  const char* on = std::getenv("DK_ENABLE_TEST_SWITCHES");
  if (!on || on[0] != '1') return 0;
  unsigned m = 0;
  for (const auto& v : vars)
    if (std::getenv(v.name)) m |= v.bit;
  return m;
}

std::mutex g_lds_mutex;
struct LdsAllowed { const void* kernel; int device, bytes; };
std::vector<LdsAllowed> g_lds_allowed;  // what has been set so far
}  // namespace

unsigned test_switches() {
  unsigned m = g_switches.load(std::memory_order_relaxed);
  if (m == kSwitchesUnread) {
    m = switches_from_environment();
    unsigned expected = kSwitchesUnread;
    if (!g_switches.compare_exchange_strong(expected, m)) m = expected;  // a dk_test_switches() call came first
  }
  return m;
}

bool allow_dynamic_lds(const void* kernel, int bytes) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return false;
  std::lock_guard<std::mutex> lock(g_lds_mutex);
  for (auto& e : g_lds_allowed)
    if (e.kernel == kernel && e.device == dev) {
      if (e.bytes >= bytes) return true;
      if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
      e.bytes = bytes;  // only ever raised: a concurrent launch may rely on the old value
      return true;
    }
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  g_lds_allowed.push_back({kernel, dev, bytes});
  return true;
}

bool allow_max_dynamic_lds(const void* kernel) { return allow_dynamic_lds(kernel, kMaxDynamicLds); }

}  // namespace dk

namespace {

constexpr long kMaxElems = 2147483647L;  // plane-relative indices are 32-bit

int make_geo(const dk_conv_desc* d, Geo& g) {
  if (!d) return DK_ERR_NULL_POINTER;
  if (d->dtype < DK_F32 || d->dtype > DK_F64) return DK_ERR_BAD_DTYPE;
  if (d->batch < 0 || d->channel <= 0 || d->in_h <= 0 || d->in_w <= 0 || d->k_h <= 0 ||
      d->k_w <= 0 || d->stride_h <= 0 || d->stride_w <= 0 || d->pad_h < 0 || d->pad_w < 0 ||
      d->dil_h <= 0 || d->dil_w <= 0 || d->scope_h <= 0 || d->scope_w <= 0 || d->groups <= 0)
    return DK_ERR_BAD_SHAPE;
  if (d->channel % d->groups != 0) return DK_ERR_BAD_SHAPE;
  if (d->layout != DK_LAYOUT_NCHW && d->layout != DK_LAYOUT_NHWC) return DK_ERR_BAD_SHAPE;
  if (d->rotation_clip < DK_CLIP_NONE || d->rotation_clip > DK_CLIP_COORD ||
      (d->rotation_clip != DK_CLIP_NONE && !(d->clip_min <= d->clip_max)))
    return DK_ERR_BAD_SHAPE;
  // K.cpp:42-43
  const long oh = ((long)d->in_h + 2L * d->pad_h - ((long)d->dil_h * (d->k_h - 1) + 1)) / d->stride_h + 1;
  const long ow = ((long)d->in_w + 2L * d->pad_w - ((long)d->dil_w * (d->k_w - 1) + 1)) / d->stride_w + 1;
  if ((long)d->in_h + 2L * d->pad_h < (long)d->dil_h * (d->k_h - 1) + 1 ||
      (long)d->in_w + 2L * d->pad_w < (long)d->dil_w * (d->k_w - 1) + 1 || oh <= 0 || ow <= 0)
    return DK_ERR_BAD_SHAPE;
  // element counts as saturating products: the factors are only known to be positive 32-bit
  // numbers here, and four of them can exceed 64 bits
  auto count = [](std::initializer_list<long> f) {
    long p = 1;
    for (long v : f) p = (v != 0 && p > (1L << 62) / v) ? (1L << 62) : p * v;
    return p;
  };
  const long taps = count({d->k_h, d->k_w});
  if (count({d->batch, d->channel, d->in_h, d->in_w}) > kMaxElems ||
      count({d->batch, d->channel, oh, ow}) > kMaxElems ||
      count({d->batch, d->groups, 2, taps, oh, ow}) > kMaxElems ||
      count({d->batch, d->channel, taps, oh, ow}) > 4 * kMaxElems ||
      count({d->channel, d->scope_h, d->scope_w}) > kMaxElems)
    return DK_ERR_TOO_LARGE;
  g.batch = d->batch;
  g.channel = d->channel;
  g.in_h = d->in_h;
  g.in_w = d->in_w;
  g.k_h = d->k_h;
  g.k_w = d->k_w;
  g.stride_h = d->stride_h;
  g.stride_w = d->stride_w;
  g.pad_h = d->pad_h;
  g.pad_w = d->pad_w;
  g.dil_h = d->dil_h;
  g.dil_w = d->dil_w;
  g.out_h = (int)oh;
  g.out_w = (int)ow;
  g.scope_h = d->scope_h;
  g.scope_w = d->scope_w;
  g.groups = d->groups;
  g.centre_h = (d->scope_h - d->k_h) / 2.0;  // K.cu:338-341
  g.centre_w = (d->scope_w - d->k_w) / 2.0;
  g.clip_mode = d->rotation_clip;
  g.clip_lo = d->clip_min;
  g.clip_hi = d->clip_max;
  return DK_OK;
}

int launch_status() { return hipGetLastError() == hipSuccess ? DK_OK : DK_ERR_LAUNCH; }

// Calls f.template operator()<T>() with T the element type tagged by `dtype`.
template <typename F>
int by_dtype(int dtype, F&& f) {
  switch (dtype) {
    case DK_F32: f.template operator()<float>(); break;
    case DK_F16: f.template operator()<__half>(); break;
    case DK_BF16: f.template operator()<bf16_t>(); break;
    case DK_F64: f.template operator()<double>(); break;
    default: return DK_ERR_BAD_DTYPE;
  }
  return launch_status();
}

// The tuned kernels exist for the 16- and 32-bit types only.
template <typename T> constexpr bool kHasFast = !std::is_same<T, double>::value;

template <typename T> const T* in(const void* p) { return static_cast<const T*>(p); }
template <typename T> T* out(void* p) { return static_cast<T*>(p); }

// The filter gradient of an empty batch is all zeros: the ordered reduction over zero partial
// buffers writes them (a kernel, not a memset, so the call can be captured into a graph).
int zero_filter_grad(const Geo& g, int dtype, void* filter_grad, hipStream_t s) {
  const long count = (long)g.channel * g.scope_h * g.scope_w;
  return by_dtype(dtype, [&]<typename T>() {
    using CT = compute_t<T>;
    launch_reduce_partials<CT, T>(static_cast<const CT*>(nullptr), 0, count, out<T>(filter_grad), s);
  });
}

size_t local_filter_ws(const Geo& g, int dtype, int layout = DK_LAYOUT_NCHW) {
  if (layout == DK_LAYOUT_NHWC) return nhwc_supported(g, dtype) ? nhwc_grad_filter_workspace(g, dtype) : 0;
  const size_t a = dtype == DK_F64 ? 0 : fast_local_grad_filter_workspace(g);
  return a ? a : generic_grad_filter_workspace(g, dtype);
}

}  // namespace

// ---- the filter gradient for callers that cannot allocate ---------------------------------
//
// The per-workgroup partial sums live in a file-scope device array instead of a caller's
// workspace.  Each GPU holds its own copy of the array at its own address; the address is looked
// up once per device (first call with that device current) and kept.  Host code never uses the
// array's name as a pointer: kernels, and anything else that needs the memory, get `ptr`.
static __device__ __align__(256) unsigned char dk_static_scratch[DK_STATIC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<void*> g_static_scratch[kMaxDevices];

int static_scratch_of_current_device(void** ptr) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return DK_ERR_LAUNCH;
  if (dev < 0 || dev >= kMaxDevices) return DK_ERR_UNSUPPORTED;
  void* p = g_static_scratch[dev].load(std::memory_order_acquire);
  if (!p) {
    // two threads racing here both get the same address
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(dk_static_scratch)) != hipSuccess || !p) return DK_ERR_LAUNCH;
    g_static_scratch[dev].store(p, std::memory_order_release);
  }
  *ptr = p;
  return DK_OK;
}
// by_dtype without float64, which these kernels do not take
template <typename F>
int by_tensor_dtype(int dtype, F&& f) {
  return by_dtype(dtype, [&]<typename T>() {
    if constexpr (!std::is_same_v<T, double>) f.template operator()<T>();
  });
}

}  // namespace

extern "C" {

int dk_version(void) { return (0 << 16) | 3; }

size_t dk_conv_desc_size(void) { return sizeof(dk_conv_desc); }
size_t dk_nd_desc_size(void) { return sizeof(dk_nd_desc); }
size_t dk_offset_conv_desc_size(void) { return sizeof(dk_offset_conv_desc); }

unsigned dk_test_switches(unsigned mask) {
  const unsigned before = test_switches();
  g_switches.store(mask & ~kSwitchesUnread, std::memory_order_relaxed);
  return before;
}

const char* dk_status_string(int status) {
  switch (status) {
    case DK_OK: return "ok";
    case DK_ERR_NULL_POINTER: return "null pointer argument";
    case DK_ERR_BAD_SHAPE: return "invalid shape (non-positive size, empty output, or channel % groups != 0)";
    case DK_ERR_BAD_DTYPE: return "unknown dtype tag";
    case DK_ERR_TOO_LARGE: return "tensor has 2^31 or more elements";
    case DK_ERR_WORKSPACE: return "workspace missing or too small";
    case DK_ERR_LAUNCH: return "HIP kernel launch failed";
    case DK_ERR_UNSUPPORTED: return "unsupported configuration";
    case DK_ERR_SCRATCH_LIMIT: return "problem needs more scratch memory than the library's static buffer holds";
    default: return "unknown status";
  }
}

int dk_conv_out_size(const dk_conv_desc* desc, int32_t* out_h, int32_t* out_w) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (out_h) *out_h = g.out_h;
  if (out_w) *out_w = g.out_w;
  return DK_OK;
}

int dk_sample_depthwise_layout_supported(const dk_conv_desc* desc) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  return desc->layout == DK_LAYOUT_NHWC ? (nhwc_supported(g, desc->dtype) ? 1 : 0) : 1;
}

// ---- local ------------------------------------------------------------------------------

int dk_sample_depthwise_forward(const dk_conv_desc* desc, const void* input, const void* rotation,
                                const void* filter, void* output, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!input || !rotation || !filter || !output) return DK_ERR_NULL_POINTER;
  if (desc->layout == DK_LAYOUT_NHWC && !nhwc_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (desc->layout == DK_LAYOUT_NHWC)
    return by_dtype(desc->dtype, [&]<typename T>() {
      nhwc_gather<T>(g, false, in<T>(input), in<T>(rotation), in<T>(filter), out<T>(output), s);
    });
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_local_gather<T>(g, false, in<T>(input), in<T>(rotation), in<T>(filter), out<T>(output), s)) return;
    generic_forward<T>(g, false, in<T>(input), (const T*)nullptr, in<T>(rotation), in<T>(filter), out<T>(output), s);
  });
}

int dk_sample_depthwise_backward_data(const dk_conv_desc* desc, const void* out_grad,
                                      const void* rotation, const void* filter, void* in_grad,
                                      void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!out_grad || !rotation || !filter || !in_grad) return DK_ERR_NULL_POINTER;
  if (desc->layout == DK_LAYOUT_NHWC && !nhwc_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (desc->layout == DK_LAYOUT_NHWC)
    return by_dtype(desc->dtype, [&]<typename T>() {
      nhwc_gather<T>(g, true, in<T>(out_grad), in<T>(rotation), in<T>(filter), out<T>(in_grad), s);
    });
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_local_gather<T>(g, true, in<T>(out_grad), in<T>(rotation), in<T>(filter), out<T>(in_grad), s)) return;
    generic_local_grad_input<T>(g, in<T>(out_grad), in<T>(rotation), in<T>(filter), out<T>(in_grad), s);
  });
}

size_t dk_sample_depthwise_backward_filter_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return local_filter_ws(g, desc->dtype, desc->layout);
}

int dk_sample_depthwise_backward_filter(const dk_conv_desc* desc, const void* out_grad,
                                        const void* input, const void* rotation, void* filter_grad,
                                        void* workspace, size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!out_grad || !input || !rotation || !filter_grad) return DK_ERR_NULL_POINTER;
  if (desc->layout == DK_LAYOUT_NHWC && !nhwc_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  const size_t need = local_filter_ws(g, desc->dtype, desc->layout);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (g.batch == 0) return zero_filter_grad(g, desc->dtype, filter_grad, s);
  if (desc->layout == DK_LAYOUT_NHWC)
    return by_dtype(desc->dtype, [&]<typename T>() {
      nhwc_grad_filter<T>(g, in<T>(out_grad), in<T>(input), in<T>(rotation), out<T>(filter_grad), workspace, s);
    });
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_local_grad_filter<T>(g, in<T>(out_grad), in<T>(input), in<T>(rotation), out<T>(filter_grad), workspace, s)) return;
    generic_grad_filter<T>(g, false, in<T>(out_grad), in<T>(input), (const T*)nullptr, in<T>(rotation),
                           out<T>(filter_grad), workspace, s);
  });
}

size_t dk_sample_depthwise_backward_rotation_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  if (desc->layout == DK_LAYOUT_NHWC) return nhwc_supported(g, desc->dtype) ? nhwc_grad_rotation_workspace(g, desc->dtype) : 0;
  return desc->dtype == DK_F64 ? 0 : fast_local_grad_rotation_workspace(g);
}

int dk_sample_depthwise_backward_rotation(const dk_conv_desc* desc, const void* out_grad,
                                          const void* input, const void* rotation,
                                          const void* filter, void* rotation_grad, void* workspace,
                                          size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!out_grad || !input || !rotation || !filter || !rotation_grad) return DK_ERR_NULL_POINTER;
  if (desc->layout == DK_LAYOUT_NHWC && !nhwc_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  const size_t need = dk_sample_depthwise_backward_rotation_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (desc->layout == DK_LAYOUT_NHWC)
    return by_dtype(desc->dtype, [&]<typename T>() {
      nhwc_grad_rotation<T>(g, in<T>(out_grad), in<T>(input), in<T>(rotation), in<T>(filter), out<T>(rotation_grad), workspace, s);
    });
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_local_grad_rotation<T>(g, in<T>(out_grad), in<T>(input), in<T>(rotation), in<T>(filter),
                                      out<T>(rotation_grad), workspace, s)) return;
    generic_grad_rotation<T>(g, false, in<T>(out_grad), in<T>(input), (const T*)nullptr, in<T>(rotation),
                             in<T>(filter), out<T>(rotation_grad), s);
  });
}

// ---- the filter gradient for callers that cannot allocate ---------------------------------

int dk_sample_depthwise_backward_filter_static(const dk_conv_desc* desc, const void* out_grad,
                                               const void* input, const void* rotation,
                                               void* filter_grad, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!out_grad || !input || !rotation || !filter_grad) return DK_ERR_NULL_POINTER;
  if (local_filter_ws(g, desc->dtype, desc->layout) > (size_t)DK_STATIC_SCRATCH_BYTES) return DK_ERR_SCRATCH_LIMIT;
  void* ptr = nullptr;
  const int st = static_scratch_of_current_device(&ptr);
  if (st != DK_OK) return st;
  // Every partial sum the reduction reads is written by this call's kernels first, so nothing
  // of an earlier call's contents has to be cleared.
  return dk_sample_depthwise_backward_filter(desc, out_grad, input, rotation, filter_grad, ptr,
                                             DK_STATIC_SCRATCH_BYTES, stream);
}

// Small layers: the gradients in one launch (dk_local_small.hip), which has no partial sums of its own
static bool backward_in_one_launch(const Geo& g, const dk_conv_desc* desc) {
  const bool channels_last = desc->layout == DK_LAYOUT_NHWC;
  return desc->dtype != DK_F64 && (!channels_last || nhwc_supported(g, desc->dtype)) &&
         local_small_backward_supported(g, channels_last, desc->dtype == DK_F32);
}

static size_t backward_need(const Geo& g, const dk_conv_desc* desc, bool rotation, bool filter) {
  if (backward_in_one_launch(g, desc)) return 0;
  // The rotation and the filter gradient run one after the other on the stream and share the buffer.
  return std::max(filter ? dk_sample_depthwise_backward_filter_workspace(desc) : 0,
                  rotation ? dk_sample_depthwise_backward_rotation_workspace(desc) : 0);
}

size_t dk_sample_depthwise_backward_workspace(const dk_conv_desc* desc) {
  Geo g;
  return make_geo(desc, g) == DK_OK ? backward_need(g, desc, true, true) : 0;
}

int dk_sample_depthwise_backward(const dk_conv_desc* desc, const void* out_grad, const void* input,
                                 const void* rotation, const void* filter, void* in_grad,
                                 void* rotation_grad, void* filter_grad, void* workspace,
                                 size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (!out_grad || !input || !rotation || !filter) return DK_ERR_NULL_POINTER;
  const size_t need = backward_need(g, desc, rotation_grad != nullptr, filter_grad != nullptr);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (backward_in_one_launch(g, desc)) {
    // (float32 channels-last layers above stride 1: the input gradient, like that of larger layers of few channels or pixels, is the
    // table kernel's to the bit, a launch of its own)
    const bool apart = in_grad && desc->layout == DK_LAYOUT_NHWC && desc->dtype == DK_F32 && (g.stride_h > 1 || g.stride_w > 1);
    const int st = by_tensor_dtype(desc->dtype, [&]<typename T>() {
      local_small_backward<T>(g, desc->layout == DK_LAYOUT_NHWC, in<T>(out_grad), in<T>(input), in<T>(rotation), in<T>(filter),
                              apart ? nullptr : out<T>(in_grad), out<T>(rotation_grad), out<T>(filter_grad), static_cast<hipStream_t>(stream));
    });
    return apart && st == DK_OK ? dk_sample_depthwise_backward_data(desc, out_grad, rotation, filter, in_grad, stream) : st;
  }
  // Filter gradient first, input gradient last: measured 4 % faster than the reference's order
  // (input, rotation, filter) on a 245 MB layer -- the two kernels that read out_grad, input and
  // rotation run back to back and the input gradient's 115 MB of writes do not push those
  // operands out of the 256 MB memory-side cache in between.
  int st = DK_OK;
  if (filter_grad && st == DK_OK)
    st = dk_sample_depthwise_backward_filter(desc, out_grad, input, rotation, filter_grad, workspace,
                                             workspace_bytes, stream);
  if (rotation_grad && st == DK_OK)
    st = dk_sample_depthwise_backward_rotation(desc, out_grad, input, rotation, filter, rotation_grad, workspace,
                                               workspace_bytes, stream);
  if (in_grad && st == DK_OK)
    st = dk_sample_depthwise_backward_data(desc, out_grad, rotation, filter, in_grad, stream);
  return st;
}

// ---- deformable --------------------------------------------------------------------------

int dk_deformable_sample_depthwise_forward(const dk_conv_desc* desc, const void* input,
                                           const void* offset, const void* rotation,
                                           const void* filter, void* output, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!input || !offset || !filter || !output) return DK_ERR_NULL_POINTER;  // rotation may be NULL: all zeros
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_deform_forward<T>(g, in<T>(input), in<T>(offset), in<T>(rotation), in<T>(filter), out<T>(output), s)) return;
    generic_forward<T>(g, true, in<T>(input), in<T>(offset), in<T>(rotation), in<T>(filter), out<T>(output), s);
  });
}

size_t dk_deformable_sample_depthwise_backward_data_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return std::max(generic_deform_grad_input_workspace(g, desc->dtype), fast_deform_grad_input_workspace(g));
}

int dk_deformable_sample_depthwise_backward_data(const dk_conv_desc* desc, const void* out_grad,
                                                 const void* offset, const void* rotation,
                                                 const void* filter, void* in_grad, void* workspace,
                                                 size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !offset || !filter || !in_grad) return DK_ERR_NULL_POINTER;  // rotation may be NULL: all zeros
  const size_t need = dk_deformable_sample_depthwise_backward_data_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_deform_grad_input<T>(g, in<T>(out_grad), in<T>(offset), in<T>(rotation), in<T>(filter),
                                    out<T>(in_grad), workspace, s)) return;
    generic_deform_grad_input<T>(g, in<T>(out_grad), in<T>(offset), in<T>(rotation), in<T>(filter),
                                 out<T>(in_grad), workspace, s);
  });
}

size_t dk_deformable_sample_depthwise_backward_filter_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return std::max(generic_grad_filter_workspace(g, desc->dtype), fast_deform_grad_filter_workspace(g));
}

int dk_deformable_sample_depthwise_backward_filter(const dk_conv_desc* desc, const void* out_grad,
                                                   const void* input, const void* offset,
                                                   const void* rotation, void* filter_grad,
                                                   void* workspace, size_t workspace_bytes,
                                                   void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !filter_grad) return DK_ERR_NULL_POINTER;  // rotation may be NULL: all zeros
  const size_t need = dk_deformable_sample_depthwise_backward_filter_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (g.batch == 0) return zero_filter_grad(g, desc->dtype, filter_grad, s);
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (fast_deform_grad_filter<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation),
                                     out<T>(filter_grad), workspace, s)) return;
    generic_grad_filter<T>(g, true, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation),
                           out<T>(filter_grad), workspace, s);
  });
}

size_t dk_deformable_sample_depthwise_backward_offset_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return fast_deform_grad_coord_workspace(g, false);
}

int dk_deformable_sample_depthwise_backward_offset(const dk_conv_desc* desc, const void* out_grad,
                                                   const void* input, const void* offset,
                                                   const void* rotation, const void* filter,
                                                   void* offset_grad, void* workspace,
                                                   size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !filter || !offset_grad) return DK_ERR_NULL_POINTER;  // rotation may be NULL: all zeros
  const size_t need = fast_deform_grad_coord_workspace(g, false);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (need && fast_deform_grad_coord<T>(g, false, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation),
                                            in<T>(filter), out<T>(offset_grad), workspace, s)) return;
    generic_grad_offset<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation), in<T>(filter),
                           out<T>(offset_grad), s);
  });
}

size_t dk_deformable_sample_depthwise_backward_rotation_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return fast_deform_grad_coord_workspace(g, true);
}

int dk_deformable_sample_depthwise_backward_rotation(const dk_conv_desc* desc, const void* out_grad,
                                                     const void* input, const void* offset,
                                                     const void* rotation, const void* filter,
                                                     void* rotation_grad, void* workspace,
                                                     size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !rotation || !filter || !rotation_grad) return DK_ERR_NULL_POINTER;
  const size_t need = fast_deform_grad_coord_workspace(g, true);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      if (need && fast_deform_grad_coord<T>(g, true, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation),
                                            in<T>(filter), out<T>(rotation_grad), workspace, s)) return;
    generic_grad_rotation<T>(g, true, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation),
                             in<T>(filter), out<T>(rotation_grad), s);
  });
}

size_t dk_deformable_sample_depthwise_backward_offset_rotation_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return std::max(fast_deform_grad_coords_workspace(g),
                  std::max(fast_deform_grad_coord_workspace(g, false), fast_deform_grad_coord_workspace(g, true)));
}

int dk_deformable_sample_depthwise_backward_offset_rotation(const dk_conv_desc* desc, const void* out_grad,
                                                            const void* input, const void* offset,
                                                            const void* rotation, const void* filter,
                                                            void* offset_grad, void* rotation_grad,
                                                            void* workspace, size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !rotation || !filter || !offset_grad || !rotation_grad) return DK_ERR_NULL_POINTER;
  const size_t need = dk_deformable_sample_depthwise_backward_offset_rotation_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool fused = false;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      fused = fast_deform_grad_coords_workspace(g) != 0 &&
              fast_deform_grad_coords<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation), in<T>(filter),
                                         out<T>(offset_grad), out<T>(rotation_grad), workspace, s);
  });
  if (st != DK_OK || fused) return st;
  // one after the other, sharing the workspace (stream order)
  const int so = dk_deformable_sample_depthwise_backward_offset(desc, out_grad, input, offset, rotation, filter,
                                                                offset_grad, workspace, workspace_bytes, stream);
  if (so != DK_OK) return so;
  return dk_deformable_sample_depthwise_backward_rotation(desc, out_grad, input, offset, rotation, filter,
                                                          rotation_grad, workspace, workspace_bytes, stream);
}

size_t dk_deformable_sample_depthwise_backward_offset_filter_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return std::max(std::max(plain_deform_grad_offset_filter_workspace(g), tile_deform_grads_workspace(g, false)),
                  std::max(dk_deformable_sample_depthwise_backward_offset_workspace(desc),
                           dk_deformable_sample_depthwise_backward_filter_workspace(desc)));
}

int dk_deformable_sample_depthwise_backward_offset_filter(const dk_conv_desc* desc, const void* out_grad, const void* input,
                                                          const void* offset, const void* rotation, const void* filter,
                                                          void* offset_grad, void* filter_grad, void* workspace,
                                                          size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !filter || !offset_grad || !filter_grad) return DK_ERR_NULL_POINTER;  // rotation may be NULL: all zeros
  const size_t need = dk_deformable_sample_depthwise_backward_offset_filter_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool fused = false;
  if (!rotation && g.batch > 0) {
    const int st = by_dtype(desc->dtype, [&]<typename T>() {
      if constexpr (kHasFast<T>)
        fused = plain_deform_grad_offset_filter<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(filter),
                                                   out<T>(offset_grad), out<T>(filter_grad), static_cast<float*>(workspace), s) ||
                tile_deform_grads<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), nullptr, in<T>(filter), out<T>(offset_grad),
                                     nullptr, out<T>(filter_grad), static_cast<float*>(workspace), s);
    });
    if (st != DK_OK || fused) return st;
  }
  // one after the other, sharing the workspace (stream order)
  const int so = dk_deformable_sample_depthwise_backward_offset(desc, out_grad, input, offset, rotation, filter, offset_grad,
                                                                workspace, workspace_bytes, stream);
  if (so != DK_OK) return so;
  return dk_deformable_sample_depthwise_backward_filter(desc, out_grad, input, offset, rotation, filter_grad, workspace,
                                                        workspace_bytes, stream);
}

size_t dk_deformable_sample_depthwise_backward_parameters_workspace(const dk_conv_desc* desc) {
  Geo g;
  if (make_geo(desc, g) != DK_OK) return 0;
  return std::max(tile_deform_grads_workspace(g, true), std::max(dk_deformable_sample_depthwise_backward_offset_rotation_workspace(desc),
                                                           dk_deformable_sample_depthwise_backward_filter_workspace(desc)));
}

int dk_deformable_sample_depthwise_backward_parameters(const dk_conv_desc* desc, const void* out_grad, const void* input,
                                                       const void* offset, const void* rotation, const void* filter,
                                                       void* offset_grad, void* rotation_grad, void* filter_grad,
                                                       void* workspace, size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !offset || !rotation || !filter || !offset_grad || !rotation_grad || !filter_grad) return DK_ERR_NULL_POINTER;
  const size_t need = dk_deformable_sample_depthwise_backward_parameters_workspace(desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool fused = false;
  if (g.batch > 0) {
    const int st = by_dtype(desc->dtype, [&]<typename T>() {
      if constexpr (kHasFast<T>)
        fused = tile_deform_grads<T>(g, in<T>(out_grad), in<T>(input), in<T>(offset), in<T>(rotation), in<T>(filter), out<T>(offset_grad),
                                     out<T>(rotation_grad), out<T>(filter_grad), static_cast<float*>(workspace), s);
    });
    if (st != DK_OK || fused) return st;
  }
  // one after the other, sharing the workspace (stream order)
  const int so = dk_deformable_sample_depthwise_backward_offset_rotation(desc, out_grad, input, offset, rotation, filter, offset_grad,
                                                                         rotation_grad, workspace, workspace_bytes, stream);
  if (so != DK_OK) return so;
  return dk_deformable_sample_depthwise_backward_filter(desc, out_grad, input, offset, rotation, filter_grad, workspace,
                                                        workspace_bytes, stream);
}

// ---- offset branch -----------------------------------------------------------------------

// ---- depthwise convolution with one kernel per image and channel ---------------------------

// The kernel tensor's strides as the kernels take them; false for a layout whose offsets do not fit
// (negative strides, or a span of 2^31 elements or more).
static bool kernel_strides(const Geo& g, const int64_t* given, long (&ws)[4], const long** out) {
  *out = nullptr;
  if (!given) return true;
  const long ext[4] = {g.batch, g.channel, g.k_h, g.k_w};
  long span = 0;
  for (int i = 0; i < 4; ++i) {
    if (given[i] < 0 || given[i] >= kMaxElems) return false;
    ws[i] = (long)given[i];
    span += (ext[i] - 1) * ws[i];
  }
  if (span >= kMaxElems) return false;
  *out = ws;
  return true;
}

int dk_image_depthwise_supported(const dk_conv_desc* desc) {
  Geo g;
  return make_geo(desc, g) == DK_OK && desc->layout == DK_LAYOUT_NCHW && image_conv_supported(g, desc->dtype);
}

int dk_image_depthwise_forward(const dk_conv_desc* desc, const void* input, const void* weight,
                               const int64_t* weight_strides, void* output, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!input || !weight || !output) return DK_ERR_NULL_POINTER;
  if (!image_conv_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  long ws_buf[4];
  const long* ws;
  if (!kernel_strides(g, weight_strides, ws_buf, &ws)) return DK_ERR_BAD_SHAPE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool ok = true;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    ok = image_conv_forward<T>(g, ws, in<T>(input), in<T>(weight), out<T>(output), s);
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

int dk_image_depthwise_backward_data_add(const dk_conv_desc* desc, const void* out_grad, const void* weight,
                                         const int64_t* weight_strides, const float* plane_grad, void* in_grad,
                                         void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !weight || !in_grad) return DK_ERR_NULL_POINTER;
  if (!image_conv_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  long ws_buf[4];
  const long* ws;
  if (!kernel_strides(g, weight_strides, ws_buf, &ws)) return DK_ERR_BAD_SHAPE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool ok = true;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    ok = image_conv_grad_input<T>(g, ws, in<T>(out_grad), in<T>(weight), plane_grad, out<T>(in_grad), s);
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

int dk_image_depthwise_backward_data(const dk_conv_desc* desc, const void* out_grad, const void* weight,
                                     const int64_t* weight_strides, void* in_grad, void* stream) {
  return dk_image_depthwise_backward_data_add(desc, out_grad, weight, weight_strides, nullptr, in_grad, stream);
}

int dk_image_depthwise_backward_weight(const dk_conv_desc* desc, const void* out_grad, const void* input,
                                       void* weight_grad, const int64_t* weight_strides, void* stream) {
  Geo g;
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  if (desc->layout != DK_LAYOUT_NCHW) return DK_ERR_UNSUPPORTED;
  if (!out_grad || !input || !weight_grad) return DK_ERR_NULL_POINTER;
  if (!image_conv_supported(g, desc->dtype)) return DK_ERR_UNSUPPORTED;
  long ws_buf[4];
  const long* ws;
  if (!kernel_strides(g, weight_strides, ws_buf, &ws)) return DK_ERR_BAD_SHAPE;
  if (g.batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  bool ok = true;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    ok = image_conv_grad_weight<T>(g, ws, in<T>(out_grad), in<T>(input), out<T>(weight_grad), s);
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

// ---- the per-image kernels of the global layer ---------------------------------------------

static int check_global_kernels(const dk_conv_desc* desc, Geo& g) {
  const int rc = make_geo(desc, g);
  if (rc != DK_OK) return rc;
  return desc->layout == DK_LAYOUT_NCHW && global_kernels_supported(g, desc->dtype) ? DK_OK : DK_ERR_UNSUPPORTED;
}

int dk_global_kernels_supported(const dk_conv_desc* desc) {
  Geo g;
  return check_global_kernels(desc, g) == DK_OK;
}

int dk_global_kernels_forward(const dk_conv_desc* desc, const void* input, const void* fc_weight, const void* fc_bias,
                              const void* weight, void* pooled, void* coord, void* clamped, void* kernels, void* stream) {
  Geo g;
  const int rc = check_global_kernels(desc, g);
  if (rc != DK_OK) return rc;
  if (!input || !fc_weight || !fc_bias || !weight || !pooled || !coord || !clamped || !kernels) return DK_ERR_NULL_POINTER;
  if (g.batch == 0) return DK_OK;
  return by_tensor_dtype(desc->dtype, [&]<typename T>() {
    global_kernels_forward<T>(g, in<T>(input), in<T>(fc_weight), in<T>(fc_bias), in<T>(weight), out<T>(pooled), out<T>(coord),
                              out<T>(clamped), out<T>(kernels), static_cast<hipStream_t>(stream));
  });
}

size_t dk_global_kernels_backward_workspace(const dk_conv_desc* desc) {
  Geo g;
  return check_global_kernels(desc, g) == DK_OK ? global_kernels_backward_workspace(g, desc->dtype) : 0;
}

int dk_global_kernels_backward(const dk_conv_desc* desc, const void* kernels_grad, const void* pooled, const void* coord,
                               const void* clamped, const void* weight, const void* fc_weight, void* weight_grad,
                               void* fc_weight_grad, void* fc_bias_grad, float* pooled_grad, void* workspace,
                               size_t workspace_bytes, void* stream) {
  Geo g;
  const int rc = check_global_kernels(desc, g);
  if (rc != DK_OK) return rc;
  if (!kernels_grad || !pooled || !coord || !clamped || !weight || !fc_weight) return DK_ERR_NULL_POINTER;
  if (!workspace || workspace_bytes < global_kernels_backward_workspace(g, desc->dtype)) return DK_ERR_WORKSPACE;
  if (g.batch == 0) return DK_ERR_UNSUPPORTED;  // nothing to sum: the caller's zeros
  return by_tensor_dtype(desc->dtype, [&]<typename T>() {
    global_kernels_backward<T>(g, desc->dtype, in<T>(kernels_grad), in<T>(pooled), in<T>(coord), in<T>(clamped), in<T>(weight),
                               in<T>(fc_weight), out<T>(weight_grad), out<T>(fc_weight_grad), out<T>(fc_bias_grad),
                               pooled_grad, workspace, static_cast<hipStream_t>(stream));
  });
}

// Tensors on planes the 16-bit matrix-instruction kernels cover: 16-bit elements as they are, float32 ones as
// bfloat16 (hi, lo) pairs
static bool offset_conv_on_16_bit_matrix(const dk_offset_conv_desc* d) {
  if (d->dtype == DK_F32 && path_disabled(kNoOffsetPairs)) return false;
  return offset_conv16_supported(d->in_channels, d->out_channels, d->h, d->w);
}

// forward: the call is (or asks about) the forward, the one pass that has a stride-2 kernel
static int check_offset_conv(const dk_offset_conv_desc* d, bool forward = false) {
  if (!d) return DK_ERR_NULL_POINTER;
  if (d->batch < 0 || d->in_channels <= 0 || d->out_channels <= 0 || d->h <= 0 || d->w <= 0) return DK_ERR_BAD_SHAPE;
  if (d->stride < 0 || d->stride > 2) return DK_ERR_BAD_SHAPE;
  if (d->dtype != DK_F32 && d->dtype != DK_F16 && d->dtype != DK_BF16) return d->dtype == DK_F64 ? DK_ERR_UNSUPPORTED : DK_ERR_BAD_DTYPE;
  if ((long)d->batch * d->in_channels * d->h * d->w > kMaxElems) return DK_ERR_TOO_LARGE;
  if (d->stride == 2)
    return forward && (d->dtype != DK_F32 || (!path_disabled(kNoOffsetPairs) && d->in_channels % 16 == 0)) &&
                   offset_conv16_s2_supported(d->in_channels, d->out_channels, d->h, d->w)
               ? DK_OK
               : DK_ERR_UNSUPPORTED;
  // 16-bit tensors: any number of channels.  (float32 ones in sixteens only: as bfloat16 pairs they are further from the float64
  // convolution than the framework's kernels, which serve the others.)  us both gradients, library / here: 80 x 577 x 7^2 float16
  // 55 / 40, 76 x 61 x 28^2 bfloat16 81 / 55, 11 x 41 x 112^2 float16 96 / 62, 64 x 250 x 28^2 bfloat16 stride 2 111 / 51.
  if (!offset_conv_supported(ceil_div(d->in_channels, 16) * 16, d->out_channels, d->h, d->w)) return DK_ERR_UNSUPPORTED;
  return d->in_channels % 16 == 0 || (d->dtype != DK_F32 && offset_conv_on_16_bit_matrix(d)) ? DK_OK : DK_ERR_UNSUPPORTED;
}

int dk_offset_conv_supported(const dk_offset_conv_desc* desc) { return check_offset_conv(desc, true) == DK_OK; }

int dk_offset_conv_worthwhile(const dk_offset_conv_desc* desc) {
  if (check_offset_conv(desc, true) != DK_OK) return 0;
  if (desc->stride == 2)  // as below, on the output plane
    return (long)desc->batch * ((((desc->h - 1) / 2 + 1) * (desc->w / 2) + 447) / 448) >= 64;
  // forward and input gradient on 16-bit matrix instructions are ahead of the library's on every plane they cover
  // once there are workgroups ((image, 448-pixel tile) items) for a quarter of the CUs
  if (offset_conv_on_16_bit_matrix(desc))
    return (long)desc->batch * ((desc->h * desc->w + 447) / 448) >= 64;
  return offset_conv_worthwhile(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w);
}

static size_t offset_conv_forward_need(const dk_offset_conv_desc* d) {
  const bool pairs = d->dtype == DK_F32;
  if (d->stride == 2) return offset_conv16_s2_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w, pairs);
  return offset_conv_on_16_bit_matrix(d)
             ? offset_conv16_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w, pairs)
             : offset_conv_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w);
}

size_t dk_offset_conv_forward_workspace(const dk_offset_conv_desc* desc) {
  if (check_offset_conv(desc, true) != DK_OK) return 0;
  return offset_conv_forward_need(desc);
}

int dk_offset_conv_forward(const dk_offset_conv_desc* desc, const void* input, const void* weight,
                           const void* bias, void* output, void* workspace, size_t workspace_bytes,
                           void* stream) {
  const int rc = check_offset_conv(desc, true);
  if (rc != DK_OK) return rc;
  if (!input || !weight || !bias || !output) return DK_ERR_NULL_POINTER;
  const size_t need = offset_conv_forward_need(desc);
  if (!workspace || workspace_bytes < need) return DK_ERR_WORKSPACE;
  bool ok = false;
  const bool matrix16 = offset_conv_on_16_bit_matrix(desc);
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>) {
      if (desc->stride == 2) {
        ok = offset_conv16_s2_forward<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w,
                                         in<T>(input), in<T>(weight), in<T>(bias), out<T>(output), workspace,
                                         static_cast<hipStream_t>(stream));
        return;
      }
      if (matrix16) {
        ok = offset_conv16_forward<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w, in<T>(input),
                                      in<T>(weight), in<T>(bias), out<T>(output), workspace, static_cast<hipStream_t>(stream));
        return;
      }
      ok = offset_conv_forward<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w, in<T>(input),
                                  in<T>(weight), in<T>(bias), out<T>(output), workspace, static_cast<hipStream_t>(stream));
    }
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

static int check_offset_conv_backward_input(const dk_offset_conv_desc* d) {
  const int rc = check_offset_conv(d, true);  // (stride 2: what holds for its forward holds for this pass)
  if (rc != DK_OK) return rc;
  if ((long)d->batch * d->out_channels * d->h * d->w > kMaxElems) return DK_ERR_TOO_LARGE;
  if (d->stride == 2) return DK_OK;
  return offset_conv_on_16_bit_matrix(d) ? DK_OK : DK_ERR_UNSUPPORTED;
}

static size_t offset_conv_backward_input_need(const dk_offset_conv_desc* d) {
  const bool pairs = d->dtype == DK_F32;
  return d->stride == 2 ? offset_conv16_s2_backward_input_workspace(d->in_channels, d->out_channels, pairs)
                        : offset_conv16_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w, pairs);
}

int dk_offset_conv_backward_input_worthwhile(const dk_offset_conv_desc* desc) {
  if (check_offset_conv_backward_input(desc) != DK_OK || !dk_offset_conv_worthwhile(desc)) return 0;
  if (desc->dtype == DK_F32 && desc->stride != 2) return desc->in_channels >= 64 && desc->w >= 14;
  return 1;
}

size_t dk_offset_conv_backward_input_workspace(const dk_offset_conv_desc* desc) {
  if (check_offset_conv_backward_input(desc) != DK_OK) return 0;
  return offset_conv_backward_input_need(desc);
}

int dk_offset_conv_backward_input(const dk_offset_conv_desc* desc, const void* out_grad, const void* weight,
                                  void* input_grad, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_offset_conv_backward_input(desc);
  if (rc != DK_OK) return rc;
  if (!out_grad || !weight || !input_grad) return DK_ERR_NULL_POINTER;
  if (!workspace || workspace_bytes < offset_conv_backward_input_need(desc)) return DK_ERR_WORKSPACE;
  bool ok = false;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>) {
      if (desc->stride == 2)
        ok = offset_conv16_s2_backward_input<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w,
                                                in<T>(out_grad), in<T>(weight), out<T>(input_grad), workspace,
                                                static_cast<hipStream_t>(stream));
      else
        ok = offset_conv16_backward_input<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w,
                                             in<T>(out_grad), in<T>(weight), out<T>(input_grad), workspace,
                                             static_cast<hipStream_t>(stream));
    }
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

// The weight gradient on the 16-bit matrix instructions: 16-bit tensors, and float32 ones as bfloat16 pairs
static bool offset_wgrad_on_16_bit_matrix(const dk_offset_conv_desc* d) {
  if (path_disabled(kNoOffsetWgrad16) || (d->dtype == DK_F32 && path_disabled(kNoOffsetPairs))) return false;
  return offset_wgrad16_supported(d->in_channels, d->out_channels, d->h, d->w, d->stride == 2 ? 2 : 1);
}

static int check_offset_conv_backward_weight(const dk_offset_conv_desc* d) {
  if (!d) return DK_ERR_NULL_POINTER;
  if (d->stride == 2) {
    const int rc = check_offset_conv(d, true);  // shapes and dtypes as for the stride-2 forward
    if (rc != DK_OK) return rc;
    return offset_wgrad_on_16_bit_matrix(d) ? DK_OK : DK_ERR_UNSUPPORTED;
  }
  if (d->in_channels % 16 != 0 && !offset_wgrad_on_16_bit_matrix(d)) return DK_ERR_UNSUPPORTED;
  return check_offset_conv(d);
}

static size_t offset_conv_backward_weight_need(const dk_offset_conv_desc* d) {
  if (offset_wgrad_on_16_bit_matrix(d))
    return offset_wgrad16_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w, d->stride == 2 ? 2 : 1,
                                    d->dtype == DK_F32);
  return offset_conv_wgrad_workspace(d->batch, d->in_channels, d->out_channels, d->h, d->w);
}

size_t dk_offset_conv_backward_weight_workspace(const dk_offset_conv_desc* desc) {
  if (check_offset_conv_backward_weight(desc) != DK_OK) return 0;
  return offset_conv_backward_weight_need(desc);
}

int dk_offset_conv_backward_weight(const dk_offset_conv_desc* desc, const void* out_grad, const void* input,
                                   void* weight_grad, void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_offset_conv_backward_weight(desc);
  if (rc != DK_OK) return rc;
  if (!out_grad || !input || !weight_grad) return DK_ERR_NULL_POINTER;
  const size_t need = offset_conv_backward_weight_need(desc);
  if (need == 0) return DK_ERR_UNSUPPORTED;  // fewer than 15 outputs on the fp32 matrix-instruction kernel
  if (!workspace || workspace_bytes < need) return DK_ERR_WORKSPACE;
  const bool matrix16 = offset_wgrad_on_16_bit_matrix(desc);
  bool ok = false;
  const int st = by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>) {
      if (matrix16)
        ok = offset_wgrad16<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w,
                               desc->stride == 2 ? 2 : 1, in<T>(input), in<T>(out_grad), out<T>(weight_grad), workspace,
                               static_cast<hipStream_t>(stream));
      else
        ok = offset_conv_wgrad<T>(desc->batch, desc->in_channels, desc->out_channels, desc->h, desc->w, in<T>(input),
                                  in<T>(out_grad), out<T>(weight_grad), workspace, static_cast<hipStream_t>(stream));
    }
  });
  return ok ? st : DK_ERR_UNSUPPORTED;
}

size_t dk_offset_conv_backward_bias_workspace(const dk_offset_conv_desc* desc) {
  if (!desc || desc->batch < 0 || desc->out_channels <= 0) return 0;
  return offset_conv_bias_grad_workspace(desc->batch, desc->out_channels);
}

int dk_offset_conv_backward_bias(const dk_offset_conv_desc* desc, const void* out_grad, void* bias_grad,
                                 void* workspace, size_t workspace_bytes, void* stream) {
  if (!desc) return DK_ERR_NULL_POINTER;
  if (desc->batch < 0 || desc->out_channels <= 0 || desc->h <= 0 || desc->w <= 0) return DK_ERR_BAD_SHAPE;
  if (desc->dtype != DK_F32 && desc->dtype != DK_F16 && desc->dtype != DK_BF16)
    return desc->dtype == DK_F64 ? DK_ERR_UNSUPPORTED : DK_ERR_BAD_DTYPE;
  if ((long)desc->batch * desc->out_channels * desc->h * desc->w > kMaxElems) return DK_ERR_TOO_LARGE;
  if (!out_grad || !bias_grad) return DK_ERR_NULL_POINTER;
  const size_t need = offset_conv_bias_grad_workspace(desc->batch, desc->out_channels);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  return by_dtype(desc->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>)
      offset_conv_bias_grad<T>(desc->batch, desc->out_channels, desc->h * desc->w, in<T>(out_grad), out<T>(bias_grad),
                               workspace, static_cast<hipStream_t>(stream));
  });
}

static int check_offset_conv_direct(const dk_offset_conv_desc* d) {
  if (!d) return DK_ERR_NULL_POINTER;
  if (d->batch < 0 || d->in_channels <= 0 || d->out_channels <= 0 || d->h <= 0 || d->w <= 0) return DK_ERR_BAD_SHAPE;
  if (d->stride < 0 || d->stride > 2) return DK_ERR_BAD_SHAPE;
  if (d->dtype != DK_F32 && d->dtype != DK_F16 && d->dtype != DK_BF16) return d->dtype == DK_F64 ? DK_ERR_UNSUPPORTED : DK_ERR_BAD_DTYPE;
  return offset_conv_direct_supported(d->batch, d->in_channels, d->out_channels, d->h, d->w) ? DK_OK : DK_ERR_UNSUPPORTED;
}

// Channels-times-pixels of the calls that these kernels are for, or 0: too few images for the matrix-instruction kernels, or
// (`general`) 16-bit tensors on a plane that those have no kernel for (float32 ones keep the library's results there), or whose
// channels are no multiple of sixteen.
static long offset_conv_direct_work(const dk_offset_conv_desc* desc, bool* general) {
  if (check_offset_conv_direct(desc) != DK_OK || dk_offset_conv_worthwhile(desc)) return 0;
  *general = !dk_offset_conv_supported(desc) || desc->in_channels % 16 != 0;
  if (*general && desc->dtype == DK_F32) return 0;
  const long stride = desc->stride == 2 ? 2 : 1, pixels = ((desc->h - 1) / stride + 1) * ((desc->w - 1) / stride + 1);
  return pixels * desc->batch * desc->in_channels;
}

// Measured through the operator against the library convolution, us here / library: 1 x 192 x 28^2 float32 13 / 31; 15 x 192 x 28^2
// stride 2 22 / 66; 63 x 608 x 7^2 52 / 101 (1.9 M pixel-channels); above that the vector unit falls behind: 30 x 384 x 14^2 bfloat16
// (2.3 M) 55 / 49.  A wave's channels are a serial chain, so many of them lose to the library where it has a kernel that suits:
//   stride 2 on planes from 56 on (the lanes' reads are far apart): 1 x 304 x 56^2 32 / 34, 1 x 336 x 56^2 37 / 33, 1 x 768 x 56^2 bfloat16 81 / 38
//   multiples of 128 channels: 1 x 640 x 14^2 39 / 47, 4 x 768 x 7^2 51 / 37; stride 2 8 x 384 x 28^2 35 / 40, 8 x 640 x 14^2 58 / 49, 8 x 768 x
//   14^2 69 / 38 (others: 8 x 736 x 14^2 67 / 163, 4 x 944 x 7^2 61 / 144)
//   one image in 16 bits: 832 channels of 14^2 48 / 52, 864 channels 51 / 48, 960 channels at stride 2 57 / 48 (four images 61 / 87)
//   two pixels per lane (more than 8192 pixels): float32 16 x 96 x 28^2 26 / 27, 144 channels 36 / 34; float16 64 channels 22 / 22, 96 channels
//   30 / 23; bfloat16 144 channels 39 / 107
int dk_offset_conv_direct_worthwhile(const dk_offset_conv_desc* desc) {
  bool general;
  const long work = offset_conv_direct_work(desc, &general);
  if (work == 0 || work > 2000000) return 0;
  if (general) return 0;  // (the framework's: see offset_conv in dk_torch.cpp)
  const int c = desc->in_channels;
  const bool half = desc->dtype != DK_F32, strided = desc->stride == 2;
  if (strided && desc->w >= 56 && c > 304) return 0;
  if (c % 128 == 0 && c > (strided ? 384 : 640)) return 0;
  if (half && desc->batch == 1 && c > 840) return 0;
  if (!strided && work / c > 8192 && desc->dtype != DK_BF16) return c <= (half ? 64 : 128);
  return 1;
}

// The input and the weight gradient: 1 x 192 x 28^2 float32 33 / 73, 63 x 608 x 7^2 94 / 96; 30 x 384 x 14^2 bfloat16 (2.3 M) 96 / 86.  At stride 2
// the input has four times the pixels: 15 x 192 x 28^2 (560 k) 67 / 93, 8 x 384 x 28^2 (600 k) 71 / 98; 16 x 960 x 14^2 (750 k) 103 / 98, 16 x
// 384 x 28^2 (1.2 M) 98 / 97, 8 x 288 x 56^2 (1.8 M) 124 / 98.
int dk_offset_conv_direct_backward_worthwhile(const dk_offset_conv_desc* desc) {
  bool general;
  const long work = offset_conv_direct_work(desc, &general);
  // other planes: 9 x 240 x 12 x 13 float16 40 / 48, 10 x 60 x 10 x 11 bfloat16 21 / 62, stride 2 7 x 37 x 57 x 55 bfloat16 37 / 66, 13 x 32 x 103 x 30
  // float16 (324 k) 47 / 49; 60 x 16 x 40 x 20 (48000 pixels, a channel's walk over which is serial) 78 / 49, 10 x 547 x 14^2 (1.1 M)
  // 82 / 51
  if (work > 0 && general) return work <= (desc->stride == 2 ? 370000 : 600000) && work / desc->in_channels <= 16384;
  return work > 0 && work <= (desc->stride == 2 ? 620000 : 2000000);
}

// pass 0: forward (a, b = input, weight), 1: input gradient (out_grad, weight), 2: weight gradient (out_grad, input)
static int offset_conv_direct(const dk_offset_conv_desc* d, int pass, const void* a, const void* b, const void* bias, void* res, void* stream) {
  const int rc = check_offset_conv_direct(d);
  if (rc != DK_OK) return rc;
  if (!a || !b || !res || (pass == 0 && !bias)) return DK_ERR_NULL_POINTER;
  const int stride = d->stride == 2 ? 2 : 1;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(d->dtype, [&]<typename T>() {
    if constexpr (kHasFast<T>) {
      if (pass == 0)
        offset_conv_direct_forward<T>(d->batch, d->in_channels, d->out_channels, d->h, d->w, stride, in<T>(a), in<T>(b), in<T>(bias), out<T>(res), s);
      else if (pass == 1)
        offset_conv_direct_backward_input<T>(d->batch, d->in_channels, d->out_channels, d->h, d->w, stride, in<T>(a), in<T>(b), out<T>(res), s);
      else
        offset_conv_direct_backward_weight<T>(d->batch, d->in_channels, d->out_channels, d->h, d->w, stride, in<T>(a), in<T>(b), out<T>(res), s);
    }
  });
}

int dk_offset_conv_direct_forward(const dk_offset_conv_desc* desc, const void* input, const void* weight, const void* bias,
                                  void* output, void* stream) {
  return offset_conv_direct(desc, 0, input, weight, bias, output, stream);
}

int dk_offset_conv_direct_backward_input(const dk_offset_conv_desc* desc, const void* out_grad, const void* weight,
                                         void* input_grad, void* stream) {
  return offset_conv_direct(desc, 1, out_grad, weight, nullptr, input_grad, stream);
}

int dk_offset_conv_direct_backward_weight(const dk_offset_conv_desc* desc, const void* out_grad, const void* input,
                                          void* weight_grad, void* stream) {
  return offset_conv_direct(desc, 2, out_grad, input, nullptr, weight_grad, stream);
}

// ---- N-d linear sample --------------------------------------------------------------------

static int check_nd(const dk_nd_desc* d) {
  if (!d) return DK_ERR_NULL_POINTER;
  if (d->dtype < DK_F32 || d->dtype > DK_F64) return DK_ERR_BAD_DTYPE;
  if (d->dims < 1 || d->dims > DK_ND_MAX_DIMS) return DK_ERR_UNSUPPORTED;
  if (d->batch < 0 || d->channel <= 0) return DK_ERR_BAD_SHAPE;
  long prod = d->channel;
  for (int i = 0; i < d->dims; ++i) {
    if (d->shape[i] <= 0) return DK_ERR_BAD_SHAPE;
    prod *= d->shape[i];
    if (prod > kMaxElems) return DK_ERR_TOO_LARGE;
  }
  if (d->batch * d->channel > 16L * kMaxElems) return DK_ERR_TOO_LARGE;
  return DK_OK;
}

size_t dk_nd_linear_sample_forward_workspace(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_forward_workspace(*desc);
}

size_t dk_nd_linear_sample_order_bytes(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_order_bytes(*desc);
}

size_t dk_nd_linear_sample_order_workspace(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_sort_workspace(*desc);
}

int dk_nd_linear_sample_order(const dk_nd_desc* desc, const void* coord, void* order, void* workspace,
                              size_t workspace_bytes, void* stream) {
  const int rc = check_nd(desc);
  if (rc != DK_OK) return rc;
  if (nd_order_bytes(*desc) == 0) return DK_ERR_UNSUPPORTED;
  if (!coord || !order) return DK_ERR_NULL_POINTER;
  const size_t need = nd_sort_workspace(*desc);
  if (!workspace || workspace_bytes < need) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    nd_order<T>(*desc, in<T>(coord), static_cast<int*>(order), workspace, s);
  });
}

int dk_nd_linear_sample_forward(const dk_nd_desc* desc, const void* data, const void* coord, const void* order,
                                void* output, void* workspace, size_t workspace_bytes,
                                void* stream) {
  const int rc = check_nd(desc);
  if (rc != DK_OK) return rc;
  if (!data || !coord || !output) return DK_ERR_NULL_POINTER;
  const size_t need = nd_forward_workspace(*desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  if (desc->batch == 0) return DK_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    nd_forward<T>(*desc, in<T>(data), in<T>(coord), out<T>(output), workspace, static_cast<const int*>(order), s);
  });
}

size_t dk_nd_linear_sample_backward_data_workspace(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_grad_data_workspace(*desc);
}

int dk_nd_linear_sample_backward_data(const dk_nd_desc* desc, const void* out_grad,
                                      const void* coord, const void* order, void* in_grad, void* workspace,
                                      size_t workspace_bytes, void* stream) {
  const int rc = check_nd(desc);
  if (rc != DK_OK) return rc;
  if (!in_grad || (desc->batch > 0 && (!out_grad || !coord))) return DK_ERR_NULL_POINTER;
  const size_t need = nd_grad_data_workspace(*desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    nd_grad_data<T>(*desc, in<T>(out_grad), in<T>(coord), out<T>(in_grad), workspace, static_cast<const int*>(order), s);
  });
}

size_t dk_nd_linear_sample_backward_coord_workspace(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_data_cl_workspace(*desc);
}

int dk_nd_linear_sample_backward_coord(const dk_nd_desc* desc, const void* out_grad,
                                       const void* data, const void* coord, const void* order, void* coord_grad,
                                       void* workspace, size_t workspace_bytes, void* stream) {
  const int rc = check_nd(desc);
  if (rc != DK_OK) return rc;
  if (desc->batch == 0) return DK_OK;
  if (!out_grad || !data || !coord || !coord_grad) return DK_ERR_NULL_POINTER;
  const size_t need = nd_data_cl_workspace(*desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    nd_grad_coord<T>(*desc, in<T>(out_grad), in<T>(data), in<T>(coord), out<T>(coord_grad), workspace,
                     static_cast<const int*>(order), s);
  });
}

size_t dk_nd_linear_sample_backward_workspace(const dk_nd_desc* desc) {
  if (check_nd(desc) != DK_OK) return 0;
  return nd_backward_workspace(*desc);
}

int dk_nd_linear_sample_backward(const dk_nd_desc* desc, const void* out_grad, const void* data, const void* coord,
                                 const void* order, void* in_grad, void* coord_grad, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  const int rc = check_nd(desc);
  if (rc != DK_OK) return rc;
  // (an empty batch: the data's gradient is zeros, and there is nothing else to read or write)
  if (!in_grad || (desc->batch > 0 && (!out_grad || !data || !coord || !coord_grad))) return DK_ERR_NULL_POINTER;
  const size_t need = nd_backward_workspace(*desc);
  if (need && (!workspace || workspace_bytes < need)) return DK_ERR_WORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return by_dtype(desc->dtype, [&]<typename T>() {
    nd_backward<T>(*desc, in<T>(out_grad), in<T>(data), in<T>(coord), out<T>(in_grad), out<T>(coord_grad), workspace,
                   static_cast<const int*>(order), s);
  });
}

}  // extern "C"
