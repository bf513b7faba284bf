// The autograd operators over the C ABI (include/dk_hip.h) as native code: argument checks, descriptors, result and
// workspace tensors, and the backward nodes.  The kernels of a small layer take 5 - 15 us each; the same host path in
// Python (an autograd.Function per operator, whose backward runs on the engine's device thread and waits for the
// interpreter lock) took 142 us per forward + backward of a [2, 32, 28, 28] layer whose six kernels sum to 48 us.
//
// Counterparts of the reference's functions/filter_sample_depthwise.py:19-206 and functions/nd_linear_sample.py:18-62
// (the two extension modules' pybind functions are the C ABI's); the Python files of the same names keep the signatures.
// What a forward call keeps for its backward pass goes through SavedVariable (version checks; saved-tensor hooks, which
// may offload or pack it), except the sampler's order of the points: bytes of the library's own layout.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include <array>
#include <cmath>
#include <limits>

#include "../../include/dk_hip.h"

namespace {

using at::Tensor;
using torch::autograd::edge_list;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
using Pair = std::array<int64_t, 2>;
using OptTensor = std::optional<Tensor>;

// A failing native call; the user gets it as the package's DkError (a RuntimeError, handed in by _lib.py): from a forward
// call by the module's exception translator, from a backward node by OpNode::apply.
struct DkFailure : std::runtime_error {
  using std::runtime_error::runtime_error;
};
PyObject* g_error_class = nullptr;  // read with the interpreter lock held
void set_python_error(const DkFailure& e) { PyErr_SetString(g_error_class ? g_error_class : PyExc_RuntimeError, e.what()); }

void check(int status, const char* what) {
  if (status != DK_OK)
    throw DkFailure(std::string(what) + " failed: " + dk_status_string(status) + " (status " + std::to_string(status) + ")");
}

int dtype_tag(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return DK_F32;
    case at::kHalf: return DK_F16;
    case at::kBFloat16: return DK_BF16;
    case at::kDouble: return DK_F64;
    default: TORCH_CHECK_TYPE(false, "unsupported dtype ", t.scalar_type(), " (float32, float16, bfloat16, float64)");
  }
}

// The operators exist on the GPU only, as in the reference (functions/filter_sample_depthwise.py:43-44).
void require_gpu(std::initializer_list<const Tensor*> tensors) {
  const Tensor* first = nullptr;
  for (const Tensor* t : tensors)
    if (t->defined()) {
      TORCH_CHECK_NOT_IMPLEMENTED(t->is_cuda(), "deformable-kernel operators are implemented for GPU tensors only");
      if (!first) first = t;
      TORCH_CHECK_VALUE(t->device() == first->device(), "all tensors must be on the same device");
      TORCH_CHECK_TYPE(t->scalar_type() == first->scalar_type(), "all tensors must have the same dtype (got ",
                       first->scalar_type(), " and ", t->scalar_type(), ")");
    }
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
const void* in(const Tensor& t) { return t.defined() ? t.const_data_ptr() : nullptr; }
void* out(const Tensor& t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }

struct Workspace {
  Tensor buf;
  size_t bytes;
  Workspace(size_t n, const Tensor& like) : bytes(n) {
    if (n) buf = at::empty({(int64_t)n}, like.options().dtype(at::kByte));
  }
  void* ptr() const { return buf.defined() ? buf.mutable_data_ptr() : nullptr; }
};

bool channels_last(const Tensor& t) {  // stored channels-last and not also in the default order
  return t.dim() == 4 && !t.is_contiguous() && t.is_contiguous(at::MemoryFormat::ChannelsLast);
}

// Base of the backward nodes.  Their results are not differentiable a second time: asking for it raises.  An undefined
// upstream gradient stands for zeros, as in a Python Function: the inputs get gradients of zeros.
struct OpNode : Node {
  virtual variable_list backward(const variable_list& grads) = 0;
  virtual void release() = 0;  // gives back what the forward call kept
  // (one thread's backward pass may end while another's is inside apply on the same graph)
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    release();
  }
  variable_list apply(variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    variable_list results;
    {
      at::AutoGradMode no_grad(false);
      if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
      const c10::DeviceGuard device(grads[0].device());
      try {
        results = backward(grads);
      } catch (const DkFailure& e) {
        // the engine hands a Python error through as it is, and anything else as a RuntimeError
        py::gil_scoped_acquire gil;
        set_python_error(e);
        python_error error;
        error.persist();
        throw error;
      }
    }
    if (!at::GradMode::is_enabled() || !grads[0].requires_grad()) return results;
    for (Tensor& t : results)
      if (t.defined()) t = t.detach().requires_grad_();
    return torch::autograd::DelayedError("trying to differentiate twice a function that was marked with @once_differentiable",
                                         (int64_t)results.size())
        .apply(std::move(results));
  }
  bool need(size_t i) const { return task_should_compute_output(i); }
};

// Runs `forward` without recording and hooks the node that `save` fills to its result if an input requires grad.
// An input with a forward-mode tangent is refused: the kernels have no such derivative, and the result would lose it.
// So is a call inside a functorch transform (vmap, grad, jvp, functionalize): the node would hang on the transform's
// wrapper of the result, and what the transform hands back has lost it.
template <typename N, typename Forward, typename Save>
Tensor record(std::initializer_list<const Tensor*> inputs, Forward&& forward, Save&& save) {
  TORCH_CHECK_NOT_IMPLEMENTED(!c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode),
                              "deformable-kernel operators do not run inside functorch transforms (torch.func, torch.vmap)");
  for (const Tensor* t : inputs)
    TORCH_CHECK_NOT_IMPLEMENTED(!t->defined() || !t->_fw_grad(0).defined(),
                                "deformable-kernel operators have no forward-mode derivative (no jvp)");
  bool tracked = false;
  if (at::GradMode::is_enabled())
    for (const Tensor* t : inputs) tracked = tracked || (t->defined() && t->requires_grad());
  Tensor result;
  std::shared_ptr<N> node;
  {
    at::AutoGradMode no_grad(false);
    const c10::DeviceGuard device((*inputs.begin())->device());
    result = forward();
    if (tracked) {
      node = std::shared_ptr<N>(new N(), torch::autograd::deleteNode);
      save(*node);
    }
  }
  if (tracked) {
    edge_list edges;
    edges.reserve(inputs.size());
    for (const Tensor* t : inputs) edges.push_back(t->defined() ? torch::autograd::impl::gradient_edge(*t) : torch::autograd::Edge());
    node->set_next_edges(std::move(edges));
    torch::autograd::set_history(result, node);
  }
  return result;
}

// ---- the two depthwise operators --------------------------------------------------------------

struct ConvArgs {
  Pair kernel, stride, padding, dilation;
  int64_t groups;
  int clip_mode;
  double clip_lo, clip_hi;
};

dk_conv_desc conv_desc(const Tensor& input, int64_t scope_h, int64_t scope_w, const ConvArgs& a, int layout = DK_LAYOUT_NCHW) {
  dk_conv_desc d{};
  d.batch = (int32_t)input.size(0), d.channel = (int32_t)input.size(1);
  d.in_h = (int32_t)input.size(2), d.in_w = (int32_t)input.size(3);
  d.k_h = (int32_t)a.kernel[0], d.k_w = (int32_t)a.kernel[1];
  d.stride_h = (int32_t)a.stride[0], d.stride_w = (int32_t)a.stride[1];
  d.pad_h = (int32_t)a.padding[0], d.pad_w = (int32_t)a.padding[1];
  d.dil_h = (int32_t)a.dilation[0], d.dil_w = (int32_t)a.dilation[1];
  d.scope_h = (int32_t)scope_h, d.scope_w = (int32_t)scope_w;
  d.groups = (int32_t)a.groups;
  d.dtype = dtype_tag(input);
  d.rotation_clip = a.clip_mode;
  d.clip_min = (float)a.clip_lo, d.clip_max = (float)a.clip_hi;
  d.layout = layout;
  return d;
}

// Shapes of the operators' arguments; returns the output plane (functions/filter_sample_depthwise.py:90-102).
Pair check_conv_shapes(const Tensor& input, const Tensor& rotation, const Tensor& weight, const Tensor& offset, const ConvArgs& a) {
  TORCH_CHECK_VALUE(input.dim() == 4 && weight.dim() == 4, "input must be [N, C, H, W] and weight [C, 1, S_h, S_w]");
  const int64_t n = input.size(0), c = input.size(1);
  Pair o{};
  for (int d = 0; d < 2; ++d) {
    TORCH_CHECK_VALUE(a.stride[d] > 0, "stride must be positive");
    const int64_t span = input.size(d + 2) + 2 * a.padding[d] - (a.dilation[d] * (a.kernel[d] - 1) + 1);
    o[d] = (span >= 0 ? span / a.stride[d] : -1) + 1;
  }
  TORCH_CHECK_VALUE(n > 0 && c > 0 && o[0] > 0 && o[1] > 0, "convolution input is too small (output would be ", n, "x", c, "x",
                    o[0], "x", o[1], ")");
  TORCH_CHECK_VALUE(weight.size(0) == c && weight.size(1) == 1, "weight must be [C, 1, S_h, S_w] with C = ", c, ", got ",
                    weight.sizes());
  TORCH_CHECK_VALUE(a.groups >= 1 && c % a.groups == 0, "channels (", c, ") must be divisible by rotation_groups (", a.groups, ")");
  const int64_t taps2 = a.kernel[0] * a.kernel[1] * 2;
  if (rotation.defined())
    TORCH_CHECK_VALUE(rotation.sizes() == at::IntArrayRef({n, a.groups * taps2, o[0], o[1]}), "rotation must be [", n, ", ",
                      a.groups * taps2, ", ", o[0], ", ", o[1], "], got ", rotation.sizes());
  if (offset.defined())
    TORCH_CHECK_VALUE(offset.sizes() == at::IntArrayRef({n, taps2, o[0], o[1]}), "offset must be [", n, ", ", taps2, ", ", o[0],
                      ", ", o[1], "], got ", offset.sizes());
  return o;
}

struct SampleDepthwiseFunctionBackward : OpNode {
  SavedVariable input, rotation, weight;
  dk_conv_desc desc;
  std::string name() const override { return "SampleDepthwiseFunctionBackward"; }
  void release() override {
    input.reset_data(), rotation.reset_data(), weight.reset_data();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), r = rotation.unpack(), w = weight.unpack();
    require_gpu({&grads[0], &x});
    const Tensor g = grads[0].contiguous(desc.layout == DK_LAYOUT_NHWC ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous);
    variable_list res(3);
    // one native call for the whole backward pass: the gradients that are not needed are passed as NULL and skipped
    if (need(0)) res[0] = at::empty_like(x);
    if (need(1)) res[1] = at::empty_like(r);
    if (need(2)) res[2] = at::empty_like(w);
    const Workspace ws(need(1) || need(2) ? dk_sample_depthwise_backward_workspace(&desc) : 0, x);
    check(dk_sample_depthwise_backward(&desc, in(g), in(x), in(r), in(w), out(res[0]), out(res[1]), out(res[2]), ws.ptr(), ws.bytes,
                                       stream_of(x)),
          "sample_depthwise backward");
    return res;
  }
};

Tensor sample_depthwise(const Tensor& input, const Tensor& rotation, const Tensor& weight, const Pair& kernel, const Pair& stride,
                        const Pair& padding, const Pair& dilation, int64_t groups, int clip_mode, double clip_lo, double clip_hi) {
  require_gpu({&input, &rotation, &weight});
  const ConvArgs a{kernel, stride, padding, dilation, groups, clip_mode, clip_lo, clip_hi};
  const Pair o = check_conv_shapes(input, rotation, weight, Tensor(), a);
  // A channels-last input runs the library's channels-last kernels and gets a channels-last output (and gradients): no
  // layout change around the operator.  The reference's kernels take planar tensors only.  Geometries whose channels-last
  // tables do not fit LDS (e.g. 64 rotation groups) take the planar kernels on a planar copy, and the output goes back.
  const bool wants_nhwc = channels_last(input);
  dk_conv_desc desc = conv_desc(input, weight.size(2), weight.size(3), a, wants_nhwc ? DK_LAYOUT_NHWC : DK_LAYOUT_NCHW);
  if (wants_nhwc && dk_sample_depthwise_layout_supported(&desc) != 1) desc.layout = DK_LAYOUT_NCHW;
  const auto fmt = desc.layout == DK_LAYOUT_NHWC ? at::MemoryFormat::ChannelsLast : at::MemoryFormat::Contiguous;
  Tensor x, r, w;
  return record<SampleDepthwiseFunctionBackward>(
      {&input, &rotation, &weight},
      [&] {
        x = input.contiguous(fmt), r = rotation.contiguous(fmt), w = weight.contiguous();
        Tensor res = at::empty({input.size(0), input.size(1), o[0], o[1]}, input.options().memory_format(fmt));
        check(dk_sample_depthwise_forward(&desc, in(x), in(r), in(w), out(res), stream_of(x)), "sample_depthwise forward");
        return wants_nhwc && desc.layout != DK_LAYOUT_NHWC ? res.contiguous(at::MemoryFormat::ChannelsLast) : res;
      },
      [&](SampleDepthwiseFunctionBackward& n) {
        n.input = SavedVariable(x, false), n.rotation = SavedVariable(r, false), n.weight = SavedVariable(w, false);
        n.desc = desc;
      });
}

struct DeformableSampleDepthwiseFunctionBackward : OpNode {
  SavedVariable input, offset, rotation, weight;
  bool has_rotation = false;
  dk_conv_desc desc;
  std::string name() const override { return "DeformableSampleDepthwiseFunctionBackward"; }
  void release() override {
    input.reset_data(), offset.reset_data(), rotation.reset_data(), weight.reset_data();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), f = offset.unpack(), r = has_rotation ? rotation.unpack() : Tensor(), w = weight.unpack();
    require_gpu({&grads[0], &x});
    const Tensor g = grads[0].contiguous();
    void* const s = stream_of(x);
    variable_list res(4);
    const bool need_offset = need(1), need_rotation = has_rotation && need(2), need_filter = need(3);
    if (need(0)) {
      res[0] = at::empty_like(x);
      const Workspace ws(dk_deformable_sample_depthwise_backward_data_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_data(&desc, in(g), in(f), in(r), in(w), out(res[0]), ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_data");
    }
    if (need_offset) res[1] = at::empty_like(f);
    if (need_rotation) res[2] = at::empty_like(r);
    if (need_filter) res[3] = at::empty_like(w);
    if (need_offset && need_filter && !has_rotation) {
      // one call for both (one pass over the samples where the library has that kernel)
      const Workspace ws(dk_deformable_sample_depthwise_backward_offset_filter_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_offset_filter(&desc, in(g), in(x), in(f), nullptr, in(w), out(res[1]), out(res[3]),
                                                                  ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_offset_filter");
      return res;
    }
    if (need_offset && need_rotation && need_filter) {
      const Workspace ws(dk_deformable_sample_depthwise_backward_parameters_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_parameters(&desc, in(g), in(x), in(f), in(r), in(w), out(res[1]), out(res[2]),
                                                               out(res[3]), ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_parameters");
      return res;
    }
    if (need_offset && need_rotation) {
      // one call for both coordinate gradients (one pass over the input where the library has that kernel)
      const Workspace ws(dk_deformable_sample_depthwise_backward_offset_rotation_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_offset_rotation(&desc, in(g), in(x), in(f), in(r), in(w), out(res[1]), out(res[2]),
                                                                    ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_offset_rotation");
    } else if (need_offset) {
      const Workspace ws(dk_deformable_sample_depthwise_backward_offset_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_offset(&desc, in(g), in(x), in(f), in(r), in(w), out(res[1]), ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_offset");
    } else if (need_rotation) {
      const Workspace ws(dk_deformable_sample_depthwise_backward_rotation_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_rotation(&desc, in(g), in(x), in(f), in(r), in(w), out(res[2]), ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_rotation");
    }
    if (need_filter) {
      const Workspace ws(dk_deformable_sample_depthwise_backward_filter_workspace(&desc), x);
      check(dk_deformable_sample_depthwise_backward_filter(&desc, in(g), in(x), in(f), in(r), out(res[3]), ws.ptr(), ws.bytes, s),
            "deform_sample_depthwise backward_filter");
    }
    return res;
  }
};

// rotation absent: no kernel-space offsets (DeformKernelConv2d / DeformConv2d); the library then reads no rotation tensor,
// where the reference's module hands over a tensor of zeros
Tensor deform_sample_depthwise(const Tensor& input, const Tensor& offset, const OptTensor& rotation_arg, const Tensor& weight,
                               const Pair& kernel, const Pair& stride, const Pair& padding, const Pair& dilation, int64_t groups,
                               int clip_mode, double clip_lo, double clip_hi) {
  const Tensor rotation = rotation_arg ? *rotation_arg : Tensor();
  require_gpu({&input, &offset, &rotation, &weight});
  const ConvArgs a{kernel, stride, padding, dilation, groups, clip_mode, clip_lo, clip_hi};
  const Pair o = check_conv_shapes(input, rotation, weight, offset, a);
  const dk_conv_desc desc = conv_desc(input, weight.size(2), weight.size(3), a);
  Tensor x, f, r, w;
  return record<DeformableSampleDepthwiseFunctionBackward>(
      {&input, &offset, &rotation, &weight},
      [&] {
        x = input.contiguous(), f = offset.contiguous(), w = weight.contiguous();
        if (rotation.defined()) r = rotation.contiguous();
        Tensor res = at::empty({input.size(0), input.size(1), o[0], o[1]}, input.options());
        check(dk_deformable_sample_depthwise_forward(&desc, in(x), in(f), in(r), in(w), out(res), stream_of(x)),
              "deform_sample_depthwise forward");
        return res;
      },
      [&](DeformableSampleDepthwiseFunctionBackward& n) {
        n.input = SavedVariable(x, false), n.offset = SavedVariable(f, false), n.weight = SavedVariable(w, false);
        n.has_rotation = r.defined();
        if (n.has_rotation) n.rotation = SavedVariable(r, false);
        n.desc = desc;
      });
}

// ---- N-d sampler --------------------------------------------------------------------------------

struct NdLinearSampleFunctionBackward : OpNode {
  SavedVariable input, coord;
  Tensor order;  // the points' order by cell
  dk_nd_desc desc;
  std::string name() const override { return "NdLinearSampleFunctionBackward"; }
  void release() override {
    input.reset_data(), coord.reset_data();
    order.reset();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), p = coord.unpack();
    require_gpu({&grads[0], &x});
    const Tensor g = grads[0].contiguous();
    void* const s = stream_of(x);
    variable_list res(2);
    if (need(0) && need(1)) {
      res[0] = at::empty_like(x), res[1] = at::empty_like(p);
      const Workspace ws(dk_nd_linear_sample_backward_workspace(&desc), x);
      check(dk_nd_linear_sample_backward(&desc, in(g), in(x), in(p), in(order), out(res[0]), out(res[1]), ws.ptr(), ws.bytes, s),
            "nd_linear_sample backward");
      return res;
    }
    if (need(0)) {
      res[0] = at::empty_like(x);
      const Workspace ws(dk_nd_linear_sample_backward_data_workspace(&desc), x);
      check(dk_nd_linear_sample_backward_data(&desc, in(g), in(p), in(order), out(res[0]), ws.ptr(), ws.bytes, s),
            "nd_linear_sample backward_data");
    }
    if (need(1)) {
      res[1] = at::empty_like(p);
      const Workspace ws(dk_nd_linear_sample_backward_coord_workspace(&desc), x);
      check(dk_nd_linear_sample_backward_coord(&desc, in(g), in(x), in(p), in(order), out(res[1]), ws.ptr(), ws.bytes, s),
            "nd_linear_sample backward_coord");
    }
    return res;
  }
};

Tensor nd_linear_sample(const Tensor& input, const Tensor& coord) {
  require_gpu({&input, &coord});
  const int64_t dims = input.dim() - 1;
  TORCH_CHECK_VALUE(coord.dim() == 2 && coord.size(1) == dims, "coord must be [B, ", dims, "] for input of shape ", input.sizes(),
                    ", got ", coord.sizes());
  TORCH_CHECK_VALUE(dims >= 1 && dims <= DK_ND_MAX_DIMS, "nd_linear_sample supports 1..", DK_ND_MAX_DIMS,
                    " sampling dimensions, got ", dims);
  dk_nd_desc desc{};
  desc.batch = coord.size(0), desc.channel = (int32_t)input.size(0), desc.dims = (int32_t)dims;
  for (int d = 0; d < DK_ND_MAX_DIMS; ++d) desc.shape[d] = d < dims ? (int32_t)input.size(d + 1) : 1;
  desc.dtype = dtype_tag(input);
  Tensor x, p, order;
  return record<NdLinearSampleFunctionBackward>(
      {&input, &coord},
      [&] {
        x = input.contiguous(), p = coord.contiguous();
        Tensor res = at::empty({coord.size(0), input.size(0)}, input.options());
        void* const s = stream_of(x);
        // many points per cell: the kernels work on the points sorted by cell; sort once, here, and keep the order for
        // the backward pass
        if (const size_t bytes = dk_nd_linear_sample_order_bytes(&desc)) {
          order = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
          const Workspace ws(dk_nd_linear_sample_order_workspace(&desc), x);
          check(dk_nd_linear_sample_order(&desc, in(p), out(order), ws.ptr(), ws.bytes, s), "nd_linear_sample order");
        }
        const Workspace ws(dk_nd_linear_sample_forward_workspace(&desc), x);
        check(dk_nd_linear_sample_forward(&desc, in(x), in(p), in(order), out(res), ws.ptr(), ws.bytes, s), "nd_linear_sample forward");
        return res;
      },
      [&](NdLinearSampleFunctionBackward& n) {
        n.input = SavedVariable(x, false), n.coord = SavedVariable(p, false);
        n.order = order;
        n.desc = desc;
      });
}

// ---- offset branch ------------------------------------------------------------------------------

dk_offset_conv_desc offset_desc(const Tensor& input, const Tensor& weight, const Tensor& plane, int64_t stride) {
  dk_offset_conv_desc d{};
  d.batch = (int32_t)input.size(0), d.in_channels = (int32_t)input.size(1), d.out_channels = (int32_t)weight.size(0);
  d.h = (int32_t)plane.size(2), d.w = (int32_t)plane.size(3);
  d.dtype = dtype_tag(input);
  d.stride = (int32_t)stride;
  return d;
}

// Tensors the library's kernels take: on the GPU, all float32 or all float16 or all bfloat16
bool offset_conv_native_tensors(const Tensor& input, const Tensor& weight, const Tensor& bias) {
  const auto t = input.scalar_type();
  return input.is_cuda() && weight.is_cuda() && weight.scalar_type() == t && (t == at::kFloat || t == at::kHalf || t == at::kBFloat16) &&
         (!bias.defined() || (bias.is_cuda() && bias.scalar_type() == t)) && input.dim() == 4 && weight.dim() == 4;
}

bool offset_conv_covered(const Tensor& input, const Tensor& weight, const Pair& stride, const Pair& padding, const Pair& dilation,
                         int (*query)(const dk_offset_conv_desc*)) {
  if (weight.size(2) != 3 || weight.size(3) != 3 || weight.size(1) != input.size(1)) return false;
  if (!(stride == Pair{1, 1} || stride == Pair{2, 2}) || padding != Pair{1, 1} || dilation != Pair{1, 1}) return false;
  const dk_offset_conv_desc d = offset_desc(input, weight, input, stride[0]);
  return query(&d) != 0;
}

struct OffsetConvFunctionBackward : OpNode {
  SavedVariable input, weight;
  Pair stride, padding, dilation;
  bool native = false, direct = false, forced = false, has_bias = false;
  std::string name() const override { return "OffsetConvFunctionBackward"; }
  void release() override {
    input.reset_data(), weight.reset_data();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), w = weight.unpack(), g = grads[0].contiguous();
    void* const s = stream_of(x);
    variable_list res(3);
    const dk_offset_conv_desc d = offset_desc(x, w, x, stride[0]);
    // a workspace query of 0 says "this pass is not covered"; the input gradient's other query, that the framework's
    // kernel is the faster one on this shape
    const bool native_weight = need(1) && native && dk_offset_conv_backward_weight_workspace(&d) > 0;
    const bool native_input = need(0) && native && dk_offset_conv_backward_input_workspace(&d) > 0 &&
                              (forced || dk_offset_conv_backward_input_worthwhile(&d));
    const bool lib_input = need(0) && !native_input && !direct, lib_weight = need(1) && !native_weight && !direct;
    if (direct && need(0)) {
      res[0] = at::empty_like(x);
      check(dk_offset_conv_direct_backward_input(&d, in(g), in(w), out(res[0]), s), "offset_conv input gradient");
    }
    if (direct && need(1)) {
      res[1] = at::empty_like(w);
      check(dk_offset_conv_direct_backward_weight(&d, in(g), in(x), out(res[1]), s), "offset_conv weight gradient");
    }
    if (lib_input || lib_weight) {  // the framework's routine, without its bias gradient
      auto r = at::convolution_backward(g, x, w, std::nullopt, stride, padding, dilation, false, at::IntArrayRef({0, 0}), 1,
                                        {lib_input, lib_weight, false});
      if (lib_input) res[0] = std::get<0>(r);
      if (lib_weight) res[1] = std::get<1>(r);
    }
    if (native_input) {
      res[0] = at::empty_like(x);
      const Workspace ws(dk_offset_conv_backward_input_workspace(&d), x);
      check(dk_offset_conv_backward_input(&d, in(g), in(w), out(res[0]), ws.ptr(), ws.bytes, s), "offset_conv input gradient");
    }
    if (native_weight) {
      res[1] = at::empty_like(w);
      const Workspace ws(dk_offset_conv_backward_weight_workspace(&d), x);
      check(dk_offset_conv_backward_weight(&d, in(g), in(x), out(res[1]), ws.ptr(), ws.bytes, s), "offset_conv weight gradient");
    }
    if (has_bias && need(2)) {
      res[2] = at::empty({w.size(0)}, g.options());
      const dk_offset_conv_desc b = offset_desc(x, w, g, 1);
      const Workspace ws(dk_offset_conv_backward_bias_workspace(&b), x);
      check(dk_offset_conv_backward_bias(&b, in(g), out(res[2]), ws.ptr(), ws.bytes, s), "offset_conv bias gradient");
    }
    return res;
  }
};

Tensor offset_conv(const Tensor& input, const Tensor& weight, const OptTensor& bias_arg, const Pair& stride, const Pair& padding,
                   const Pair& dilation, bool force) {
  const Tensor bias = bias_arg ? *bias_arg : Tensor();
  if (!offset_conv_native_tensors(input, weight, bias)) return at::conv2d(input, weight, bias_arg, stride, padding, dilation);
  const bool native = offset_conv_covered(input, weight, stride, padding, dilation, force ? dk_offset_conv_supported : dk_offset_conv_worthwhile);
  // few images: one launch per pass on the vector unit
  const bool direct = !native && offset_conv_covered(input, weight, stride, padding, dilation, dk_offset_conv_direct_worthwhile);
  // Channels in sixteens; layers of others have the framework's forward.  A 16-bit offset that rounds the other way moves its
  // sample by its last bit, and where it crosses a cell's border the slope jumps: the offsets of a trained layer stay what
  // they were, the gradients of the convolution itself are the library's.
  const bool own_forward = native && (force || input.size(1) % 16 == 0);
  const bool direct_grads = !native && offset_conv_covered(input, weight, stride, padding, dilation, dk_offset_conv_direct_backward_worthwhile);
  Tensor x, w;
  return record<OffsetConvFunctionBackward>(
      {&input, &weight, &bias},
      [&] {
        x = input.contiguous(), w = weight.contiguous();
        if (!own_forward && !direct) return at::conv2d(x, w, bias_arg, stride, padding, dilation);
        const Tensor b = bias.defined() ? bias.contiguous() : at::zeros({w.size(0)}, x.options());
        const int64_t st = stride[0];
        Tensor res = at::empty({x.size(0), w.size(0), (x.size(2) - 1) / st + 1, (x.size(3) - 1) / st + 1}, x.options());
        const dk_offset_conv_desc d = offset_desc(x, w, x, st);
        if (direct) {
          check(dk_offset_conv_direct_forward(&d, in(x), in(w), in(b), out(res), stream_of(x)), "offset_conv forward");
          return res;
        }
        const Workspace ws(dk_offset_conv_forward_workspace(&d), x);
        check(dk_offset_conv_forward(&d, in(x), in(w), in(b), out(res), ws.ptr(), ws.bytes, stream_of(x)), "offset_conv forward");
        return res;
      },
      [&](OffsetConvFunctionBackward& n) {
        n.input = SavedVariable(x, false), n.weight = SavedVariable(w, false);
        n.stride = stride, n.padding = padding, n.dilation = dilation;
        n.native = native, n.direct = direct_grads, n.forced = force, n.has_bias = bias.defined();
      });
}

bool offset_conv_supported(const Tensor& input, const Tensor& weight, const OptTensor& bias, const Pair& stride, const Pair& padding,
                           const Pair& dilation, bool worthwhile) {
  return offset_conv_native_tensors(input, weight, bias ? *bias : Tensor()) &&
         offset_conv_covered(input, weight, stride, padding, dilation, worthwhile ? dk_offset_conv_worthwhile : dk_offset_conv_supported);
}

// ---- depthwise convolution with one kernel per image and channel; the global layer ----------------

using Strides = std::array<int64_t, 4>;

// Whether the tensor's elements occupy numel() distinct consecutive slots in some axis order (so that empty_strided with
// the same strides gives a tensor of the same layout)
bool dense(const Tensor& t) {
  std::array<bool, 4> used{};
  int64_t expect = 1;
  for (int k = 0; k < 4; ++k) {
    int pick = -1;
    for (int d = 0; d < 4; ++d)
      if (!used[d] && t.size(d) != 1 && (pick < 0 || t.stride(d) < t.stride(pick))) pick = d;
    if (pick < 0) return true;
    if (t.stride(pick) != expect) return false;
    expect *= t.size(pick);
    used[pick] = true;
  }
  return true;
}

Tensor empty_out(const Tensor& input, const dk_conv_desc& desc) {
  int32_t oh = 0, ow = 0;
  check(dk_conv_out_size(&desc, &oh, &ow), "convolution shape");
  return at::empty({input.size(0), input.size(1), oh, ow}, input.options());
}

struct ImageDepthwiseConvFunctionBackward : OpNode {
  SavedVariable input, weight;
  dk_conv_desc desc;
  std::string name() const override { return "ImageDepthwiseConvFunctionBackward"; }
  void release() override {
    input.reset_data(), weight.reset_data();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), w = weight.unpack(), g = grads[0].contiguous();
    const Strides st{w.stride(0), w.stride(1), w.stride(2), w.stride(3)};
    const int64_t* strides = w.is_contiguous() ? nullptr : st.data();
    variable_list res(2);
    if (need(0)) {
      res[0] = at::empty_like(x);
      check(dk_image_depthwise_backward_data(&desc, in(g), in(w), strides, out(res[0]), stream_of(x)), "image_depthwise_conv grad input");
    }
    if (need(1)) {
      // same layout as the kernels: a permuted view of the sampler's output gets a gradient whose rows are the sampler's
      // rows, so no transposing copy runs on the way back either
      res[1] = at::empty_strided(w.sizes(), w.strides(), w.options());
      check(dk_image_depthwise_backward_weight(&desc, in(g), in(x), out(res[1]), strides, stream_of(x)), "image_depthwise_conv grad weight");
    }
    return res;
  }
};

Tensor image_depthwise_conv(const Tensor& input, const Tensor& weight, const Pair& stride, const Pair& padding, const Pair& dilation) {
  require_gpu({&input, &weight});
  TORCH_CHECK_VALUE(input.dim() == 4 && weight.dim() == 4,
                    "input must be [N, C, H, W] and weight [N * C, 1, k_h, k_w] or [N, C, k_h, k_w]");
  const int64_t n = input.size(0), c = input.size(1);
  TORCH_CHECK_VALUE((weight.size(0) == n * c && weight.size(1) == 1) || (weight.size(0) == n && weight.size(1) == c), "weight of shape ",
                    weight.sizes(), " does not hold one kernel per image and channel of an input of shape ", input.sizes());
  const dk_conv_desc desc = conv_desc(input, 1, 1, ConvArgs{{weight.size(2), weight.size(3)}, stride, padding, dilation, 1, DK_CLIP_NONE, 0.0, 0.0});
  Tensor x, w;
  return record<ImageDepthwiseConvFunctionBackward>(
      {&input, &weight},
      [&] {
        x = input.contiguous();
        // [N * C, 1, k, k], or a layout with gaps or repeats
        w = (weight.size(1) == 1 && c != 1) || !dense(weight) ? weight.contiguous() : weight;
        const Strides st{w.stride(0), w.stride(1), w.stride(2), w.stride(3)};
        Tensor res = empty_out(x, desc);
        check(dk_image_depthwise_forward(&desc, in(x), in(w), w.is_contiguous() ? nullptr : st.data(), out(res), stream_of(x)),
              "image_depthwise_conv forward");
        return res;
      },
      [&](ImageDepthwiseConvFunctionBackward& m) {
        m.input = SavedVariable(x, false), m.weight = SavedVariable(w, false);
        m.desc = desc;
      });
}

struct GlobalDeformConvFunctionBackward : OpNode {
  SavedVariable input, weight, fc_weight;
  SavedVariable saved_pooled, saved_coord, saved_kernels;  // made by the forward call
  dk_conv_desc desc;
  std::string name() const override { return "GlobalDeformConvFunctionBackward"; }
  void release() override {
    input.reset_data(), weight.reset_data(), fc_weight.reset_data();
    saved_pooled.reset_data(), saved_coord.reset_data(), saved_kernels.reset_data();
  }
  variable_list backward(const variable_list& grads) override {
    const Tensor x = input.unpack(), w = weight.unpack(), fw = fc_weight.unpack(), g = grads[0].contiguous();
    const Tensor pooled = saved_pooled.unpack(), coord = saved_coord.unpack(), kernels = saved_kernels.unpack();
    const int64_t c = x.size(1), k = desc.k_h;
    const Strides strides{k * k * c, 1, k * c, c};
    void* const s = stream_of(x);
    variable_list res(4);
    const Tensor gk = at::empty_like(kernels);
    check(dk_image_depthwise_backward_weight(&desc, in(g), in(x), out(gk), strides.data(), s), "global_deform_conv grad kernels");
    const Tensor gpool = need(0) ? at::empty(pooled.sizes(), pooled.options().dtype(at::kFloat)) : Tensor();
    if (need(1)) res[1] = at::empty_like(w);
    if (need(2)) res[2] = at::empty_like(fw);
    if (need(3)) res[3] = at::empty({fw.size(0)}, fw.options());
    const Workspace ws(dk_global_kernels_backward_workspace(&desc), x);
    check(dk_global_kernels_backward(&desc, in(gk), in(pooled), in(coord[0]), in(coord[1]), in(w), in(fw), out(res[1]), out(res[2]),
                                     out(res[3]), static_cast<float*>(out(gpool)), ws.ptr(), ws.bytes, s),
          "global_deform_conv grad parameters");
    if (need(0)) {
      res[0] = at::empty_like(x);
      check(dk_image_depthwise_backward_data_add(&desc, in(g), in(kernels), strides.data(), static_cast<const float*>(in(gpool)), out(res[0]), s),
            "global_deform_conv grad input");
    }
    return res;
  }
};

dk_conv_desc global_desc(const Tensor& input, const Tensor& weight, int64_t k, const Pair& stride, const Pair& padding, const Pair& dilation) {
  return conv_desc(input, weight.size(2), weight.size(3), ConvArgs{{k, k}, stride, padding, dilation, 1, DK_CLIP_NONE, 0.0, 0.0});
}

bool global_deform_conv_supported(const Tensor& input, const Tensor& weight, const Tensor& fc_weight, const OptTensor& fc_bias,
                                  int64_t k, const Pair& stride, const Pair& padding, const Pair& dilation) {
  if (!fc_bias) return false;
  for (const Tensor* t : {&input, &weight, &fc_weight, &*fc_bias})
    if (!t->is_cuda() || t->scalar_type() != input.scalar_type() || t->device() != input.device()) return false;
  const auto t = input.scalar_type();
  if ((t != at::kFloat && t != at::kHalf && t != at::kBFloat16) || input.dim() != 4 || weight.dim() != 4 || input.size(0) == 0)
    return false;
  if (weight.size(0) != input.size(1) || weight.size(1) != 1 ||
      fc_weight.sizes() != at::IntArrayRef({2 * k * k, input.size(1)}) || fc_bias->sizes() != at::IntArrayRef({2 * k * k}))
    return false;
  const dk_conv_desc desc = global_desc(input, weight, k, stride, padding, dilation);
  return dk_global_kernels_supported(&desc) && dk_image_depthwise_supported(&desc);
}

Tensor global_deform_conv(const Tensor& input, const Tensor& weight, const Tensor& fc_weight, const Tensor& fc_bias, int64_t k,
                          const Pair& stride, const Pair& padding, const Pair& dilation) {
  require_gpu({&input, &weight, &fc_weight, &fc_bias});
  TORCH_CHECK_VALUE(global_deform_conv_supported(input, weight, fc_weight, fc_bias, k, stride, padding, dilation),
                    "global_deform_conv: shapes the library's kernels do not cover (global_deform_conv_supported)");
  const dk_conv_desc desc = global_desc(input, weight, k, stride, padding, dilation);
  Tensor x, w, fw, pooled, coord, kernels;
  return record<GlobalDeformConvFunctionBackward>(
      {&input, &weight, &fc_weight, &fc_bias},
      [&] {
        x = input.contiguous(), w = weight.contiguous(), fw = fc_weight.contiguous();
        const Tensor fb = fc_bias.contiguous();
        const int64_t n = x.size(0), c = x.size(1), taps = k * k;
        pooled = at::empty({n, c}, x.options());
        coord = at::empty({2, n, taps, 2}, x.options());  // as predicted, and clamped to the scope
        kernels = at::empty({n, taps, c}, x.options());
        const Strides strides{taps * c, 1, k * c, c};
        Tensor res = empty_out(x, desc);
        check(dk_global_kernels_forward(&desc, in(x), in(fw), in(fb), in(w), out(pooled), out(coord[0]), out(coord[1]), out(kernels),
                                        stream_of(x)),
              "global_deform_conv kernels");
        check(dk_image_depthwise_forward(&desc, in(x), in(kernels), strides.data(), out(res), stream_of(x)), "global_deform_conv forward");
        return res;
      },
      [&](GlobalDeformConvFunctionBackward& n) {
        n.input = SavedVariable(x, false), n.weight = SavedVariable(w, false), n.fc_weight = SavedVariable(fw, false);
        n.saved_pooled = SavedVariable(pooled, false), n.saved_coord = SavedVariable(coord, false);
        n.saved_kernels = SavedVariable(kernels, false);
        n.desc = desc;
      });
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("set_error_class", [](py::object cls) { g_error_class = cls.release().ptr(); });  // (never given back: outlives the shutdown order)
  py::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const DkFailure& e) {
      set_python_error(e);
    }
  });
  // The operators run without the interpreter lock, as the framework's own do: a call may wait in the allocator, load a
  // code object or search for a convolution.  (Saved-tensor hooks and Python dispatch take the lock themselves.)
  const py::call_guard<py::gil_scoped_release> unlocked;
  m.def("sample_depthwise", &sample_depthwise, unlocked);
  m.def("deform_sample_depthwise", &deform_sample_depthwise, unlocked);
  m.def("nd_linear_sample", &nd_linear_sample, unlocked);
  m.def("offset_conv", &offset_conv, unlocked);
  m.def("offset_conv_supported", &offset_conv_supported);
  m.def("image_depthwise_conv", &image_depthwise_conv, unlocked);
  m.def("global_deform_conv", &global_deform_conv, unlocked);
  m.def("global_deform_conv_supported", &global_deform_conv_supported);
  m.attr("conv_desc_size") = sizeof(dk_conv_desc);
}
