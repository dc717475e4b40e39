// Native host side of medvision_amd.ops: argument checks, allocation, workspace and autograd nodes around the C
// entry points of libmedvision_hip.
//
// Small calls of these operators last 5 - 20 us on the GPU, about what the same steps cost in Python (12 us for a
// resampling call, 70 - 150 us for a training step whose backward node has to take the interpreter's lock in the
// autograd thread).  Here a forward call costs ~4 us and backward nodes never enter the interpreter.
// Errors keep the types and texts of the Python layer.
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/numpy.h>

#include <optional>

#include "../../include/medvision_hip.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

[[noreturn]] void raise(PyObject *type, const std::string &text) {
  py::gil_scoped_acquire gil;
  PyErr_SetString(type, text.c_str());
  throw py::error_already_set();
}

// None of the operators has a forward-mode derivative: a dual tensor is refused instead of losing its tangent (it need
// not require a gradient, so the short ways around the autograd nodes would take it).
void no_forward_mode(const Tensor &t) {
  if (t.defined() && t._fw_grad(/*level=*/0).defined())
    raise(PyExc_NotImplementedError, "forward-mode AD is not implemented for this operator");
}

// (std::runtime_error becomes RuntimeError without the C++ backtrace that TORCH_CHECK appends)
#define MVB_CHECK(cond, ...) \
  do {                       \
    if (!(cond)) throw std::runtime_error(c10::str(__VA_ARGS__)); \
  } while (0)

void check(int status) {
  if (status != MV_OK) throw std::runtime_error(mv_last_error());
}

std::string dtype_name(const Tensor &t) {
  py::gil_scoped_acquire gil;
  return py::str(py::cast(t).attr("dtype")).cast<std::string>();
}

int dtype_code(const Tensor &t) {
  switch (t.scalar_type()) {
    case at::kFloat: return MV_F32;
    case at::kHalf: return MV_F16;
    case at::kBFloat16: return MV_BF16;
    case at::kDouble: return MV_F64;
    default: throw std::runtime_error("unsupported dtype " + dtype_name(t));
  }
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void same_device(const Tensor &ref, const Tensor &t, const char *name) {
  MVB_CHECK(!t.defined() || t.device() == ref.device(), name, " is on ", t.device().str(), ", expected ", ref.device().str(),
            " like the input tensor");
}

Tensor bytes_on(const Tensor &like, size_t n) {
  return n ? at::empty({static_cast<int64_t>(n)}, like.options().dtype(at::kByte)) : Tensor();
}

// sampling_ratio, order, im2col_step: any number, as int() takes it
int64_t whole(double v) {
  MVB_CHECK(v > -9e18 && v < 9e18, "expected a whole number, got ", v);
  return static_cast<int64_t>(v);
}

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

using Dims = std::array<int, 3>;

// "output_size": one integer or a tuple of ndim integers
Dims parse_size(const py::handle &size, int ndim) {
  Dims out{1, 1, 1};
  if (PyLong_Check(size.ptr())) {
    for (int a = 3 - ndim; a < 3; ++a) out[a] = static_cast<int>(PyLong_AsLong(size.ptr()));
  } else if (PyTuple_Check(size.ptr())) {
    if (PyTuple_GET_SIZE(size.ptr()) != ndim) raise(PyExc_AssertionError, "");
    for (int a = 0; a < ndim; ++a) {
      PyObject *v = PyTuple_GET_ITEM(size.ptr(), a);
      if (!PyLong_Check(v)) raise(PyExc_AssertionError, "");
      out[3 - ndim + a] = static_cast<int>(PyLong_AsLong(v));
    }
  } else {
    raise(PyExc_TypeError, "\"output_size\" must be an integer or tuple of integers");
  }
  if (PyErr_Occurred()) throw py::error_already_set();
  return out;
}

// stride / padding / dilation of a layer: one integer for all axes or one per axis
Dims per_axis(const py::handle &value, int ndim, int absent) {
  Dims out{absent, absent, absent};
  if (PySequence_Check(value.ptr())) {
    const py::sequence seq = py::reinterpret_borrow<py::sequence>(value);
    if (static_cast<int>(seq.size()) != ndim) raise(PyExc_TypeError, "one value per axis is needed");
    for (int a = 0; a < ndim; ++a) out[3 - ndim + a] = seq[a].cast<int>();
  } else {
    const int v = value.cast<int>();
    for (int a = 3 - ndim; a < 3; ++a) out[a] = v;
  }
  return out;
}

// ---- RoIAlign, RoIAlignRotated and the affine engines -----------------------------------------------------------
enum RoiKind { kPlain, kRotated, kAffine };

struct RoiCall {
  int kind, ndim, ratio, order;
  bool aligned;
  float scale;
  Dims out;
  const char *what() const { return kind == kPlain ? "RoIAlign" : kind == kRotated ? "RoIAlignRotated" : "affine"; }
  int columns() const { return kind == kPlain ? 1 + 2 * ndim : ndim == 2 ? 6 : 10; }
};

Tensor prepared_rois(const RoiCall &c, const Tensor &rois, const Tensor &features) {
  MVB_CHECK(rois.dim() == 2 && rois.size(1) == c.columns(), "wrong roi size! size_rois should be ", c.columns());
  const auto want = features.scalar_type() == at::kDouble ? at::kDouble : at::kFloat;
  if (rois.scalar_type() == want && rois.device() == features.device() && rois.is_contiguous()) return rois;
  return rois.to(features.options().dtype(want)).contiguous();
}

// [N, C, D, H, W] of a feature tensor or gradient (images: D = 1)
std::array<int, 5> five_dims(const at::IntArrayRef &s, int ndim) {
  if (ndim == 2) return {int(s[0]), int(s[1]), 1, int(s[2]), int(s[3])};
  return {int(s[0]), int(s[1]), int(s[2]), int(s[3]), int(s[4])};
}

Tensor roi_forward(const RoiCall &c, const Tensor &input, const Tensor &rois_in, const Tensor &prepared) {
  MVB_CHECK(input.is_cuda(), c.what(), " is not implemented on CPU");
  const Tensor features = input.contiguous();
  const Tensor rois = prepared_rois(c, rois_in, features);
  MVB_CHECK(features.dim() == c.ndim + 2, "expected a ", c.ndim + 2, "-d feature tensor, got ", features.dim(), "-d");
  const bool labels = features.scalar_type() == at::kInt && c.kind == kAffine;
  const int code = labels ? static_cast<int>(MV_I32) : dtype_code(features);
  const auto d = five_dims(features.sizes(), c.ndim);
  const int n = static_cast<int>(rois.size(0));
  const c10::DeviceGuard guard(features.device());
  const Tensor output = c.ndim == 2 ? at::empty({n, d[1], c.out[1], c.out[2]}, features.options())
                                    : at::empty({n, d[1], c.out[0], c.out[1], c.out[2]}, features.options());
  void *const stream = stream_of(features);
  if (prepared.defined()) {
    same_device(features, prepared, "prepared");
    MVB_CHECK(static_cast<size_t>(prepared.numel()) ==
                  mv_roi_align_prepared_bytes(code, c.ndim, d[0], d[1], d[2], d[3], d[4]),
              "prepared copy does not belong to features of this shape");
    // four bytes per roi for the order the rois are worked in; what heads the copy does not serve need
    const size_t bytes = std::max<size_t>(4 * static_cast<size_t>(n),
        mv_roi_align_forward_workspace_bytes(code, c.ndim, d[1], n, c.out[0], c.out[1], c.out[2], c.ratio));
    const Tensor ws = bytes_on(features, bytes);
    check(mv_roi_align_forward_prepared(ptr(features), ptr(prepared), ptr(rois), ptr(output), code, c.ndim, d[0], d[1],
                                        d[2], d[3], d[4], n, c.out[0], c.out[1], c.out[2], c.scale, c.ratio, c.order,
                                        ptr(ws), bytes, stream));
    return output;
  }
  const size_t bytes = mv_roi_align_forward_workspace_bytes_for_input(code, c.ndim, d[0], d[1], d[2], d[3], d[4], n,
                                                                      c.out[0], c.out[1], c.out[2], c.ratio);
  const Tensor ws = bytes_on(features, bytes);
  int status;
  if (c.kind == kPlain && c.ndim == 2)
    status = mv_roi_align_2d_forward(ptr(features), ptr(rois), ptr(output), code, d[0], d[1], d[3], d[4], n, c.out[1],
                                     c.out[2], c.scale, c.ratio, c.order, ptr(ws), bytes, stream);
  else if (c.kind == kPlain)
    status = mv_roi_align_3d_forward(ptr(features), ptr(rois), ptr(output), code, d[0], d[1], d[2], d[3], d[4], n,
                                     c.out[0], c.out[1], c.out[2], c.scale, c.ratio, c.order, ptr(ws), bytes, stream);
  else if (c.ndim == 2)
    status = (c.kind == kRotated ? mv_roi_align_rotated_2d_forward : mv_affine_2d)(
        ptr(features), ptr(rois), ptr(output), code, d[0], d[1], d[3], d[4], n, c.out[1], c.out[2], c.scale, c.ratio,
        c.aligned, c.order, ptr(ws), bytes, stream);
  else
    status = (c.kind == kRotated ? mv_roi_align_rotated_3d_forward : mv_affine_3d)(
        ptr(features), ptr(rois), ptr(output), code, d[0], d[1], d[2], d[3], d[4], n, c.out[0], c.out[1], c.out[2],
        c.scale, c.ratio, c.aligned, c.order, ptr(ws), bytes, stream);
  check(status);
  return output;
}

Tensor roi_backward(const RoiCall &c, const Tensor &grad_output, const Tensor &rois_in, at::IntArrayRef feature_size) {
  MVB_CHECK(grad_output.is_cuda(), c.what(), " is not implemented on CPU");
  const c10::DeviceGuard guard(grad_output.device());
  const Tensor g = grad_output.contiguous();
  const Tensor rois = prepared_rois(c, rois_in, g);
  const int code = dtype_code(g);
  const auto d = five_dims(feature_size, c.ndim);
  const int n = static_cast<int>(rois.size(0));
  const Tensor grad_input = at::empty(feature_size, g.options());
  const size_t bytes = mv_roi_align_backward_write_workspace_bytes(code, c.ndim, c.kind == kRotated, d[0], d[1], d[2], d[3], d[4], n,
                                                                   c.out[0], c.out[1], c.out[2], c.ratio, c.order);
  const Tensor ws = bytes_on(g, bytes);
  check(mv_roi_align_backward_replace(ptr(g), ptr(rois), ptr(grad_input), code, c.ndim, c.kind == kRotated, d[0], d[1], d[2],
                                      d[3], d[4], n, c.out[0], c.out[1], c.out[2], c.scale, c.ratio, c.aligned, c.order,
                                      ptr(ws), bytes, stream_of(g)));
  return grad_input;
}

struct RoiAlignFunction : torch::autograd::Function<RoiAlignFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &features, const Tensor &rois,
                        const std::optional<Tensor> &prepared, const RoiCall &call) {
    ctx->save_for_backward({rois});
    ctx->saved_data["size"] = features.sizes();
    ctx->saved_data["call"] = std::vector<int64_t>{call.kind, call.ndim, call.ratio, call.order, call.aligned};
    ctx->saved_data["scale"] = static_cast<double>(call.scale);
    return roi_forward(call, features, rois, prepared.value_or(Tensor()));
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    if (!ctx->needs_input_grad(0) || !grads[0].defined()) return {Tensor(), Tensor(), Tensor(), Tensor()};
    const at::NoGradGuard no_grad;
    const auto call = ctx->saved_data["call"].toIntVector();
    RoiCall c{int(call[0]), int(call[1]), int(call[2]), int(call[3]), call[4] != 0,
              static_cast<float>(ctx->saved_data["scale"].toDouble()), {1, 1, 1}};
    for (int a = 0; a < c.ndim; ++a) c.out[3 - c.ndim + a] = static_cast<int>(grads[0].size(2 + a));
    return {roi_backward(c, grads[0], ctx->get_saved_variables()[0], ctx->saved_data["size"].toIntVector()), Tensor(),
            Tensor(), Tensor()};
  }
};

// features that need no gradient (or a call under no_grad) get no node
Tensor roi_align(int ndim, bool rotated, const Tensor &features, const Tensor &rois, const py::object &output_size,
                 double spatial_scale, double sampling_ratio, bool aligned, double order, const std::optional<Tensor> &prepared) {
  const RoiCall c{rotated ? kRotated : kPlain, ndim, static_cast<int>(whole(sampling_ratio)), static_cast<int>(whole(order)), aligned, static_cast<float>(spatial_scale),
                  parse_size(output_size, ndim)};
  no_forward_mode(features);
  no_forward_mode(rois);
  const py::gil_scoped_release no_gil;
  if (!(at::GradMode::is_enabled() && (features.requires_grad() || rois.requires_grad()))) {
    const at::NoGradGuard no_grad;
    return roi_forward(c, features, rois, prepared.value_or(Tensor()));
  }
  return RoiAlignFunction::apply(features, rois, prepared, c);
}

Tensor affine(int ndim, const Tensor &features, const Tensor &rois, const py::object &out_size, double spatial_scale,
              double sampling_ratio, bool aligned, double given_order) {
  const int order = static_cast<int>(whole(given_order));
  RoiCall c{kAffine, ndim, static_cast<int>(whole(sampling_ratio)), order, aligned, static_cast<float>(spatial_scale), parse_size(out_size, ndim)};
  const auto t = features.scalar_type();
  // (int32: label maps at order 0, sampled as they are -- the reference resamples a float copy of them)
  if (!(t == at::kFloat || t == at::kHalf || t == at::kBFloat16 || t == at::kDouble || (t == at::kInt && order == 0)))
    raise(PyExc_AssertionError, "input must be a floating tensor but got " + dtype_name(features));
  if ((order != 0 && order != 1 && order != 3) || order != given_order)
    raise(PyExc_AssertionError, c10::str("order ", given_order, " is not supported!"));
  if (order == 0) c.ratio = 1;   // never average nearest-neighbour samples (reference cuda_fun_tools.py:72-74)
  const py::gil_scoped_release no_gil;
  const at::NoGradGuard no_grad;
  return roi_forward(c, features, rois, Tensor());
}

// The same for a sample [C, *spatial] as for a batch of one
Tensor affine_sample(int ndim, const Tensor &sample, const Tensor &rois, const py::object &out_size, double sampling_ratio, double order) {
  return affine(ndim, sample.unsqueeze(0), rois, out_size, 1.0, sampling_ratio, true, order).squeeze(0);
}

// ---- deformable convolution -----------------------------------------------------------------------------------------
struct DcnCall {
  int nd, groups, dg;
  Dims stride, pad, dil;
};

struct DcnShape {
  int nd;
  mv_dcn3d_shape v;
  mv_dcn2d_shape i;
  std::vector<int64_t> out;   // [B, Cout, *spatial]
  int taps;
};

DcnShape dcn_shape(const DcnCall &c, const Tensor &input, const Tensor &weight) {
  MVB_CHECK(input.is_contiguous(), "input tensor has to be contiguous");
  MVB_CHECK(weight.is_contiguous(), "weight tensor has to be contiguous");
  MVB_CHECK(input.dim() == c.nd + 2 && weight.dim() == c.nd + 2, "expected ", c.nd + 2, "-d input and weight tensors");
  const auto x = five_dims(input.sizes(), c.nd), w = five_dims(weight.sizes(), c.nd);
  const int C = x[1], Cout = w[0], ck = w[1];
  MVB_CHECK(c.groups > 0 && c.dg > 0, "groups must be positive");   // (divided by below)
  MVB_CHECK(C == ck * c.groups, "Input shape and kernel channels wont match: (", C, " vs ", ck * c.groups, ").");
  MVB_CHECK(C % c.groups == 0 && Cout % c.groups == 0, "channels(", C, ") and channels_out(", Cout, ") must divide group(",
            c.groups, ")");
  MVB_CHECK(C % c.dg == 0, "channels(", C, ") must divide deformable_group(", c.dg, ")");
  DcnShape s{};
  s.nd = c.nd;
  s.v = {x[0], C, x[2], x[3], x[4], Cout, w[2], w[3], w[4], c.stride[0], c.stride[1], c.stride[2],
         c.pad[0], c.pad[1], c.pad[2], c.dil[0], c.dil[1], c.dil[2], c.groups, c.dg};
  s.i = {x[0], C, x[3], x[4], Cout, w[3], w[4], c.stride[1], c.stride[2], c.pad[1], c.pad[2], c.dil[1], c.dil[2],
         c.groups, c.dg};
  s.taps = w[2] * w[3] * w[4];
  int d = 1, h = 1, wd = 1;
  check(c.nd == 3 ? mv_dcn3d_output_dims(&s.v, &d, &h, &wd) : mv_dcn2d_output_dims(&s.i, &h, &wd));
  s.out = {x[0], Cout};
  if (c.nd == 3) s.out.push_back(d);
  s.out.push_back(h);
  s.out.push_back(wd);
  return s;
}

std::string shape_text(at::IntArrayRef s) {
  std::string t = "(";
  for (size_t i = 0; i < s.size(); ++i) t += (i ? ", " : "") + std::to_string(s[i]);
  return t + ")";
}

void check_aux(const DcnShape &s, const Tensor &t, int channels, const char *name) {
  std::vector<int64_t> want = s.out;
  want[1] = channels;
  MVB_CHECK(t.sizes() == at::IntArrayRef(want), name, " has shape ", shape_text(t.sizes()), ", expected ", shape_text(want));
}

Tensor dcn_forward(const DcnCall &c, const Tensor &input, const Tensor &offset_in, const Tensor &mask_in,
                   const Tensor &weight, const Tensor &bias_in) {
  const DcnShape s = dcn_shape(c, input, weight);
  same_device(input, offset_in, "offset");
  same_device(input, mask_in, "mask");
  same_device(input, weight, "weight");
  same_device(input, bias_in, "bias");
  const Tensor bias = bias_in.defined() ? bias_in.contiguous() : bias_in;
  const Tensor offset = offset_in.to(input.scalar_type()).contiguous();
  const Tensor mask = mask_in.defined() ? mask_in.to(input.scalar_type()).contiguous() : mask_in;
  check_aux(s, offset, c.dg * c.nd * s.taps, "offset");
  if (mask.defined()) check_aux(s, mask, c.dg * s.taps, "mask");
  MVB_CHECK(weight.scalar_type() == input.scalar_type() && (!bias.defined() || bias.scalar_type() == input.scalar_type()),
            "input, weight and bias must share one dtype");
  const int code = dtype_code(input);
  const c10::DeviceGuard guard(input.device());
  const Tensor output = at::empty(s.out, input.options());
  const Tensor ws = bytes_on(input, c.nd == 3 ? mv_dcn3d_forward_workspace_bytes(&s.v, code)
                                              : mv_dcn2d_forward_workspace_bytes(&s.i, code));
  void *const stream = stream_of(input);
  check(c.nd == 3 ? mv_dcn3d_forward(ptr(input), ptr(offset), ptr(mask), ptr(weight), ptr(bias), ptr(output), &s.v, code,
                                     ptr(ws), stream)
                  : mv_dcn2d_forward(ptr(input), ptr(offset), ptr(mask), ptr(weight), ptr(bias), ptr(output), &s.i, code,
                                     ptr(ws), stream));
  return output;
}

struct DcnGrads {
  Tensor input, offset, mask, weight, bias;
};

DcnGrads dcn_backward(const DcnCall &c, const Tensor &input, const Tensor &offset_in, const Tensor &mask_in,
                      const Tensor &weight, const Tensor &bias, const Tensor &grad_in) {
  const c10::DeviceGuard guard(input.device());
  const DcnShape s = dcn_shape(c, input, weight);
  same_device(input, grad_in, "grad_output");
  const Tensor offset = offset_in.to(input.scalar_type()).contiguous();
  const Tensor mask = mask_in.defined() ? mask_in.to(input.scalar_type()).contiguous() : mask_in;
  const Tensor grad = grad_in.to(input.scalar_type()).contiguous();
  MVB_CHECK(grad.sizes() == at::IntArrayRef(s.out), "Input shape and grad_out shape wont match: (", shape_text(s.out), " vs ",
            shape_text(grad.sizes()), ").");
  DcnGrads g;
  g.input = at::empty_like(input);
  g.weight = at::empty_like(weight);
  if (bias.defined()) g.bias = at::empty_like(bias, at::MemoryFormat::Contiguous);
  g.offset = at::empty_like(offset);
  if (mask.defined()) g.mask = at::empty_like(mask);
  const int code = dtype_code(input);
  const Tensor ws = bytes_on(input, c.nd == 3 ? mv_dcn3d_backward_workspace_bytes(&s.v, code)
                                              : mv_dcn2d_backward_workspace_bytes(&s.i, code));
  void *const stream = stream_of(input);
  check(c.nd == 3 ? mv_dcn3d_backward_write(ptr(input), ptr(offset), ptr(mask), ptr(weight), ptr(grad), ptr(g.input), ptr(g.offset),
                                      ptr(g.mask), ptr(g.weight), ptr(g.bias), &s.v, code, ptr(ws), stream)
                  : mv_dcn2d_backward_write(ptr(input), ptr(offset), ptr(mask), ptr(weight), ptr(grad), ptr(g.input), ptr(g.offset),
                                      ptr(g.mask), ptr(g.weight), ptr(g.bias), &s.i, code, ptr(ws), stream));
  return g;
}

struct DeformConvFunction : torch::autograd::Function<DeformConvFunction> {
  static Tensor forward(AutogradContext *ctx, const Tensor &input_in, const Tensor &offset,
                        const std::optional<Tensor> &mask_in, const Tensor &weight_in,
                        const std::optional<Tensor> &bias_in, const DcnCall &c) {
    Tensor input = input_in, weight = weight_in, bias = bias_in.value_or(Tensor());
    const Tensor mask = mask_in.value_or(Tensor());
    if (offset.scalar_type() == at::kHalf || offset.scalar_type() == at::kBFloat16) {   // autocast: follow the offset branch
      input = input.to(offset.scalar_type());
      weight = weight.to(offset.scalar_type());
      if (bias.defined()) bias = bias.to(offset.scalar_type());
    }
    const Tensor output = dcn_forward(c, input, offset, mask, weight, bias);
    ctx->save_for_backward({input, offset, mask, weight, bias});
    ctx->saved_data["call"] = std::vector<int64_t>{c.nd, c.groups, c.dg, c.stride[0], c.stride[1], c.stride[2], c.pad[0],
                                                   c.pad[1], c.pad[2], c.dil[0], c.dil[1], c.dil[2]};
    return output;
  }
  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    if (!grads[0].defined()) return variable_list(6);
    variable_list out;
    {
      const at::NoGradGuard no_grad;
      MVB_CHECK(grads[0].is_cuda(), "Not implemented on the CPU");
      const auto v = ctx->saved_data["call"].toIntVector();
      const DcnCall c{int(v[0]), int(v[1]), int(v[2]), {int(v[3]), int(v[4]), int(v[5])}, {int(v[6]), int(v[7]), int(v[8])},
                      {int(v[9]), int(v[10]), int(v[11])}};
      const auto saved = ctx->get_saved_variables();
      const DcnGrads g = dcn_backward(c, saved[0], saved[1], saved[2], saved[3], saved[4], grads[0]);
      out = {g.input, g.offset, g.mask, g.weight, g.bias, Tensor()};
    }
    // the gradients cannot be differentiated again: say so when someone tries
    if (at::GradMode::is_enabled() && grads[0].requires_grad()) {
      for (Tensor &t : out) {
        if (!t.defined()) continue;
        auto once = std::make_shared<torch::autograd::DelayedError>(
            "trying to differentiate twice a function that was marked with @once_differentiable", 1);
        t.set_requires_grad(true);
        t = (*once)(variable_list{t})[0];
      }
    }
    return out;
  }
};

void im2col_step_check(int64_t batch, int64_t im2col_step) {
  const int64_t step = std::min(batch, im2col_step);
  MVB_CHECK(step != 0 && batch % step == 0, "batch(", batch, ") must divide im2col_step(", step, ")");
}

// DCNv2: scalar stride / padding / dilation, optional bias
Tensor modulated_deform_conv(int nd, const Tensor &input, const Tensor &offset, const Tensor &mask, const Tensor &weight,
                             const std::optional<Tensor> &bias, int stride, int padding, int dilation, int groups, int dg) {
  if (!input.is_cuda()) raise(PyExc_NotImplementedError, "");
  const int s0 = nd == 3 ? stride : 1, p0 = nd == 3 ? padding : 0, d0 = nd == 3 ? dilation : 1;
  const DcnCall c{nd, groups, dg, {s0, stride, stride}, {p0, padding, padding}, {d0, dilation, dilation}};
  for (const Tensor &t : {input, offset, mask, weight, bias.value_or(Tensor())}) no_forward_mode(t);
  const py::gil_scoped_release no_gil;
  return DeformConvFunction::apply(input, offset, mask, weight, bias, c);
}

// DCNv1: the bias is always added
Tensor deform_conv(int nd, const Tensor &input, const Tensor &offset, const Tensor &weight, const Tensor &bias,
                   const py::object &stride, const py::object &padding, const py::object &dilation, int groups, int dg,
                   double im2col_step) {
  const DcnCall c{nd, groups, dg, per_axis(stride, nd, 1), per_axis(padding, nd, 0), per_axis(dilation, nd, 1)};
  for (const Tensor &t : {input, offset, weight, bias}) no_forward_mode(t);
  const py::gil_scoped_release no_gil;
  MVB_CHECK(input.is_cuda(), "Not implemented on the CPU");
  im2col_step_check(input.size(0), whole(im2col_step));
  return DeformConvFunction::apply(input, offset, std::nullopt, weight, bias, c);
}

// ---- displacement-field warp ------------------------------------------------------------------------------------------
Tensor deform_warp(const Tensor &img_in, const Tensor &offset_in, double given_order) {
  const int order = given_order == 0.0 || given_order == 1.0 || given_order == 3.0 ? static_cast<int>(given_order) : -1;
  const py::gil_scoped_release no_gil;
  const at::NoGradGuard no_grad;
  MVB_CHECK(img_in.is_cuda(), "Not implemented on the CPU");
  const int ndim = static_cast<int>(img_in.dim()) - 2;
  MVB_CHECK(ndim == 2 || ndim == 3, "expected a 4-d or 5-d image, got ", img_in.dim(), "-d");
  const c10::DeviceGuard guard(img_in.device());
  const Tensor img = img_in.contiguous();
  const bool labels = img.scalar_type() == at::kInt;   // label maps: order 0 picks voxels, so they are warped as they are
  MVB_CHECK(!labels || order == 0, "int32 label maps are warped at order 0 only");
  const Tensor offset = offset_in.to(img.options().dtype(labels ? at::kFloat : img.scalar_type())).contiguous();
  std::vector<int64_t> want = img.sizes().vec();
  if (want.size() > 1) want[1] = ndim;
  MVB_CHECK(offset.sizes() == at::IntArrayRef(want), "offset must have shape [B, ", ndim, ", *spatial]");
  MVB_CHECK(order >= 0, "order ", given_order, " is not supported (0 nearest, 1 linear, 3 cubic)");
  const int code = labels ? static_cast<int>(MV_I32) : dtype_code(img);
  const Tensor out = at::empty_like(img);
  const auto d = five_dims(img.sizes(), ndim);
  void *const stream = stream_of(img);
  check(ndim == 2 ? mv_deform_warp_2d(ptr(img), ptr(offset), ptr(out), code, d[0], d[1], d[3], d[4], order, stream)
                  : mv_deform_warp_3d(ptr(img), ptr(offset), ptr(out), code, d[0], d[1], d[2], d[3], d[4], order, stream));
  return out;
}

// A volume [B,C,D,H,W], or a sample [C,D,H,W] as a batch of one, warped by the field that its control grids [B,3,z,y,x] give over the
// window [border, points - border]; nothing where that has to be done in two calls.
std::optional<Tensor> elastic_warp(const Tensor &given, const Tensor &grid, double border) {
  const py::gil_scoped_release no_gil;
  const at::NoGradGuard no_grad;
  const bool sample = given.dim() == 4;
  const Tensor img_in = sample ? given.unsqueeze(0) : given;
  if (!img_in.is_cuda() || img_in.dim() != 5 || grid.dim() != 5 || grid.device() != img_in.device() || grid.scalar_type() != at::kFloat ||
      grid.size(0) != img_in.size(0) || grid.size(1) != 3 || img_in.numel() == 0)
    return std::nullopt;
  const auto type = img_in.scalar_type();
  if (type != at::kInt && type != at::kFloat && type != at::kHalf && type != at::kBFloat16) return std::nullopt;
  for (const Tensor &t : {img_in, grid})
    for (int64_t n : t.sizes())
      if (n > std::numeric_limits<int>::max()) return std::nullopt;
  const int code = type == at::kInt ? static_cast<int>(MV_I32) : dtype_code(img_in);
  const auto d = five_dims(img_in.sizes(), 3);
  const auto g = five_dims(grid.sizes(), 3);
  const float edge = static_cast<float>(border);
  if (!mv_elastic_warp_3d_applies(code, d[0], d[2], d[3], d[4], g[2], g[3], g[4], edge)) return std::nullopt;
  const c10::DeviceGuard guard(img_in.device());
  const Tensor img = img_in.contiguous(), points = grid.contiguous();
  const Tensor out = at::empty_like(img);
  check(mv_elastic_warp_3d(ptr(img), ptr(points), ptr(out), code, d[0], d[1], d[2], d[3], d[4], g[2], g[3], g[4], edge, stream_of(img)));
  return sample ? out.squeeze(0) : out;
}

// ---- helpers of the augmentation stages ----------------------------------------------------------------------------
// A host array (rois, a control grid) on the device, without waiting for what is queued there.  float64 stays float64,
// every other type becomes float32.
Tensor upload(const py::array &given, const at::Device &device) {
  const bool wide = py::isinstance<py::array_t<double>>(given);
  const py::array array = wide ? py::array(py::array_t<double, py::array::c_style | py::array::forcecast>(given))
                               : py::array(py::array_t<float, py::array::c_style | py::array::forcecast>(given));
  const auto type = wide ? at::kDouble : at::kFloat;
  const std::vector<int64_t> shape(array.shape(), array.shape() + array.ndim());
  const size_t bytes = static_cast<size_t>(array.nbytes());
  const void *data = array.data();
  const py::gil_scoped_release no_gil;
  const at::NoGradGuard no_grad;
  if (!device.is_cuda() || bytes > MV_UPLOAD_MAX_BYTES)
    return at::from_blob(const_cast<void *>(data), shape, type).to(device, type, false, true);
  const c10::DeviceGuard guard(device);
  const Tensor out = at::empty(shape, at::TensorOptions().dtype(type).device(device));
  check(mv_upload(data, ptr(out), bytes, stream_of(out)));
  return out;
}

// The roi of one window of one sample, as geometry.window_rois has it (its float32 arithmetic, in its order), on the device
Tensor window_roi(int dim, const std::vector<double> &start, const std::vector<double> &end, const std::vector<double> &scales,
                  const std::vector<double> &shifts, double rotate, const at::Device &device) {
  const size_t n = static_cast<size_t>(dim);
  MVB_CHECK((dim == 2 || dim == 3) && start.size() == n && end.size() == n && scales.size() == n && shifts.size() == n,
            "expected one value per axis");
  float row[10] = {};
  const int columns = dim == 2 ? 6 : 10;
  for (size_t a = 0; a < n; a++) {
    const float s = static_cast<float>(start[a]), e = static_cast<float>(end[a]), scale = static_cast<float>(scales[a]), shift = static_cast<float>(shifts[a]);
    const float extent = e - s, middle = (s + e) / 2.f, moved = extent * shift;
    row[1 + a] = middle - moved / scale;
    row[1 + n + a] = extent / scale;
  }
  row[columns - 1] = static_cast<float>(rotate);
  const py::gil_scoped_release no_gil;
  const at::NoGradGuard no_grad;
  const c10::OptionalDeviceGuard guard(device.is_cuda() ? std::optional<at::Device>(device) : std::nullopt);
  const Tensor out = at::empty({1, columns}, at::TensorOptions().dtype(at::kFloat).device(device));
  if (device.is_cuda()) check(mv_upload(row, ptr(out), columns * sizeof(float), stream_of(out)));
  else std::memcpy(out.data_ptr(), row, columns * sizeof(float));
  return out;
}

// torch.cuda.max_memory_allocated() in MiB, without building the whole tree of statistics (18 us)
double peak_mib() {
  auto *allocator = c10::hip::HIPCachingAllocator::get();
  if (!allocator->initialized()) return 0.0;
  return allocator->getDeviceStats(c10::hip::current_device()).allocated_bytes[0].peak / 1048576.0;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("roi_align", &roi_align);
  m.def("affine", &affine);
  m.def("affine_sample", &affine_sample);
  m.def("modulated_deform_conv", &modulated_deform_conv);
  m.def("deform_conv", &deform_conv);
  m.def("deform_warp", &deform_warp);
  m.def("elastic_warp", &elastic_warp);
  m.def("upload", &upload);
  m.def("window_roi", &window_roi);
  m.def("peak_mib", &peak_mib);
}
