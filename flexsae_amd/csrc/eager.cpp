// Ordinary eager calls without Python between the launches: the checks of a call, its allocations, the C-ABI entry points and
// the autograd nodes of the two losses, as an extension module of CPython over torch's C++ interface.
//
// A small step is host work: with the same steps in Python (ctypes, torch.empty, an autograd.Function whose backward takes the
// interpreter's lock on autograd's device thread) B=64, K=32, F=4096, D=256 fp32 takes 160 us (TopK) and 195 us
// (hierarchical) for 35-45 us of kernels; the figures with this module stand at the entry points in ops.py.
//
// A function here returns None for a call that is not its business (tensors that are not plain, something around the call that
// has to see the ops, arguments that a check refuses): the caller then goes through the ops, which see, resolve or refuse it.
// A backward whose surroundings or gradient are not plain calls back into ops.py with what was saved.
#include <dlfcn.h>

#include <atomic>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/flexsae_amd.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;

// ---- the library ---------------------------------------------------------------------------
#define FLEXSAE_ENTRIES(X)                                                                                              \
  X(abi_version) X(fwd_workspace_bytes) X(topk_fwd_best_workspace_bytes) X(topk_fwd) X(hier_fwd)                        \
  X(topk_bwd_from_indices_workspace_bytes) X(topk_bwd_from_indices) X(hier_bwd_workspace_bytes) X(hier_bwd)             \
  X(hier_fwd_bwd_workspace_bytes_flags) X(hier_step) X(finish_grads)
struct Library {
#define X(name) decltype(&flexsae_##name) name = nullptr;
  FLEXSAE_ENTRIES(X)
#undef X
} lib;

// What the Python side keeps: callbacks, the flags of the devices (never freed: the interpreter is gone when statics are) and
// settings.
PyObject *general_backward = nullptr;  // (kind, grad, saved, needs, numbers, dW) -> (gradients, dW left)
PyObject *raise_status = nullptr;      // (status, entry point)
constexpr int kMaxDevices = 64;
Tensor *const status_flags = new Tensor[kMaxDevices];
std::atomic<int> topk_bwd_flags{0};
std::atomic<bool> lists_in_python{false};  // a shared_pair_list() block is active: backwards look there first

[[noreturn]] void throw_python() {  // what the interpreter has raised
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "unexpected result of a callback");
  python_error e;
  e.persist();
  throw e;
}

void check(int status, const char *entry) {
  if (status == FLEXSAE_OK) return;
  pybind11::gil_scoped_acquire gil;
  PyObject *r = PyObject_CallFunction(raise_status, "is", status, entry);
  Py_XDECREF(r);
  throw_python();
}

// ---- which calls ---------------------------------------------------------------------------
// A tensor on the GPU whose values are its memory and which nothing but autograd looks at.
bool plain_tensor(const Tensor &t) {
  static const uint64_t usual =
      (c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
       c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::DispatchKeySet(c10::DispatchKey::AutocastCUDA))
          .raw_repr();
  return t.defined() && t.is_cuda() && (t.key_set().raw_repr() & ~usual) == 0 && !t._fw_grad(0).defined();
}

// Nothing around the call that has to see the ops: modes, transforms, tracers.
bool plain_surroundings() {
  static const c10::DispatchKeySet watching(
      {c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode,
       c10::DispatchKey::Functionalize, c10::DispatchKey::Python, c10::DispatchKey::PreDispatch, c10::DispatchKey::Tracer,
       c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchVmapMode});
  return c10::impl::TorchDispatchModeTLS::stack_len() == 0 && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
         !c10::impl::tls_local_dispatch_key_set().included_.has_any(watching);
}

bool plain_backward(const Tensor &grad) {
  return !c10::GradMode::is_enabled() && plain_tensor(grad) && plain_surroundings();
}

int dtype_of(c10::ScalarType t) {
  switch (t) {
    case c10::ScalarType::Float: return FLEXSAE_F32;
    case c10::ScalarType::BFloat16: return FLEXSAE_BF16;
    case c10::ScalarType::Half: return FLEXSAE_F16;
    default: return -1;
  }
}

struct Inputs {
  Tensor indices, weight, vals, bias, target;
};

// The checks of _validate in ops.py (which says what is wrong with what fails here).  A bias that is not defined is not asked for.
bool usable(const Inputs &in) {
  for (const Tensor *t : {&in.indices, &in.weight, &in.vals, &in.bias, &in.target})
    if (t->defined() || t != &in.bias)
      if (!plain_tensor(*t) || t->device() != in.weight.device() || t->dim() != (t == &in.bias ? 1 : 2)) return false;
  const int64_t B = in.indices.size(0), K = in.indices.size(1), F = in.weight.size(0), D = in.weight.size(1);
  if (in.vals.size(0) != B || in.vals.size(1) != K || (in.bias.defined() && in.bias.size(0) != D) || in.target.size(0) != B ||
      in.target.size(1) != D)
    return false;
  if (B < 1 || K < 1 || F < 1 || D < 1 || F >= (int64_t{1} << 31) || D >= (int64_t{1} << 29) ||
      B > ((int64_t{1} << 32) - 1) / K)
    return false;
  if (in.indices.scalar_type() != c10::ScalarType::Long) return false;
  for (const Tensor *t : {&in.weight, &in.vals, &in.bias, &in.target})
    if (t->defined() && dtype_of(t->scalar_type()) < 0) return false;
  const int device = in.weight.device().index();
  return device >= 0 && device < kMaxDevices && status_flags[device].defined();
}

// What hooks have handed back for the saved tensors of a backward may be anything.
bool usable_fp32(const Tensor &t, const Tensor &weight, at::IntArrayRef sizes) {
  return plain_tensor(t) && t.device() == weight.device() && t.sizes() == sizes && t.scalar_type() == c10::ScalarType::Float;
}

// ... of a backward of its own: indices, weight, vals, resid
bool usable_saved(const variable_list &saved) {
  return usable({saved[0], saved[1], saved[2], Tensor(), saved[3]}) && saved[3].scalar_type() == c10::ScalarType::Float;
}

// ... of a step: its inputs
bool usable_inputs(const variable_list &saved) { return usable({saved[0], saved[1], saved[2], saved[3], saved[4]}); }

flexsae_shape shape_of(const Tensor &indices, const Tensor &weight, const Tensor &vals, int bias_dtype, int target_dtype) {
  return {indices.size(0), indices.size(1), weight.size(0), weight.size(1), dtype_of(weight.scalar_type()),
          dtype_of(vals.scalar_type()), bias_dtype, target_dtype};
}

flexsae_shape shape_of(const Inputs &in) {
  return shape_of(in.indices, in.weight, in.vals, dtype_of(in.bias.scalar_type()), dtype_of(in.target.scalar_type()));
}

// Contiguous and 16-byte aligned, as the vector accesses of the kernels need.
Tensor prepared(const Tensor &t) {
  const Tensor c = t.contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 ? c.clone() : c;
}

Inputs prepared(const Inputs &in) {
  return {prepared(in.indices), prepared(in.weight), prepared(in.vals), prepared(in.bias), prepared(in.target)};
}

Tensor make(const Tensor &like, at::IntArrayRef sizes, c10::ScalarType type) {
  return at::empty(sizes, like.options().dtype(type).requires_grad(false));
}

Tensor make_workspace(const Tensor &like, size_t bytes) {
  return make(like, {static_cast<int64_t>(bytes)}, c10::ScalarType::Byte);
}

int *flag_of(const Tensor &t) { return status_flags[t.device().index()].data_ptr<int>(); }
void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
bool capturing(const Tensor &t) {
  const c10::DeviceGuard guard(t.device());
  return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}
const int64_t *index_ptr(const Tensor &t) { return t.const_data_ptr<int64_t>(); }
float *f32(const Tensor &t) { return t.data_ptr<float>(); }

// The upstream gradient as one fp32 number on the device.
Tensor grad_scalar(const Tensor &grad, const c10::Device &device) {
  const Tensor g = grad.detach();
  if (g.scalar_type() == c10::ScalarType::Float && g.device() == device && g.numel() == 1) return g;
  return g.to(device, c10::ScalarType::Float).reshape({1}).contiguous();
}

// ---- the steps -----------------------------------------------------------------------------
// (loss, resid)
std::pair<Tensor, Tensor> forward(bool topk, const Inputs &given) {
  const c10::DeviceGuard guard(given.weight.device());
  const Inputs in = prepared(given);
  const flexsae_shape s = shape_of(in);
  const size_t bytes = topk ? lib.topk_fwd_best_workspace_bytes(&s) : lib.fwd_workspace_bytes(&s);
  const Tensor workspace = make_workspace(in.weight, bytes);
  Tensor loss = make(in.weight, {}, c10::ScalarType::Float);
  Tensor resid = make(in.weight, {s.B, s.D}, c10::ScalarType::Float);
  check((topk ? lib.topk_fwd : lib.hier_fwd)(&s, index_ptr(in.indices), in.weight.data_ptr(), in.vals.data_ptr(),
                                             in.bias.data_ptr(), in.target.data_ptr(), f32(loss), f32(resid),
                                             workspace.data_ptr(), bytes, flag_of(in.weight), stream_of(in.weight)),
        topk ? "flexsae_topk_fwd" : "flexsae_hier_fwd");
  return {loss, resid};
}

// (dW, dvals, dbias), dvals and dbias times grad (undefined: one) in the leaves' types; dW_unit (undefined: none) times it in
// the weight's, in place where it has that type
std::tuple<Tensor, Tensor, Tensor> finish(const Tensor &grad, const Tensor &weight, const Tensor &dW_unit, const Tensor &dvals,
                                          c10::ScalarType vals_type, const Tensor &dbias, c10::ScalarType bias_type) {
  const Tensor g = grad.defined() ? grad_scalar(grad, weight.device()) : Tensor();
  Tensor dW;
  if (dW_unit.defined())
    dW = dW_unit.scalar_type() == weight.scalar_type() ? dW_unit : make(weight, dW_unit.sizes(), weight.scalar_type());
  Tensor out_v = make(weight, dvals.sizes(), vals_type), out_b = make(weight, dbias.sizes(), bias_type);
  check(lib.finish_grads(dW.defined() ? dW.data_ptr() : nullptr, dtype_of(weight.scalar_type()),
                         dW.defined() ? dW_unit.data_ptr() : nullptr,
                         dtype_of((dW.defined() ? dW_unit : weight).scalar_type()), dW.defined() ? dW.numel() : 0,
                         out_v.data_ptr(), dtype_of(vals_type), f32(dvals), dvals.numel(), out_b.data_ptr(),
                         dtype_of(bias_type), f32(dbias), dbias.numel(), g.defined() ? f32(g) : nullptr, stream_of(weight)),
        "flexsae_finish_grads");
  return {dW, out_v, out_b};
}

// How a training step of the hierarchical loss runs: what ops.py has decided about it.
struct StepPlan {
  bool need_dw;
  int64_t slice_cols;
  int64_t flags;     // of the call
  int64_t ws_flags;  // of the workspace query
  Tensor stats;      // pinned memory for what the pair list says about the indices (undefined: not wanted) ...
  int64_t tag;       // ... and the mark that it has arrived
};

struct Step {
  Tensor loss, dvals, dbias, dW;
};

// grad (undefined: the unit gradient, of fp16 weights in fp32): dW is the gradient for it in the weight's type.
// step: dW is not formed, the weights move by it.
Step hier_step(const Inputs &given, const StepPlan &p, const Tensor &grad = Tensor(), const Tensor &step = Tensor()) {
  const c10::DeviceGuard guard(given.weight.device());
  const Inputs in = prepared(given);
  const flexsae_shape s = shape_of(in);
  const size_t bytes = lib.hier_fwd_bwd_workspace_bytes_flags(&s, p.slice_cols, static_cast<int>(p.ws_flags));
  const Tensor workspace = make_workspace(in.weight, bytes);
  const bool half = in.weight.scalar_type() == c10::ScalarType::Half;
  const auto type = half && !grad.defined() ? c10::ScalarType::Float : in.weight.scalar_type();
  Step r;
  r.loss = make(in.weight, {}, c10::ScalarType::Float);
  if (p.need_dw && !step.defined()) r.dW = make(in.weight, {s.F, s.D}, type);
  r.dvals = make(in.weight, {s.B, s.K}, c10::ScalarType::Float);
  r.dbias = make(in.weight, {s.D}, c10::ScalarType::Float);
  const Tensor g = grad.defined() ? grad_scalar(grad, in.weight.device()) : Tensor();
  const Tensor by = step.defined() ? grad_scalar(step, in.weight.device()) : Tensor();
  const int status = lib.hier_step(
      &s, index_ptr(in.indices), in.weight.data_ptr(), in.vals.data_ptr(), in.bias.data_ptr(), in.target.data_ptr(),
      g.defined() ? f32(g) : nullptr, by.defined() ? f32(by) : nullptr, f32(r.loss),
      r.dW.defined() ? r.dW.data_ptr() : nullptr, dtype_of(type), f32(r.dvals), f32(r.dbias), workspace.data_ptr(), bytes,
      static_cast<int>(p.flags) | (p.need_dw ? 0 : FLEXSAE_BWD_NO_DW),
      p.stats.defined() ? static_cast<uint32_t *>(p.stats.data_ptr()) : nullptr, static_cast<uint32_t>(p.tag),
      flag_of(in.weight), stream_of(in.weight));
  // (a call that was refused, here or by an allocation above, has left the weights alone)
  if (step.defined() && (status == FLEXSAE_OK || status == FLEXSAE_ERR_LAUNCH))
    torch::autograd::impl::bump_version(given.weight);
  check(status, "flexsae_hier_step");
  return r;
}

// ---- autograd ------------------------------------------------------------------------------
enum Kind { kTopk = 0, kHier = 1, kSliced = 2, kLate = 3 };

void save_plan(AutogradContext *ctx, const StepPlan &plan) {
  ctx->saved_data["need_dw"] = static_cast<int64_t>(plan.need_dw);
  ctx->saved_data["cols"] = plan.slice_cols;
  ctx->saved_data["flags"] = plan.flags;
  ctx->saved_data["ws_flags"] = plan.ws_flags;
}

StepPlan saved_plan(AutogradContext *ctx) {
  return {ctx->saved_data["need_dw"].toInt() != 0, ctx->saved_data["cols"].toInt(), ctx->saved_data["flags"].toInt(),
          ctx->saved_data["ws_flags"].toInt(), Tensor(), 0};
}

// A backward that is not plain, by ops.py; dW: the unit gradient, which it may take or leave.
variable_list backward_in_python(AutogradContext *ctx, Kind kind, const Tensor &grad, const variable_list &saved,
                                 std::initializer_list<int64_t> numbers, Tensor *dW, size_t n_inputs) {
  pybind11::gil_scoped_acquire gil;
  auto tuple_of = [](size_t n, auto item) {
    auto t = pybind11::reinterpret_steal<pybind11::object>(PyTuple_New(static_cast<Py_ssize_t>(n)));
    for (size_t i = 0; i < n; ++i) PyTuple_SET_ITEM(t.ptr(), static_cast<Py_ssize_t>(i), item(i));
    return t;
  };
  const auto py_saved = tuple_of(saved.size(), [&](size_t i) { return THPVariable_Wrap(saved[i]); });
  const auto py_needs = tuple_of(5, [&](size_t i) { return PyBool_FromLong(ctx->needs_input_grad(i)); });
  const auto py_numbers = tuple_of(numbers.size(), [&](size_t i) { return PyLong_FromLongLong(numbers.begin()[i]); });
  const auto py_grad = pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(grad));
  const auto py_dw = dW && dW->defined() ? pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(*dW))
                                         : pybind11::reinterpret_borrow<pybind11::object>(Py_None);
  const auto r = pybind11::reinterpret_steal<pybind11::object>(
      PyObject_CallFunction(general_backward, "iOOOOO", static_cast<int>(kind), py_grad.ptr(), py_saved.ptr(),
                            py_needs.ptr(), py_numbers.ptr(), py_dw.ptr()));
  if (!r.ptr()) throw_python();
  PyObject *const grads = PyTuple_GetItem(r.ptr(), 0), *const left = PyTuple_GetItem(r.ptr(), 1);
  if (!grads || !left || !PyTuple_Check(grads) || PyTuple_GET_SIZE(grads) != 5) throw_python();
  if (dW) *dW = left == Py_None ? Tensor() : THPVariable_Unpack(left);
  variable_list out(n_inputs);
  for (Py_ssize_t i = 0; i < 5; ++i) {
    PyObject *const g = PyTuple_GET_ITEM(grads, i);
    if (g != Py_None) out[static_cast<size_t>(i)] = THPVariable_Unpack(g);
  }
  return out;
}

struct TopkLoss : torch::autograd::Function<TopkLoss> {
  static Variable forward(AutogradContext *ctx, const Variable &indices, const Variable &weight, const Variable &vals,
                          const Variable &bias, const Variable &target) {
    auto [loss, resid] = ::forward(true, {indices, weight, vals, bias, target});
    ctx->save_for_backward({indices, weight, vals, resid});
    ctx->set_materialize_grads(false);
    ctx->saved_data["bias"] = static_cast<int64_t>(bias.scalar_type());
    ctx->saved_data["target"] = static_cast<int64_t>(target.scalar_type());
    return loss;
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &grad = grads[0];
    if (!grad.defined()) return variable_list(5);
    const int64_t bias_type = ctx->saved_data["bias"].toInt(), target_type = ctx->saved_data["target"].toInt();
    if (!plain_backward(grad) || lists_in_python || !usable_saved(saved))
      return backward_in_python(ctx, kTopk, grad, saved,
                                {dtype_of(static_cast<c10::ScalarType>(bias_type)),
                                 dtype_of(static_cast<c10::ScalarType>(target_type))},
                                nullptr, 5);
    const Tensor indices = prepared(saved[0]), weight = prepared(saved[1]), vals = prepared(saved[2]), resid = prepared(saved[3]);
    const c10::DeviceGuard guard(weight.device());
    const Tensor g = grad_scalar(grad, weight.device());
    const flexsae_shape s = shape_of(indices, weight, vals, FLEXSAE_F32, FLEXSAE_F32);
    // (the slice width only sizes the partial sums of frequent latents: up to 256 MiB of them)
    const int64_t per_col = s.B * s.K / 32 * 4, cols = (int64_t{256} << 20) / (per_col > 1 ? per_col : 1);
    const size_t bytes = lib.topk_bwd_from_indices_workspace_bytes(&s, cols > 1 ? cols : 1);
    const auto leaf_bias = static_cast<c10::ScalarType>(bias_type);
    Tensor dW = at::empty_like(weight);
    Tensor dvals = make(weight, {s.B, s.K}, vals.scalar_type()), dbias = make(weight, {s.D}, leaf_bias);
    const Tensor workspace = make_workspace(weight, bytes);
    check(lib.topk_bwd_from_indices(&s, index_ptr(indices), weight.data_ptr(), vals.data_ptr(), f32(resid), f32(g),
                                    dW.data_ptr(), s.weight_dtype, dvals.data_ptr(), s.vals_dtype, dbias.data_ptr(),
                                    dtype_of(leaf_bias), workspace.data_ptr(), bytes, topk_bwd_flags, flag_of(weight),
                                    stream_of(weight)),
          "flexsae_topk_bwd_from_indices");
    Tensor dtarget;
    if (ctx->needs_input_grad(4))
      dtarget = (resid * (grad.to(c10::ScalarType::Float) * (-2.0 / static_cast<double>(s.B * s.D))))
                    .to(static_cast<c10::ScalarType>(target_type));
    return {Tensor(), dW, dvals, dbias, dtarget};
  }
};

struct HierLoss : torch::autograd::Function<HierLoss> {
  static Variable forward(AutogradContext *ctx, const Variable &indices, const Variable &weight, const Variable &vals,
                          const Variable &bias, const Variable &target, int64_t slice_cols) {
    auto [loss, resid] = ::forward(false, {indices, weight, vals, bias, target});
    ctx->save_for_backward({indices, weight, vals, resid});
    ctx->set_materialize_grads(false);
    ctx->saved_data["bias"] = static_cast<int64_t>(bias.scalar_type());
    ctx->saved_data["cols"] = slice_cols;
    return loss;
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &grad = grads[0];
    if (!grad.defined()) return variable_list(6);
    const auto leaf_bias = static_cast<c10::ScalarType>(ctx->saved_data["bias"].toInt());
    if (!plain_backward(grad) || lists_in_python || !usable_saved(saved))
      return backward_in_python(ctx, kHier, grad, saved, {dtype_of(leaf_bias)}, nullptr, 6);
    const Tensor indices = prepared(saved[0]), weight = prepared(saved[1]), vals = prepared(saved[2]), resid = prepared(saved[3]);
    const c10::DeviceGuard guard(weight.device());
    const Tensor g = grad_scalar(grad, weight.device());
    const flexsae_shape s = shape_of(indices, weight, vals, FLEXSAE_F32, FLEXSAE_F32);
    const size_t bytes = lib.hier_bwd_workspace_bytes(&s, ctx->saved_data["cols"].toInt());
    const Tensor workspace = make_workspace(weight, bytes);
    Tensor dW = at::empty_like(weight);
    Tensor dvals = make(weight, {s.B, s.K}, c10::ScalarType::Float), dbias = make(weight, {s.D}, c10::ScalarType::Float);
    check(lib.hier_bwd(&s, index_ptr(indices), weight.data_ptr(), vals.data_ptr(), f32(resid), f32(g), dW.data_ptr(),
                       s.weight_dtype, f32(dvals), f32(dbias), workspace.data_ptr(), bytes, 0, flag_of(weight),
                       stream_of(weight)),
          "flexsae_hier_bwd");
    if (vals.scalar_type() != c10::ScalarType::Float || leaf_bias != c10::ScalarType::Float)
      std::tie(std::ignore, dvals, dbias) = finish(Tensor(), weight, Tensor(), dvals, vals.scalar_type(), dbias, leaf_bias);
    return {Tensor(), dW, dvals, dbias, Tensor(), Tensor()};
  }
};

struct SlicedLoss : torch::autograd::Function<SlicedLoss> {
  static Variable forward(AutogradContext *ctx, const Variable &indices, const Variable &weight, const Variable &vals,
                          const Variable &bias, const Variable &target, const StepPlan &plan) {
    Step r = hier_step({indices, weight, vals, bias, target}, plan);
    ctx->save_for_backward({indices, weight, vals, bias, target, r.dvals, r.dbias});
    ctx->set_materialize_grads(false);
    // the unit gradient is no saved tensor: the backward scales it in place and hands the very buffer on
    if (plan.need_dw) ctx->saved_data["dW"] = r.dW;
    save_plan(ctx, plan);
    return r.loss;
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    auto saved = ctx->get_saved_variables();
    const Tensor &grad = grads[0];
    if (!grad.defined()) return variable_list(6);
    const auto at = ctx->saved_data.find("dW");
    Tensor dW = at != ctx->saved_data.end() ? at->second.toTensor() : Tensor();
    const StepPlan plan = saved_plan(ctx);
    if (!plain_backward(grad) || (lists_in_python && !dW.defined()) || !usable_inputs(saved) ||
        !usable_fp32(saved[5], saved[1], saved[2].sizes()) || !usable_fp32(saved[6], saved[1], saved[3].sizes()) ||
        (dW.defined() && dW.device() != saved[1].device())) {
      auto out = backward_in_python(ctx, kSliced, grad, saved, {plan.need_dw, plan.flags}, &dW, 6);
      if (dW.defined()) ctx->saved_data["dW"] = dW;
      else ctx->saved_data.erase("dW");
      return out;
    }
    Tensor dvals = prepared(saved[5]), dbias = prepared(saved[6]);
    if (ctx->needs_input_grad(1)) {
      TORCH_CHECK(plan.need_dw, "the step ran without dW but weight requires a gradient");
      ctx->saved_data.erase("dW");  // the buffer now belongs to whoever receives the gradient
      if (!dW.defined()) {          // a second backward through a retained graph: the buffer went with the first one
        Step again = hier_step({saved[0], saved[1], saved[2], saved[3], saved[4]}, plan);
        dW = again.dW;
        dvals = again.dvals;
        dbias = again.dbias;
      }
    } else {
      dW = Tensor();
    }
    const c10::DeviceGuard guard(saved[1].device());
    auto [w, v, b] = finish(grad, saved[1], dW, dvals, saved[2].scalar_type(), dbias, saved[3].scalar_type());
    return {Tensor(), w, v, b, Tensor(), Tensor()};
  }
};

// The loss alone in the forward, the step with the upstream gradient in the backward (_late_step in ops.py).
struct LateLoss : torch::autograd::Function<LateLoss> {
  static Variable forward(AutogradContext *ctx, const Variable &indices, const Variable &weight, const Variable &vals,
                          const Variable &bias, const Variable &target, const StepPlan &plan) {
    auto [loss, resid] = ::forward(false, {indices, weight, vals, bias, target});
    ctx->save_for_backward({indices, weight, vals, bias, target});
    ctx->set_materialize_grads(false);
    save_plan(ctx, plan);
    if (plan.stats.defined()) ctx->saved_data["stats"] = plan.stats;
    ctx->saved_data["tag"] = plan.tag;
    return loss;
  }

  static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &grad = grads[0];
    if (!grad.defined()) return variable_list(6);
    StepPlan plan = saved_plan(ctx);
    if (!plain_backward(grad) || lists_in_python || !usable_inputs(saved))
      return backward_in_python(ctx, kLate, grad, saved, {plan.need_dw, plan.flags}, nullptr, 6);
    const auto at = ctx->saved_data.find("stats");
    // (a graph under capture would write them again at every replay, as those of the forward's step)
    if (at != ctx->saved_data.end() && !capturing(saved[1])) {
      plan.stats = at->second.toTensor();
      plan.tag = ctx->saved_data["tag"].toInt();
      ctx->saved_data.erase("stats");
    }
    const Step r = hier_step({saved[0], saved[1], saved[2], saved[3], saved[4]}, plan, grad);
    const c10::DeviceGuard guard(saved[1].device());
    auto [w, v, b] = finish(grad, saved[1], Tensor(), r.dvals, saved[2].scalar_type(), r.dbias, saved[3].scalar_type());
    return {Tensor(), r.dW, v, b, Tensor(), Tensor()};
  }
};

// ---- the module ----------------------------------------------------------------------------
bool take_inputs(PyObject *const *args, Inputs &in) {
  Tensor *const to[5] = {&in.indices, &in.weight, &in.vals, &in.bias, &in.target};
  for (int i = 0; i < 5; ++i) {
    if (!THPVariable_CheckExact(args[i])) return false;
    *to[i] = THPVariable_Unpack(args[i]);
  }
  return plain_surroundings() && usable(in);
}

int64_t number(PyObject *o) {
  const int64_t v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) throw_python();
  return v;
}

bool arguments(Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "expected %zd arguments, got %zd", want, n);
  return false;
}

// topk_loss(indices, weight, vals, bias, target) -> loss
PyObject *py_topk_loss(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Inputs in;
  if (!arguments(n, 5)) return nullptr;
  if (!take_inputs(args, in)) Py_RETURN_NONE;
  Tensor loss;
  {
    pybind11::gil_scoped_release no_gil;
    const bool grad = c10::GradMode::is_enabled() && (in.weight.requires_grad() || in.vals.requires_grad() ||
                                                      in.bias.requires_grad() || in.target.requires_grad());
    loss = grad ? TopkLoss::apply(in.indices, in.weight, in.vals, in.bias, in.target) : forward(true, in).first;
  }
  return THPVariable_Wrap(loss);
  END_HANDLE_TH_ERRORS
}

// hier_loss(indices, weight, vals, bias, target, slice_cols) -> loss: forward, and a backward of its own
PyObject *py_hier_loss(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Inputs in;
  if (!arguments(n, 6)) return nullptr;
  if (!take_inputs(args, in)) Py_RETURN_NONE;
  const int64_t cols = number(args[5]);
  Tensor loss;
  {
    pybind11::gil_scoped_release no_gil;
    const bool grad = c10::GradMode::is_enabled() && (in.weight.requires_grad() || in.vals.requires_grad() ||
                                                      in.bias.requires_grad() || in.target.requires_grad());
    loss = grad ? HierLoss::apply(in.indices, in.weight, in.vals, in.bias, in.target, cols) : forward(false, in).first;
  }
  return THPVariable_Wrap(loss);
  END_HANDLE_TH_ERRORS
}

// need_dw (or the step of an update), slice_cols, flags, ws_flags, stats, tag
constexpr Py_ssize_t kPlanArguments = 6;
StepPlan take_plan(PyObject *const *args, bool need_dw) {
  StepPlan plan = {need_dw, number(args[1]), number(args[2]), number(args[3]), Tensor(), number(args[5])};
  if (THPVariable_Check(args[4])) plan.stats = THPVariable_Unpack(args[4]);
  return plan;
}

template <typename Loss>
PyObject *step_loss(PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Inputs in;
  if (!arguments(n, 5 + kPlanArguments)) return nullptr;
  if (!take_inputs(args, in)) Py_RETURN_NONE;
  const StepPlan plan = take_plan(args + 5, number(args[5]) != 0);
  Tensor loss;
  {
    pybind11::gil_scoped_release no_gil;
    loss = Loss::apply(in.indices, in.weight, in.vals, in.bias, in.target, plan);
  }
  return THPVariable_Wrap(loss);
  END_HANDLE_TH_ERRORS
}

// hier_sliced(indices, weight, vals, bias, target, need_dw, slice_cols, flags, ws_flags, stats, tag) -> loss: the training step
PyObject *py_hier_sliced(PyObject *, PyObject *const *args, Py_ssize_t n) { return step_loss<SlicedLoss>(args, n); }
// hier_late(the same): the loss, and the step in the backward
PyObject *py_hier_late(PyObject *, PyObject *const *args, Py_ssize_t n) { return step_loss<LateLoss>(args, n); }

// hier_sgd(indices, weight, vals, bias, target, step, slice_cols, flags, ws_flags, stats, tag) -> (loss, dvals, dbias)
PyObject *py_hier_sgd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Inputs in;
  if (!arguments(n, 5 + kPlanArguments)) return nullptr;
  if (!take_inputs(args, in) || !THPVariable_CheckExact(args[5])) Py_RETURN_NONE;
  const Tensor step = THPVariable_Unpack(args[5]);
  if (!plain_tensor(step) || in.weight.is_inference() || !in.weight.is_contiguous() ||
      reinterpret_cast<uintptr_t>(in.weight.data_ptr()) % 16 || in.weight.size(1) % 4 || in.indices.size(1) > 256)
    Py_RETURN_NONE;
  const StepPlan plan = take_plan(args + 5, true);
  Step r;
  {
    pybind11::gil_scoped_release no_gil;
    const c10::AutoGradMode no_grad(false);
    in.vals = in.vals.detach();
    in.bias = in.bias.detach();
    r = hier_step(in, plan, Tensor(), step);
  }
  return Py_BuildValue("NNN", THPVariable_Wrap(r.loss), THPVariable_Wrap(r.dvals), THPVariable_Wrap(r.dbias));
  END_HANDLE_TH_ERRORS
}

// set_flag(device, flag)
PyObject *py_set_flag(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments(n, 2)) return nullptr;
  const int64_t device = number(args[0]);
  if (device >= 0 && device < kMaxDevices && THPVariable_Check(args[1])) status_flags[device] = THPVariable_Unpack(args[1]);
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// settings(topk_bwd_flags, lists_in_python)
PyObject *py_settings(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments(n, 2)) return nullptr;
  topk_bwd_flags = static_cast<int>(number(args[0]));
  lists_in_python = number(args[1]) != 0;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// init(path of the library, general_backward, raise_status)
PyObject *py_init(PyObject *, PyObject *const *args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (!arguments(n, 3)) return nullptr;
  const char *const path = PyUnicode_AsUTF8(args[0]);
  if (!path) return nullptr;
  void *const handle = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!handle) return PyErr_Format(PyExc_OSError, "%s", dlerror());
#define X(name)                                                                                                  \
  if (!(lib.name = reinterpret_cast<decltype(lib.name)>(dlsym(handle, "flexsae_" #name))))                       \
    return PyErr_Format(PyExc_OSError, "%s does not export flexsae_" #name, path);
  FLEXSAE_ENTRIES(X)
#undef X
  if (lib.abi_version() != FLEXSAE_ABI_VERSION) return PyErr_Format(PyExc_OSError, "%s has another ABI version", path);
  Py_INCREF(args[1]);
  Py_INCREF(args[2]);
  general_backward = args[1];
  raise_status = args[2];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define FLEXSAE_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FLEXSAE_METHOD(init),       FLEXSAE_METHOD(set_flag),    FLEXSAE_METHOD(settings),
                         FLEXSAE_METHOD(topk_loss),  FLEXSAE_METHOD(hier_loss),   FLEXSAE_METHOD(hier_sliced),
                         FLEXSAE_METHOD(hier_late),  FLEXSAE_METHOD(hier_sgd),    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_eager", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// build_id, torch_version: what the module was built from and against, for whoever loads it to compare
PyMODINIT_FUNC PyInit__eager() {
  PyObject *const m = PyModule_Create(&module);
  if (m && (PyModule_AddStringConstant(m, "build_id", FLEXSAE_BUILD_ID) < 0 ||
            PyModule_AddStringConstant(m, "torch_version", FLEXSAE_TORCH_VERSION) < 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
