// The host side of the op and layer calls on GPU tensors, in C++: what nv_norms/ops.py and
// nv_norms/layers.py do in Python (output and workspace allocation, tensor descriptors, the current
// stream, the call of the C ABI, the autograd node), without the interpreter.  At small sizes that
// host work is all a call costs: a forward and a backward op call 47 us through ctypes, 12 us here
// (4.8 and 7.3), a layer's forward without gradients 28 -> 6.5 us.  A layer's forward and its gradients by
// torch.autograd.grad, steps back to back, at [32, 1024] float32: 94 -> 35 us where the engine's thread
// stays awake between steps (torch's own layer_norm: 34 us), 187 -> 62 us where it has to be woken, which
// differs from one process to the next.
//
// Every function here takes the plain case only: exact torch.Tensor (or Parameter) objects,
// contiguous, on one GPU, of a storage type and rank that the C ABI has, with nobody listening to the
// calls (a tracer, a dispatch or torch-function mode, a functorch transform).  For anything else it
// returns None and the caller goes the way it went before, which words the errors; a status of the
// C ABI that is not OK comes back as an int, and the caller raises it.  The autograd node, which has no
// such caller, goes that way itself.
//
// Counterpart in the reference: the OpKernels' Compute methods (fused_layer_norm_op.cc:295-458,
// fused_instance_norm_op.cc:328-534) and the registered gradients (nv_norm_ops.py:27-67).
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SequenceNumber.h>
#include <ATen/TracerMode.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/HIPContextLight.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <ATen/record_function.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/utils/object_ptr.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include <algorithm>
#include <array>
#include <string>
#include <utility>
#include <vector>

#include "../../include/atex_norms.h"

namespace {

// The C ABI, from the library that nv_norms/_capi.py has loaded.
struct Abi {
  decltype(&atexn_last_error) last_error = nullptr;
  decltype(&atexn_layer_norm_resolve_axes) ln_axes = nullptr;
  decltype(&atexn_instance_norm_resolve_format) in_format = nullptr;
  decltype(&atexn_fused_layer_norm_workspace_bytes) ln_fwd_ws = nullptr;
  decltype(&atexn_fused_layer_norm) ln_fwd = nullptr;
  decltype(&atexn_fused_layer_norm_grad_workspace_bytes) ln_bwd_ws = nullptr;
  decltype(&atexn_fused_layer_norm_grad) ln_bwd = nullptr;
  decltype(&atexn_fused_instance_norm_workspace_bytes) in_fwd_ws = nullptr;
  decltype(&atexn_fused_instance_norm) in_fwd = nullptr;
  decltype(&atexn_fused_instance_norm_grad_workspace_bytes) in_bwd_ws = nullptr;
  decltype(&atexn_fused_instance_norm_grad) in_bwd = nullptr;
} g_abi;

template <typename F>
bool bind(void* lib, const char* name, F& f) {
  f = reinterpret_cast<F>(dlsym(lib, name));
  if (f == nullptr) PyErr_Format(PyExc_ImportError, "%s is missing from the library", name);
  return f != nullptr;
}

// Which op, and its attribute: normalised axes (LayerNorm) or data format (InstanceNorm).
struct Attr {
  bool layer_norm = true;
  std::vector<int> axes;
  std::string format;
};

// A valid attribute as a number that a saved_data entry holds without an allocation, and back: how many
// axes, which are the last ones, or whether the channels come first.
int64_t as_number(const Attr& a, int rank) {
  if (!a.layer_norm) return a.format[1] == 'C';
  unsigned seen = 0;
  for (const int v : a.axes) seen |= 1u << (v < 0 ? v + rank : v);
  return __builtin_popcount(seen);
}
Attr from_number(bool layer_norm, int64_t n) {
  Attr a;
  a.layer_norm = layer_norm;
  if (!layer_norm) a.format = n != 0 ? "NC..." : "N...C";
  else for (int64_t i = n; i > 0; --i) a.axes.push_back(static_cast<int>(-i));
  return a;
}

// False: not the plain case.
bool describe(const at::Tensor& t, const c10::Device& device, atexn_tensor& d) {
  if (!t.defined() || t.device() != device || t.layout() != c10::kStrided || !t.has_storage()) return false;
  switch (t.scalar_type()) {
    case at::kFloat: d.dtype = ATEXN_F32; break;
    case at::kHalf: d.dtype = ATEXN_F16; break;
    case at::kBFloat16: d.dtype = ATEXN_BF16; break;
    default: return false;
  }
  const auto sizes = t.sizes();
  if (sizes.size() > ATEXN_MAX_RANK || !t.is_contiguous()) return false;
  d.rank = static_cast<int>(sizes.size());
  for (size_t i = 0; i < sizes.size(); ++i) d.dims[i] = sizes[i];
  d.data = t.numel() != 0 ? t.data_ptr() : nullptr;
  d.device = ATEXN_DEVICE_GPU;
  return true;
}
void describe_new(const at::Tensor& t, atexn_tensor& d) {
  (void)describe(t, t.device(), d);
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType type, const c10::Device& device) {
  return at::Tensor(at::detail::empty_cuda(sizes, type, device, std::nullopt));
}

struct Workspace {
  c10::DataPtr data;
  size_t bytes;
  explicit Workspace(size_t n) : bytes(n) {
    // (of the caching allocator, on the current stream: given back when the call returns, to be
    // used again by what follows on that stream)
    if (n != 0) data = at::cuda::getCUDADeviceAllocator()->allocate(n);
  }
};

struct Result {
  bool plain = true;
  int status = ATEXN_OK;
  std::array<at::Tensor, 3> out;
};

Result forward(const Attr& a, const at::Tensor& x, const at::Tensor& scale, const at::Tensor& offset, float eps) {
  Result r;
  atexn_tensor xd{}, sd{}, od{}, yd{}, md{}, rd{};
  const c10::Device device = x.device();
  if (!device.is_cuda() || !describe(x, device, xd) || !describe(scale, device, sd) || !describe(offset, device, od)) {
    r.plain = false;
    return r;
  }
  const c10::DeviceGuard guard(device);
  std::array<int64_t, 2> stat{};
  int stat_rank = 1;
  const int n_axes = static_cast<int>(a.axes.size());
  if (a.layer_norm) {
    int64_t d = 0;
    r.status = g_abi.ln_axes(xd.rank, xd.dims, a.axes.data(), n_axes, &stat[0], &d);
  } else {
    int layout = 0;
    int64_t d = 0;
    stat_rank = 2;
    r.status = g_abi.in_format(xd.rank, xd.dims, a.format.c_str(), &layout, &stat[0], &stat[1], &d);
  }
  if (r.status != ATEXN_OK) return r;
  const at::IntArrayRef stat_sizes(stat.data(), stat_rank);
  r.out = {empty(x.sizes(), x.scalar_type(), device), empty(stat_sizes, at::kFloat, device),
           empty(stat_sizes, at::kFloat, device)};
  describe_new(r.out[0], yd);
  describe_new(r.out[1], md);
  describe_new(r.out[2], rd);
  void* stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
  if (a.layer_norm) {
    const Workspace ws(g_abi.ln_fwd_ws(&xd, a.axes.data(), n_axes));
    r.status = g_abi.ln_fwd(&xd, &sd, &od, eps, a.axes.data(), n_axes, &yd, &md, &rd, ws.data.get(), ws.bytes, stream);
  } else {
    const Workspace ws(g_abi.in_fwd_ws(&xd, a.format.c_str()));
    r.status = g_abi.in_fwd(&xd, &sd, &od, eps, a.format.c_str(), &yd, &md, &rd, ws.data.get(), ws.bytes, stream);
  }
  return r;
}

Result backward(const Attr& a, const at::Tensor& dy, const at::Tensor& x, const at::Tensor& scale,
                const at::Tensor& mean, const at::Tensor& inv_std) {
  Result r;
  atexn_tensor dyd{}, xd{}, sd{}, md{}, rd{}, dxd{}, dgd{}, dbd{};
  const c10::Device device = x.device();
  if (!device.is_cuda() || !describe(dy, device, dyd) || !describe(x, device, xd) || !describe(scale, device, sd) ||
      !describe(mean, device, md) || !describe(inv_std, device, rd)) {
    r.plain = false;
    return r;
  }
  const c10::DeviceGuard guard(device);
  r.out = {empty(x.sizes(), x.scalar_type(), device), empty(scale.sizes(), at::kFloat, device),
           empty(scale.sizes(), at::kFloat, device)};
  describe_new(r.out[0], dxd);
  describe_new(r.out[1], dgd);
  describe_new(r.out[2], dbd);
  void* stream = c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(device.index()).stream();
  const int n_axes = static_cast<int>(a.axes.size());
  if (a.layer_norm) {
    const Workspace ws(g_abi.ln_bwd_ws(&xd, a.axes.data(), n_axes));
    r.status = g_abi.ln_bwd(&dyd, &xd, &sd, &md, &rd, a.axes.data(), n_axes, &dxd, &dgd, &dbd, ws.data.get(), ws.bytes,
                            stream);
  } else {
    const Workspace ws(g_abi.in_bwd_ws(&xd, a.format.c_str()));
    r.status = g_abi.in_bwd(&dyd, &xd, &sd, &md, &rd, a.format.c_str(), &dxd, &dgd, &dbd, ws.data.get(), ws.bytes, stream);
  }
  return r;
}

// The gradient op through nv_norms/ops.py, for what is not the plain case and for errors, which it words.
std::array<at::Tensor, 3> gradients_in_python(const Attr& a, const at::Tensor& dy, const at::Tensor& x, const at::Tensor& gamma,
                                              const at::Tensor& mean, const at::Tensor& inv_std) {
  const pybind11::gil_scoped_acquire gil;
  auto raise = [] {
    python_error e;
    e.persist();
    throw python_error(std::move(e));
  };
  THPObjectPtr ops(PyImport_ImportModule("atex_amd.nv_norms.ops"));
  if (!ops) raise();
  THPObjectPtr attr(a.layer_norm ? PyList_New(static_cast<Py_ssize_t>(a.axes.size())) : PyUnicode_FromString(a.format.c_str()));
  if (!attr) raise();
  for (size_t i = 0; i < a.axes.size(); ++i) PyList_SET_ITEM(attr.get(), static_cast<Py_ssize_t>(i), PyLong_FromLong(a.axes[i]));
  std::array<THPObjectPtr, 5> t;
  const at::Tensor* const from[5] = {&dy, &x, &gamma, &mean, &inv_std};
  for (int i = 0; i < 5; ++i) {
    t[i] = THPObjectPtr(THPVariable_Wrap(*from[i]));
    if (!t[i]) raise();
  }
  THPObjectPtr out(PyObject_CallMethod(ops.get(), a.layer_norm ? "fused_layer_norm_grad_op" : "fused_instance_norm_grad_op",
                                             "OOOOOO", t[0].get(), t[1].get(), t[2].get(), t[3].get(), t[4].get(), attr.get()));
  if (!out) raise();
  std::array<at::Tensor, 3> r;
  for (int i = 0; i < 3; ++i) r[i] = THPVariable_Unpack(PyTuple_GetItem(out.get(), i));
  return r;
}

// What the gradient's nodes return: n tensors, the first three defined.
torch::autograd::variable_list gradients(const Attr& a, const at::Tensor& grad, const at::Tensor& x, const at::Tensor& gamma,
                                         const at::Tensor& mean, const at::Tensor& inv_std, size_t n) {
  const at::Tensor dy = grad.defined() ? grad.contiguous() : at::zeros_like(x);
  Result r = backward(a, dy, x, gamma, mean, inv_std);
  if (!r.plain || r.status != ATEXN_OK) r.out = gradients_in_python(a, dy, x, gamma, mean, inv_std);
  torch::autograd::variable_list out(n);
  std::move(r.out.begin(), r.out.end(), out.begin());
  return out;
}

// The gradient of y (mean and inv_std are not differentiable) as torch's own C++ autograd function.  It is
// what compiled autograd can take apart; eager backwards go through the node below, which does the same
// in 5 us less (an autograd step of a small layer: 34 us, 40 with this function's node).
template <bool LAYER_NORM>
struct FusedNorm : torch::autograd::Function<FusedNorm<LAYER_NORM>> {
  static constexpr bool is_traceable = false;  // the backward calls the C ABI: data, not proxies

  // y: what the node is attached to
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& gamma,
                            const at::Tensor& /*beta*/, const Attr* a, const at::Tensor* y, const at::Tensor* mean,
                            const at::Tensor* inv_std) {
    ctx->save_for_backward({x, gamma, *mean, *inv_std});
    ctx->set_materialize_grads(false);
    ctx->saved_data["attr"] = as_number(*a, static_cast<int>(x.dim()));
    return *y;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    const torch::autograd::variable_list saved = ctx->get_saved_variables();
    const Attr a = from_number(LAYER_NORM, ctx->saved_data["attr"].toInt());
    return gradients(a, grads[0], saved[0], saved[1], saved[2], saved[3], /*n=*/7);
  }
};

template <bool LAYER_NORM>
struct FusedNormBackward : public torch::autograd::Node {
  Attr attr;
  torch::autograd::SavedVariable x, gamma, mean, inv_std;
  mutable std::shared_ptr<torch::autograd::Node> compiled;  // FusedNorm's node over the same tensors, if asked for

  std::string name() const override { return LAYER_NORM ? "FusedLayerNormBackward" : "FusedInstanceNormBackward"; }
  void release_variables() override {
    std::lock_guard<std::mutex> lock(mutex_);
    x.reset_data();
    gamma.reset_data();
    mean.reset_data();
    inv_std.reset_data();
    if (compiled) compiled->release_variables();
  }
  torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
    std::lock_guard<std::mutex> lock(mutex_);
    const at::Tensor xv = x.unpack(), gv = gamma.unpack(), mv = mean.unpack(), rv = inv_std.unpack();
    return gradients(attr, grads[0], xv, gv, mv, rv, /*n=*/3);
  }
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override {
    if (!compiled) {
      const at::Tensor xv = x.unpack(), gv = gamma.unpack(), mv = mean.unpack(), rv = inv_std.unpack();
      // y and beta stand for tensors that no longer exist: one element in the shape of x, and a value
      // that has a gradient whatever x and gamma have
      const at::Tensor y = at::empty_strided(xv.sizes(), std::vector<int64_t>(xv.dim(), 0), xv.options());
      const at::AutoGradMode on(true);
      compiled = FusedNorm<LAYER_NORM>::apply(xv, gv, at::empty_like(gv).requires_grad_(true), &attr, &y, &mv, &rv).grad_fn();
      compiled->set_next_edges(torch::autograd::edge_list(next_edges()));
    }
    compiled->compiled_args(args);
  }
  torch::autograd::variable_list apply_with_saved(const torch::autograd::variable_list& inputs,
                                                  torch::dynamo::autograd::SwapSavedVariables& saved) override {
    return compiled->apply_with_saved(inputs, saved);
  }
};

// ------------------------------------------------------------------------------ arguments
PyTypeObject* g_device_context = nullptr;  // torch.utils._device.DeviceContext

// Whether a torch-function mode is on that may want to see the calls.  A default device (a with-block of
// torch.device, torch.set_default_device) is such a mode, but one that only completes calls that name no
// device, and there are none.
bool function_mode_watches() {
  if (!at::impl::torch_function_mode_enabled()) return false;
  for (int64_t i = 0; i < at::impl::PythonTorchFunctionTLS::stack_len(); ++i) {
    PyObject* const mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
    if (Py_TYPE(mode) != g_device_context) return true;
  }
  return false;
}
// False: somebody records, intercepts or transforms the calls of this thread.  What is done here
// never reaches the dispatcher, so they would not see it (a traced layer would come out as a
// constant).
bool unobserved() {
  return !at::tracer::impl::is_dispatch_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
         !function_mode_watches();
}
bool tensor_arg(PyObject* o, at::Tensor& t) {
  if (!THPVariable_CheckExact(o)) return false;
  t = THPVariable_Unpack(o);
  return true;
}
bool int_arg(PyObject* o, int& v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long n = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow != 0 || n < INT_MIN || n > INT_MAX) return false;
  v = static_cast<int>(n);
  return true;
}
// The attribute of an op call: a tuple or list of ints, or an int, for LayerNorm's axes; a str for
// InstanceNorm's data format.
template <bool LAYER_NORM>
bool attr_arg(PyObject* o, Attr& a) {
  a.layer_norm = LAYER_NORM;
  if constexpr (!LAYER_NORM) {
    if (!PyUnicode_CheckExact(o)) return false;
    Py_ssize_t n = 0;
    const char* s = PyUnicode_AsUTF8AndSize(o, &n);
    if (s == nullptr) {
      PyErr_Clear();
      return false;
    }
    a.format.assign(s, static_cast<size_t>(n));
    return true;
  } else {
    int v = 0;
    if (int_arg(o, v)) {
      a.axes.assign(1, v);
      return true;
    }
    const bool tuple = PyTuple_CheckExact(o);
    if (!tuple && !PyList_CheckExact(o)) return false;
    const Py_ssize_t n = tuple ? PyTuple_GET_SIZE(o) : PyList_GET_SIZE(o);
    if (n < 1 || n > ATEXN_MAX_RANK) return false;
    a.axes.reserve(static_cast<size_t>(n));
    for (Py_ssize_t i = 0; i < n; ++i) {
      if (!int_arg(tuple ? PyTuple_GET_ITEM(o, i) : PyList_GET_ITEM(o, i), v)) return false;
      a.axes.push_back(v);
    }
    return true;
  }
}
PyObject* answer(Result& r) {
  if (!r.plain) Py_RETURN_NONE;
  if (r.status != ATEXN_OK) return PyLong_FromLong(r.status);
  PyObject* t = PyTuple_New(3);
  if (t == nullptr) return nullptr;
  for (int i = 0; i < 3; ++i) {
    PyObject* o = THPVariable_Wrap(std::move(r.out[i]));
    if (o == nullptr) {
      Py_DECREF(t);
      return nullptr;
    }
    PyTuple_SET_ITEM(t, i, o);
  }
  return t;
}

// *_fwd(x, scale, offset, attribute, epsilon) -> (y, mean, inv_std) | status | None
template <bool LAYER_NORM>
PyObject* norm_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  at::Tensor x, scale, offset;
  Attr a;
  if (n != 5 || !unobserved() || !PyFloat_CheckExact(args[4]) || !tensor_arg(args[0], x) || !tensor_arg(args[1], scale) ||
      !tensor_arg(args[2], offset) || !attr_arg<LAYER_NORM>(args[3], a)) {
    Py_RETURN_NONE;
  }
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[4]));
  Result r;
  {
    pybind11::gil_scoped_release no_gil;
    r = forward(a, x, scale, offset, eps);
  }
  return answer(r);
  END_HANDLE_TH_ERRORS
}

// *_bwd(dy, x, scale, mean, inv_std, attribute) -> (dx, dgamma, dbeta) | status | None
template <bool LAYER_NORM>
PyObject* norm_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  at::Tensor dy, x, scale, mean, inv_std;
  Attr a;
  if (n != 6 || !unobserved() || !tensor_arg(args[0], dy) || !tensor_arg(args[1], x) || !tensor_arg(args[2], scale) ||
      !tensor_arg(args[3], mean) || !tensor_arg(args[4], inv_std) || !attr_arg<LAYER_NORM>(args[5], a)) {
    Py_RETURN_NONE;
  }
  Result r;
  {
    pybind11::gil_scoped_release no_gil;
    r = backward(a, dy, x, scale, mean, inv_std);
  }
  return answer(r);
  END_HANDLE_TH_ERRORS
}

// *_apply(x, gamma, beta, attribute, epsilon): *_fwd with y attached to the autograd graph
template <bool LAYER_NORM>
PyObject* norm_apply(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  at::Tensor x, gamma, beta;
  Attr a;
  if (n != 5 || !unobserved() || !PyFloat_CheckExact(args[4]) || !tensor_arg(args[0], x) || !tensor_arg(args[1], gamma) ||
      !tensor_arg(args[2], beta) || !attr_arg<LAYER_NORM>(args[3], a) || !x.is_cuda()) {
    Py_RETURN_NONE;
  }
  // (forward-mode derivatives are not the node's business: the way round Python refuses them)
  for (const at::Tensor* t : {&x, &gamma, &beta}) {
    if (t->_fw_grad(/*level=*/0).defined()) Py_RETURN_NONE;
  }
  const float eps = static_cast<float>(PyFloat_AS_DOUBLE(args[4]));
  Result r;
  {
    pybind11::gil_scoped_release no_gil;
    // (what a profiler shows of the Python autograd function)
    at::RecordFunction record(at::RecordScope::FUNCTION);
    if (record.isActive()) {
      const char* const name = LAYER_NORM ? "_FusedLayerNormFn" : "_FusedInstanceNormFn";
      const int64_t sequence = static_cast<int64_t>(at::sequence_number::peek());  // the node's, below
      if (record.needsInputs()) {
        const std::array<c10::IValue, 3> inputs{x, gamma, beta};
        record.before(name, c10::ArrayRef<const c10::IValue>(inputs.data(), inputs.size()), sequence);
      } else {
        record.before(name, sequence);
      }
    }
    r = forward(a, x, gamma, beta, eps);
    if (r.plain && r.status == ATEXN_OK && torch::autograd::compute_requires_grad(x, gamma, beta)) {
      auto node = std::shared_ptr<FusedNormBackward<LAYER_NORM>>(new FusedNormBackward<LAYER_NORM>(), torch::autograd::deleteNode);
      node->set_next_edges(torch::autograd::collect_next_edges(x, gamma, beta));
      node->attr = std::move(a);
      node->x = torch::autograd::SavedVariable(x, false);
      node->gamma = torch::autograd::SavedVariable(gamma, false);
      node->mean = torch::autograd::SavedVariable(r.out[1], false);
      node->inv_std = torch::autograd::SavedVariable(r.out[2], false);
      torch::autograd::set_history(r.out[0], node);
    }
  }
  return answer(r);
  END_HANDLE_TH_ERRORS
}

// load(path): the C ABI's library (already in the process)
PyObject* load(PyObject*, PyObject* path) {
  const char* p = PyUnicode_AsUTF8(path);
  if (p == nullptr) return nullptr;
  void* lib = dlopen(p, RTLD_NOW | RTLD_LOCAL);
  if (lib == nullptr) return PyErr_Format(PyExc_ImportError, "%s", dlerror());
  const bool ok = bind(lib, "atexn_last_error", g_abi.last_error) && bind(lib, "atexn_layer_norm_resolve_axes", g_abi.ln_axes) &&
                  bind(lib, "atexn_instance_norm_resolve_format", g_abi.in_format) &&
                  bind(lib, "atexn_fused_layer_norm_workspace_bytes", g_abi.ln_fwd_ws) &&
                  bind(lib, "atexn_fused_layer_norm", g_abi.ln_fwd) &&
                  bind(lib, "atexn_fused_layer_norm_grad_workspace_bytes", g_abi.ln_bwd_ws) &&
                  bind(lib, "atexn_fused_layer_norm_grad", g_abi.ln_bwd) &&
                  bind(lib, "atexn_fused_instance_norm_workspace_bytes", g_abi.in_fwd_ws) &&
                  bind(lib, "atexn_fused_instance_norm", g_abi.in_fwd) &&
                  bind(lib, "atexn_fused_instance_norm_grad_workspace_bytes", g_abi.in_bwd_ws) &&
                  bind(lib, "atexn_fused_instance_norm_grad", g_abi.in_bwd);
  if (!ok) return nullptr;
  THPObjectPtr device(PyImport_ImportModule("torch.utils._device"));
  PyObject* const context = device ? PyObject_GetAttrString(device.get(), "DeviceContext") : nullptr;  // (kept)
  if (context == nullptr) return nullptr;
  g_device_context = reinterpret_cast<PyTypeObject*>(context);
  Py_RETURN_NONE;
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f));
}
PyMethodDef methods[] = {
    {"load", load, METH_O, "load(path): takes the entry points of the C ABI from the library at path."},
    {"layer_norm_fwd", fast(norm_fwd<true>), METH_FASTCALL,
     "layer_norm_fwd(x, scale, offset, axis, epsilon) -> (y, mean, inv_std), a status or None."},
    {"layer_norm_bwd", fast(norm_bwd<true>), METH_FASTCALL,
     "layer_norm_bwd(dy, x, scale, mean, inv_std, axis) -> (dx, dgamma, dbeta), a status or None."},
    {"layer_norm_apply", fast(norm_apply<true>), METH_FASTCALL, "layer_norm_fwd with y attached to the autograd graph."},
    {"instance_norm_fwd", fast(norm_fwd<false>), METH_FASTCALL,
     "instance_norm_fwd(x, scale, offset, data_format, epsilon) -> (y, mean, inv_std), a status or None."},
    {"instance_norm_bwd", fast(norm_bwd<false>), METH_FASTCALL,
     "instance_norm_bwd(dy, x, scale, mean, inv_std, data_format) -> (dx, dgamma, dbeta), a status or None."},
    {"instance_norm_apply", fast(norm_apply<false>), METH_FASTCALL,
     "instance_norm_fwd with y attached to the autograd graph."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_host", "Host side of the fused normalization ops on torch GPU tensors.",
                      -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_host(void) { return PyModule_Create(&module); }
