// PyTorch-side autograd node of the WTConv layer in C++ (host code only; the kernels live behind the C ABI of
// include/wtconv_hip.h, whose entry points this module receives as addresses from the ctypes loader, so that the
// process holds one copy of the library).
//
// Why C++: an eager training step of a small plane spends more time in PyTorch's Python autograd machinery than on
// the GPU -- a torch.autograd.Function with the 9-13 differentiable inputs of this layer (the reference's own
// parameter structure, wtconv/wtconv2d.py:19-31) costs ~13 us of host time per input and pass.  The node below does
// the same work as wtconv_amd/functional.py (_forward_impl / _backward_impl) without the interpreter: allocate
// the outputs, fill the parameter tables, call the library on the current stream.
//
// Only the canonical case is handled here: every parameter on the device of x, contiguous, all in one of the three
// kernel dtypes.  layer() returns None for anything else and the caller takes the Python path, which converts.
#include <torch/extension.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/PyInterpreter.h>

#include <chrono>
#include <mutex>
#include <optional>
#include <vector>

#include "../../include/wtconv_hip.h"
#include "../../include/wtconv_ops.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The C ABI as function pointers (filled once by bind()).
struct Abi {
  int (*fwd2)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwd2)(const void*, const void*, void*, const wtconv_params*, const wtconv_typed_grads*, int, int, int, int, int,
              int, int, int, void*, size_t, void*);
  int (*bwdin2)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwdpar2)(const void*, const void*, const wtconv_params*, const wtconv_typed_grads*, int, int, int, int, int, int,
                 int, int, void*, size_t, void*);
  size_t (*ws2)(int, int, int, int, int, int, int);
  int (*fwd1)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwd1)(const void*, const void*, void*, const wtconv_params*, const wtconv_typed_grads*, int, int, int, int, int,
              int, int, void*, size_t, void*);
  int (*bwdin1)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwdpar1)(const void*, const void*, const wtconv_params*, const wtconv_typed_grads*, int, int, int, int, int, int,
                 int, void*, size_t, void*);
  size_t (*ws1)(int, int, int, int, int, int);
  const char* (*last_error)();
  int (*haar2)(const void*, void*, long long, int, int, int, int, void*);
  int (*haar1)(const void*, void*, long long, int, int, int, void*);
  int (*haar2c)(const void*, void*, long long, int, int, int, int, const void*, int, unsigned*, void*);
  int (*haar1c)(const void*, void*, long long, int, int, int, const void*, int, unsigned*, void*);
  int (*mlp_ok)(int, int, int, int);
  size_t (*mlp_ws)(int, int, int, int);
  int (*mlp)(const void*, const void*, void*, const wtconv_mlp_params*, int, int, int, int, float, int, int, void*, size_t,
             void*);
  int (*patch_ok)(int, int, int, int, int, int);
  size_t (*patch_ws)(int, int, int, int, int, int);
  int (*patch)(int, const void*, void*, const wtconv_patch_params*, int, int, int, int, int, float, int, int, void*, size_t,
               void*);
  int (*mlpt_ok)(long long, int, int);
  int (*mlpt_fwd)(const void*, void*, void*, void*, const wtconv_mlp_params*, long long, int, int, int, int, void*);
  size_t (*mlpt_ws)(long long, int, int, int);
  int (*mlpt_bwd)(const void*, const void*, const void*, const void*, const wtconv_mlp_params*, void*, const wtconv_mlp_grads*,
                  long long, int, int, int, int, void*, size_t, void*);
  int (*norm)(const void*, void*, const void*, const void*, int, int, int, float, int, int, int, void*);
  int (*residual)(const void*, const void*, const void*, void*, int, int, int, int, int, void*);
  size_t (*block_ws)(int, int, int, int);
  int (*norm_bwd)(const void*, const void*, const void*, void*, void*, void*, int, int, int, int, float, int, int, int, void*,
                  size_t, void*);
  int (*residual_bwd)(const void*, const void*, const void*, void*, void*, int, int, int, int, int, int, void*, size_t, void*);
  int (*pool_ok)(int, int, int);
  int (*pool)(const void*, void*, const void*, const void*, int, int, int, float, int, int, void*);
  bool bound = false;
} abi;

template <typename F>
void take(F& slot, uintptr_t addr) { slot = reinterpret_cast<F>(addr); }

// What the look-ups below compare with, imported by bind(): an import within a call could let another thread in while a
// static's initialisation is under way.
struct Python {
  PyObject *module, *device_context, *linear, *gelu;
} python;

// Addresses in the order of the names in wtconv_amd/_ext.py.
void bind(const std::vector<uintptr_t>& a) {
  TORCH_CHECK(a.size() == 32, "bind: expected 32 addresses, got ", a.size());
  take(abi.fwd2, a[0]); take(abi.bwd2, a[1]); take(abi.bwdin2, a[2]); take(abi.bwdpar2, a[3]); take(abi.ws2, a[4]);
  take(abi.fwd1, a[5]); take(abi.bwd1, a[6]); take(abi.bwdin1, a[7]); take(abi.bwdpar1, a[8]); take(abi.ws1, a[9]);
  take(abi.last_error, a[10]);
  take(abi.haar2, a[11]); take(abi.haar1, a[12]); take(abi.haar2c, a[13]); take(abi.haar1c, a[14]);
  take(abi.mlp_ok, a[15]); take(abi.mlp_ws, a[16]); take(abi.mlp, a[17]);
  take(abi.patch_ok, a[18]); take(abi.patch_ws, a[19]); take(abi.patch, a[20]);
  take(abi.mlpt_ok, a[21]); take(abi.mlpt_fwd, a[22]); take(abi.mlpt_ws, a[23]); take(abi.mlpt_bwd, a[24]);
  take(abi.norm, a[25]); take(abi.residual, a[26]); take(abi.block_ws, a[27]); take(abi.norm_bwd, a[28]); take(abi.residual_bwd, a[29]);
  take(abi.pool_ok, a[30]); take(abi.pool, a[31]);
  const py::object nn = py::module_::import("torch.nn");
  python = {py::module_::import("torch.nn.modules.module").release().ptr(),
            py::module_::import("torch.utils._device").attr("DeviceContext").cast<py::object>().release().ptr(),
            nn.attr("Linear").cast<py::object>().release().ptr(), nn.attr("GELU").cast<py::object>().release().ptr()};
  abi.bound = true;
}

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return WTCONV_F32;
    case at::kBFloat16: return WTCONV_BF16;
    case at::kHalf: return WTCONV_F16;
    default: return -1;
  }
}

void fail(int rc, const char* what) {
  const char* msg = abi.last_error ? abi.last_error() : "";
  TORCH_CHECK_VALUE(rc != WTCONV_E_ARG, msg && *msg ? msg : what);
  TORCH_CHECK(false, (msg && *msg) ? msg : what, " (code ", rc, ")");
}

struct Shape { int B, C, H, W; };      // 1-D rows: H = 1, W = N

size_t workspace_bytes(int dims, const Shape& s, int K, int L, int pass) {
  size_t n = dims == 2 ? abi.ws2(s.B, s.C, s.H, s.W, K, L, pass) : abi.ws1(s.B, s.C, s.W, K, L, pass);
  return n < 256 ? 256 : n;
}

template <typename Table>
void fill(Table& t, const Tensor& base_w, const Tensor& base_b, const Tensor& base_s, at::TensorList wt, int L) {
  t = Table{};
  t.base_weight = static_cast<decltype(t.base_weight)>(base_w.data_ptr());
  t.base_bias = base_b.defined() ? static_cast<decltype(t.base_bias)>(base_b.data_ptr()) : nullptr;
  t.base_scale = static_cast<decltype(t.base_scale)>(base_s.data_ptr());
  for (int l = 0; l < L; ++l) {
    t.wt_weight[l] = static_cast<decltype(t.base_weight)>(wt[l].data_ptr());
    t.wt_scale[l] = static_cast<decltype(t.base_weight)>(wt[L + l].data_ptr());
  }
}

// Device memory of one call, given back to PyTorch's stream-ordered allocator when the launches are queued.
c10::DataPtr scratch(const Tensor& like, size_t bytes) { return c10::GetAllocator(like.device().type())->allocate(bytes); }

// A tensor over part of `flat`'s storage (what narrow().view() gives, without two trips through the dispatcher).
Tensor part_of(const Tensor& flat, int64_t at, at::IntArrayRef sizes) {
  Tensor t = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(flat.storage()), flat.key_set(), flat.dtype());
  t.unsafeGetTensorImpl()->set_sizes_contiguous(sizes);
  t.unsafeGetTensorImpl()->set_storage_offset(flat.storage_offset() + at);
  return t;
}

constexpr int kMaxTensors = 3 + 2 * WTCONV_MAX_LEVELS;

// The parameters of a layer: base weight, base bias (may be undefined), base scale, L level weights, L level scales.
struct LayerParams {
  Tensor t[kMaxTensors];
  int L = 0;
  int count() const { return 3 + 2 * L; }
  // values of tensor i
  int64_t numel(int i, int64_t C, int dims, int64_t K) const {
    const int64_t taps = dims == 2 ? K * K : K, S = dims == 2 ? 4 : 2;
    return i == 0 ? C * taps : i < 3 ? C : i < 3 + L ? S * C * taps : S * C;
  }
  at::TensorList levels() const { return at::TensorList(t + 3, 2 * L); }
};

Shape shape_of(const Tensor& x, int dims) {
  return dims == 2 ? Shape{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3)}
                   : Shape{(int)x.size(0), (int)x.size(1), 1, (int)x.size(2)};
}

Tensor layer_forward(const Tensor& x, const LayerParams& lp, int dims, int K) {
  const c10::DeviceGuard guard(x.device());      // (PyTorch on ROCm names the device type "cuda")
  const Shape s = shape_of(x, dims);
  Tensor out = at::empty(x.sizes(), x.options().requires_grad(false));
  const size_t wsz = workspace_bytes(dims, s, K, lp.L, 0);
  const c10::DataPtr ws = scratch(x, wsz);
  wtconv_params p;
  fill(p, lp.t[0], lp.t[1], lp.t[2], lp.levels(), lp.L);
  void* stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  const int dt = dtype_code(x.scalar_type()), pdt = dtype_code(lp.t[0].scalar_type());
  const int rc = dims == 2 ? abi.fwd2(x.const_data_ptr(), out.mutable_data_ptr(), &p, s.B, s.C, s.H, s.W, K, lp.L, dt, pdt,
                                      ws.get(), wsz, stream)
                           : abi.fwd1(x.const_data_ptr(), out.mutable_data_ptr(), &p, s.B, s.C, s.W, K, lp.L, dt, pdt,
                                      ws.get(), wsz, stream);
  if (rc) fail(rc, "wtconv forward");
  return out;
}

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }

// A tensor that a node saved, as the kernels read it: hooks on saved tensors may give it back with other strides, at an
// address of less alignment (`align`: copied then, too), or as another tensor altogether.
[[gnu::noinline, gnu::cold]] void another_came_back(const Tensor& t, const at::Device& dev, at::ScalarType type, int64_t numel) {
  TORCH_CHECK(false, "wtconv backward: ", numel, " values of type ", type, " on ", dev, " were saved, and ", t.numel(), " of type ",
              t.scalar_type(), " on ", t.device(), " came back");
}
inline void make_readable(Tensor& t, const at::Device& dev, at::ScalarType type, int64_t numel, bool align) {
  if (!t.defined()) return;
  if (t.device() != dev || t.scalar_type() != type || t.numel() != numel) another_came_back(t, dev, type, numel);
  if (!t.is_contiguous()) t = t.contiguous();
  if (align && !aligned16(t)) t = t.clone();
}
inline Tensor readable(const torch::autograd::SavedVariable& v, const torch::autograd::Node& node, at::ScalarType type, int64_t numel) {
  Tensor t = v.unpack();
  make_readable(t, node.input_metadata(0).device(), type, numel, true);
  return t;
}

// The type of a node's results: that of the activations.
at::ScalarType made_type(const torch::autograd::Node& node) { return c10::typeMetaToScalarType(node.input_metadata(0).dtype()); }

// Results that come from raw pointers and carry no graph: a derivative of theirs is refused.  (Detached: a result may be the
// caller's own upstream gradient, passed on, whose history is not ours to write.)
void refuse_second_derivatives(variable_list& res, const char* what) {
  for (Tensor& t : res)
    if (t.defined()) {
      t = t.detach();
      auto err = std::make_shared<torch::autograd::Error>(
          std::string("the backward pass of ") + what + " is not differentiable (double backward / create_graph=True through "
          "this layer is not supported)", torch::autograd::edge_list());
      torch::autograd::create_gradient_edge(t, err);
    }
}

// Gradients of x and of the parameters: edges 0 and 1..count() of the node.
struct WTConvNode : public torch::autograd::Node {
  torch::autograd::SavedVariable x_, p_[kMaxTensors];
  int dims_ = 0, K_ = 0, L_ = 0;
  Shape shape_ = {};
  at::ScalarType ptype_ = at::kFloat;

  std::string name() const override { return "WTConvLayerBackward"; }

  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    x_.reset_data();
    for (int i = 0; i < 3 + 2 * L_; ++i) p_[i].reset_data();
  }

  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    const int dims = dims_, K = K_, L = L_;
    const Shape s = shape_;
    const at::Device dev = input_metadata(0).device();
    Tensor x = x_.unpack();
    make_readable(x, dev, made_type(*this), static_cast<int64_t>(s.B) * s.C * s.H * s.W, false);
    LayerParams lp;
    lp.L = L;
    const int n = lp.count();
    for (int i = 0; i < n; ++i) {
      lp.t[i] = p_[i].unpack();
      make_readable(lp.t[i], dev, ptype_, lp.numel(i, s.C, dims, K), false);
    }
    variable_list res(1 + n);
    if (!grads[0].defined()) return res;
    const bool need_x = task_should_compute_output(0);
    bool need_params = false;
    for (int i = 1; i <= n; ++i) need_params = need_params || task_should_compute_output(i);
    if (!need_x && !need_params) return res;
    // Under create_graph=True every result that something differentiable went into is refused a second derivative
    // (the gradients come from raw pointers and carry no graph) instead of being treated as a constant.
    bool twice = false;
    if (at::GradMode::is_enabled()) {
      twice = grads[0].requires_grad() || x.requires_grad();
      for (int i = 0; i < n; ++i) twice = twice || (lp.t[i].defined() && lp.t[i].requires_grad());
    }
    const at::NoGradGuard no_grad;
    Tensor g = grads[0];
    if (g.scalar_type() != x.scalar_type()) g = g.to(x.scalar_type());
    if (!g.is_contiguous()) g = g.contiguous();
    const c10::DeviceGuard guard(x.device());
    const int pass = need_x && need_params ? 3 : (need_x ? 1 : 2);
    const size_t wsz = workspace_bytes(dims, s, K, L, pass);
    const c10::DataPtr ws = scratch(x, wsz);
    wtconv_params p;
    fill(p, lp.t[0], lp.t[1], lp.t[2], lp.levels(), L);
    void* stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    const int dt = dtype_code(x.scalar_type()), pdt = dtype_code(lp.t[0].scalar_type());
    Tensor grad_x;
    if (need_x) grad_x = at::empty(x.sizes(), x.options().requires_grad(false));
    // parameter gradients are written, in the parameters' type, into one flat buffer (one allocation for the 3 + 2 L
    // tensors), of which each parameter gets its part
    int64_t pos[kMaxTensors], total = 0;
    Tensor flat;
    wtconv_typed_grads gt = {};
    gt.dtype = pdt;
    if (need_params) {
      for (int i = 0; i < n; ++i) {
        pos[i] = total;
        if (lp.t[i].defined()) total += lp.t[i].numel();
      }
      flat = at::empty({total}, x.options().dtype(lp.t[0].scalar_type()).requires_grad(false));
      char* f = static_cast<char*>(flat.mutable_data_ptr());
      const size_t size = flat.element_size();
      gt.base_weight = f + pos[0] * size;
      gt.base_bias = lp.t[1].defined() ? f + pos[1] * size : nullptr;
      gt.base_scale = f + pos[2] * size;
      for (int l = 0; l < L; ++l) {
        gt.wt_weight[l] = f + pos[3 + l] * size;
        gt.wt_scale[l] = f + pos[3 + L + l] * size;
      }
    }
    const void *xp = x.const_data_ptr(), *gp = g.const_data_ptr();
    void* gxp = need_x ? grad_x.mutable_data_ptr() : nullptr;
    int rc;
    if (dims == 2) {
      rc = pass == 3   ? abi.bwd2(xp, gp, gxp, &p, &gt, s.B, s.C, s.H, s.W, K, L, dt, pdt, ws.get(), wsz, stream)
           : pass == 1 ? abi.bwdin2(gp, gxp, &p, s.B, s.C, s.H, s.W, K, L, dt, pdt, ws.get(), wsz, stream)
                       : abi.bwdpar2(xp, gp, &p, &gt, s.B, s.C, s.H, s.W, K, L, dt, pdt, ws.get(), wsz, stream);
    } else {
      rc = pass == 3   ? abi.bwd1(xp, gp, gxp, &p, &gt, s.B, s.C, s.W, K, L, dt, pdt, ws.get(), wsz, stream)
           : pass == 1 ? abi.bwdin1(gp, gxp, &p, s.B, s.C, s.W, K, L, dt, pdt, ws.get(), wsz, stream)
                       : abi.bwdpar1(xp, gp, &p, &gt, s.B, s.C, s.W, K, L, dt, pdt, ws.get(), wsz, stream);
    }
    if (rc) fail(rc, "wtconv backward");
    res[0] = std::move(grad_x);
    if (need_params) {
      for (int i = 0; i < n; ++i)
        if (lp.t[i].defined() && task_should_compute_output(1 + i)) res[1 + i] = part_of(flat, pos[i], lp.t[i].sizes());
    }
    if (twice) refuse_second_derivatives(res, "the WTConv layer");
    return res;
  }
};

bool canonical(const Tensor& t, const at::Device& dev, at::ScalarType pd) {
  return t.device() == dev && t.scalar_type() == pd && t.is_contiguous();
}

// The tensors of a list or tuple, as levels lp.t[at...]; false if it is neither or holds anything else.
bool take_levels(PyObject* seq, LayerParams& lp, int L, int at) {
  const bool list = PyList_CheckExact(seq);
  if (!list && !PyTuple_CheckExact(seq)) return false;
  if ((list ? PyList_GET_SIZE(seq) : PyTuple_GET_SIZE(seq)) != L) return false;
  for (int i = 0; i < L; ++i) {
    PyObject* o = list ? PyList_GET_ITEM(seq, i) : PyTuple_GET_ITEM(seq, i);
    if (!THPVariable_Check(o)) return false;
    lp.t[at + i] = THPVariable_Unpack(o);
  }
  return true;
}

// layer(x, base_weight, base_bias or None, base_scale, level weights, level scales, dims, K, L): the layer with its C++
// autograd node, or None when the arguments are not the canonical ones (the caller then takes the Python path, which
// converts what can be converted and says what is wrong with the rest).  A plain CPython function: the argument
// conversions of pybind11 cost more than the checks below.
PyObject* layer(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 9, "layer: expected 9 arguments, got ", nargs);
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  const int dims = static_cast<int>(PyLong_AsLong(args[6]));
  const long K = PyLong_AsLong(args[7]), L = PyLong_AsLong(args[8]);
  if (PyErr_Occurred()) return nullptr;
  if ((dims != 1 && dims != 2) || L < 1 || L > WTCONV_MAX_LEVELS || K < 1 || K % 2 == 0) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i)
    if (!THPVariable_Check(args[i]) && !(i == 2 && args[i] == Py_None)) Py_RETURN_NONE;
  const Tensor& x_in = THPVariable_Unpack(args[0]);
  if (!x_in.is_cuda() || x_in.dim() != dims + 2 || dtype_code(x_in.scalar_type()) < 0 || x_in.numel() == 0) Py_RETURN_NONE;
  LayerParams lp;
  lp.L = static_cast<int>(L);
  lp.t[0] = THPVariable_Unpack(args[1]);
  if (args[2] != Py_None) lp.t[1] = THPVariable_Unpack(args[2]);
  lp.t[2] = THPVariable_Unpack(args[3]);
  if (!take_levels(args[4], lp, lp.L, 3) || !take_levels(args[5], lp, lp.L, 3 + lp.L)) Py_RETURN_NONE;
  const at::ScalarType pd = lp.t[0].scalar_type();
  const at::Device dev = x_in.device();
  if (dtype_code(pd) < 0) Py_RETURN_NONE;
  const int64_t C = x_in.size(1);
  bool record = at::GradMode::is_enabled(), any = x_in.requires_grad();
  for (int i = 0; i < lp.count(); ++i) {
    const Tensor& t = lp.t[i];
    if (!t.defined()) continue;
    if (!canonical(t, dev, pd) || t.numel() != lp.numel(i, C, dims, K) || t._fw_grad(0).defined()) Py_RETURN_NONE;
    any = any || t.requires_grad();
  }
  if (x_in._fw_grad(0).defined()) Py_RETURN_NONE;      // forward-mode differentiation: refused by the Python function
  record = record && any;
  Tensor out;
  {
    const pybind11::gil_scoped_release nogil;
    Tensor x = x_in;
    if (!x.is_contiguous()) {
      const at::NoGradGuard no_grad;
      x = x.contiguous();
    }
    out = layer_forward(x, lp, dims, static_cast<int>(K));
    if (record) {
      const std::shared_ptr<WTConvNode> node(new WTConvNode(), torch::autograd::deleteNode);
      torch::autograd::edge_list next;
      next.reserve(1 + lp.count());
      auto edge = [&](const Tensor& t) {
        next.push_back(t.defined() ? torch::autograd::impl::gradient_edge(t) : torch::autograd::Edge());
      };
      edge(x_in);
      for (int i = 0; i < lp.count(); ++i) edge(lp.t[i]);
      node->set_next_edges(std::move(next));
      node->x_ = torch::autograd::SavedVariable(x, false);
      for (int i = 0; i < lp.count(); ++i) node->p_[i] = torch::autograd::SavedVariable(lp.t[i], false);
      node->dims_ = dims;
      node->K_ = static_cast<int>(K);
      node->L_ = lp.L;
      node->shape_ = shape_of(x, dims);
      node->ptype_ = pd;
      torch::autograd::set_history(out, node);
    }
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- the single-level Haar transforms (wtconv_amd/wavelet.py), with the check of the filter bank they are handed.

// Words of pinned host memory that a kernel writes its verdict into while the caller waits: one page, taken when the
// first bank is checked, its words lent for one call each.  A word that a queued kernel may still write is not lent
// again before that has happened: the next call would take the write for its own kernel's.
class VerdictPool {
 public:
  unsigned* lend() {
    const std::lock_guard<std::mutex> lock(m_);
    if (page_ == nullptr) {
      if (hipHostMalloc(reinterpret_cast<void**>(&page_), kWords * kStride * sizeof(unsigned),
                        hipHostMallocCoherent | hipHostMallocMapped | hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        page_ = nullptr;
        return nullptr;
      }
      for (int i = 0; i < kWords; ++i) free_.push_back(page_ + i * kStride);
    }
    for (size_t i = 0; i < parked_.size();) {
      if (*static_cast<volatile unsigned*>(parked_[i]) == 0u) { ++i; continue; }
      free_.push_back(parked_[i]);
      parked_[i] = parked_.back();
      parked_.pop_back();
    }
    if (free_.empty()) return nullptr;
    unsigned* w = free_.back();
    free_.pop_back();
    *static_cast<volatile unsigned*>(w) = 0u;
    return w;
  }
  void give_back(unsigned* w) {
    const std::lock_guard<std::mutex> lock(m_);
    free_.push_back(w);
  }
  // a word whose kernel has not written it yet, as far as the caller knows
  void park(unsigned* w) {
    const std::lock_guard<std::mutex> lock(m_);
    parked_.push_back(w);
  }

 private:
  static constexpr int kWords = 64, kStride = 16;      // a cache line each
  std::mutex m_;
  unsigned* page_ = nullptr;
  std::vector<unsigned*> free_, parked_;
};
VerdictPool verdicts;

// One call's word: given back when nothing can write it any more, parked otherwise (also when the call throws).
struct VerdictWord {
  unsigned* const w;
  bool settled = false;
  explicit VerdictWord(unsigned* word) : w(word) {}
  VerdictWord(const VerdictWord&) = delete;
  ~VerdictWord() {
    if (settled) verdicts.give_back(w);
    else verdicts.park(w);
  }
};

// Waits for the kernel that writes *w.  It writes early, so this is a short spin; should nothing arrive in two seconds
// (a long queue ahead of it on the stream), the stream is waited for instead.
unsigned await_verdict(const unsigned* w, hipStream_t stream) {
  const volatile unsigned* v = w;
  const auto begin = std::chrono::steady_clock::now();
  for (unsigned spins = 0;; ++spins) {
    if (const unsigned got = *v) return got;
    __builtin_ia32_pause();
    if ((spins & 0xfffu) == 0xfffu && std::chrono::steady_clock::now() - begin > std::chrono::seconds(2)) break;
  }
  TORCH_CHECK(hipStreamSynchronize(stream) == hipSuccess, "the stream failed while a filter bank was being checked");
  return *v;
}

class HaarNode : public torch::autograd::Function<HaarNode> {
 public:
  // bank / verdict: addresses (0 = no check)
  static Tensor forward(AutogradContext* ctx, const Tensor& x, int64_t dims, bool inverse, int64_t bank,
                        int64_t bank_dtype, int64_t verdict) {
    ctx->saved_data["dims"] = dims;
    ctx->saved_data["inverse"] = inverse;
    const c10::DeviceGuard guard(x.device());
    const int64_t b = x.size(0), c = x.size(1);
    const int64_t h = dims == 2 ? (inverse ? 2 * x.size(3) : x.size(2)) : 1;
    const int64_t w = inverse ? 2 * x.size(dims == 2 ? 4 : 3) : x.size(dims == 2 ? 3 : 2);
    Tensor out = dims == 2 ? (inverse ? at::empty({b, c, h, w}, x.options()) : at::empty({b, c, 4, h / 2, w / 2}, x.options()))
                           : (inverse ? at::empty({b, c, w}, x.options()) : at::empty({b, c, 2, w / 2}, x.options()));
    void* stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    const int dt = dtype_code(x.scalar_type());
    int rc;
    if (verdict == 0)
      rc = dims == 2 ? abi.haar2(x.data_ptr(), out.data_ptr(), b * c, h, w, dt, inverse, stream)
                     : abi.haar1(x.data_ptr(), out.data_ptr(), b * c, w, dt, inverse, stream);
    else
      rc = dims == 2 ? abi.haar2c(x.data_ptr(), out.data_ptr(), b * c, h, w, dt, inverse, reinterpret_cast<const void*>(bank),
                                  bank_dtype, reinterpret_cast<unsigned*>(verdict), stream)
                     : abi.haar1c(x.data_ptr(), out.data_ptr(), b * c, w, dt, inverse, reinterpret_cast<const void*>(bank),
                                  bank_dtype, reinterpret_cast<unsigned*>(verdict), stream);
    if (rc) fail(rc, "wtconv haar");
    return out;
  }

  // The transforms are orthogonal: each one's backward is the other.
  static variable_list backward(AutogradContext* ctx, variable_list grad_outputs) {
    variable_list res(6);
    if (grad_outputs[0].defined())
      res[0] = HaarNode::apply(grad_outputs[0].contiguous(), ctx->saved_data["dims"].toInt(),
                               !ctx->saved_data["inverse"].toBool(), int64_t{0}, int64_t{0}, int64_t{0});
    return res;
  }
};

// The transform of a contiguous GPU tensor.  With a bank: the result if it is db1's, False if it is another one, None
// if it is not one that a kernel can look at (host memory, another dtype, strided) and nothing was done.
py::object haar(const Tensor& x, const std::optional<Tensor>& bank, int64_t dims, bool inverse) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (!bank.has_value()) {
    Tensor out;
    {
      py::gil_scoped_release nogil;
      out = HaarNode::apply(x, dims, inverse, int64_t{0}, int64_t{0}, int64_t{0});
    }
    return py::cast(out);
  }
  const int bdt = dtype_code(bank->scalar_type());
  if (bdt < 0 || bank->device() != x.device() || !bank->is_contiguous() || x.numel() == 0) return py::none();
  if (x._fw_grad(0).defined()) return py::none();      // (refused, but only behind the launch)
  const hipStream_t stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
  hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
  TORCH_CHECK(hipStreamIsCapturing(stream, &capturing) == hipSuccess && capturing == hipStreamCaptureStatusNone,
              "a filter bank in GPU memory cannot be checked while the stream is being captured");
  unsigned* w = verdicts.lend();
  if (w == nullptr) return py::none();
  Tensor out;
  unsigned got;
  {
    py::gil_scoped_release nogil;
    VerdictWord word(w);
    try {
      out = HaarNode::apply(x, dims, inverse, reinterpret_cast<int64_t>(bank->data_ptr()), int64_t{bdt},
                            reinterpret_cast<int64_t>(w));
    } catch (...) {      // (the kernel may have been queued)
      word.settled = hipStreamSynchronize(stream) == hipSuccess;
      if (!word.settled) (void)hipGetLastError();
      throw;
    }
    got = await_verdict(w, stream);
    word.settled = true;
  }
  if (got != 1u) return py::bool_(false);
  return py::cast(out);
}

// The block behind its WTConv layer in one kernel (inference): undefined if the kernels do not take these tensors, or autograd
// would record the call.  b1, b2 and gamma may be undefined.
Tensor fused_mlp(const Tensor& x, const Tensor& shortcut, const Tensor& norm_w, const Tensor& norm_b, double eps, const Tensor& w1,
                 const Tensor& b1, const Tensor& w2, const Tensor& b2, const Tensor& gamma) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (x.dim() != 4 || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || !x.is_contiguous()) return Tensor();
  if (shortcut.sizes() != x.sizes() || !b1.defined() || !b2.defined()) return Tensor();
  const int64_t B = x.size(0), C = x.size(1), HW = x.size(2) * x.size(3);
  if (w1.dim() != 2 || w2.dim() != 2 || w1.size(1) != C || w2.size(0) != C || w1.size(0) != w2.size(1)) return Tensor();
  const int64_t hidden = w1.size(0);
  if (norm_w.numel() != C || norm_b.numel() != C || b1.numel() != hidden || b2.numel() != C) return Tensor();
  if (gamma.defined() && gamma.numel() != C) return Tensor();
  const bool grad = at::GradMode::is_enabled();
  if (grad && x.requires_grad()) return Tensor();
  if (x._fw_grad(0).defined()) return Tensor();
  uintptr_t bits = 0;
  for (const Tensor* t : {&shortcut, &norm_w, &norm_b, &w1, &b1, &w2, &b2, &gamma}) {
    if (!t->defined()) continue;
    if (!canonical(*t, x.device(), at::kBFloat16) || (grad && t->requires_grad()) || t->_fw_grad(0).defined()) return Tensor();
    if (t != &shortcut) bits |= reinterpret_cast<uintptr_t>(t->const_data_ptr());
  }
  if (bits % 16 || x.numel() == 0 || B * HW > (1LL << 30) || !abi.mlp_ok(B, C, HW, hidden)) return Tensor();
  const c10::DeviceGuard guard(x.device());
  Tensor out = at::empty(x.sizes(), x.options());
  const size_t wsz = abi.mlp_ws(B, C, HW, hidden);
  c10::DataPtr ws;
  if (wsz) ws = scratch(x, wsz);
  const wtconv_mlp_params p = {norm_w.const_data_ptr(), norm_b.const_data_ptr(), w1.const_data_ptr(), b1.const_data_ptr(),
                               w2.const_data_ptr(), b2.const_data_ptr(), gamma.defined() ? gamma.const_data_ptr() : nullptr};
  const int rc = abi.mlp(x.const_data_ptr(), shortcut.const_data_ptr(), out.mutable_data_ptr(), &p, B, C, HW, hidden,
                         static_cast<float>(eps), WTCONV_BF16, WTCONV_BF16, ws.get(), wsz,
                         c10::hip::getCurrentHIPStream(x.device().index()).stream());
  if (rc) fail(rc, "wtconv block mlp");
  return out;
}

// (x, shortcut, norm weight, norm bias, eps, fc1 weight, fc1 bias, fc2 weight, fc2 bias, gamma)
PyObject* block_mlp(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 10, "block_mlp: expected 10 arguments, got ", nargs);
  Tensor t[10];
  for (int i = 0; i < 10; ++i) {
    if (i == 4 || (args[i] == Py_None && (i == 6 || i == 8 || i == 9))) continue;
    TORCH_CHECK_TYPE(THPVariable_Check(args[i]), "block_mlp: argument ", i, " is no tensor");
    t[i] = THPVariable_Unpack(args[i]);
  }
  const double eps = PyFloat_AsDouble(args[4]);
  if (eps == -1. && PyErr_Occurred()) return nullptr;
  const Tensor out = fused_mlp(t[0], t[1], t[2], t[3], eps, t[5], t[6], t[7], t[8], t[9]);
  if (!out.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

// ---- modules, looked into without the interpreter: a block at inference asks for some forty attributes, which cost as much
// host time as two launches (one image, 14 x 14 x 384: a block 20.9 -> 16.3 us of host time, of these the MLP 11.9 -> 8.1;
// WTConvNeXt-T on one image, which the host bounds, 500 -> 442 us).

// A name that lives as long as the process.
PyObject* name_of(const char* s) { return PyUnicode_InternFromString(s); }

// A module's own attributes (borrowed); nullptr if it has none.
PyObject* own_dict(PyObject* module) {
  PyObject** at = _PyObject_GetDictPtr(module);
  return at != nullptr && *at != nullptr && PyDict_Check(*at) ? *at : nullptr;
}

// module.<name>, an ordinary parameter or sub-module (of the dict `kind`) first, else as Python looks it up; throws.
py::object member(PyObject* module, PyObject* kind, PyObject* name) {
  if (PyObject* own = own_dict(module))
    if (PyObject* of = PyDict_GetItemWithError(own, kind))
      if (PyDict_Check(of))
        if (PyObject* v = PyDict_GetItemWithError(of, name))
          if (v != Py_None) return py::reinterpret_borrow<py::object>(v);
  if (PyErr_Occurred()) throw py::error_already_set();
  PyObject* v = PyObject_GetAttr(module, name);
  if (v == nullptr) throw py::error_already_set();
  return py::reinterpret_steal<py::object>(v);
}
py::object parameter(PyObject* module, PyObject* name) {
  static PyObject* const kind = name_of("_parameters");
  return member(module, kind, name);
}
py::object submodule(PyObject* module, PyObject* name) {
  static PyObject* const kind = name_of("_modules");
  return member(module, kind, name);
}

// An attribute that the module itself holds, or as Python looks it up; throws.
py::object attribute(PyObject* module, PyObject* name) {
  if (PyObject* own = own_dict(module))
    if (PyObject* v = PyDict_GetItemWithError(own, name)) return py::reinterpret_borrow<py::object>(v);
  if (PyErr_Occurred()) throw py::error_already_set();
  PyObject* v = PyObject_GetAttr(module, name);
  if (v == nullptr) throw py::error_already_set();
  return py::reinterpret_steal<py::object>(v);
}

bool truth(PyObject* o) {
  const int t = PyObject_IsTrue(o);
  if (t < 0) throw py::error_already_set();
  return t != 0;
}

// Whether something expects to see these modules called, or the functions they call: hooks of the modules or of all
// modules, a `forward` put on a module itself, a dispatch or function mode (FLOP counters, tracers).  The function mode
// of a default device only looks at factory functions.
bool watched_modules(PyObject* const* modules, Py_ssize_t n) {
  static PyObject* const all[] = {name_of("_global_forward_hooks"), name_of("_global_forward_pre_hooks")};
  static PyObject* const one[] = {name_of("_forward_hooks"), name_of("_forward_pre_hooks")};
  static PyObject* const forward = name_of("forward");
  for (PyObject* name : all) {
    const py::object hooks = py::reinterpret_steal<py::object>(PyObject_GetAttr(python.module, name));
    if (!hooks) throw py::error_already_set();
    if (truth(hooks.ptr())) return true;
  }
  if (c10::impl::TorchDispatchModeTLS::stack_len()) return true;
  for (Py_ssize_t i = 0; i < n; ++i) {
    for (PyObject* name : one)
      if (truth(attribute(modules[i], name).ptr())) return true;
    PyObject* own = own_dict(modules[i]);
    if (own == nullptr) return true;
    const int has = PyDict_Contains(own, forward);
    if (has < 0) throw py::error_already_set();
    if (has) return true;
  }
  for (int64_t i = 0, m = at::impl::PythonTorchFunctionTLS::stack_len(); i < m; ++i) {
    PyObject* mode = at::impl::PythonTorchFunctionTLS::get_stack_at(i)->ptr(getPyInterpreter());
    if (reinterpret_cast<PyObject*>(Py_TYPE(mode)) != python.device_context) return true;
  }
  return false;
}

PyObject* watched(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  return PyBool_FromLong(watched_modules(args, nargs));
  END_HANDLE_TH_ERRORS
}

// Base weight, bias and scale, level weights and level scales of a WTConv2d / WTConv1d, as layer() takes them; None if the
// module is built another way (lists of modules that are no plain dicts).  A look-up of a parameter may run Python code
// (parametrizations), and that may replace any sub-module, or let another thread do so: a part is looked up in its turn, in
// the order in which Python reads them, and held while it is read.
PyObject* layer_params(PyObject*, PyObject* module) {
  HANDLE_TH_ERRORS
  static PyObject* const modules = name_of("_modules");
  static PyObject* const weight = name_of("weight");
  static PyObject* const bias = name_of("bias");
  static PyObject* const parts[] = {name_of("base_conv"), name_of("base_scale"), name_of("wavelet_convs"), name_of("wavelet_scale")};
  auto held = [](PyObject* borrowed) {
    if (borrowed == nullptr && PyErr_Occurred()) throw py::error_already_set();
    return py::reinterpret_borrow<py::object>(borrowed);
  };
  auto dict_of = [&](PyObject* m) -> py::object {
    PyObject* own = own_dict(m);
    const py::object of = own != nullptr ? held(PyDict_GetItemWithError(own, modules)) : py::object();
    return of && PyDict_CheckExact(of.ptr()) ? of : py::object();
  };
  const py::object sub = dict_of(module);
  auto part = [&](int i) { return held(PyDict_GetItemWithError(sub.ptr(), parts[i])); };
  auto list = [&](int i) {
    const py::object p = part(i);
    return p ? dict_of(p.ptr()) : py::object();
  };
  if (!sub || !part(0) || !part(1) || !list(2) || !list(3)) Py_RETURN_NONE;
  const py::object base = part(0), base_w = parameter(base.ptr(), weight), base_b = parameter(base.ptr(), bias);
  const py::object scale = part(1);
  if (!scale) Py_RETURN_NONE;
  const py::object base_s = parameter(scale.ptr(), weight);
  py::object levels[2];
  for (int k = 0; k < 2; ++k) {
    const py::object dict = list(2 + k);
    if (!dict) Py_RETURN_NONE;
    const py::object of = py::reinterpret_steal<py::object>(PyDict_Values(dict.ptr()));
    if (!of) throw py::error_already_set();
    const Py_ssize_t n = PyList_GET_SIZE(of.ptr());
    levels[k] = py::reinterpret_steal<py::object>(PyList_New(n));
    if (!levels[k]) throw py::error_already_set();
    for (Py_ssize_t i = 0; i < n; ++i)
      PyList_SET_ITEM(levels[k].ptr(), i, parameter(PyList_GET_ITEM(of.ptr(), i), weight).release().ptr());
  }
  return PyTuple_Pack(5, base_w.ptr(), base_b.ptr(), base_s.ptr(), levels[0].ptr(), levels[1].ptr());
  END_HANDLE_TH_ERRORS
}

// What block_mlp() is called with, from (x, shortcut, norm, mlp, gamma); None where the block's passes have to be the modules'
// own: another activation than the exact GELU, observers, a tensor of a subclass, a LayerNorm without parameters.
PyObject* mlp_args(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 5, "mlp_args: expected 5 arguments, got ", nargs);
  static PyObject* const weight = name_of("weight");
  static PyObject* const bias = name_of("bias");
  static PyObject* const parts[] = {name_of("fc1"), name_of("act"), name_of("fc2")};
  static PyObject* const approximate = name_of("approximate");
  static PyObject* const eps_name = name_of("eps");
  PyObject *norm = args[2], *mlp = args[3];
  const py::object fc1 = submodule(mlp, parts[0]), act = submodule(mlp, parts[1]), fc2 = submodule(mlp, parts[2]);
  auto is = [](const py::object& o, PyObject* type) { return reinterpret_cast<PyObject*>(Py_TYPE(o.ptr())) == type; };
  if (!is(fc1, python.linear) || !is(fc2, python.linear) || !is(act, python.gelu)) Py_RETURN_NONE;
  const py::object kind = attribute(act.ptr(), approximate);
  if (!PyUnicode_Check(kind.ptr()) || PyUnicode_CompareWithASCIIString(kind.ptr(), "none") != 0) Py_RETURN_NONE;
  PyObject* modules[] = {norm, mlp, fc1.ptr(), act.ptr(), fc2.ptr()};
  if (watched_modules(modules, 5)) Py_RETURN_NONE;
  const py::object found[] = {parameter(norm, weight),      parameter(norm, bias),      attribute(norm, eps_name),
                              parameter(fc1.ptr(), weight), parameter(fc1.ptr(), bias), parameter(fc2.ptr(), weight),
                              parameter(fc2.ptr(), bias)};
  PyObject* given[] = {args[0], args[1], found[0].ptr(), found[1].ptr(), found[2].ptr(), found[3].ptr(), found[4].ptr(), found[5].ptr(),
                       found[6].ptr(), args[4]};
  if (given[2] == Py_None || given[3] == Py_None) Py_RETURN_NONE;
  for (int i = 0; i < 10; ++i)
    if (i != 4 && given[i] != Py_None && !THPVariable_CheckExact(given[i])) Py_RETURN_NONE;
  PyObject* out = PyTuple_New(10);
  if (out == nullptr) throw py::error_already_set();
  for (int i = 0; i < 10; ++i) {
    Py_INCREF(given[i]);
    PyTuple_SET_ITEM(out, i, given[i]);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// ---- a block's MLP in training: fc2(gelu(fc1(x))) over the last extent of x.

// Gradients of x, fc1's weight and bias, fc2's weight and bias: edges 0..4 of the node.
struct MlpNode : public torch::autograd::Node {
  torch::autograd::SavedVariable x_, w1_, b1_, w2_, h_, act_;
  int64_t pixels_ = 0, C_ = 0, hidden_ = 0;
  bool twice_ = false;      // whether second derivatives are answered

  std::string name() const override { return "WTConvMlpBackward"; }

  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    for (auto* v : {&x_, &w1_, &b1_, &w2_, &h_, &act_}) v->reset_data();
  }

  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    const int64_t C = C_, hidden = hidden_, pixels = pixels_;
    auto saved = [&](const torch::autograd::SavedVariable& v, int64_t numel) { return readable(v, *this, at::kBFloat16, numel); };
    const Tensor x = saved(x_, pixels * C), w1 = saved(w1_, hidden * C), w2 = saved(w2_, C * hidden), h = saved(h_, pixels * hidden),
                 act = saved(act_, pixels * hidden);
    variable_list res(5);
    if (!grads[0].defined()) return res;
    const bool need_x = task_should_compute_output(0);
    const bool need_1 = task_should_compute_output(1) || task_should_compute_output(2);
    const bool need_2 = task_should_compute_output(3) || task_should_compute_output(4);
    if (!need_x && !need_1 && !need_2) return res;
    const bool twice = at::GradMode::is_enabled() &&
                       (grads[0].requires_grad() || x.requires_grad() || w1.requires_grad() || w2.requires_grad());
    if (twice && twice_) return recorded(grads[0].to(x.scalar_type()), x, w1, b1_.unpack(), w2);
    const at::NoGradGuard no_grad;
    Tensor g = grads[0];
    if (g.scalar_type() != x.scalar_type()) g = g.to(x.scalar_type());
    if (!g.is_contiguous()) g = g.contiguous();
    if (!aligned16(g)) g = g.clone();
    const c10::DeviceGuard guard(x.device());
    const int want = (need_x ? WTCONV_MLP_DX : 0) | (need_1 ? WTCONV_MLP_FC1 : 0) | (need_2 ? WTCONV_MLP_FC2 : 0);
    const size_t wsz = abi.mlpt_ws(pixels, C, hidden, want);
    const c10::DataPtr ws = scratch(x, wsz);
    if (need_x) res[0] = at::empty(x.sizes(), x.options().requires_grad(false));
    // (one allocation for the parameters' gradients; their sizes are multiples of 32)
    const int64_t sizes[4] = {hidden * C, hidden, C * hidden, C};
    Tensor flat = at::empty({(need_1 ? sizes[0] + sizes[1] : 0) + (need_2 ? sizes[2] + sizes[3] : 0)}, x.options().requires_grad(false));
    void* to[4] = {nullptr, nullptr, nullptr, nullptr};
    int64_t pos[4], at_elem = 0;
    for (int i = 0; i < 4; ++i) {
      pos[i] = at_elem;
      if (i < 2 ? !need_1 : !need_2) continue;
      to[i] = static_cast<at::BFloat16*>(flat.mutable_data_ptr()) + at_elem;
      at_elem += sizes[i];
    }
    const wtconv_mlp_params p = {nullptr, nullptr, w1.const_data_ptr(), nullptr, w2.const_data_ptr(), nullptr, nullptr};
    const wtconv_mlp_grads gt = {to[0], to[1], to[2], to[3]};
    const int rc = abi.mlpt_bwd(x.const_data_ptr(), h.const_data_ptr(), act.const_data_ptr(), g.const_data_ptr(), &p,
                                need_x ? res[0].mutable_data_ptr() : nullptr, &gt, pixels, C, hidden, WTCONV_BF16, WTCONV_BF16,
                                ws.get(), wsz, c10::hip::getCurrentHIPStream(x.device().index()).stream());
    if (rc) fail(rc, "wtconv mlp backward");
    for (int i = 0; i < 4; ++i)
      if (task_should_compute_output(1 + i))
        res[1 + i] = i == 0 ? part_of(flat, pos[0], {hidden, C}) : i == 2 ? part_of(flat, pos[2], {C, hidden}) : part_of(flat, pos[i], {sizes[i]});
    if (twice) refuse_second_derivatives(res, "the block's MLP");
    return res;
  }

  // The gradients by operators that autograd records, all of them products of two matrices.
  variable_list recorded(const Tensor& g_in, const Tensor& x_in, const Tensor& w1, const Tensor& b1, const Tensor& w2) {
    const Tensor g = g_in.reshape({pixels_, C_}), x = x_in.reshape({pixels_, C_});
    const Tensor h = at::addmm(b1, x, w1.t()), dh = at::gelu_backward(at::mm(g, w2), h);
    variable_list res(5);
    if (task_should_compute_output(0)) res[0] = at::mm(dh, w1).reshape(x_in.sizes());
    if (task_should_compute_output(1)) res[1] = at::mm(dh.t(), x);
    if (task_should_compute_output(2)) res[2] = dh.sum(0);
    if (task_should_compute_output(3)) res[3] = at::mm(g.t(), at::gelu(h));
    if (task_should_compute_output(4)) res[4] = g.sum(0);
    return res;
  }
};

// The MLP with its C++ autograd node, where autograd records it: None otherwise, or if there are no kernels for these arguments.
// `twice`: second derivatives are answered, not refused.
py::object mlp(const Tensor& x, const Tensor& w1, const Tensor& b1, const Tensor& w2, const Tensor& b2, bool twice) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (!at::GradMode::is_enabled() || x.dim() < 2 || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || !x.is_contiguous() || x.numel() == 0)
    return py::none();
  if (w1.dim() != 2 || w2.dim() != 2 || w1.size(1) != x.size(-1) || w2.size(0) != x.size(-1) || w1.size(0) != w2.size(1)) return py::none();
  const int64_t C = w1.size(1), hidden = w1.size(0), pixels = x.numel() / C;
  if (b1.numel() != hidden || b2.numel() != C || !abi.mlpt_ok(pixels, C, hidden)) return py::none();
  bool any = x.requires_grad();
  for (const Tensor* t : {&w1, &b1, &w2, &b2}) {
    if (!canonical(*t, x.device(), at::kBFloat16) || !aligned16(*t) || t->_fw_grad(0).defined()) return py::none();
    any = any || t->requires_grad();
  }
  if (!any || !aligned16(x) || x._fw_grad(0).defined()) return py::none();
  Tensor y;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(x.device());
    Tensor h, act;
    {
      const at::NoGradGuard no_grad;
      std::vector<int64_t> wide = x.sizes().vec();
      wide.back() = hidden;
      const at::TensorOptions opt = x.options().requires_grad(false);
      y = at::empty(x.sizes(), opt);
      h = at::empty(wide, opt);
      act = at::empty(wide, opt);
    }
    const wtconv_mlp_params p = {nullptr, nullptr, w1.const_data_ptr(), b1.const_data_ptr(), w2.const_data_ptr(), b2.const_data_ptr(), nullptr};
    const int rc = abi.mlpt_fwd(x.const_data_ptr(), h.mutable_data_ptr(), act.mutable_data_ptr(), y.mutable_data_ptr(), &p, pixels, C,
                                hidden, WTCONV_BF16, WTCONV_BF16, c10::hip::getCurrentHIPStream(x.device().index()).stream());
    if (rc) fail(rc, "wtconv mlp forward");
    const std::shared_ptr<MlpNode> node(new MlpNode(), torch::autograd::deleteNode);
    torch::autograd::edge_list next;
    next.reserve(5);
    for (const Tensor* t : {&x, &w1, &b1, &w2, &b2}) next.push_back(torch::autograd::impl::gradient_edge(*t));
    node->set_next_edges(std::move(next));
    node->x_ = torch::autograd::SavedVariable(x, false);
    node->w1_ = torch::autograd::SavedVariable(w1, false);
    if (twice) node->b1_ = torch::autograd::SavedVariable(b1, false);
    node->w2_ = torch::autograd::SavedVariable(w2, false);
    node->h_ = torch::autograd::SavedVariable(h, false);
    node->act_ = torch::autograd::SavedVariable(act, false);
    node->twice_ = twice;
    node->pixels_ = pixels;
    node->C_ = C;
    node->hidden_ = hidden;
    torch::autograd::set_history(y, node);
  }
  return py::cast(y);
}

// ---- the two passes a block makes around its WTConv layer: LayerNorm over the channels of x (B, C, H, W), to (B, H, W, C) or
// (B, C, H, W), and shortcut (B, C, H, W) + gamma * y (B, H, W, C).

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

bool block_dtype(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }

c10::DataPtr block_workspace(const Tensor& x, size_t* bytes) {
  *bytes = abi.block_ws(x.size(0), x.size(1), x.size(2) * x.size(3), dtype_code(x.scalar_type()));
  TORCH_CHECK(*bytes > 0, "block backward: no tile plan for C=", x.size(1), ", HW=", x.size(2) * x.size(3));
  return scratch(x, *bytes);
}

// The upstream gradient as the kernels take it (zeros where there is none).
Tensor upstream(const Tensor& g, at::IntArrayRef sizes, const at::TensorOptions& opt) {
  if (!g.defined()) return at::zeros(sizes, opt);
  const Tensor t = g.scalar_type() == c10::typeMetaToScalarType(opt.dtype()) ? g : g.to(opt.dtype());
  return t.contiguous();
}

// Gradients of x, weight and bias: edges 0..2 of the node.
struct NormNode : public torch::autograd::Node {
  torch::autograd::SavedVariable x_, weight_;
  int64_t B_ = 0, C_ = 0, H_ = 0, W_ = 0;
  at::ScalarType ptype_ = at::kFloat;
  double eps_ = 0;
  bool nhwc_ = false;

  std::string name() const override { return "WTConvChannelNormBackward"; }

  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    x_.reset_data();
    weight_.reset_data();
  }

  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    const int64_t B = B_, C = C_, H = H_, W = W_;
    const Tensor x = readable(x_, *this, made_type(*this), B * C * H * W), weight = readable(weight_, *this, ptype_, C);
    const bool twice = at::GradMode::is_enabled() &&
                       ((grads[0].defined() && grads[0].requires_grad()) || x.requires_grad() || weight.requires_grad());
    const at::NoGradGuard no_grad;
    const c10::DeviceGuard guard(x.device());
    const at::TensorOptions opt = x.options().requires_grad(false);
    const Tensor g = nhwc_ ? upstream(grads[0], {B, H, W, C}, opt) : upstream(grads[0], {B, C, H, W}, opt);
    Tensor dx = at::empty(x.sizes(), opt), flat = at::empty({2 * C}, weight.options().requires_grad(false));
    size_t wsz;
    const c10::DataPtr ws = block_workspace(x, &wsz);
    char* f = static_cast<char*>(flat.mutable_data_ptr());
    const int pdt = dtype_code(weight.scalar_type());
    const int rc = abi.norm_bwd(x.const_data_ptr(), g.const_data_ptr(), weight.const_data_ptr(), dx.mutable_data_ptr(), f,
                                f + C * flat.element_size(), pdt, B, C, H * W, static_cast<float>(eps_),
                                dtype_code(x.scalar_type()), pdt, nhwc_, ws.get(), wsz, stream_of(x));
    if (rc) fail(rc, "wtconv channel norm backward");
    variable_list res(3);
    if (task_should_compute_output(0)) res[0] = std::move(dx);
    for (int i = 0; i < 2; ++i)
      if (task_should_compute_output(1 + i)) res[1 + i] = part_of(flat, i * C, weight.sizes());
    if (twice) refuse_second_derivatives(res, "the channel norm");
    return res;
  }
};

// LayerNorm over the channels; None if the kernels do not take these arguments.
py::object channel_norm(const Tensor& x, const Tensor& weight, const Tensor& bias, double eps, bool nhwc) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (!x.is_cuda() || x.dim() != 4 || !block_dtype(x.scalar_type()) || !x.is_contiguous() || x.numel() == 0) return py::none();
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3);
  for (const Tensor* t : {&weight, &bias})
    if (!canonical(*t, x.device(), weight.scalar_type()) || !block_dtype(t->scalar_type()) || t->numel() != C || t->dim() != 1 ||
        t->_fw_grad(0).defined())
      return py::none();
  if (x._fw_grad(0).defined()) return py::none();
  const bool record = at::GradMode::is_enabled() && (x.requires_grad() || weight.requires_grad() || bias.requires_grad());
  Tensor out;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(x.device());
    const at::TensorOptions opt = x.options().requires_grad(false);
    out = nhwc ? at::empty({B, H, W, C}, opt) : at::empty({B, C, H, W}, opt);
    const int rc = abi.norm(x.const_data_ptr(), out.mutable_data_ptr(), weight.const_data_ptr(), bias.const_data_ptr(), B, C, H * W,
                            static_cast<float>(eps), dtype_code(x.scalar_type()), dtype_code(weight.scalar_type()), nhwc, stream_of(x));
    if (rc) fail(rc, "wtconv channel norm");
    if (record) {
      const std::shared_ptr<NormNode> node(new NormNode(), torch::autograd::deleteNode);
      torch::autograd::edge_list next;
      next.reserve(3);
      for (const Tensor* t : {&x, &weight, &bias}) next.push_back(torch::autograd::impl::gradient_edge(*t));
      node->set_next_edges(std::move(next));
      node->x_ = torch::autograd::SavedVariable(x, false);
      node->weight_ = torch::autograd::SavedVariable(weight, false);
      node->B_ = B;
      node->C_ = C;
      node->H_ = H;
      node->W_ = W;
      node->ptype_ = weight.scalar_type();
      node->eps_ = eps;
      node->nhwc_ = nhwc;
      torch::autograd::set_history(out, node);
    }
  }
  return py::cast(out);
}

// Gradients of y, shortcut and gamma: edges 0..2 of the node.
struct ResidualNode : public torch::autograd::Node {
  torch::autograd::SavedVariable y_, gamma_;
  int64_t B_ = 0, C_ = 0, H_ = 0, W_ = 0;
  at::ScalarType ptype_ = at::kFloat;

  std::string name() const override { return "WTConvBlockResidualBackward"; }

  void release_variables() override {
    const std::lock_guard<std::mutex> lock(mutex_);
    y_.reset_data();
    gamma_.reset_data();
  }

  variable_list apply(variable_list&& grads) override {
    const std::lock_guard<std::mutex> lock(mutex_);
    const int64_t B = B_, C = C_, H = H_, W = W_;
    const Tensor y = readable(y_, *this, made_type(*this), B * C * H * W), gamma = readable(gamma_, *this, ptype_, C);
    const bool twice = at::GradMode::is_enabled() &&
                       ((grads[0].defined() && grads[0].requires_grad()) || y.requires_grad() || gamma.requires_grad());
    const at::NoGradGuard no_grad;
    const c10::DeviceGuard guard(y.device());
    const at::TensorOptions opt = y.options().requires_grad(false);
    Tensor g = upstream(grads[0], {B, C, H, W}, opt);
    variable_list res(3);
    if (task_should_compute_output(0) || task_should_compute_output(2)) {
      Tensor dy = at::empty(y.sizes(), opt), dgamma = at::empty(gamma.sizes(), gamma.options().requires_grad(false));
      size_t wsz;
      const c10::DataPtr ws = block_workspace(g, &wsz);
      const int pdt = dtype_code(gamma.scalar_type());
      const int rc = abi.residual_bwd(g.const_data_ptr(), y.const_data_ptr(), gamma.const_data_ptr(), dy.mutable_data_ptr(),
                                      dgamma.mutable_data_ptr(), pdt, B, C, H * W, dtype_code(y.scalar_type()), pdt, ws.get(), wsz,
                                      stream_of(y));
      if (rc) fail(rc, "wtconv block residual backward");
      if (task_should_compute_output(0)) res[0] = std::move(dy);
      if (task_should_compute_output(2)) res[2] = std::move(dgamma);
    }
    if (task_should_compute_output(1)) res[1] = std::move(g);
    if (twice) refuse_second_derivatives(res, "the block's layer scale and shortcut");
    return res;
  }
};

// shortcut + gamma * y; None if the kernels do not take these arguments, or autograd records and there is no gamma.
py::object block_residual(const Tensor& y, const Tensor& shortcut, const std::optional<Tensor>& gamma) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (!y.is_cuda() || y.dim() != 4 || shortcut.dim() != 4 || !block_dtype(y.scalar_type()) || y.numel() == 0) return py::none();
  const int64_t B = y.size(0), H = y.size(1), W = y.size(2), C = y.size(3);
  if (!y.is_contiguous() || !canonical(shortcut, y.device(), y.scalar_type()) || shortcut.sizes() != at::IntArrayRef({B, C, H, W}))
    return py::none();
  if (y._fw_grad(0).defined() || shortcut._fw_grad(0).defined()) return py::none();
  bool record = at::GradMode::is_enabled(), any = y.requires_grad() || shortcut.requires_grad();
  if (gamma.has_value()) {
    if (!canonical(*gamma, y.device(), gamma->scalar_type()) || !block_dtype(gamma->scalar_type()) || gamma->numel() != C ||
        gamma->_fw_grad(0).defined())
      return py::none();
    any = any || gamma->requires_grad();
  }
  record = record && any;
  if (record && !gamma.has_value()) return py::none();
  Tensor out;
  {
    py::gil_scoped_release nogil;
    const c10::DeviceGuard guard(y.device());
    out = at::empty(shortcut.sizes(), shortcut.options().requires_grad(false));
    const int rc = abi.residual(y.const_data_ptr(), shortcut.const_data_ptr(), gamma.has_value() ? gamma->const_data_ptr() : nullptr,
                                out.mutable_data_ptr(), B, C, H * W, dtype_code(y.scalar_type()),
                                gamma.has_value() ? dtype_code(gamma->scalar_type()) : WTCONV_F32, stream_of(y));
    if (rc) fail(rc, "wtconv block residual");
    if (record) {
      const std::shared_ptr<ResidualNode> node(new ResidualNode(), torch::autograd::deleteNode);
      torch::autograd::edge_list next;
      next.reserve(3);
      for (const Tensor* t : {&y, &shortcut, &*gamma}) next.push_back(torch::autograd::impl::gradient_edge(*t));
      node->set_next_edges(std::move(next));
      node->y_ = torch::autograd::SavedVariable(y, false);
      node->gamma_ = torch::autograd::SavedVariable(*gamma, false);
      node->B_ = B;
      node->C_ = C;
      node->H_ = H;
      node->W_ = W;
      node->ptype_ = gamma->scalar_type();
      torch::autograd::set_history(out, node);
    }
  }
  return py::cast(out);
}

// Stem (convolution, then LayerNorm over the channels) or downsample (LayerNorm, then convolution) in one kernel
// (inference): None if no kernel takes these arguments or autograd would record the call.
py::object patch_conv(const Tensor& x, const Tensor& conv_w, const Tensor& conv_b, const Tensor& norm_w, const Tensor& norm_b,
                      double eps, bool stem) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (x.dim() != 4 || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || !x.is_contiguous() || x.numel() == 0) return py::none();
  const int64_t B = x.size(0), C = x.size(1), H = x.size(2), W = x.size(3), P = stem ? 4 : 2;
  if (conv_w.dim() != 4 || conv_w.size(1) != C || conv_w.size(2) != P || conv_w.size(3) != P) return py::none();
  const int64_t cout = conv_w.size(0), normed = stem ? cout : C;
  if (conv_b.numel() != cout || norm_w.numel() != normed || norm_b.numel() != normed) return py::none();
  const bool grad = at::GradMode::is_enabled();
  if (grad && x.requires_grad()) return py::none();
  uintptr_t bits = reinterpret_cast<uintptr_t>(x.const_data_ptr());
  for (const Tensor* t : {&conv_w, &conv_b, &norm_w, &norm_b}) {
    if (!canonical(*t, x.device(), at::kBFloat16) || (grad && t->requires_grad())) return py::none();
    bits |= reinterpret_cast<uintptr_t>(t->const_data_ptr());
  }
  if (bits % 16 || x.numel() > (1LL << 40) || !abi.patch_ok(stem, B, C, H, W, cout)) return py::none();
  for (const Tensor* t : {&x, &conv_w, &conv_b, &norm_w, &norm_b})
    if (t->_fw_grad(0).defined()) return py::none();      // forward-mode differentiation: PyTorch's own operators
  const c10::DeviceGuard guard(x.device());
  Tensor out = at::empty({B, cout, H / P, W / P}, x.options());
  const size_t wsz = abi.patch_ws(stem, B, C, H, W, cout);
  c10::DataPtr ws;
  if (wsz) ws = scratch(x, wsz);
  const wtconv_patch_params p = {conv_w.const_data_ptr(), conv_b.const_data_ptr(), norm_w.const_data_ptr(), norm_b.const_data_ptr()};
  const int rc = abi.patch(stem, x.const_data_ptr(), out.mutable_data_ptr(), &p, B, C, H, W, cout, static_cast<float>(eps),
                           WTCONV_BF16, WTCONV_BF16, ws.get(), wsz, c10::hip::getCurrentHIPStream(x.device().index()).stream());
  if (rc) fail(rc, "wtconv patch conv");
  return py::cast(out);
}

// ---- the head: mean over the pixels, LayerNorm over the channels; (B, C), or None if the kernel does not take these arguments.
// (x, weight, bias, eps)
PyObject* pool_norm(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  TORCH_CHECK(nargs == 4, "pool_norm: expected 4 arguments, got ", nargs);
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  for (int i = 0; i < 3; ++i)
    if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
  const Tensor &x = THPVariable_Unpack(args[0]), &weight = THPVariable_Unpack(args[1]), &bias = THPVariable_Unpack(args[2]);
  const double eps = PyFloat_AsDouble(args[3]);
  if (eps == -1. && PyErr_Occurred()) return nullptr;
  if (!x.is_cuda() || !x.has_storage() || x.dim() != 4 || !block_dtype(x.scalar_type()) || !x.is_contiguous() || x.numel() == 0)
    Py_RETURN_NONE;
  const int64_t B = x.size(0), C = x.size(1), HW = x.size(2) * x.size(3);
  const bool grad = at::GradMode::is_enabled();
  if ((grad && x.requires_grad()) || x._fw_grad(0).defined()) Py_RETURN_NONE;
  for (const Tensor* t : {&weight, &bias})
    if (!canonical(*t, x.device(), weight.scalar_type()) || !block_dtype(t->scalar_type()) || t->numel() != C || t->dim() != 1 ||
        (grad && t->requires_grad()) || t->_fw_grad(0).defined())
      Py_RETURN_NONE;
  if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 4 || x.numel() > (1LL << 40) || B > (1LL << 30) || C > (1LL << 20) ||
      HW > (1LL << 20) || !abi.pool_ok(B, C, HW))
    Py_RETURN_NONE;
  const c10::DeviceGuard guard(x.device());
  Tensor out = at::empty({B, C}, x.options().requires_grad(false));
  const int rc = abi.pool(x.const_data_ptr(), out.mutable_data_ptr(), weight.const_data_ptr(), bias.const_data_ptr(), B, C, HW,
                          static_cast<float>(eps), dtype_code(x.scalar_type()), dtype_code(weight.scalar_type()), stream_of(x));
  if (rc) fail(rc, "wtconv pool norm");
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", &bind, "hand over the addresses of the C-ABI entry points");
  static PyMethodDef functions[] = {
      {"layer", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&layer)), METH_FASTCALL,
       "WTConv layer (2-D or 1-D) with a C++ autograd node; None if the arguments are not canonical"},
      {"pool_norm", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&pool_norm)), METH_FASTCALL,
       "mean over the pixels and LayerNorm over the channels; None if not taken"},
      {"watched", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&watched)), METH_FASTCALL,
       "whether something expects to see these modules called"},
      {"layer_params", &layer_params, METH_O, "the parameters of a WTConv module as layer() takes them; None if it is built otherwise"},
      {"mlp_args", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&mlp_args)), METH_FASTCALL,
       "the arguments of block_mlp from x, shortcut, the modules norm and mlp, and gamma; None where the modules are to be called"},
      {"block_mlp", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&block_mlp)), METH_FASTCALL,
       "LayerNorm, MLP, layer scale and shortcut of a WTConvNeXt block; None if not taken"},
      {nullptr, nullptr, 0, nullptr}};
  if (PyModule_AddFunctions(m.ptr(), functions) != 0) throw py::error_already_set();
  m.def("mlp", &mlp, "a block's MLP with a C++ autograd node; None if not taken", py::arg("x"), py::arg("fc1_weight"), py::arg("fc1_bias"),
        py::arg("fc2_weight"), py::arg("fc2_bias"), py::arg("twice") = false);
  m.def("channel_norm", &channel_norm, "LayerNorm over the channels with a C++ autograd node; None if not taken");
  m.def("block_residual", &block_residual, "layer scale and shortcut with a C++ autograd node; None if not taken");
  m.def("patch_conv", &patch_conv, "stem or downsample of a WTConvNeXt in one kernel; None if not taken");
  m.def("haar", &haar, "single-level Haar transform with a C++ autograd node, and the check of the bank it is handed");
}
