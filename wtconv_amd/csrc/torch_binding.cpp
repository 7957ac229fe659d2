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

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>

#include <chrono>
#include <mutex>
#include <optional>
#include <vector>

#include "../../include/wtconv_hip.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The C ABI as function pointers (filled once by bind()).
struct Abi {
  int (*fwd2)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwd2)(const void*, const void*, void*, const wtconv_params*, const wtconv_param_grads*, int, int, int, int, int,
              int, int, int, void*, size_t, void*);
  int (*bwdin2)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwdpar2)(const void*, const void*, const wtconv_params*, const wtconv_param_grads*, int, int, int, int, int, int,
                 int, int, void*, size_t, void*);
  size_t (*ws2)(int, int, int, int, int, int, int);
  int (*fwd1)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwd1)(const void*, const void*, void*, const wtconv_params*, const wtconv_param_grads*, int, int, int, int, int,
              int, int, void*, size_t, void*);
  int (*bwdin1)(const void*, void*, const wtconv_params*, int, int, int, int, int, int, int, void*, size_t, void*);
  int (*bwdpar1)(const void*, const void*, const wtconv_params*, const wtconv_param_grads*, int, int, int, int, int, int,
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
  bool bound = false;
} abi;

template <typename F>
void take(F& slot, uintptr_t addr) { slot = reinterpret_cast<F>(addr); }

// Addresses in the order of the names in wtconv_amd/_ext.py.
void bind(const std::vector<uintptr_t>& a) {
  TORCH_CHECK(a.size() == 18, "bind: expected 18 addresses, got ", a.size());
  take(abi.fwd2, a[0]); take(abi.bwd2, a[1]); take(abi.bwdin2, a[2]); take(abi.bwdpar2, a[3]); take(abi.ws2, a[4]);
  take(abi.fwd1, a[5]); take(abi.bwd1, a[6]); take(abi.bwdin1, a[7]); take(abi.bwdpar1, a[8]); take(abi.ws1, a[9]);
  take(abi.last_error, a[10]);
  take(abi.haar2, a[11]); take(abi.haar1, a[12]); take(abi.haar2c, a[13]); take(abi.haar1c, a[14]);
  take(abi.mlp_ok, a[15]); take(abi.mlp_ws, a[16]); take(abi.mlp, a[17]);
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
  if (rc == WTCONV_E_ARG) throw py::value_error(std::string(msg && *msg ? msg : what));
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

class WTConvNode : public torch::autograd::Function<WTConvNode> {
 public:
  // wt = the L level weights followed by the L level scales.
  static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& base_w,
                        const std::optional<Tensor>& base_b_opt, const Tensor& base_s, at::TensorList wt,
                        int64_t dims, int64_t K, int64_t L) {
    const Tensor x = x_in.contiguous();
    const Tensor base_b = base_b_opt.has_value() ? *base_b_opt : Tensor();
    const c10::DeviceGuard guard(x.device());      // (PyTorch on ROCm names the device type "cuda")
    const Shape s = dims == 2 ? Shape{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3)}
                              : Shape{(int)x.size(0), (int)x.size(1), 1, (int)x.size(2)};
    Tensor out = at::empty_like(x, at::MemoryFormat::Contiguous);
    const size_t wsz = workspace_bytes(dims, s, K, L, 0);
    Tensor ws = at::empty({static_cast<int64_t>(wsz)}, x.options().dtype(at::kByte));
    wtconv_params p;
    fill(p, base_w, base_b, base_s, wt, L);
    void* stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    const int dt = dtype_code(x.scalar_type()), pdt = dtype_code(base_w.scalar_type());
    const int rc = dims == 2 ? abi.fwd2(x.data_ptr(), out.data_ptr(), &p, s.B, s.C, s.H, s.W, K, L, dt, pdt,
                                        ws.data_ptr(), wsz, stream)
                             : abi.fwd1(x.data_ptr(), out.data_ptr(), &p, s.B, s.C, s.W, K, L, dt, pdt, ws.data_ptr(),
                                        wsz, stream);
    if (rc) fail(rc, "wtconv forward");
    variable_list saved = {x, base_w, base_b, base_s};
    saved.insert(saved.end(), wt.begin(), wt.end());
    ctx->save_for_backward(saved);
    ctx->saved_data["dims"] = dims;
    ctx->saved_data["K"] = K;
    ctx->saved_data["L"] = L;
    return out;
  }

  static variable_list backward(AutogradContext* ctx, variable_list grad_outputs) {
    const variable_list saved = ctx->get_saved_variables();
    const int dims = ctx->saved_data["dims"].toInt(), K = ctx->saved_data["K"].toInt(), L = ctx->saved_data["L"].toInt();
    const Tensor &x = saved[0], &base_w = saved[1], &base_b = saved[2], &base_s = saved[3];
    const at::TensorList wt(saved.data() + 4, 2 * L);
    const bool has_bias = base_b.defined();
    // one result per argument of forward: x, base_w, base_b, base_s, 2L level tensors, dims, K, L
    variable_list res(4 + 2 * L + 3);
    Tensor g = grad_outputs[0];
    if (!g.defined()) return res;
    // needs_input_grad counts the tensor arguments only (a missing bias is not one of them)
    const int nt = 3 + (has_bias ? 1 : 0) + 2 * L;
    const bool need_x = ctx->needs_input_grad(0);
    bool need_params = false;
    for (int i = 1; i < nt; ++i) need_params = need_params || ctx->needs_input_grad(i);
    if (!need_x && !need_params) return res;
    if (g.scalar_type() != x.scalar_type()) g = g.to(x.scalar_type());
    g = g.contiguous();
    const c10::DeviceGuard guard(x.device());      // (PyTorch on ROCm names the device type "cuda")
    const Shape s = dims == 2 ? Shape{(int)x.size(0), (int)x.size(1), (int)x.size(2), (int)x.size(3)}
                              : Shape{(int)x.size(0), (int)x.size(1), 1, (int)x.size(2)};
    const int pass = need_x && need_params ? 3 : (need_x ? 1 : 2);
    const size_t wsz = workspace_bytes(dims, s, K, L, pass);
    Tensor ws = at::empty({static_cast<int64_t>(wsz)}, x.options().dtype(at::kByte));
    wtconv_params p;
    fill(p, base_w, base_b, base_s, wt, L);
    void* stream = c10::hip::getCurrentHIPStream(x.device().index()).stream();
    const int dt = dtype_code(x.scalar_type()), pdt = dtype_code(base_w.scalar_type());
    Tensor grad_x;
    if (need_x) grad_x = at::empty_like(x, at::MemoryFormat::Contiguous);
    // parameter gradients are written as fp32 into one flat buffer (one allocation for the 5 + 2 L tensors): fp32
    // parameters get views of it in their own shapes, others views of one cast of it
    const bool f32 = base_w.scalar_type() == at::kFloat;
    std::vector<Tensor> views(3 + 2 * L);      // base_w, base_b, base_s, levels
    Tensor flat;
    wtconv_param_grads gt;
    if (need_params) {
      std::vector<const Tensor*> plist = {&base_w, &base_b, &base_s};
      for (int i = 0; i < 2 * L; ++i) plist.push_back(&wt[i]);
      int64_t total = 0;
      for (const Tensor* t : plist) total += t->defined() ? t->numel() : 0;
      flat = at::empty({total}, x.options().dtype(at::kFloat));
      int64_t pos = 0;
      for (size_t i = 0; i < plist.size(); ++i)
        if (plist[i]->defined()) {
          views[i] = flat.narrow(0, pos, plist[i]->numel());
          if (f32) views[i] = views[i].view(plist[i]->sizes());
          pos += plist[i]->numel();
        }
      const at::TensorList lv(views.data() + 3, 2 * L);
      fill(gt, views[0], views[1], views[2], lv, L);
    }
    int rc;
    if (dims == 2) {
      if (pass == 3)
        rc = abi.bwd2(x.data_ptr(), g.data_ptr(), grad_x.data_ptr(), &p, &gt, s.B, s.C, s.H, s.W, K, L, dt, pdt,
                      ws.data_ptr(), wsz, stream);
      else if (pass == 1)
        rc = abi.bwdin2(g.data_ptr(), grad_x.data_ptr(), &p, s.B, s.C, s.H, s.W, K, L, dt, pdt, ws.data_ptr(), wsz, stream);
      else
        rc = abi.bwdpar2(x.data_ptr(), g.data_ptr(), &p, &gt, s.B, s.C, s.H, s.W, K, L, dt, pdt, ws.data_ptr(), wsz, stream);
    } else {
      if (pass == 3)
        rc = abi.bwd1(x.data_ptr(), g.data_ptr(), grad_x.data_ptr(), &p, &gt, s.B, s.C, s.W, K, L, dt, pdt, ws.data_ptr(),
                      wsz, stream);
      else if (pass == 1)
        rc = abi.bwdin1(g.data_ptr(), grad_x.data_ptr(), &p, s.B, s.C, s.W, K, L, dt, pdt, ws.data_ptr(), wsz, stream);
      else
        rc = abi.bwdpar1(x.data_ptr(), g.data_ptr(), &p, &gt, s.B, s.C, s.W, K, L, dt, pdt, ws.data_ptr(), wsz, stream);
    }
    if (rc) fail(rc, "wtconv backward");
    // The gradients come from raw pointers and carry no graph.  Under create_graph=True every result that something
    // differentiable went into gets a node that raises when it is differentiated (what once_differentiable does for
    // the Python function): a second-order term is refused instead of being treated as a constant.
    bool twice = false;
    if (at::GradMode::is_enabled()) {
      twice = grad_outputs[0].requires_grad();
      for (const Tensor& t : saved) twice = twice || (t.defined() && t.requires_grad());
    }
    auto refuse = [&](Tensor& t) {
      if (!twice || !t.defined()) return;
      auto err = std::make_shared<torch::autograd::Error>(
          "the backward pass of the WTConv layer is not differentiable (double backward / create_graph=True through "
          "this layer is not supported)", torch::autograd::edge_list());
      torch::autograd::create_gradient_edge(t, err);
    };
    res[0] = grad_x;
    refuse(res[0]);
    if (need_params) {
      if (!f32) {
        const Tensor cast = flat.to(base_w.scalar_type());
        int64_t pos = 0;
        std::vector<const Tensor*> plist = {&base_w, &base_b, &base_s};
        for (int i = 0; i < 2 * L; ++i) plist.push_back(&wt[i]);
        for (size_t i = 0; i < plist.size(); ++i)
          if (plist[i]->defined()) {
            views[i] = cast.narrow(0, pos, plist[i]->numel()).view(plist[i]->sizes());
            pos += plist[i]->numel();
          }
      }
      res[1] = views[0];
      res[2] = views[1];
      res[3] = views[2];
      for (int i = 0; i < 2 * L; ++i) res[4 + i] = views[3 + i];
      for (int i = 1; i < 4 + 2 * L; ++i) refuse(res[i]);
    }
    return res;
  }
};

bool canonical(const Tensor& t, const at::Device& dev, at::ScalarType pd) {
  return t.device() == dev && t.scalar_type() == pd && t.is_contiguous();
}

// The layer with its C++ autograd node, or None when the arguments need the conversions of the Python path.
py::object layer(const Tensor& x, const Tensor& base_w, const std::optional<Tensor>& base_b, const Tensor& base_s,
                 const std::vector<Tensor>& wt_ws, const std::vector<Tensor>& wt_ss, int64_t dims, int64_t K, int64_t L) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (!x.is_cuda() || dtype_code(x.scalar_type()) < 0) return py::none();
  const at::ScalarType pd = base_w.scalar_type();
  if (dtype_code(pd) < 0) return py::none();
  if (static_cast<int64_t>(wt_ws.size()) != L || static_cast<int64_t>(wt_ss.size()) != L) return py::none();
  const at::Device dev = x.device();
  if (!canonical(base_w, dev, pd) || !canonical(base_s, dev, pd)) return py::none();
  if (base_b.has_value() && base_b->defined() && !canonical(*base_b, dev, pd)) return py::none();
  std::vector<Tensor> wt;
  wt.reserve(2 * L);
  for (const Tensor& t : wt_ws) { if (!canonical(t, dev, pd)) return py::none(); wt.push_back(t); }
  for (const Tensor& t : wt_ss) { if (!canonical(t, dev, pd)) return py::none(); wt.push_back(t); }
  const std::optional<Tensor> bias = (base_b.has_value() && base_b->defined()) ? base_b : std::nullopt;
  Tensor out;
  {
    py::gil_scoped_release nogil;
    out = WTConvNode::apply(x, base_w, bias, base_s, at::TensorList(wt), dims, K, L);
  }
  return py::cast(out);
}

// ---- the single-level Haar transforms (wtconv_amd/wavelet.py), with the check of the filter bank they are handed.

// Words of pinned host memory that a kernel writes its verdict into while the caller waits: one page, taken when the
// first bank is checked, its words lent for one call each.
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

 private:
  static constexpr int kWords = 64, kStride = 16;      // a cache line each
  std::mutex m_;
  unsigned* page_ = nullptr;
  std::vector<unsigned*> free_;
};
VerdictPool verdicts;

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
    // (an exception of the launch itself leaves nothing that would write the word)
    try {
      out = HaarNode::apply(x, dims, inverse, reinterpret_cast<int64_t>(bank->data_ptr()), int64_t{bdt},
                            reinterpret_cast<int64_t>(w));
    } catch (...) {
      verdicts.give_back(w);
      throw;
    }
    got = await_verdict(w, stream);
    verdicts.give_back(w);
  }
  if (got != 1u) return py::bool_(false);
  return py::cast(out);
}

// The block behind its WTConv layer in one kernel (inference): None if the kernel does not take these arguments or
// autograd would record the call.
py::object block_mlp(const Tensor& x, const Tensor& shortcut, const Tensor& norm_w, const Tensor& norm_b, double eps,
                     const Tensor& w1, const std::optional<Tensor>& b1, const Tensor& w2, const std::optional<Tensor>& b2,
                     const std::optional<Tensor>& gamma) {
  TORCH_CHECK(abi.bound, "wtconv binding used before bind()");
  if (x.dim() != 4 || !x.is_cuda() || x.scalar_type() != at::kBFloat16 || !x.is_contiguous()) return py::none();
  if (shortcut.sizes() != x.sizes() || !b1.has_value() || !b2.has_value()) return py::none();
  const int64_t B = x.size(0), C = x.size(1), HW = x.size(2) * x.size(3);
  if (w1.dim() != 2 || w2.dim() != 2 || w1.size(1) != C || w2.size(0) != C || w1.size(0) != w2.size(1)) return py::none();
  const int64_t hidden = w1.size(0);
  if (norm_w.numel() != C || norm_b.numel() != C || b1->numel() != hidden || b2->numel() != C) return py::none();
  if (gamma.has_value() && gamma->numel() != C) return py::none();
  const bool grad = at::GradMode::is_enabled();
  if (grad && x.requires_grad()) return py::none();
  const Tensor* all[] = {&shortcut, &norm_w, &norm_b, &w1, &*b1, &w2, &*b2, gamma.has_value() ? &*gamma : nullptr};
  uintptr_t bits = 0;
  for (const Tensor* t : all) {
    if (t == nullptr) continue;
    if (!canonical(*t, x.device(), at::kBFloat16) || (grad && t->requires_grad())) return py::none();
    if (t != &shortcut) bits |= reinterpret_cast<uintptr_t>(t->data_ptr());
  }
  if (bits % 16 || x.numel() == 0 || B * HW > (1LL << 30) || !abi.mlp_ok(B, C, HW, hidden)) return py::none();
  const c10::DeviceGuard guard(x.device());
  Tensor out = at::empty_like(x, at::MemoryFormat::Contiguous);
  const size_t wsz = abi.mlp_ws(B, C, HW, hidden);
  Tensor ws;
  if (wsz) ws = at::empty({static_cast<int64_t>(wsz)}, x.options().dtype(at::kByte));
  const wtconv_mlp_params p = {norm_w.data_ptr(), norm_b.data_ptr(), w1.data_ptr(), b1->data_ptr(), w2.data_ptr(),
                               b2->data_ptr(), gamma.has_value() ? gamma->data_ptr() : nullptr};
  const int rc = abi.mlp(x.data_ptr(), shortcut.data_ptr(), out.data_ptr(), &p, B, C, HW, hidden, static_cast<float>(eps),
                         WTCONV_BF16, WTCONV_BF16, wsz ? ws.data_ptr() : nullptr, wsz,
                         c10::hip::getCurrentHIPStream(x.device().index()).stream());
  if (rc) fail(rc, "wtconv block mlp");
  return py::cast(out);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("bind", &bind, "hand over the addresses of the C-ABI entry points");
  m.def("layer", &layer, "WTConv layer (2-D or 1-D) with a C++ autograd node; None if the arguments are not canonical");
  m.def("block_mlp", &block_mlp, "LayerNorm, MLP, layer scale and shortcut of a WTConvNeXt block; None if not taken");
  m.def("haar", &haar, "single-level Haar transform with a C++ autograd node, and the check of the bank it is handed");
}
