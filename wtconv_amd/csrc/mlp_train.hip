// Host side of the MLP's products (kernels_product.h): argument checks, tile shapes, the split of the weight gradients,
// launches.
#include <initializer_list>

#include "common.h"
#include "host_util.h"
#include "kernels_product.h"
#include "../../include/wtconv_ops.h"

using namespace wt;

namespace {

size_t round_up256(size_t v) { return (v + 255) / 256 * 256; }

template <typename S, int END>
int launch_product(const ProductArgs& a, hipStream_t stream) {
  auto kern = product_kernel<S, END>;
  if (int e = allow_lds(kern, S::kLdsBytes)) return e;
  WT_LAUNCH(kern, dim3((a.M + S::BM - 1) / S::BM * (a.N / S::BN)), dim3(S::kThreads), S::kLdsBytes, stream, a);
  return 0;
}

// Tiles of 64 pixels x 128 outputs: three workgroups a CU (48 KB of LDS) hide each other's loads, GELU and stores, which
// larger tiles with fewer fragment reads do not make up for.  Measured, both products of the forward pass, us: 12544 pixels of
// 384 channels 64 (128 x 128 tiles 64, 256 x 128 70, 64 x 128 in four stages of 32: 75), of 768 channels 171 (186, 194,
// 224); the library's, with GELU, 82 and 161.  Where those leave compute units without work, 64 x 64 with a stage more on
// its way: 800 pixels of 384 channels 16.8 (64 x 128: 22.4).
using Large = ProductShape<64, 128, 1, 4, 64, 2>;
using Large32 = ProductShape<64, 128, 1, 4, 32, 2>;      // (96 channels go by in steps of 32)
using Small = ProductShape<64, 64, 2, 2, 64, 3>;
using Small32 = ProductShape<64, 64, 2, 2, 32, 3>;
using Channels192 = ProductShape<128, 192, 2, 2, 64, 2>;
using Channels96 = ProductShape<64, 96, 4, 1, 64, 2>;

// Whether the tiles of a shape give every compute unit two workgroups.
template <typename S>
bool fills(const ProductArgs& a) { return static_cast<long long>((a.M + S::BM - 1) / S::BM) * (a.N / S::BN) >= 2LL * compute_units(); }

template <int END>
int product_to_hidden(const ProductArgs& a, hipStream_t stream) {
  if (a.K % 64) return fills<Large32>(a) ? launch_product<Large32, END>(a, stream) : launch_product<Small32, END>(a, stream);
  return fills<Large>(a) ? launch_product<Large, END>(a, stream) : launch_product<Small, END>(a, stream);
}
template <int END>
int product_to_channels(const ProductArgs& a, hipStream_t stream) {
  if (a.N % 128 == 0 && fills<Large>(a)) return launch_product<Large, END>(a, stream);
  if (a.N % 192 == 0 && fills<Channels192>(a)) return launch_product<Channels192, END>(a, stream);
  return a.N % 64 == 0 ? launch_product<Small, END>(a, stream) : launch_product<Channels96, END>(a, stream);
}

bool takes(long long M, int C, int hidden) {
  if (M <= 0 || C <= 0 || hidden <= 0 || hidden % 128 != 0 || (C % 96 != 0 && C % 128 != 0)) return false;
  // 32-bit: pixel indices, the offsets inside a tile, the threads that add up the weight gradients (half as many as they have
  // values), and the threads of a product (four per 64 values)
  if (M > (1 << 30) || hidden > (1 << 16) || C > (1 << 16)) return false;
  return static_cast<long long>(C) * hidden <= (1LL << 31) && M * (C > hidden ? C : hidden) <= (1LL << 35);
}

// Whether the kernels are the faster way, and not the library's products with passes for biases, GELU and its derivative between
// them.  What they save grows with the pixels, what they lose with the weights: their tiles reach about half of the rate of
// the library's on large products.  Measured, time of a forward and backward pass over that of the library's passes (graph
// replay), by pixels:
//                             1    49   256  1024  2048  3136  6272 12544 25088 50176
//   384 -> 1536   (0.6 M)  0.83  0.77        0.55        0.49        0.50        0.58
//   512 -> 2048   (1.0 M)  1.03  0.94  0.70  0.62  0.56  0.57  0.67  0.64  0.70  0.73
//  1024 -> 2048   (2.1 M)  1.16        0.72  0.67  0.66  0.79  0.84  0.87  0.88  0.93
//   768 -> 3072   (2.4 M)  1.12  0.94  0.75  0.68  0.67  0.81  0.82  0.88  0.92  1.05
//  1536 -> 1536   (2.4 M)  1.02        0.75  0.67  0.70  0.77  0.77  0.77  0.93  1.07
//   896 -> 3584   (3.2 M)  1.08        0.79  0.79  0.82  0.86  0.85  1.01  1.03  1.11
//   768 -> 4096   (3.1 M)  1.21        0.83  0.75  0.79  0.93  0.98  0.96  1.03  1.19
//  1024 -> 4096   (4.2 M)  1.24  1.08  0.85  0.80  0.85  0.98  1.08  1.15  1.14  1.26
//  1536 -> 6144   (9.4 M)  1.56  1.26  1.00  1.04        1.20        1.51
//  2048 -> 8192    (17 M)  2.20  1.85  1.32  1.40        1.64        1.76
// (Fewer pixels than about 48 are a little slower from a million weights on, but for as long as launching the library's eleven
// passes takes the host three times as long as either takes the device, which a caller without a graph waits for: 79 us
// against 225 with one pixel of 512 channels.)
bool pays(long long M, int C, int hidden) {
  const long long weights = static_cast<long long>(C) * hidden;
  const long long most = weights <= (2LL << 20) ? 1LL << 30 : weights <= (5LL << 19) ? 1 << 15 : weights <= (13LL << 18) ? 6500 : 2048;
  return weights <= (4LL << 20) && M <= most;
}

struct GradPlan {
  int tiles = 0, shares = 0, stages = 0;
  size_t partial = 0, bias = 0;
};

// Shares of the pixels: as many as give every compute unit two workgroups and no more, of four stages at least, since each
// leaves a record of its whole tile (64 KB, as much as two stages read).  Measured, both weight gradients with their
// biases, us: 12544 pixels of 384 channels 44 (library 150, and 42 for the biases), of 768 channels 197; 800 pixels of 384
// channels 13.8 (17 with shares of a stage).
template <typename S>
GradPlan grad_plan_of(int M, int C, int hidden, int jobs) {
  GradPlan p;
  p.tiles = hidden / S::BH * (C / S::BC);
  const int all = (M + S::BK - 1) / S::BK;
  int want = 2 * compute_units() / (p.tiles * jobs);
  if (want > all / 4) want = all / 4;
  if (want < 1) want = 1;
  p.stages = (all + want - 1) / want;
  p.shares = (all + p.stages - 1) / p.stages;
  p.partial = round_up256(sizeof(float) * S::kTileFloats * p.tiles * jobs * p.shares);
  p.bias = round_up256(sizeof(float) * (C + hidden) * p.shares);
  return p;
}

using Grad128 = WeightGradShape<128, 128, 64, 2>;
using Grad192 = WeightGradShape<128, 192, 64, 2>;
using Grad96 = WeightGradShape<128, 96, 64, 2>;

GradPlan grad_plan(int M, int C, int hidden, int jobs) {
  return C % 128 == 0 ? grad_plan_of<Grad128>(M, C, hidden, jobs)
         : C % 192 == 0 ? grad_plan_of<Grad192>(M, C, hidden, jobs) : grad_plan_of<Grad96>(M, C, hidden, jobs);
}

template <typename S>
int launch_grads(const WeightGradArgs& a, const GradPlan& p, hipStream_t stream) {
  auto kern = weight_grad_kernel<S>;
  if (int e = allow_lds(kern, S::kLdsBytes)) return e;
  WT_LAUNCH(kern, dim3(p.tiles * a.jobs * p.shares), dim3(256), S::kLdsBytes, stream, a);
  const int threads = a.jobs * p.tiles * (S::kTileFloats / 4) + (a.C + a.hidden) / 4;
  WT_LAUNCH(wgrad_sum_kernel<S>, dim3((threads + 255) / 256), dim3(256), 0, stream, a);
  return 0;
}

// What a backward call keeps in its workspace: dh, the transposed weights, the records.
struct BackwardPlan {
  bool dh = false;
  int jobs = 0, first_job = 0;
  size_t at_w1t = 0, at_w2t = 0, at_partial = 0, at_bias = 0, bytes = 0;
  GradPlan grads;
};
BackwardPlan backward_plan(int M, int C, int hidden, int want) {
  BackwardPlan p;
  const bool dx = want & WTCONV_MLP_DX, one = want & WTCONV_MLP_FC1, two = want & WTCONV_MLP_FC2;
  p.dh = dx || one;
  p.jobs = (one ? 1 : 0) + (two ? 1 : 0);
  p.first_job = two ? 0 : 1;
  const size_t weights = round_up256(sizeof(bf16_t) * static_cast<size_t>(C) * hidden);
  size_t at = p.dh ? round_up256(sizeof(bf16_t) * static_cast<size_t>(M) * hidden) : 0;
  p.at_w2t = at;
  if (p.dh) at += weights;
  p.at_w1t = at;
  if (dx) at += weights;
  if (p.jobs) {
    p.grads = grad_plan(M, C, hidden, p.jobs);
    p.at_partial = at;
    at += p.grads.partial;
    p.at_bias = at;
    at += p.grads.bias;
  }
  p.bytes = at;
  return p;
}

bool aligned(std::initializer_list<const void*> ptrs) {
  uintptr_t bits = 0;
  for (const void* p : ptrs) bits |= reinterpret_cast<uintptr_t>(p);
  return bits % 16 == 0;
}

}  // namespace

extern "C" int wtconv_mlp_supported(long long pixels, int C, int hidden) {
  return takes(pixels, C, hidden) && pays(pixels, C, hidden) ? 1 : 0;
}

extern "C" int wtconv_mlp_forward(const void* x, void* h, void* act, void* y, const wtconv_mlp_params* w, long long pixels,
                                  int C, int hidden, int dtype, int param_dtype, void* stream) {
  const char* fn = "wtconv_mlp_forward";
  if (x == nullptr || act == nullptr || y == nullptr || w == nullptr) return fail(WTCONV_E_ARG, "%s: null pointer", fn);
  if (!w->fc1_weight || !w->fc1_bias || !w->fc2_weight || !w->fc2_bias) return fail(WTCONV_E_ARG, "%s: null parameter", fn);
  if (dtype != WTCONV_BF16 || param_dtype != WTCONV_BF16) return fail(WTCONV_E_UNSUPPORTED, "%s: bfloat16 only", fn);
  if (!takes(pixels, C, hidden)) return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d, hidden=%d", fn, C, hidden);
  if (!aligned({x, h, act, y, w->fc1_weight, w->fc1_bias, w->fc2_weight, w->fc2_bias}))
    return fail(WTCONV_E_ARG, "%s: tensors must be 16-byte aligned", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  ProductArgs a = {};
  a.pix = static_cast<const bf16_t*>(x);
  a.w = static_cast<const bf16_t*>(w->fc1_weight);
  a.bias = static_cast<const bf16_t*>(w->fc1_bias);
  a.out = static_cast<bf16_t*>(act);
  a.pre = static_cast<bf16_t*>(h);
  a.M = static_cast<int>(pixels); a.N = hidden; a.K = C;
  if (int e = product_to_hidden<kEndGelu>(a, s)) return e;
  a.pix = static_cast<const bf16_t*>(act);
  a.w = static_cast<const bf16_t*>(w->fc2_weight);
  a.bias = static_cast<const bf16_t*>(w->fc2_bias);
  a.out = static_cast<bf16_t*>(y);
  a.pre = nullptr;
  a.N = C; a.K = hidden;
  if (int e = product_to_channels<kEndBias>(a, s)) return e;
  return check_launch(fn);
}

extern "C" size_t wtconv_mlp_backward_workspace_bytes(long long pixels, int C, int hidden, int want) {
  if (!takes(pixels, C, hidden)) return 0;
  return backward_plan(static_cast<int>(pixels), C, hidden, want).bytes;
}

extern "C" int wtconv_mlp_backward(const void* x, const void* h, const void* act, const void* dy, const wtconv_mlp_params* w,
                                   void* dx, const wtconv_mlp_grads* g, long long pixels, int C, int hidden, int dtype,
                                   int param_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const char* fn = "wtconv_mlp_backward";
  if (x == nullptr || h == nullptr || act == nullptr || dy == nullptr || w == nullptr || g == nullptr)
    return fail(WTCONV_E_ARG, "%s: null pointer", fn);
  if (!w->fc1_weight || !w->fc2_weight) return fail(WTCONV_E_ARG, "%s: null parameter", fn);
  if ((g->fc1_weight == nullptr && g->fc1_bias != nullptr) || (g->fc2_weight == nullptr && g->fc2_bias != nullptr))
    return fail(WTCONV_E_ARG, "%s: a bias gradient comes with its weight's", fn);
  if (dtype != WTCONV_BF16 || param_dtype != WTCONV_BF16) return fail(WTCONV_E_UNSUPPORTED, "%s: bfloat16 only", fn);
  if (!takes(pixels, C, hidden)) return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d, hidden=%d", fn, C, hidden);
  if (!aligned({x, h, act, dy, dx, w->fc1_weight, w->fc2_weight, g->fc1_weight, g->fc1_bias, g->fc2_weight, g->fc2_bias}))
    return fail(WTCONV_E_ARG, "%s: tensors must be 16-byte aligned", fn);
  const int M = static_cast<int>(pixels);
  const int want = (dx ? WTCONV_MLP_DX : 0) | (g->fc1_weight ? WTCONV_MLP_FC1 : 0) | (g->fc2_weight ? WTCONV_MLP_FC2 : 0);
  const BackwardPlan p = backward_plan(M, C, hidden, want);
  if (p.bytes > 0 && (workspace == nullptr || workspace_bytes < p.bytes || reinterpret_cast<uintptr_t>(workspace) % 16))
    return fail(WTCONV_E_WORKSPACE, "%s: workspace too small or misaligned", fn);
  hipStream_t s = static_cast<hipStream_t>(stream);
  unsigned char* ws = static_cast<unsigned char*>(workspace);
  bf16_t *dh = reinterpret_cast<bf16_t*>(ws), *w1t = reinterpret_cast<bf16_t*>(ws + p.at_w1t), *w2t = reinterpret_cast<bf16_t*>(ws + p.at_w2t);
  if (p.dh) {
    TransposeArgs t = {};
    t.src[0] = static_cast<const bf16_t*>(w->fc2_weight); t.dst[0] = w2t; t.rows[0] = C; t.cols[0] = hidden;
    t.src[1] = static_cast<const bf16_t*>(w->fc1_weight); t.dst[1] = w1t; t.rows[1] = hidden; t.cols[1] = C;
    WT_LAUNCH(transpose_weights_kernel, dim3(((C + 63) / 64) * ((hidden + 63) / 64), 1, dx ? 2 : 1), dim3(256), 0, s, t);
    ProductArgs a = {};
    a.pix = static_cast<const bf16_t*>(dy);
    a.w = w2t;
    a.out = dh;
    a.pre = const_cast<bf16_t*>(static_cast<const bf16_t*>(h));
    a.M = M; a.N = hidden; a.K = C;
    if (int e = product_to_hidden<kEndDerivative>(a, s)) return e;
    if (dx) {
      a.pix = dh;
      a.w = w1t;
      a.out = static_cast<bf16_t*>(dx);
      a.pre = nullptr;
      a.N = C; a.K = hidden;
      if (int e = product_to_channels<kEndPlain>(a, s)) return e;
    }
  }
  if (p.jobs) {
    WeightGradArgs a = {};
    a.hid[0] = static_cast<const bf16_t*>(act); a.chan[0] = static_cast<const bf16_t*>(dy);
    a.hid[1] = dh; a.chan[1] = static_cast<const bf16_t*>(x);
    a.partial = reinterpret_cast<float*>(ws + p.at_partial);
    a.bias_partial = reinterpret_cast<float*>(ws + p.at_bias);
    a.dw[0] = static_cast<bf16_t*>(g->fc2_weight); a.dw[1] = static_cast<bf16_t*>(g->fc1_weight);
    a.db[0] = static_cast<bf16_t*>(g->fc2_bias); a.db[1] = static_cast<bf16_t*>(g->fc1_bias);
    a.M = M; a.hidden = hidden; a.C = C;
    a.shares = p.grads.shares; a.stages = p.grads.stages;
    a.jobs = p.jobs; a.first_job = p.first_job;
    const int e = C % 128 == 0 ? launch_grads<Grad128>(a, p.grads, s)
                  : C % 192 == 0 ? launch_grads<Grad192>(a, p.grads, s) : launch_grads<Grad96>(a, p.grads, s);
    if (e) return e;
  }
  return check_launch(fn);
}
