// Host side of the fused block kernel (kernels_mlp.h): argument checks, the split over the hidden units, launches.
#include "common.h"
#include "host_util.h"
#include "kernels_mlp.h"

using namespace wt;

namespace {

// Channel counts with a kernel, and their shapes: two pixel tiles a wave (half the LDS reads) while the registers allow
// two waves a SIMD or more -- alone on its SIMD a wave issues at less than half the rate.
#define WT_MLP_SHAPES(X) X(96, 2, 4, 3, 32, 3) X(128, 2, 4, 2, 32, 3) X(192, 2, 4, 2, 32, 3) X(256, 1, 8, 2, 32, 3) \
                         X(384, 1, 8, 2, 32, 3)

struct MlpPlan {
  int tiles = 0, splits = 0, padded = 0;
};

template <typename S>
MlpPlan plan_of(int pixels, int hidden) {
  MlpPlan p;
  p.tiles = (pixels + S::PX - 1) / S::PX;
  p.padded = p.tiles * S::PX;
  // A few pixels make a few workgroups, each with the whole of both weight matrices to go through: the hidden units are
  // then dealt to several workgroups, as many as fill the compute units once, and their sums meet in a second launch.
  const int nslice = hidden / S::HC, cus = compute_units();
  int splits = p.tiles >= cus ? 1 : cus / p.tiles;
  if (splits > nslice) splits = nslice;
  const int per = (nslice + splits - 1) / splits;
  p.splits = (nslice + per - 1) / per;
  return p;
}

template <typename S>
int launch(MlpArgs a, size_t workspace_bytes, hipStream_t stream) {
  const char* fn = "wtconv_block_mlp";
  const MlpPlan p = plan_of<S>(a.pixels, a.hidden);
  a.padded = p.padded;
  a.splits = p.splits;
  if (p.splits > 1 && (a.partial == nullptr || workspace_bytes < sizeof(float) * p.splits * S::C * static_cast<size_t>(p.padded)))
    return fail(WTCONV_E_WORKSPACE, "%s: workspace too small", fn);
  const int per = (a.hidden / S::HC + p.splits - 1) / p.splits;
  const size_t lds = S::lds_bytes(per * S::HC);
  if (lds > static_cast<size_t>(kLdsLimitBytes)) return fail(WTCONV_E_UNSUPPORTED, "%s: %d hidden units exceed the LDS", fn, a.hidden);
  const uintptr_t bits = reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.shortcut) | reinterpret_cast<uintptr_t>(a.out);
  a.vec = a.HW % 8 == 0 && bits % 16 == 0 ? 8 : (a.HW % 4 == 0 && bits % 8 == 0 ? 4 : 1);
  if (int e = allow_lds(block_mlp_kernel<S>, lds)) return e;
  WT_LAUNCH(block_mlp_kernel<S>, dim3(p.tiles, p.splits), dim3(S::kThreads), lds, stream, a);
  if (p.splits > 1)
    WT_LAUNCH(block_mlp_combine_kernel, dim3((a.pixels + 255) / 256, S::C), dim3(256), 0, stream, a, S::C);
  return check_launch(fn);
}

bool takes(int B, int C, int HW, int hidden) {
  // (fewer pixels than the tile of one wave: most of every product would be padding)
  if (B <= 0 || HW <= 0 || static_cast<long long>(B) * HW < 32 || hidden <= 0 || hidden % 64 != 0 || hidden > 4096) return false;
  // pixel indices and the offsets inside the images that a workgroup touches are 32-bit
  if (static_cast<long long>(B) * HW > (1LL << 30) || (256LL + 2LL * HW) * C > (1LL << 31)) return false;
#define WT_CASE(c, ...) if (C == c) return MlpShape<c, __VA_ARGS__>::lds_bytes(hidden) <= static_cast<size_t>(kLdsLimitBytes);
  WT_MLP_SHAPES(WT_CASE)
#undef WT_CASE
  return false;
}

}  // namespace

extern "C" int wtconv_block_mlp_supported(int B, int C, int HW, int hidden) { return takes(B, C, HW, hidden) ? 1 : 0; }

extern "C" size_t wtconv_block_mlp_workspace_bytes(int B, int C, int HW, int hidden) {
  if (!takes(B, C, HW, hidden)) return 0;
  MlpPlan p;
#define WT_CASE(c, ...) if (C == c) p = plan_of<MlpShape<c, __VA_ARGS__>>(B * HW, hidden);
  WT_MLP_SHAPES(WT_CASE)
#undef WT_CASE
  return p.splits > 1 ? sizeof(float) * p.splits * C * static_cast<size_t>(p.padded) : 0;
}

extern "C" int wtconv_block_mlp(const void* x, const void* shortcut, void* out, const wtconv_mlp_params* w, int B, int C,
                                int HW, int hidden, float eps, int dtype, int param_dtype, void* workspace,
                                size_t workspace_bytes, void* stream) {
  const char* fn = "wtconv_block_mlp";
  if (x == nullptr || shortcut == nullptr || out == nullptr || w == nullptr) return fail(WTCONV_E_ARG, "%s: null pointer", fn);
  if (!w->norm_weight || !w->norm_bias || !w->fc1_weight || !w->fc1_bias || !w->fc2_weight || !w->fc2_bias)
    return fail(WTCONV_E_ARG, "%s: null parameter", fn);
  if (out == x) return fail(WTCONV_E_ARG, "%s: in-place use is not supported", fn);
  if (dtype != WTCONV_BF16 || param_dtype != WTCONV_BF16) return fail(WTCONV_E_UNSUPPORTED, "%s: bfloat16 only", fn);
  if (!takes(B, C, HW, hidden)) return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d, hidden=%d", fn, C, hidden);
  uintptr_t bits = 0;
  for (const void* p : {w->norm_weight, w->norm_bias, w->fc1_weight, w->fc1_bias, w->fc2_weight, w->fc2_bias, w->gamma})
    bits |= reinterpret_cast<uintptr_t>(p);
  if (bits % 16) return fail(WTCONV_E_ARG, "%s: parameters must be 16-byte aligned", fn);
  MlpArgs a = {};
  a.x = static_cast<const bf16_t*>(x);
  a.shortcut = static_cast<const bf16_t*>(shortcut);
  a.out = static_cast<bf16_t*>(out);
  a.norm_w = static_cast<const bf16_t*>(w->norm_weight);
  a.norm_b = static_cast<const bf16_t*>(w->norm_bias);
  a.w1 = static_cast<const bf16_t*>(w->fc1_weight);
  a.b1 = static_cast<const bf16_t*>(w->fc1_bias);
  a.w2 = static_cast<const bf16_t*>(w->fc2_weight);
  a.b2 = static_cast<const bf16_t*>(w->fc2_bias);
  a.gamma = static_cast<const bf16_t*>(w->gamma);
  a.partial = static_cast<float*>(workspace);
  a.eps = eps;
  a.HW = HW;
  a.hidden = hidden;
  a.pixels = B * HW;
  hipStream_t s = static_cast<hipStream_t>(stream);
#define WT_CASE(c, ...) if (C == c) return launch<MlpShape<c, __VA_ARGS__>>(a, workspace_bytes, s);
  WT_MLP_SHAPES(WT_CASE)
#undef WT_CASE
  return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d", fn, C);
}
