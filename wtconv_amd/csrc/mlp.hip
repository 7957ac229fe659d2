// Host side of the fused block kernel (kernels_mlp.h): argument checks, the split over the hidden units, launches.
#include "common.h"
#include "host_util.h"
#include "kernels_mlp.h"
#include "kernels_mlp_few.h"

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

constexpr int kMaxHidden = 4096;
template <typename S> constexpr size_t kRoomBytes = S::HC * sizeof(float);

// Whether LDS has room for one more slice of bias, with as many workgroups a CU as without.
template <typename S>
constexpr bool has_room(int hidden_here) {
#ifdef WT_EMULATE      // (exactly what is asked for)
  return false;
#else
  const size_t limit = kLdsLimitBytes, lds = S::lds_bytes(hidden_here);
  return lds + kRoomBytes<S> <= limit && limit / (lds + kRoomBytes<S>) == limit / lds;
#endif
}
template <typename S>
constexpr bool always_has_room() {
  for (int h = S::HC; h <= kMaxHidden; h += S::HC)
    if (!has_room<S>(h)) return false;
  return true;
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
  const dim3 grid(p.tiles, p.splits);
  if (has_room<S>(per * S::HC)) {
    auto kern = block_mlp_kernel<S, true>;
    if (int e = allow_lds(kern, lds + kRoomBytes<S>)) return e;
    WT_LAUNCH(kern, grid, dim3(S::kThreads), lds + kRoomBytes<S>, stream, a);
  } else if constexpr (!always_has_room<S>()) {
    auto kern = block_mlp_kernel<S, false>;
    if (int e = allow_lds(kern, lds)) return e;
    WT_LAUNCH(kern, grid, dim3(S::kThreads), lds, stream, a);
  }
  if (p.splits > 1)
    WT_LAUNCH(block_mlp_combine_kernel, dim3((a.pixels + 255) / 256, S::C), dim3(256), 0, stream, a, S::C);
  return check_launch(fn);
}

// ---- few pixels: two kernels (kernels_mlp_few.h), for these channel counts and as many pixels as make them the faster way.
// Each tile of 32 pixels goes through all weights, 8 C^2 of them, on its own, while the one kernel's time hardly depends on the
// pixels before its workgroups fill the chip; the lines of equal time lie near a constant pixels * C.  Measured (graph
// replay), us, two kernels / one kernel with its combination, from 512 channels the separate passes:
//   96 channels, 3136 pixels 12.4/13.5, 6272 16.0/16.1     128, 3136 17.6/17.5          192, 784 11.2/20.1, 3136 24.3/25.1
//   256, 784 16.8/23.3, 3136 43/27.6                       384, 196 11.3/22.6, 784 24.3/28.5, 1568 38.4/31.5
//   512, 196 17.0/29.6, 784 41.1/37.2                      768, 49 15.3/41.0, 392 38.3/52.6      1024, 49 19.9/55.5, 392 66/63
#define WT_FEW_SHAPES(X) X(96, 2, 1) X(128, 2, 1) X(192, 2, 2) X(256, 2, 2) X(384, 4, 2) X(512, 4, 2) X(768, 4, 2) X(1024, 4, 2)
constexpr long long kFewPixelChannels = 320000;
constexpr int kFewTiles = 2;

int few_tiles(int pixels) { return (pixels + 16 * kFewTiles - 1) / (16 * kFewTiles); }
size_t few_workspace(int pixels, int hidden) { return sizeof(bf16_t) * 16 * kFewTiles * static_cast<size_t>(few_tiles(pixels)) * hidden; }

bool takes_few(int B, int C, int HW, int hidden) {
  if (B <= 0 || C <= 0 || HW <= 0 || hidden <= 0 || hidden % 64 != 0 || hidden > kMaxHidden) return false;
  // (fewer pixels than a tile: most of every product would be padding)
  const long long pixels = static_cast<long long>(B) * HW;
  if (pixels < 16 * kFewTiles || pixels > kFewPixelChannels / C) return false;
#define WT_CASE(c, ...) if (C == c) return true;
  WT_FEW_SHAPES(WT_CASE)
#undef WT_CASE
  return false;
}

int launch_few(const MlpArgs& m, int C, size_t workspace_bytes, hipStream_t stream) {
  const char* fn = "wtconv_block_mlp";
  const size_t need = few_workspace(m.pixels, m.hidden);
  if (m.partial == nullptr || workspace_bytes < need || reinterpret_cast<uintptr_t>(m.partial) % 16)
    return fail(WTCONV_E_WORKSPACE, "%s: workspace too small or misaligned", fn);
  FewArgs a = {};
  a.x = m.x; a.shortcut = m.shortcut; a.out = m.out;
  a.norm_w = m.norm_w; a.norm_b = m.norm_b;
  a.w1 = m.w1; a.b1 = m.b1; a.w2 = m.w2; a.b2 = m.b2; a.gamma = m.gamma;
  a.hid = reinterpret_cast<bf16_t*>(m.partial);
  a.eps = m.eps;
  a.HW = m.HW; a.C = C; a.hidden = m.hidden; a.pixels = m.pixels;
  const uintptr_t bits = reinterpret_cast<uintptr_t>(a.shortcut) | reinterpret_cast<uintptr_t>(a.out);
  a.vec = a.HW % 4 == 0 && bits % 8 == 0;
  const int tiles = few_tiles(a.pixels);
#define WT_CASE(c, ng, kg)                                                                             \
  if (C == c) {                                                                                        \
    using S = FewShape<c, kFewTiles, ng, kg>;                                                          \
    auto kern = few_hidden_kernel<S>;                                                                  \
    if (int e = allow_lds(kern, S::kLdsBytes)) return e;                                               \
    WT_LAUNCH(kern, dim3(tiles, a.hidden / (16 * ng)), dim3(S::kThreads), S::kLdsBytes, stream, a);    \
  }
  WT_FEW_SHAPES(WT_CASE)
#undef WT_CASE
  // (four waves until each has eight steps of 32 hidden units)
  if (a.hidden < 1024) {
    auto kern = few_out_kernel<kFewTiles, 4>;
    WT_LAUNCH(kern, dim3(tiles, C / 16), dim3(256), 0, stream, a);
  } else {
    auto kern = few_out_kernel<kFewTiles, 8>;
    WT_LAUNCH(kern, dim3(tiles, C / 16), dim3(512), 0, stream, a);
  }
  return check_launch(fn);
}

// Beyond those no line is drawn by size: at 96, 128, 192, 256 and 384 channels with four hidden units each, batches of 1 to 256 and planes
// of 7 x 7 to 56 x 56 and 13 x 11, the kernel takes 0.26 to 0.88 of the time of the separate passes (graph replay; less of it
// when launched one by one), and up to 0.93 with 4096 hidden units.  With 64 it took 1.08 and 1.09 of it in two of fifteen cases
// (256 channels, 16 images of 28 x 28; 384 channels, 64 of 14 x 14), 34.5 and 44.3 us.
bool takes(int B, int C, int HW, int hidden) {
  // (fewer pixels than the tile of one wave: most of every product would be padding)
  if (B <= 0 || HW <= 0 || static_cast<long long>(B) * HW < 32 || hidden <= 0 || hidden % 64 != 0 || hidden > kMaxHidden) return false;
  // pixel indices and the offsets inside the images that a workgroup touches are 32-bit
  if (static_cast<long long>(B) * HW > (1LL << 30) || (256LL + 2LL * HW) * C > (1LL << 31)) return false;
#define WT_CASE(c, ...) if (C == c) return MlpShape<c, __VA_ARGS__>::lds_bytes(hidden) <= static_cast<size_t>(kLdsLimitBytes);
  WT_MLP_SHAPES(WT_CASE)
#undef WT_CASE
  return false;
}

}  // namespace

extern "C" int wtconv_block_mlp_supported(int B, int C, int HW, int hidden) {
  return takes_few(B, C, HW, hidden) || takes(B, C, HW, hidden) ? 1 : 0;
}

extern "C" size_t wtconv_block_mlp_workspace_bytes(int B, int C, int HW, int hidden) {
  if (takes_few(B, C, HW, hidden)) return few_workspace(B * HW, hidden);
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
  const bool few = takes_few(B, C, HW, hidden);
  if (!few && !takes(B, C, HW, hidden)) return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d, hidden=%d", fn, C, hidden);
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
  if (few) return launch_few(a, C, workspace_bytes, s);
#define WT_CASE(c, ...) if (C == c) return launch<MlpShape<c, __VA_ARGS__>>(a, workspace_bytes, s);
  WT_MLP_SHAPES(WT_CASE)
#undef WT_CASE
  return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for C=%d", fn, C);
}
