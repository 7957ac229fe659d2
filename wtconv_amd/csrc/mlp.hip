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

constexpr int kMaxHidden = 4096;

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

// ---- few pixels: two kernels (kernels_mlp_few.h), for these channel counts.  (Behind the shape: few_pays's limits, the hidden
// units up to which the pixels do not matter, and the most pixels times hidden units.)
#define WT_FEW_SHAPES(X) X(96, 2, 1, 768, 2 << 20) X(128, 2, 1, 256, 1280000) X(192, 2, 2, kMaxHidden, 2 << 20)       \
                         X(256, 2, 2, kMaxHidden, 2 << 20) X(384, 4, 2, kMaxHidden, 2 << 20) X(512, 4, 2, kMaxHidden, 1280000) \
                         X(768, 4, 2, kMaxHidden, 1280000) X(1024, 4, 2, kMaxHidden, 1 << 20)
constexpr long long kFewPixelChannels = 320000;
constexpr int kFewTiles = 2;

int few_tiles(int pixels) { return (pixels + 16 * kFewTiles - 1) / (16 * kFewTiles); }
size_t few_workspace(int pixels, int hidden) { return sizeof(bf16_t) * 16 * kFewTiles * static_cast<size_t>(few_tiles(pixels)) * hidden; }

bool has_few(int B, int C, int HW, int hidden) {
  if (B <= 0 || C <= 0 || HW <= 0 || hidden <= 0 || hidden % 64 != 0 || hidden > kMaxHidden) return false;
  // (fewer pixels than a tile: most of every product would be padding)
  const long long pixels = static_cast<long long>(B) * HW;
  if (pixels < 16 * kFewTiles || pixels > kFewPixelChannels / C) return false;
#define WT_CASE(c, ...) if (C == c) return true;
  WT_FEW_SHAPES(WT_CASE)
#undef WT_CASE
  return false;
}

// Whether the two kernels are the faster way.  Each tile of 32 pixels goes through all weights on its own, 2 C times the hidden
// units, while the one kernel's time hardly depends on the pixels before its workgroups fill the chip: the lines of equal time
// lie near a constant number of pixels * hidden units.  Measured (graph replay), us, two kernels / one kernel with its combination,
// from 512 channels the separate passes, pixels by hidden units:
//    96   196 x 384 7.7/12.1   3136 x 384 12.8/14.3   196 x 768 7.7/11.9   2500 x 768 15.5/17.8   3136 x 768 17.0/16.3
//   128   196 x 512 8.0/10.8   2500 x 512 15.4/16.9   224 x 4096 16.4/18.4   312 x 4096 17.1/16.2
//   192   196 x 768 8.5/15.5   1280 x 1024 14.5/20.6   512 x 4096 18.9/24.3   1280 x 2048 22.3/24.7   784 x 4096 33.9/21.8
//   256   196 x 1024 10.2/16.2   1024 x 2048 22.4/26.0   512 x 4096 21.0/25.3   640 x 4096 30.1/26.0
//   384   196 x 1536 11.9/23.2   784 x 1536 23.7/28.0   512 x 4096 29.7/32.2   784 x 2048 32.0/30.2   784 x 4096 47.9/33.1
//   512   196 x 2048 16.1/30.6   256 x 4096 23.9/34.3   312 x 4096 35.1/38.0   392 x 4096 40.8/37.5
//   768   49 x 3072 16.4/41.8   312 x 3072 28.1/38.0   312 x 4096 36.4/41.3   392 x 4096 47.2/43.9
//  1024   49 x 4096 20.6/55.7   256 x 4096 37.6/39.9   312 x 4096 50.5/43.4
// Of 208 other sizes of 192 to 384 channels five are over 5 % slower than the faster way, at most 10 %.  With 96 and 128 channels and
// more hidden units than the first limit the line dates from a slower pair of kernels and lies too low: there 65 of 154 sizes
// would be 5 to 48 % faster as two kernels (128, 196 x 768 8.1/13.2; 96, 1024 x 2048 12.8/17.1), up to about the 2 M of the others.
bool few_pays(int pixels, int C, int hidden) {
  const long long work = static_cast<long long>(pixels) * hidden;
#define WT_CASE(c, ng, kg, any, most) if (C == c) return hidden <= any ? work <= (most) : pixels >= 224 && work <= (1 << 20);
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
#define WT_CASE(c, ng, kg, ...)                                                                        \
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

// (The calls take every size with a kernel, also one at which the separate passes are faster.)
bool uses_few(int B, int C, int HW, int hidden) {
  return has_few(B, C, HW, hidden) && (few_pays(B * HW, C, hidden) || !takes(B, C, HW, hidden));
}

}  // namespace

extern "C" int wtconv_block_mlp_supported(int B, int C, int HW, int hidden) {
  return (has_few(B, C, HW, hidden) && few_pays(B * HW, C, hidden)) || takes(B, C, HW, hidden) ? 1 : 0;
}

extern "C" size_t wtconv_block_mlp_workspace_bytes(int B, int C, int HW, int hidden) {
  if (uses_few(B, C, HW, hidden)) return few_workspace(B * HW, hidden);
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
  const bool few = uses_few(B, C, HW, hidden);
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
