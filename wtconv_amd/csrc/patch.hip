// Host side of the stem and downsample kernels (kernels_patch.h): argument checks, choice of the work split, launches.
#include "common.h"
#include "host_util.h"
#include "kernels_patch.h"
#include "../../include/wtconv_ops.h"

using namespace wt;

namespace {

// Downsample: the work splits of each channel count.  Measured, us, weights laid out included (Few / Mid / Many):
//   192 -> 384, images of 28 x 28: 1 6.2/10.3/16.6   4 10.3/10.2/16.0   16 26/13.4/16.3   64 81/23/20   256 327/78/61
//   384 -> 768, of 14 x 14:        1 9.7/16.4/37.9   8 18.0/19.0/40.7   16 29/19.6/40.4   64 104/46/41  256 354/127/80
//   96 -> 192, of 56 x 56:         1 5.0/6.8/9.9     4 8.0/7.4/9.9      16 21/10.4/10.9   64 76/30/24   256 290/106/60
// (at 256 images the input and output take 45, 23 and 11 at the rate of a copy, the separate passes about 300, 210 and 150).
// Few pixels: small tiles of pixels and channels, and K in parts, until a workgroup has little to do; they fetch rows of the weights
// as they lie, which is slow but saves a launch.  Mid: whole K, a few tiles of channels a workgroup.  Many: as many
// channels and pixels a workgroup as the registers and LDS allow, so that its weights serve more pixels.
template <int C> struct Split;
template <> struct Split<96> { using Few = PatchShape<96, 1, 2, 2, 1>; using Mid = PatchShape<96, 2, 4, 1, 1>; using Many = PatchShape<96, 4, 4, 1, 3>; };
template <> struct Split<128> { using Few = PatchShape<128, 1, 2, 2, 1>; using Mid = PatchShape<128, 2, 8, 1, 1>; using Many = PatchShape<128, 4, 8, 1, 2>; };
template <> struct Split<192> { using Few = PatchShape<192, 1, 2, 4, 1>; using Mid = PatchShape<192, 2, 8, 1, 1>; using Many = PatchShape<192, 2, 8, 1, 3>; };
template <> struct Split<256> { using Few = PatchShape<256, 1, 2, 4, 1>; using Mid = PatchShape<256, 2, 8, 1, 1>; using Many = PatchShape<256, 4, 16, 1, 2>; };
template <> struct Split<384> { using Few = PatchShape<384, 1, 2, 4, 1>; using Mid = PatchShape<384, 2, 8, 1, 1>; using Many = PatchShape<384, 2, 16, 1, 3>; };
template <> struct Split<512> { using Few = PatchShape<512, 1, 2, 4, 1>; using Mid = PatchShape<512, 2, 8, 1, 1>; using Many = PatchShape<512, 2, 8, 1, 8>; };
#define WT_PATCH_CHANNELS(X) X(96) X(128) X(192) X(256) X(384) X(512)

template <typename S>
long long workgroups(int pixels, int cout) { return static_cast<long long>((pixels + S::MP - 1) / S::MP) * (cout / S::COUT); }

// 0 Few, 1 Mid, 2 Many: as long as the finer split's workgroups are about one round of the compute units (Few's, of which
// several share one, two and a half), it ends sooner.
template <int C>
int split_of(int pixels, int cout) {
  using P = Split<C>;
  const int cus = compute_units();
  if (workgroups<typename P::Few>(pixels, cout) * 2 <= cus * 5 || cout % P::Mid::COUT) return 0;
  if (workgroups<typename P::Mid>(pixels, cout) * 4 <= cus * 5 || cout % P::Many::COUT) return 1;
  return 2;
}

// Whether that split is the faster way, and not the separate passes.  It is where the split is the one that the pixels ask for
// (Many takes 0.3 to 0.82 of their time up to 6144 output channels).  Output channels that are not whole groups of that split go
// by a finer one, which loads and normalises the input once for every 32 (Few) or 64 or 128 (Mid) of them.  Measured, time over that of the
// separate passes, by images of 14 x 14:
//   Few   96 ->  480   64 0.49   512 0.84   2048 1.01       96 ->  992   64 0.70   170 1.06     128 -> 480   512 0.92   2048 1.06
//        192 ->  224   64 0.45   512 0.88   2048 0.87      192 ->  480   64 0.76   170 1.20     192 -> 992    64 1.13
//        256 ->  224             512 0.83   2048 0.86      384 ->  224  512 0.90  2048 1.07     384 -> 416    64 0.98    170 1.28
//        512 ->  224  170 0.90   512 0.90   2048 1.22      512 ->  480   32 0.95    64 1.26     512 -> 992    16 0.64     32 1.33
//   Mid  256 -> 3200             512 0.96                  384 ->  640  512 0.86  2048 0.93     384 -> 896   256 0.93   2048 1.07
//        384 -> 2048   32 0.49    64 1.04   2048 1.41      512 ->  640  512 0.90  2048 1.03     512 -> 896   170 0.57    256 1.02
//        512 -> 1152  100 0.93   256 1.10                  512 -> 3200   32 0.59    64 1.21
template <int C>
bool pays(int pixels, int cout) {
  using P = Split<C>;
  const int cus = compute_units();
  const long long few = workgroups<typename P::Few>(pixels, cout), mid = workgroups<typename P::Mid>(pixels, cout);
  switch (split_of<C>(pixels, cout)) {
    case 0:
      if (few * 2 <= cus * 5 || few * C <= 900000) return true;
      if (cout <= 224) return C <= 256 || few * C <= 6000000;
      return C <= 128 && cout <= 480 && few * C <= 3100000;
    case 1:
      return C <= 256 || mid * 4 <= cus * 5 || mid <= (cout <= 640 ? 12000 : cout <= 896 ? 2700 : 1500);
    default:
      return true;
  }
}

template <typename S>
int launch(const PatchArgs& a, hipStream_t stream) {
  auto kern = norm_patch_kernel<S>;
  if (int e = allow_lds(kern, S::kLdsBytes)) return e;
  if (S::kLaidOut) WT_LAUNCH(patch_weights_kernel, dim3((a.cout / 16 * (S::K / 32) + 3) / 4), dim3(256), 0, stream, a, S::K);
  WT_LAUNCH(kern, dim3((a.pixels + S::MP - 1) / S::MP, a.cout / S::COUT), dim3(S::kThreads), S::kLdsBytes, stream, a);
  return 0;
}

template <int C>
int launch_split(const PatchArgs& a, hipStream_t stream) {
  switch (split_of<C>(a.pixels, a.cout)) {
    case 0: return launch<typename Split<C>::Few>(a, stream);
    case 1: return launch<typename Split<C>::Mid>(a, stream);
    default: return launch<typename Split<C>::Many>(a, stream);
  }
}

bool sizes_ok(int B, int C, int H, int W, int cout, int P) {
  if (B <= 0 || C <= 0 || H <= 0 || W <= 0 || cout <= 0 || H % P || W % P) return false;
  const long long plane = static_cast<long long>(H) * W;
  // pixel indices and the offsets inside an image are 32-bit
  return B * (plane / (P * P)) <= (1LL << 30) && plane * (C > cout ? C : cout) <= (1LL << 30);
}

bool takes_downsample(int B, int C, int H, int W, int cout) {
  if (!sizes_ok(B, C, H, W, cout, 2)) return false;
#define WT_CASE(c) if (C == c) return cout % Split<c>::Few::COUT == 0;
  WT_PATCH_CHANNELS(WT_CASE)
#undef WT_CASE
  return false;
}

// (rows of output pixels go four at a time)
bool takes_stem(int B, int C, int H, int W, int cout) {
  return sizes_ok(B, C, H, W, cout, 4) && W % 16 == 0 && C <= 4 && (cout == 96 || cout == 128);
}

template <typename S>
int launch_stem(const PatchArgs& a, hipStream_t stream) {
  auto kern = patch_norm_kernel<S>;
  const int groups = (a.pixels + S::PX - 1) / S::PX, wgs = (groups + S::kWaves - 1) / S::kWaves;
  const int most = compute_units() * resident_per_cu(kern, 64 * S::kWaves, 0);
  WT_LAUNCH(kern, dim3(wgs < most ? wgs : most), dim3(64 * S::kWaves), 0, stream, a);
  return 0;
}

}  // namespace

extern "C" int wtconv_ops_version(void) { return WTCONV_OPS_VERSION; }

extern "C" int wtconv_patch_conv_supported(int stem, int B, int C, int H, int W, int cout) {
  if (stem) return takes_stem(B, C, H, W, cout) ? 1 : 0;
  if (!takes_downsample(B, C, H, W, cout)) return 0;
#define WT_CASE(c) if (C == c) return pays<c>(B * (H / 2) * (W / 2), cout) ? 1 : 0;
  WT_PATCH_CHANNELS(WT_CASE)
#undef WT_CASE
  return 0;
}

extern "C" size_t wtconv_patch_conv_workspace_bytes(int stem, int B, int C, int H, int W, int cout) {
  if (stem || !takes_downsample(B, C, H, W, cout)) return 0;
  const int pixels = B * (H / 2) * (W / 2);
  bool laid_out = false;
#define WT_CASE(c) if (C == c) laid_out = split_of<c>(pixels, cout) > 0;
  WT_PATCH_CHANNELS(WT_CASE)
#undef WT_CASE
  return laid_out ? static_cast<size_t>(cout) * C * 4 * sizeof(bf16_t) : 0;
}

extern "C" int wtconv_patch_conv(int stem, const void* x, void* out, const wtconv_patch_params* w, int B, int C, int H, int W,
                                 int cout, float eps, int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                                 void* stream) {
  const char* fn = "wtconv_patch_conv";
  if (x == nullptr || out == nullptr || w == nullptr) return fail(WTCONV_E_ARG, "%s: null pointer", fn);
  if (!w->conv_weight || !w->conv_bias || !w->norm_weight || !w->norm_bias) return fail(WTCONV_E_ARG, "%s: null parameter", fn);
  if (out == x) return fail(WTCONV_E_ARG, "%s: in-place use is not supported", fn);
  if (dtype != WTCONV_BF16 || param_dtype != WTCONV_BF16) return fail(WTCONV_E_UNSUPPORTED, "%s: bfloat16 only", fn);
  if (stem ? !takes_stem(B, C, H, W, cout) : !takes_downsample(B, C, H, W, cout))
    return fail(WTCONV_E_UNSUPPORTED, "%s: no kernel for %d -> %d channels of %d x %d", fn, C, cout, H, W);
  uintptr_t bits = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out);
  for (const void* p : {w->conv_weight, w->conv_bias, w->norm_weight, w->norm_bias}) bits |= reinterpret_cast<uintptr_t>(p);
  if (bits % 16) return fail(WTCONV_E_ARG, "%s: tensors must be 16-byte aligned", fn);
  const size_t need = wtconv_patch_conv_workspace_bytes(stem, B, C, H, W, cout);
  if (need && (workspace == nullptr || workspace_bytes < need || reinterpret_cast<uintptr_t>(workspace) % 16))
    return fail(WTCONV_E_WORKSPACE, "%s: workspace too small or misaligned", fn);
  const int P = stem ? 4 : 2;
  PatchArgs a = {};
  a.x = static_cast<const bf16_t*>(x);
  a.out = static_cast<bf16_t*>(out);
  a.w = static_cast<const bf16_t*>(w->conv_weight);
  a.bias = static_cast<const bf16_t*>(w->conv_bias);
  a.norm_w = static_cast<const bf16_t*>(w->norm_weight);
  a.norm_b = static_cast<const bf16_t*>(w->norm_bias);
  a.eps = eps;
  a.frags = static_cast<bf16_t*>(workspace);
  a.cin = C; a.cout = cout; a.H = H; a.W = W; a.HO = H / P; a.WO = W / P;
  a.pixels = B * a.HO * a.WO;
  a.vec = (a.HO * a.WO) % 4 == 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  int rc = 0;
  if (stem) {
    rc = cout == 96 ? launch_stem<StemShape<6, 4>>(a, s) : launch_stem<StemShape<8, 2>>(a, s);
  } else {
#define WT_CASE(c) if (C == c) rc = launch_split<c>(a, s);
    WT_PATCH_CHANNELS(WT_CASE)
#undef WT_CASE
  }
  return rc ? rc : check_launch(fn);
}
