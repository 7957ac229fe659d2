// C ABI of libwtconv_hip.so (declared in include/wtconv_hip.h): argument checks, LDS
// planning and kernel launches.  Nothing here allocates, frees or synchronises.
#include <stdlib.h>
#include <string.h>

#include <mutex>

#include "common.h"
#include "host_util.h"
#include "launch.h"
#include "../../include/wtconv_ops.h"
#include "mfma2d.h"
#include "kernels1d.h"
#include "kernels1d_row.h"
#include "kernels2d.h"
#include "kernels2d_stream.h"
#include "plan.h"
#ifdef WT_EMULATE      // one translation unit for the host build
#include "conv1d.hip"
#include "plane2d.hip"
#include "stream2d.hip"
#include "wgrad2d.hip"
#endif

namespace wt {

// Threads of wgrad_finish_kernel: one per entry of a channel's record (taps of every filter + sumG) where that fits.
static inline int finish_threads(int nrec) { return nrec >= 1024 ? 1024 : (nrec + kWave - 1) / kWave * kWave; }

static inline bool known_dtype(int d) { return d == WTCONV_F32 || d == WTCONV_BF16 || d == WTCONV_F16; }

static int check_common(const char* fn, const wtconv_params* params, int B, int C, int K, int L,
                        int dtype, int pdtype) {
  if (B <= 0 || C <= 0) return fail(WTCONV_E_ARG, "%s: batch and channels must be positive (got %d, %d)", fn, B, C);
  if (K < 1 || K % 2 == 0) return fail(WTCONV_E_ARG, "%s: kernel_size must be odd and positive (got %d)", fn, K);
  if (K > wtconv_max_kernel_size())
    return fail(WTCONV_E_UNSUPPORTED, "%s: kernel_size %d exceeds the largest built kernel (%d)", fn, K,
                wtconv_max_kernel_size());
  if (L < 1 || L > kMaxLevels) return fail(WTCONV_E_ARG, "%s: wt_levels must be 1-%d (got %d)", fn, kMaxLevels, L);
  if (!known_dtype(dtype)) return fail(WTCONV_E_ARG, "%s: unknown dtype %d", fn, dtype);
  if (!known_dtype(pdtype)) return fail(WTCONV_E_ARG, "%s: unknown param dtype %d", fn, pdtype);
  if (params == nullptr || params->base_weight == nullptr || params->base_scale == nullptr)
    return fail(WTCONV_E_ARG, "%s: null parameter pointer", fn);
  for (int l = 0; l < L; ++l)
    if (params->wt_weight[l] == nullptr || params->wt_scale[l] == nullptr)
      return fail(WTCONV_E_ARG, "%s: null parameter pointer at level %d", fn, l);
  return 0;
}

// How the plane-resident parameter-gradient kernel walks a channel's B planes: pb an iteration, `bchunk` a workgroup, which
// makes `nchunk` workgroups a channel.
struct WgradSplit { int pb, bchunk, nchunk; };

static WgradSplit wgrad_split(int B, int C, int H, int W, int K, int L) {
  constexpr int kPlannedCUs = 256;      // a constant, so that workspace sizes do not depend on the device queried
  WgradSplit s = {wgrad_planes_that_fit(B, H, W, K, L), 0, 0};
  if (!wgrad_is_alone(K, L)) {
    // Two workgroups a CU, one where an iteration's planes take more than half of the LDS.  (Planned for two while one ran, the
    // chunks made two rounds, and each workgroup's fixed parts were paid twice: [23,29,75,60] fp16, K = 5, two levels
    // 43 -> 31 us, [16,40,61,69] fp32 48 -> 37, [6,58,100,85] one level 36 -> 30, [4,368,79,98] K = 3, five levels 99 -> 84.)
    const Plan2D t = make_plan2d_geometry(s.pb, 1, H, W, K, L, true, 512, s.pb);
    const bool one = static_cast<size_t>(t.plane_lds_floats) * 4 > static_cast<size_t>(kLdsLimitBytes) / 2;
    wgrad_chunks(B, C, s.pb, kPlannedCUs * (one ? 1 : 2), &s.bchunk, &s.nchunk);
    return s;
  }
  // One workgroup a CU, with as many planes an iteration as suit the chunks, of up to four rounds of the chip: the split of
  // least time by a model of it, in microseconds 13 a round (clearing LDS, a first load with nothing beside it, the
  // reduction), 4 an iteration and 1.6 per 1000 pixels in it (a third of that goes by the places for planes, a power of two,
  // of which the kernel deals each the same threads), 0.2 a chunk for the last workgroup's sums.  Of 90 drawn shapes, each
  // measured with every number of planes and one to four rounds, it takes 0.4 % longer than the best split at the geometric
  // mean and up to 5 %, once 11.  Of the time with planes for 80 KB and chunks for two workgroups a CU it takes 0.86 over 400 other
  // drawn shapes, at most 1.10 ([46,10,16,18], three levels, 24 -> 27 us; [256,270,6,5] 164 -> 180): [16,72,45,37] fp16, two levels, 59 -> 46, [41,89,13,13] three
  // levels 57 -> 34, [52,86,20,22] four 87 -> 68, [103,44,39,48] fp32, three 147 -> 117, [34,350,31,27] four 245 -> 181.
  const int fit = s.pb, most = B < 64 ? B : 64, four = 4 * kPlannedCUs / C;
  float best = 0.f;
  for (int n = 1; n <= (four < most ? four : most) || n == 1; ++n) {
    const int planes = (B + n - 1) / n, iters = (planes + fit - 1) / fit, even = (planes + iters - 1) / iters, slots = pow2_ceil(even);
    for (int pb = even;; pb = slots / 2) {
      const int its = (planes + pb - 1) / pb, nn = (B + its * pb - 1) / (its * pb), rounds = (C * nn + kPlannedCUs - 1) / kPlannedCUs;
      const float places = 0.65f * pb + 0.35f * pow2_ceil(pb);
      const float cost = rounds * (13.f + its * (4.f + places * 0.0016f * H * W)) + 0.2f * nn;
      if (s.nchunk == 0 || cost < best) { best = cost; s = {pb, its * pb, nn}; }
      if (pb != even || even == slots) break;
    }
  }
  return s;
}

static size_t fold_floats(int C, int S, int L, int KK) { return static_cast<size_t>(C) * (1 + S * L) * KK + C; }

// Folded filters as the plane kernel writes them itself (PlaneFold): each channel's table on cache lines of its own.
constexpr int kFoldInsidePlanes = 512;
static size_t folded_tables(int C, int L, int KK) { return static_cast<size_t>(C) * (((1 + 4 * L) * KK + 31) / 32 * 32); }

static int launch_fold(const wtconv_params* params, int pdtype, float* fw, float* fb, int C, int S, int L,
                       int KK, int flip, int use_bias, hipStream_t stream, unsigned* zero_words = nullptr,
                       int nzero = 0) {
  const int total = C * (1 + S * L) * KK;
  int blocks = (total + 255) / 256;
  if (blocks > 1024) blocks = 1024;
  WT_LAUNCH(fold_params_kernel, dim3(blocks), dim3(256), 0, stream, to_table(params, L), pdtype, fw, fb, C, S, L,
            KK, flip, use_bias, zero_words, zero_words != nullptr ? nzero : 0);
  return check_launch("fold_params_kernel");
}

// ---- planes that do not fit LDS: one level at a time until the rest does (kernels2d_stream.h) ----------
static size_t lds_fit_limit(size_t limit) {
#ifdef WT_EMULATE   // host emulation only: send small planes through the step kernels
  if (const char* e = getenv("WT_EMU_LDS_LIMIT")) return static_cast<size_t>(atol(e));
#endif
  return limit;
}

static size_t plane_lds_bytes(int B, int C, int H, int W, int K, int L) {
  return static_cast<size_t>(make_plan2d(B, C, H, W, K, L, false, 256).plane_lds_floats) * 4;
}

// Planes that the plane-resident kernel takes: two of them fit a CU's LDS.  With one, nothing hides its phases' latency,
// and taking the first level as a step of its own is faster, us forward: 96x96 (16 images of 64 channels, fp32, K = 5,
// three levels) 81 -> 70, 112x112 (12 images) 83 -> 70, 99x83 (16, fp16) 146 -> 82.  At three to a CU it is not: 80x80
// 53.5 resident, 56.5 in steps.
static bool plane_fits_lds(int B, int C, int H, int W, int K, int L) {
  return row_lanes(W) <= kMaxPlaneThreads && plane_lds_bytes(B, C, H, W, K, L) <= lds_fit_limit(kLdsLimitBytes / 2);
}

// The parameter-gradient kernel (512 threads) keeps planes that fit alone: 128x128 fp32 training step 179 us, 185 with
// one level more as a step.
static bool wgrad_fits_lds(int B, int C, int H, int W, int K, int L) {
  if (W > kMaxWgradWidth) return false;
  Plan2D pl = make_plan2d(B, C, H, W, K, L, true, 512);
  return static_cast<size_t>(pl.plane_lds_floats) * 4 <= lds_fit_limit(kLdsLimitBytes);
}

constexpr long long kMaxPlaneElems = 1LL << 28;

// Workgroups of stream_corr_kernel that run at once (two per CU on 256 CUs; a constant, as workspace sizes must not depend on
// the device queried): one round of them, at most one per batch item and 16 x 64 coefficients.
constexpr int kStreamResident = 512;
static int stream_chunks(int B, int C, int H, int W) {
  const long long units = static_cast<long long>(B) * ((H + 31) / 32) * ((W + 127) / 128);
  long long want = kStreamResident / C;
  if (want > units) want = units;
  return static_cast<int>(want < 1 ? 1 : want);
}

// Planes beyond LDS: how many levels are taken one at a time (kernels2d_stream.h) until what is left fits -- the layer
// itself (`depth`), its parameter gradients, which need two pyramids (`wdepth`) --, and where the workspace keeps what
// goes from step to step: LL bands of x (or grad_out) and results of the sub-layers, (B * C, h_d, w_d) each.
struct Stream2D {
  int h[kMaxLevels + 1], w[kMaxLevels + 1];
  int depth, wdepth;
  size_t ll[kMaxLevels + 1];     // offsets in floats from the start of an area of `floats`
  size_t floats;
};

static Stream2D make_stream2d(int B, int C, int H, int W, int K, int L) {
  Stream2D s = {};
  s.h[0] = H; s.w[0] = W;
  size_t off = 0;
  for (int l = 1; l <= L; ++l) {
    s.h[l] = (s.h[l - 1] + 1) / 2;
    s.w[l] = (s.w[l - 1] + 1) / 2;
    s.ll[l] = off;
    off += round_up64(static_cast<size_t>(B) * C * s.h[l] * s.w[l]);
  }
  s.floats = off;
  while (s.depth < L && !plane_fits_lds(B, C, s.h[s.depth], s.w[s.depth], K, L - s.depth)) ++s.depth;
  while (s.wdepth < L && !wgrad_fits_lds(B, C, s.h[s.wdepth], s.w[s.wdepth], K, L - s.wdepth)) ++s.wdepth;
  return s;
}

// Planes beyond LDS: the four bands of every level, which calls once kept in their workspace.  The sizes they ask for are
// never less, so that the shapes refused for want of static scratch are the same.
static size_t four_band_floats(int B, int C, int H, int W, int K, int L) {
  if (plane_lds_bytes(B, C, H, W, K, L) <= static_cast<size_t>(kLdsLimitBytes)) return 0;
  const Stream2D s = make_stream2d(B, C, H, W, K, L);
  size_t area = 0;
  for (int l = 1; l <= L; ++l) area += round_up64(static_cast<size_t>(B) * C * s.h[l] * s.w[l] * (l < L ? 5 : 4));
  return area;
}

// Partial sums of the steps, then those of the plane-resident sub-layer.
static size_t stream_records(int B, int C, int H, int W, int K, int L) {
  return round_up64(static_cast<size_t>(stream_chunks(B, C, H, W)) * C * ((1 + 4 * L) * K * K + 1));
}
static size_t stream_sub_records(const Stream2D& s, int B, int C, int K, int L) {
  if (s.wdepth == L) return 0;
  const int d = s.wdepth;
  return round_up64(static_cast<size_t>(wgrad_split(B, C, s.h[d], s.w[d], K, L - d).nchunk) * C * ((1 + 4 * (L - d)) * K * K + 1));
}

// choose_plane_shape's answer, kept for the sizes asked for last: it weighs up to twenty pairs, two microseconds of host time that
// a small call would show.
static void plane_shape(const Plan2D& pl, int K, int* tj1, int* sg_shift) {
  struct Known { int B, C, H, W, K, L, tj1, sg_shift; };
  static thread_local Known known[64] = {};
  const unsigned at = (pl.B * 31u + pl.C) * 31u + pl.H * 97u + pl.W * 7u + K * 5u + pl.L;
  Known& k = known[(at ^ at >> 6) % 64];
  if (k.B != pl.B || k.C != pl.C || k.H != pl.H || k.W != pl.W || k.K != K || k.L != pl.L) {
    k = {pl.B, pl.C, pl.H, pl.W, K, pl.L, 4, 8};
    choose_plane_shape(pl, K, &k.tj1, &k.sg_shift);
  }
  *tj1 = k.tj1;
  *sg_shift = k.sg_shift;
}

// One launch of the plane-resident kernels on planes that fit LDS; `fw` / `fb` folded parameters, those of a channel
// `fw_stride` floats from the next one's, the level filters `fw_skip` floats behind their usual place.
static int resident2d(const char* fn, const void* x, void* out, const float* fw, const float* fb, int B, int C, int H,
                      int W, int K, int L, int dtype, int fw_stride, int fw_skip, hipStream_t stream,
                      const PlaneFold& fold = PlaneFold{}) {
  Plan2D pl = make_plan2d(B, C, H, W, K, L, false, 256);
  int tj1 = 4, sg_shift = 8;
  if (plane_shape_is_static(K, H, W, L)) static_plane_shape(H, &tj1, &sg_shift);
  else plane_shape(pl, K, &tj1, &sg_shift);
  finish_plane_plan(&pl, tj1, sg_shift);
  pl.fw_stride = fw_stride;
  pl.fw_skip = fw_skip;
  if (static_cast<size_t>(pl.lds_floats) * 4 > kLdsLimitBytes)
    return fail(WTCONV_E_UNSUPPORTED,
                "%s: a %dx%d plane with %d levels needs %zu B of LDS (limit %d); plane too large for the "
                "plane-resident kernels", fn, H, W, L, static_cast<size_t>(pl.lds_floats) * 4, kLdsLimitBytes);
  if (row_lanes(W) > (1 << pl.sg_shift) || pl.block > kMaxPlaneThreads)      // (rows are walked whole)
    return fail(WTCONV_E_UNSUPPORTED, "%s: rows of %d pixels are too long for the plane-resident kernels", fn, W);
  return launch_plane2d(dtype, K, tj1, x, out, fw, fb, pl, fold, stream);
}

// The layer on planes beyond LDS.  `ll` and `res`: areas of make_stream2d (LL bands, results of the sub-layers).
static int stream2d_pass(const char* fn, const Stream2D& sp, const void* x, void* out, const float* fw, const float* fb,
                         float* ll, float* res, int B, int C, int K, int L, int dtype, hipStream_t stream) {
  const int KK = K * K, D = sp.depth, fstride = (1 + 4 * L) * KK;
  auto type_at = [&](int d) { return d == 0 ? dtype : WTCONV_F32; };
  auto in_at = [&](int d) { return d == 0 ? x : static_cast<const void*>(ll + sp.ll[d]); };
  auto base_at = [&](int d) { return d == 0 ? 0 : (1 + 4 * (d - 1)) * KK; };     // filter that is step d's base conv
  for (int d = 0; d < D && d + 1 < L; ++d)
    if (int e = launch_stream_ll(type_at(d), in_at(d), sp.h[d], sp.w[d], ll + sp.ll[d + 1], B * C, stream)) return e;
  if (D < L)
    if (int e = resident2d(fn, in_at(D), res + sp.ll[D], fw + base_at(D), nullptr, B, C, sp.h[D], sp.w[D], K, L - D,
                           WTCONV_F32, fstride, 3 * KK, stream)) return e;
  for (int d = D - 1; d >= 0; --d) {
    const StreamStep st = {B, C, sp.h[d], sp.w[d]};
    void* to = d == 0 ? out : static_cast<void*>(res + sp.ll[d]);
    if (int e = launch_stream_final(type_at(d), K, st, in_at(d), to, d + 1 < L ? res + sp.ll[d + 1] : nullptr, fw,
                                    d == 0 ? fb : nullptr, fstride, base_at(d), (1 + 4 * d) * KK, stream)) return e;
  }
  return 0;
}

// `shared_ll` (planes beyond LDS only): where to leave the LL bands for a later pass of the same call; the folded
// parameters and the results of the sub-layers then go to `shared_fw` instead of the workspace start.
// `resident`: planes that fit LDS alone run on the plane-resident kernel, which needs room for the folded parameters only.
// `tickets` (plane-resident paths only): C words this pass clears on its way, for the parameter-gradient pass that
// follows it on the stream; they must lie outside the folded parameters at the workspace start.
static int plane2d_pass(const char* fn, const void* x, void* out, const wtconv_params* params, int B, int C,
                        int H, int W, int K, int L, int dtype, int pdtype, void* ws, size_t ws_bytes,
                        void* stream_, int flip, float* shared_ll = nullptr, float* shared_fw = nullptr,
                        unsigned* tickets = nullptr, bool resident = false) {
  if (int e = check_common(fn, params, B, C, K, L, dtype, pdtype)) return e;
  if (H <= 0 || W <= 0) return fail(WTCONV_E_ARG, "%s: spatial size must be positive (got %dx%d)", fn, H, W);
  if (static_cast<long long>(H) * W > kMaxPlaneElems)   // 32-bit offsets inside a plane and its four stacked sub-bands
    return fail(WTCONV_E_UNSUPPORTED, "%s: a plane of %dx%d exceeds 2^28 elements", fn, H, W);
  if (x == nullptr || out == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
  const size_t esz = dtype == WTCONV_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(x) % esz) || (reinterpret_cast<uintptr_t>(out) % esz))
    return fail(WTCONV_E_ARG, "%s: tensor pointer not aligned to its element size", fn);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  const size_t need = resident ? fold_floats(C, 4, L, K * K) * sizeof(float)
                               : wtconv2d_workspace_bytes(B, C, H, W, K, L, flip ? WTCONV_PASS_BACKWARD_INPUT : WTCONV_PASS_FORWARD);
  if (ws == nullptr || ws_bytes < need)
    return fail(WTCONV_E_WORKSPACE, "%s: workspace of %zu B needed, %zu given", fn, need, ws_bytes);
  if (static_cast<long long>(B) * C > 0x7fffffffLL / 4)
    return fail(WTCONV_E_UNSUPPORTED, "%s: batch*channels = %lld is too large", fn, static_cast<long long>(B) * C);
  if (mfma2d_query(B, C, H, W, K, L, dtype).ok)
    return mfma2d_pass(fn, x, out, params, B, C, H, W, K, L, dtype, pdtype, stream, flip, tickets, C);
  if (!resident && !plane_fits_lds(B, C, H, W, K, L)) {
    const Stream2D sp = make_stream2d(B, C, H, W, K, L);
    float* fw = shared_ll != nullptr ? shared_fw : static_cast<float*>(ws);
    float* fb = fw + static_cast<size_t>(C) * (1 + 4 * L) * K * K;
    float* res = fw + round_up64(fold_floats(C, 4, L, K * K));
    float* ll = shared_ll != nullptr ? shared_ll : res + sp.floats;
    if (int e = launch_fold(params, pdtype, fw, fb, C, 4, L, K * K, flip, flip ? 0 : 1, stream)) return e;
    return stream2d_pass(fn, sp, x, out, fw, fb, ll, res, B, C, K, L, dtype, stream);
  }
  float* fw = static_cast<float*>(ws);
  float* fb = fw + static_cast<size_t>(C) * (1 + 4 * L) * K * K;
  // A small forward launch folds its parameters itself: the fold kernel and the gap behind it are a quarter of it, us
  // [8,32,64,64] fp32, K = 5, three levels 18.1 -> 13.9.  With more planes than one for a CU the launch is the cheaper way.
  if (!flip && tickets == nullptr && static_cast<long long>(B) * C <= kFoldInsidePlanes && !plane_shape_is_static(K, H, W, L) &&
      reinterpret_cast<uintptr_t>(ws) % 128 == 0 && ws_bytes >= folded_tables(C, L, K * K) * sizeof(float)) {
    const PlaneFold fold = {static_cast<float*>(ws), to_table(params, L), pdtype};
    return resident2d(fn, x, out, nullptr, nullptr, B, C, H, W, K, L, dtype, static_cast<int>(folded_tables(1, L, K * K)), 0,
                      stream, fold);
  }
  if (int e = launch_fold(params, pdtype, fw, fb, C, 4, L, K * K, flip, flip ? 0 : 1, stream, tickets, C)) return e;
  return resident2d(fn, x, out, fw, fb, B, C, H, W, K, L, dtype, (1 + 4 * L) * K * K, 0, stream);
}

// ---- row-resident 1-D kernels ----------------------------------------------------------
// Rows of any length run on the register-resident kernels, those longer than a workgroup in segments of about equal
// length; K = 1, whose convolutions have no neighbours to fetch, uses the tiled ones.  (Measured down to rows of four
// lanes, 64 samples: 16.9 us against 35.4 on tiles for [256,64,64] float32, K = 5, three levels.)
struct Row1DShape { int S, block; Row1D pl; };

static bool row1d_shape(int C, int N, int K, int L, Row1DShape* sh) {
  if (K < 3 || K > 7 || L < 1 || L > kMaxLevels || N <= 0) return false;
  const int S = row1d_samples(L);
  const int n = N / S + (N % S != 0 ? 1 : 0);
  const bool one = n <= kRow1dMaxLanes;
  const int hal = one ? 0 : row1d_guard(K, L, S);
  const int most = kRow1dMaxLanes - 2 * hal;
  Row1D& r = sh->pl;
  r.C = C; r.N = N; r.hal = hal;
  r.nseg = one ? 1 : (n + most - 1) / most;
  r.use = (n + r.nseg - 1) / r.nseg;
  r.nl = r.use + 2 * hal;
  sh->S = S;
  sh->block = (r.nl + 63) / 64 * 64;
  return true;
}

// Workgroups per CU the kernels with two slot regions (parameter gradients, fused backward) are planned for: what
// LDS allows, at most two waves per SIMD (they need up to 256 registers).
static int row1d_two_region_per_cu(int K, int L, const Row1DShape& sh) {
  const size_t lds = 2 * row1d_region(K, L, sh.S, sh.block) * sizeof(float);
  int per_cu = static_cast<int>(kLdsLimitBytes / lds);
  if (per_cu > 512 / sh.block) per_cu = 512 / sh.block;
  return per_cu < 1 ? 1 : per_cu;
}

static int tile1d_pass(const char* fn, const void* x, void* out, const wtconv_params* params, int B, int C,
                       int N, int K, int L, int dtype, int pdtype, void* ws, size_t ws_bytes, void* stream_,
                       int flip) {
  if (int e = check_common(fn, params, B, C, K, L, dtype, pdtype)) return e;
  if (N <= 0) return fail(WTCONV_E_ARG, "%s: length must be positive (got %d)", fn, N);
  if (x == nullptr || out == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
  const size_t esz = dtype == WTCONV_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(x) % esz) || (reinterpret_cast<uintptr_t>(out) % esz))
    return fail(WTCONV_E_ARG, "%s: tensor pointer not aligned to its element size", fn);
  Row1DShape sh = {};
  const bool row_resident = row1d_shape(C, N, K, L, &sh);
  const Plan1D pl = make_plan1d(C, N, L, false, esz, x, out, nullptr);
  const size_t need = wtconv1d_workspace_bytes(B, C, N, K, L, flip ? WTCONV_PASS_BACKWARD_INPUT : WTCONV_PASS_FORWARD);
  if (ws == nullptr || ws_bytes < need)
    return fail(WTCONV_E_WORKSPACE, "%s: workspace of %zu B needed, %zu given", fn, need, ws_bytes);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  if (row_resident) {      // (these kernels fold their channel's parameters themselves: no fold launch, no table)
    return launch_row1d(dtype, K, L, x, out, params, pdtype, flip, sh.pl, B, sh.block, stream);
  }
  float* fw = static_cast<float*>(ws);
  float* fb = fw + static_cast<size_t>(C) * (1 + 2 * L) * K;
  if (int e = launch_fold(params, pdtype, fw, fb, C, 2, L, K, flip, flip ? 0 : 1, stream)) return e;
  return launch_tile1d(dtype, x, out, fw, fb, pl, B, stream);
}

// ---- static scratch for callers that may not allocate ------------------------------------
// One array per GPU the library runs on, held until the process ends.  Host code never uses the
// array's name as an address: the device address is looked up once per device and cached.
constexpr size_t kStaticScratchBytes = 4u << 20;
constexpr int kMaxDevices = 64;
#ifndef WT_EMULATE
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];
static std::mutex g_scratch_mutex;
static void* g_scratch_ptr[kMaxDevices];

static int static_scratch(const char* fn, void** ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return fail(WTCONV_E_LAUNCH, "%s: hipGetDevice: %s", fn, hipGetErrorString(e));
  if (dev < 0 || dev >= kMaxDevices) return fail(WTCONV_E_UNSUPPORTED, "%s: device index %d", fn, dev);
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr)
      return fail(WTCONV_E_LAUNCH, "%s: hipGetSymbolAddress(scratch): %s", fn, hipGetErrorString(e));
    g_scratch_ptr[dev] = p;
  }
  *ptr = g_scratch_ptr[dev];
  return 0;
}
#else
static unsigned char scratch[kStaticScratchBytes];
static int static_scratch(const char*, void** ptr) { *ptr = scratch; return 0; }
#endif

static int check_grad_dtype(const char* fn, const wtconv_typed_grads* grads) {
  if (grads->dtype != WTCONV_F32 && grads->dtype != WTCONV_BF16 && grads->dtype != WTCONV_F16)
    return fail(WTCONV_E_ARG, "%s: unknown gradient dtype %d", fn, grads->dtype);
  return 0;
}

// The gradients of the untyped entry points: float.
struct FloatGrads {
  wtconv_typed_grads t = {};
  const wtconv_typed_grads* ptr = nullptr;
  FloatGrads(const wtconv_param_grads* g, int levels) {
    if (g == nullptr) return;
    t.dtype = WTCONV_F32;
    t.base_weight = g->base_weight; t.base_bias = g->base_bias; t.base_scale = g->base_scale;
    for (int l = 0; l < levels && l < kMaxLevels; ++l) { t.wt_weight[l] = g->wt_weight[l]; t.wt_scale[l] = g->wt_scale[l]; }
    ptr = &t;
  }
};

static int check_grad_table(const char* fn, const wtconv_params* params, const wtconv_typed_grads* grads, int L) {
  if (grads == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
  if (int e = check_grad_dtype(fn, grads)) return e;
  if (grads->base_weight == nullptr || grads->base_scale == nullptr ||
      (params->base_bias != nullptr && grads->base_bias == nullptr))
    return fail(WTCONV_E_ARG, "%s: null gradient pointer", fn);
  for (int l = 0; l < L; ++l)
    if (grads->wt_weight[l] == nullptr || grads->wt_scale[l] == nullptr)
      return fail(WTCONV_E_ARG, "%s: null gradient pointer at level %d", fn, l);
  return 0;
}

static GradTable to_grad_table(const wtconv_typed_grads* grads, int L) {
  GradTable gt = {};
  gt.dtype = grads->dtype;
  gt.base_weight = grads->base_weight;
  gt.base_bias = grads->base_bias;
  gt.base_scale = grads->base_scale;
  for (int l = 0; l < L; ++l) { gt.wt_weight[l] = grads->wt_weight[l]; gt.wt_scale[l] = grads->wt_scale[l]; }
  return gt;
}

}  // namespace wt

using namespace wt;

extern "C" {

int wtconv_abi_version(void) { return WTCONV_ABI_VERSION; }

const char* wtconv_last_error(void) { return g_err; }

int wtconv_max_kernel_size(void) { return 7; }

// Whether both passes of a backward call are made of steps (planes beyond LDS): they share the LL bands of grad_out.
static bool stream2d_backward(int B, int C, int H, int W, int K, int L) {
  return !plane_fits_lds(B, C, H, W, K, L) && !wgrad_fits_lds(B, C, H, W, K, L);
}

size_t wtconv2d_workspace_bytes(int B, int C, int H, int W, int K, int levels, int pass) {
  if (pass == WTCONV_PASS_BACKWARD) {
    if (B > 0 && C > 0 && H > 0 && W > 0 && K > 0 && levels > 0 && levels <= kMaxLevels &&
        static_cast<long long>(H) * W <= kMaxPlaneElems && stream2d_backward(B, C, H, W, K, levels)) {
      // what the parameter-gradient pass needs (its LL bands of grad_out serve both), folded parameters, sub-layers
      const size_t extra = round_up64(fold_floats(C, 4, levels, K * K)) + make_stream2d(B, C, H, W, K, levels).floats;
      const size_t both = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD_PARAMS) +
                          (extra * sizeof(float) + 255) / 256 * 256;
      const size_t input = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD_INPUT);
      return both > input ? both : input;
    }
    const size_t a = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD_INPUT);
    const size_t b = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD_PARAMS);
    return a > b ? a : b;
  }
  if (B <= 0 || C <= 0 || H <= 0 || W <= 0 || K <= 0 || levels <= 0 || levels > kMaxLevels) return 0;
  if (static_cast<long long>(H) * W > kMaxPlaneElems) return 0;
  size_t floats;
  if (pass == WTCONV_PASS_BACKWARD_PARAMS) {
    // the dtype is not an argument here: room for the bf16 matrix-core kernel's partial sums as well
    const Mfma2dWgradQuery mq = mfma2d_wgrad_query(B, C, H, W, K, levels, WTCONV_BF16);
    const size_t mfloats = mq.ok ? mq.ws_bytes / sizeof(float) : 0;
    if (wgrad_fits_lds(B, C, H, W, K, levels)) {
      floats = static_cast<size_t>(wgrad_split(B, C, H, W, K, levels).nchunk) * C * ((1 + 4 * levels) * K * K + 1);
    } else {      // partial sums, then the LL bands of x and of grad_out
      const Stream2D sp = make_stream2d(B, C, H, W, K, levels);
      floats = stream_records(B, C, H, W, K, levels) + stream_sub_records(sp, B, C, K, levels);
      const size_t area = four_band_floats(B, C, H, W, K, levels);
      floats += 2 * (area > sp.floats ? area : sp.floats);
    }
    if (mfloats > floats) floats = mfloats;
    floats = round_up64(floats) + static_cast<size_t>(C);      // one ticket word per channel behind the records
  } else {
    // the dtype is not an argument here: size for the larger of the two (fp32 tensors take
    // three split tables) whenever either could run on the matrix-core kernels
    size_t mf = 0;
    for (int dt : {WTCONV_F32, WTCONV_BF16}) {
      const Mfma2dQuery q = mfma2d_query(B, C, H, W, K, levels, dt);
      if (q.ok && q.ws_bytes > mf) mf = q.ws_bytes;
    }
    floats = fold_floats(C, 4, levels, K * K);
    if (pass == WTCONV_PASS_FORWARD && static_cast<long long>(B) * C <= kFoldInsidePlanes &&
        folded_tables(C, levels, K * K) > floats)
      floats = folded_tables(C, levels, K * K);
    if (!plane_fits_lds(B, C, H, W, K, levels)) {
      size_t area = four_band_floats(B, C, H, W, K, levels);
      const Stream2D sp = make_stream2d(B, C, H, W, K, levels);
      if (area < 2 * sp.floats) area = 2 * sp.floats;
      floats = round_up64(floats) + area;
    }
    if (mf > floats * sizeof(float)) floats = (mf + 3) / 4;
  }
  return (floats * sizeof(float) + 255) / 256 * 256;
}

int wtconv2d_forward(const void* x, void* out, const wtconv_params* params, int B, int C, int H, int W, int K,
                     int levels, int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                     void* stream) {
  return plane2d_pass("wtconv2d_forward", x, out, params, B, C, H, W, K, levels, dtype, param_dtype, workspace,
                      workspace_bytes, stream, 0);
}

size_t wtconv_static_scratch_bytes(void) { return kStaticScratchBytes; }

int wtconv2d_forward_static(const void* x, void* out, const wtconv_params* params, int B, int C, int H, int W,
                            int K, int levels, int dtype, int param_dtype, void* stream) {
  const char* fn = "wtconv2d_forward_static";
  size_t need = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_FORWARD);
  // (planes that are faster in steps, but not with this much scratch, stay in LDS where they fit)
  const bool resident = need > kStaticScratchBytes && fold_floats(C, 4, levels, K * K) * sizeof(float) <= kStaticScratchBytes &&
                        row_lanes(W) <= kMaxPlaneThreads &&
                        plane_lds_bytes(B, C, H, W, K, levels) <= static_cast<size_t>(kLdsLimitBytes);
  if (need > kStaticScratchBytes && !resident)
    return fail(WTCONV_E_UNSUPPORTED,
                "%s: this shape needs %zu B of scratch, the static buffer holds %zu B; use wtconv2d_forward with a "
                "caller-supplied workspace", fn, need, kStaticScratchBytes);
  void* ptr = nullptr;
  if (int e = static_scratch(fn, &ptr)) return e;
  return plane2d_pass(fn, x, out, params, B, C, H, W, K, levels, dtype, param_dtype, ptr, kStaticScratchBytes,
                      stream, 0, nullptr, nullptr, nullptr, resident);
}

int wtconv2d_backward_input(const void* grad_out, void* grad_x, const wtconv_params* params, int B, int C,
                            int H, int W, int K, int levels, int dtype, int param_dtype, void* workspace,
                            size_t workspace_bytes, void* stream) {
  return plane2d_pass("wtconv2d_backward_input", grad_out, grad_x, params, B, C, H, W, K, levels, dtype,
                      param_dtype, workspace, workspace_bytes, stream, 1);
}

// Where the parameter-gradient pass of a plane-resident shape keeps its channel tickets in the workspace.
static unsigned* wgrad2d_tickets(void* workspace, int B, int C, int H, int W, int K, int L) {
  const size_t need = wtconv2d_workspace_bytes(B, C, H, W, K, L, WTCONV_PASS_BACKWARD_PARAMS);
  return reinterpret_cast<unsigned*>(static_cast<char*>(workspace) + need) - C;
}

// have_g_ll (planes beyond LDS only): the LL bands of grad_out that the layer itself needs are in the workspace already.
// tickets_zeroed (plane-resident paths only): an earlier kernel on the stream has cleared the channel tickets.
static int backward_params2d(const char* fn, const void* x, const void* grad_out, const wtconv_params* params,
                             const wtconv_typed_grads* grads, int B, int C, int H, int W, int K, int levels,
                             int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                             void* stream_, bool have_g_ll, bool tickets_zeroed = false) {
  const int L = levels;
  if (int e = check_common(fn, params, B, C, K, L, dtype, param_dtype)) return e;
  if (H <= 0 || W <= 0) return fail(WTCONV_E_ARG, "%s: spatial size must be positive (got %dx%d)", fn, H, W);
  if (static_cast<long long>(H) * W > kMaxPlaneElems)   // 32-bit offsets inside a plane and its four stacked sub-bands
    return fail(WTCONV_E_UNSUPPORTED, "%s: a plane of %dx%d exceeds 2^28 elements", fn, H, W);
  if (x == nullptr || grad_out == nullptr || grads == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
  if (int e = check_grad_dtype(fn, grads)) return e;
  if (grads->base_weight == nullptr || grads->base_scale == nullptr ||
      (params->base_bias != nullptr && grads->base_bias == nullptr))
    return fail(WTCONV_E_ARG, "%s: null gradient pointer", fn);
  for (int l = 0; l < L; ++l)
    if (grads->wt_weight[l] == nullptr || grads->wt_scale[l] == nullptr)
      return fail(WTCONV_E_ARG, "%s: null gradient pointer at level %d", fn, l);
  const size_t esz = dtype == WTCONV_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(x) % esz) || (reinterpret_cast<uintptr_t>(grad_out) % esz))
    return fail(WTCONV_E_ARG, "%s: tensor pointer not aligned to its element size", fn);
  const size_t need = wtconv2d_workspace_bytes(B, C, H, W, K, L, WTCONV_PASS_BACKWARD_PARAMS);
  if (workspace == nullptr || workspace_bytes < need)
    return fail(WTCONV_E_WORKSPACE, "%s: workspace of %zu B needed, %zu given", fn, need, workspace_bytes);
  if (static_cast<long long>(B) * C > 0x7fffffffLL / 4)
    return fail(WTCONV_E_UNSUPPORTED, "%s: batch*channels = %lld is too large", fn, static_cast<long long>(B) * C);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  int nchunk;
  float* partial = static_cast<float*>(workspace);
  int e;
  SubRecords sub = {};
  const Mfma2dWgradQuery mq = mfma2d_wgrad_query(B, C, H, W, K, L, dtype);
  const bool resident = mq.ok || wgrad_fits_lds(B, C, H, W, K, L);
  // The plane-resident first-stage kernels finish their channels themselves (last workgroup of a channel): one ticket
  // word per channel at the end of the workspace, cleared by a small launch of its own.
  FinishArgs fin = {};
  if (resident) {
    fin.tickets = wgrad2d_tickets(workspace, B, C, H, W, K, L);
    fin.prm = to_table(params, L);
    fin.pdtype = param_dtype;
    fin.gt = to_grad_table(grads, L);
    if (!tickets_zeroed) {
      WT_LAUNCH(zero_tickets_kernel, dim3((C + 255) / 256), dim3(256), 0, stream, fin.tickets, C);
      if (int ze = check_launch("zero_tickets_kernel")) return ze;
    }
  }
  if (mq.ok) {
    nchunk = mq.nchunk;
    e = mfma2d_wgrad_pass(fn, x, grad_out, partial, B, C, H, W, K, L, fin, stream);
  } else if (resident) {
    const WgradSplit split = wgrad_split(B, C, H, W, K, L);
    Plan2D pl = make_plan2d(B, C, H, W, K, L, true, 512, split.pb);
    finish_wgrad_plan(&pl, K);
    nchunk = split.nchunk;
    e = launch_wgrad2d(dtype, K, L, x, grad_out, partial, pl, B, split.bchunk, nchunk, fin, stream);
  } else {
    const Stream2D sp = make_stream2d(B, C, H, W, K, L);
    nchunk = stream_chunks(B, C, H, W);
    float* sub_partial = partial + stream_records(B, C, H, W, K, L);
    float* gll = sub_partial + stream_sub_records(sp, B, C, K, L);
    float* xll = gll + sp.floats;
    const int D = sp.wdepth;
    e = 0;
    for (int d = 0; d <= D && d <= L && !e; ++d) {
      const int dt = d == 0 ? dtype : WTCONV_F32;
      const void* xd = d == 0 ? x : static_cast<const void*>(xll + sp.ll[d]);
      const void* gd = d == 0 ? grad_out : static_cast<const void*>(gll + sp.ll[d]);
      if (d == D && d < L) {       // the rest fits LDS
        const int Ls = L - d;
        const WgradSplit split = wgrad_split(B, C, sp.h[d], sp.w[d], K, Ls);
        Plan2D pl = make_plan2d(B, C, sp.h[d], sp.w[d], K, Ls, true, 512, split.pb);
        finish_wgrad_plan(&pl, K);
        sub.nchunk = split.nchunk;
        sub.partial = sub_partial;
        sub.depth = d;
        e = launch_wgrad2d(WTCONV_F32, K, Ls, xd, gd, sub_partial, pl, B, split.bchunk, sub.nchunk, FinishArgs{}, stream);
        break;
      }
      // a step; at d == L only the LL band's own filter is left, the base conv of a layer without levels
      const StreamStep st = {B, C, sp.h[d], sp.w[d]};
      const bool more = d < L;
      const bool g_there = have_g_ll && d + 1 <= sp.depth && d + 1 < L;
      const StreamCorrOut o = {partial, (1 + 4 * L) * K * K + 1, d == 0 ? 0 : 1 + 4 * (d - 1), 2 + 4 * d, d == 0 ? 1 : 0};
      e = launch_stream_corr(dt, K, st, xd, gd, more ? xll + sp.ll[d + 1] : nullptr,
                             more && !g_there ? gll + sp.ll[d + 1] : nullptr, more, o, nchunk, stream);
    }
  }
  if (e || resident) return e;
  const GradTable gt = to_grad_table(grads, L);
  const int nrec = (1 + 4 * L) * K * K + 1;
  WT_LAUNCH(wgrad_finish_kernel, dim3(C), dim3(finish_threads(nrec)), static_cast<size_t>(nrec) * sizeof(float),
            stream, partial, nchunk, to_table(params, L), param_dtype, gt, C, 4, L, K * K, sub);
  return check_launch("wgrad_finish_kernel");
}

int wtconv2d_backward_params(const void* x, const void* grad_out, const wtconv_params* params,
                             const wtconv_param_grads* grads, int B, int C, int H, int W, int K, int levels,
                             int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                             void* stream) {
  return wtconv2d_backward_params_typed(x, grad_out, params, FloatGrads(grads, levels).ptr, B, C, H, W, K, levels, dtype,
                                        param_dtype, workspace, workspace_bytes, stream);
}

int wtconv2d_backward_params_typed(const void* x, const void* grad_out, const wtconv_params* params,
                                   const wtconv_typed_grads* grads, int B, int C, int H, int W, int K, int levels,
                                   int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  return backward_params2d("wtconv2d_backward_params", x, grad_out, params, grads, B, C, H, W, K, levels, dtype,
                           param_dtype, workspace, workspace_bytes, stream, false);
}

int wtconv2d_backward(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                      const wtconv_param_grads* grads, int B, int C, int H, int W, int K, int levels, int dtype,
                      int param_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  return wtconv2d_backward_typed(x, grad_out, grad_x, params, FloatGrads(grads, levels).ptr, B, C, H, W, K, levels, dtype,
                                 param_dtype, workspace, workspace_bytes, stream);
}

int wtconv2d_backward_typed(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                            const wtconv_typed_grads* grads, int B, int C, int H, int W, int K, int levels, int dtype,
                            int param_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  // Planes beyond LDS (both passes in steps): the LL bands of grad_out are built once, in the place where the
  // parameter-gradient pass keeps them, and serve both passes.
  const bool sizes_ok = B > 0 && C > 0 && H > 0 && W > 0 && K >= 1 && K % 2 == 1 && K <= wtconv_max_kernel_size() &&
                        levels >= 1 && levels <= kMaxLevels && static_cast<long long>(H) * W <= kMaxPlaneElems;
  if (sizes_ok && !mfma2d_query(B, C, H, W, K, levels, dtype).ok && !mfma2d_wgrad_query(B, C, H, W, K, levels, dtype).ok &&
      stream2d_backward(B, C, H, W, K, levels)) {
    const size_t need = wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD);
    if (workspace == nullptr || workspace_bytes < need)
      return fail(WTCONV_E_WORKSPACE, "wtconv2d_backward: workspace of %zu B needed, %zu given", need, workspace_bytes);
    const Stream2D sp = make_stream2d(B, C, H, W, K, levels);
    float* gll = static_cast<float*>(workspace) + stream_records(B, C, H, W, K, levels) +
                 stream_sub_records(sp, B, C, K, levels);
    float* fw = static_cast<float*>(workspace) +
                wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD_PARAMS) / sizeof(float);
    if (int e = plane2d_pass("wtconv2d_backward", grad_out, grad_x, params, B, C, H, W, K, levels, dtype, param_dtype,
                             workspace, workspace_bytes, stream, 1, gll, fw))
      return e;
    return backward_params2d("wtconv2d_backward", x, grad_out, params, grads, B, C, H, W, K, levels, dtype,
                             param_dtype, workspace, workspace_bytes, stream, true);
  }
  // Otherwise the two passes run one after the other on the stream and share the workspace.  Plane-resident shapes:
  // the input-gradient pass clears the channel tickets of the parameter-gradient pass on its way (one launch fewer),
  // where they lie beyond the folded parameters that it keeps at the start of the workspace.
  if (sizes_ok && workspace != nullptr &&
      workspace_bytes >= wtconv2d_workspace_bytes(B, C, H, W, K, levels, WTCONV_PASS_BACKWARD) &&
      (mfma2d_query(B, C, H, W, K, levels, dtype).ok || plane_fits_lds(B, C, H, W, K, levels)) &&
      (mfma2d_wgrad_query(B, C, H, W, K, levels, dtype).ok || wgrad_fits_lds(B, C, H, W, K, levels))) {
    unsigned* tickets = wgrad2d_tickets(workspace, B, C, H, W, K, levels);
    const char* fold_end = static_cast<const char*>(workspace) + fold_floats(C, 4, levels, K * K) * sizeof(float);
    if (reinterpret_cast<const char*>(tickets) >= fold_end) {
      if (int e = plane2d_pass("wtconv2d_backward", grad_out, grad_x, params, B, C, H, W, K, levels, dtype, param_dtype,
                               workspace, workspace_bytes, stream, 1, nullptr, nullptr, tickets))
        return e;
      return backward_params2d("wtconv2d_backward", x, grad_out, params, grads, B, C, H, W, K, levels, dtype,
                               param_dtype, workspace, workspace_bytes, stream, false, true);
    }
  }
  if (int e = wtconv2d_backward_input(grad_out, grad_x, params, B, C, H, W, K, levels, dtype, param_dtype, workspace,
                                      workspace_bytes, stream))
    return e;
  return wtconv2d_backward_params_typed(x, grad_out, params, grads, B, C, H, W, K, levels, dtype, param_dtype, workspace,
                                        workspace_bytes, stream);
}

size_t wtconv1d_workspace_bytes(int B, int C, int N, int K, int levels, int pass) {
  if (pass == WTCONV_PASS_BACKWARD) {
    const size_t a = wtconv1d_workspace_bytes(B, C, N, K, levels, WTCONV_PASS_BACKWARD_INPUT);
    const size_t b = wtconv1d_workspace_bytes(B, C, N, K, levels, WTCONV_PASS_BACKWARD_PARAMS);
    return a > b ? a : b;
  }
  if (B <= 0 || C <= 0 || N <= 0 || K <= 0 || levels <= 0 || levels > kMaxLevels) return 0;
  size_t floats;
  if (pass == WTCONV_PASS_BACKWARD_PARAMS) {
    const Plan1D pl = make_plan1d(C, N, levels, true, 4, nullptr, nullptr, nullptr);
    int per_chunk, nchunk;
    Row1DShape sh = {};
    if (row1d_shape(C, N, K, levels, &sh))
      row1d_chunks(B * sh.pl.nseg, C, row1d_two_region_per_cu(K, levels, sh), &per_chunk, &nchunk);
    else
      wgrad_chunks1d(B, C, pl.ntiles, &per_chunk, &nchunk);
    // partial sums, then one ticket word per channel (fused backward kernel)
    floats = round_up64(static_cast<size_t>(nchunk) * C * ((1 + 2 * levels) * K + 1)) + static_cast<size_t>(C);
  } else {
    floats = fold_floats(C, 2, levels, K);
  }
  return (floats * sizeof(float) + 255) / 256 * 256;
}

int wtconv1d_forward(const void* x, void* out, const wtconv_params* params, int B, int C, int N, int K,
                     int levels, int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                     void* stream) {
  return tile1d_pass("wtconv1d_forward", x, out, params, B, C, N, K, levels, dtype, param_dtype, workspace,
                     workspace_bytes, stream, 0);
}

int wtconv1d_backward_input(const void* grad_out, void* grad_x, const wtconv_params* params, int B, int C,
                            int N, int K, int levels, int dtype, int param_dtype, void* workspace,
                            size_t workspace_bytes, void* stream) {
  return tile1d_pass("wtconv1d_backward_input", grad_out, grad_x, params, B, C, N, K, levels, dtype,
                     param_dtype, workspace, workspace_bytes, stream, 1);
}

int wtconv1d_backward_params(const void* x, const void* grad_out, const wtconv_params* params,
                             const wtconv_param_grads* grads, int B, int C, int N, int K, int levels,
                             int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                             void* stream) {
  return wtconv1d_backward_params_typed(x, grad_out, params, FloatGrads(grads, levels).ptr, B, C, N, K, levels, dtype,
                                        param_dtype, workspace, workspace_bytes, stream);
}

int wtconv1d_backward_params_typed(const void* x, const void* grad_out, const wtconv_params* params,
                                   const wtconv_typed_grads* grads, int B, int C, int N, int K, int levels,
                                   int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                                   void* stream_) {
  const char* fn = "wtconv1d_backward_params";
  const int L = levels;
  if (int e = check_common(fn, params, B, C, K, L, dtype, param_dtype)) return e;
  if (N <= 0) return fail(WTCONV_E_ARG, "%s: length must be positive (got %d)", fn, N);
  if (x == nullptr || grad_out == nullptr || grads == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
  if (int e = check_grad_dtype(fn, grads)) return e;
  if (grads->base_weight == nullptr || grads->base_scale == nullptr ||
      (params->base_bias != nullptr && grads->base_bias == nullptr))
    return fail(WTCONV_E_ARG, "%s: null gradient pointer", fn);
  for (int l = 0; l < L; ++l)
    if (grads->wt_weight[l] == nullptr || grads->wt_scale[l] == nullptr)
      return fail(WTCONV_E_ARG, "%s: null gradient pointer at level %d", fn, l);
  const size_t esz = dtype == WTCONV_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(x) % esz) || (reinterpret_cast<uintptr_t>(grad_out) % esz))
    return fail(WTCONV_E_ARG, "%s: tensor pointer not aligned to its element size", fn);
  const Plan1D pl = make_plan1d(C, N, L, true, esz, x, grad_out, nullptr);
  const size_t need = wtconv1d_workspace_bytes(B, C, N, K, L, WTCONV_PASS_BACKWARD_PARAMS);
  if (workspace == nullptr || workspace_bytes < need)
    return fail(WTCONV_E_WORKSPACE, "%s: workspace of %zu B needed, %zu given", fn, need, workspace_bytes);
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  int per_chunk, nchunk;
  Row1DShape sh = {};
  const bool row_resident = row1d_shape(C, N, K, L, &sh);
  if (row_resident)
    row1d_chunks(B * sh.pl.nseg, C, row1d_two_region_per_cu(K, L, sh), &per_chunk, &nchunk);
  else
    wgrad_chunks1d(B, C, pl.ntiles, &per_chunk, &nchunk);
  if (nchunk > 65535) return fail(WTCONV_E_UNSUPPORTED, "%s: too many chunks (%d)", fn, nchunk);
  float* partial = static_cast<float*>(workspace);
  int e;
  if (row_resident) {
    e = launch_row1d_wgrad(dtype, K, L, x, grad_out, partial, sh.pl, B, sh.block, per_chunk, nchunk, stream);
  } else {
    e = launch_wgrad1d(dtype, L, x, grad_out, partial, pl, B, per_chunk, nchunk, stream);
  }
  if (e) return e;
  const GradTable gt = to_grad_table(grads, L);
  const int nrec = (1 + 2 * L) * K + 1;
  WT_LAUNCH(wgrad_finish_kernel, dim3(C), dim3(finish_threads(nrec)), static_cast<size_t>(nrec) * sizeof(float),
            stream, partial, nchunk, to_table(params, L), param_dtype, gt, C, 2, L, K, SubRecords{});
  return check_launch("wgrad_finish_kernel");
}

int wtconv1d_backward(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                      const wtconv_param_grads* grads, int B, int C, int N, int K, int levels, int dtype,
                      int param_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  return wtconv1d_backward_typed(x, grad_out, grad_x, params, FloatGrads(grads, levels).ptr, B, C, N, K, levels, dtype,
                                 param_dtype, workspace, workspace_bytes, stream);
}

int wtconv1d_backward_typed(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                            const wtconv_typed_grads* grads, int B, int C, int N, int K, int levels, int dtype,
                            int param_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  const char* fn = "wtconv1d_backward";
  // rows that the register-resident kernels take run the whole backward pass as one kernel -- with the lanes, chunks
  // and workspace layout of the separate parameter-gradient pass, so the two share wtconv1d_workspace_bytes
  Row1DShape sh = {};
  if (row1d_shape(C, N, K, levels, &sh) && row1d_bwd_built(K, levels, sh.S)) {
    const int L = levels;
    if (int e = check_common(fn, params, B, C, K, L, dtype, param_dtype)) return e;
    if (x == nullptr || grad_out == nullptr || grad_x == nullptr) return fail(WTCONV_E_ARG, "%s: null tensor pointer", fn);
    if (int e = check_grad_table(fn, params, grads, L)) return e;
    const size_t esz = dtype == WTCONV_F32 ? 4 : 2;
    if ((reinterpret_cast<uintptr_t>(x) % esz) || (reinterpret_cast<uintptr_t>(grad_out) % esz) ||
        (reinterpret_cast<uintptr_t>(grad_x) % esz))
      return fail(WTCONV_E_ARG, "%s: tensor pointer not aligned to its element size", fn);
    const size_t need = wtconv1d_workspace_bytes(B, C, N, K, L, WTCONV_PASS_BACKWARD);
    if (workspace == nullptr || workspace_bytes < need)
      return fail(WTCONV_E_WORKSPACE, "%s: workspace of %zu B needed, %zu given", fn, need, workspace_bytes);
    if (reinterpret_cast<uintptr_t>(workspace) % 4)
      return fail(WTCONV_E_ARG, "%s: workspace not aligned", fn);
    int per_chunk, nchunk;
    row1d_chunks(B * sh.pl.nseg, C, row1d_two_region_per_cu(K, L, sh), &per_chunk, &nchunk);
    if (nchunk > 65535) return fail(WTCONV_E_UNSUPPORTED, "%s: too many chunks (%d)", fn, nchunk);
    float* partial = static_cast<float*>(workspace);
    unsigned* tickets = reinterpret_cast<unsigned*>(partial + round_up64(static_cast<size_t>(nchunk) * C * ((1 + 2 * L) * K + 1)));
    const GradTable gt = to_grad_table(grads, L);
    return launch_row1d_bwd(dtype, K, L, x, grad_out, grad_x, partial, tickets, params, param_dtype, gt, sh.pl, B, sh.block,
                            per_chunk, nchunk, static_cast<hipStream_t>(stream));
  }
  if (int e = wtconv1d_backward_input(grad_out, grad_x, params, B, C, N, K, levels, dtype, param_dtype, workspace,
                                      workspace_bytes, stream))
    return e;
  return wtconv1d_backward_params_typed(x, grad_out, params, grads, B, C, N, K, levels, dtype, param_dtype, workspace,
                                        workspace_bytes, stream);
}

}  // extern "C"
