// Host-side planning: LDS layouts and launch geometry.  Pure C++, no device code.
#pragma once

#include <stddef.h>
#include <stdint.h>

#include "host_util.h"
#include "kernels1d.h"
#include "kernels2d.h"

namespace wt {

constexpr int round_up(int v, int m) { return (v + m - 1) / m * m; }

// Strip widths of the 2-D kernels (outputs per work item along a row).
constexpr int kTJC = 1;     // coarser levels of the plane kernel: single coefficients keep the most lanes busy
                            // (measured against strips of 2: 28x28 planes 106 -> 100 us, 14x14 73 -> 71, 56x56 equal)
constexpr int kTJW = 4;     // weight-gradient correlation strips

constexpr int pow2_ceil(int v) { int p = 1; while (p < v) p *= 2; return p; }

// A row of per_row threads as walk_rows takes it.
constexpr unsigned dense_rows(int per_row) { return static_cast<unsigned>(per_row) << 21 | ((1u << 20) + per_row - 1) / per_row; }

// Rows of `used` items over the threads: dense, or a power of two of threads each where that takes `height` rows, and half as
// many, in as many passes (which is 0.2 % faster at the geometric mean, now and then a tenth or more either way: banks).
constexpr unsigned row_split(int used, int threads, int height) {
  const int p = pow2_ceil(used);
  auto passes = [&](int n, int per_row) { const int rows = threads / per_row; return rows > 0 ? (n + rows - 1) / rows : n + 1; };
  const bool even = passes(height, p) == passes(height, used) && passes((height + 1) / 2, p) == passes((height + 1) / 2, used);
  return dense_rows(even && p <= threads ? p : used);
}
constexpr int log2_int(int v) { int s = 0; while ((1 << s) < v) ++s; return s; }

// Lanes that a row of a plane takes: one for each piece of four pixels it is loaded in, which is also one for each
// coefficient of a row of level 2 (kTJC = 1; rows of coarser levels take fewer).  The kernels walk a plane by whole rows, so
// a plane has at least as many threads; flat ones (H <= 2 and W > 64, say) would get fewer by their area alone.
constexpr int kMaxPlaneThreads = 1024;
constexpr int row_lanes(int W) { return pow2_ceil((W + 3) / 4); }
static_assert(kTJC == 1, "row_lanes counts single coefficients of level 2");

// Widest plane of the weight-gradient kernel: a wave sums strips of kTJW pixels of whole rows.
constexpr int kMaxWgradWidth = kWave * kTJW;

// Fills the LDS layout of one plane.  Planes are stacked in one column: x, then the four
// sub-band planes of level 1, level 2, ...; consecutive planes are separated by one gap of
// P zero rows that serves as bottom halo of the upper and top halo of the lower plane.
// with_grad_pyramid adds the padded pyramid of grad_out used by the weight-gradient kernel
// (and drops the Z buffers it does not need).
constexpr Plan2D make_plan2d_geometry(int B, int C, int H, int W, int K, int L, bool with_grad_pyramid, int nthreads,
                                      int pb) {
  Plan2D pl = {};
  pl.B = B; pl.C = C; pl.H = H; pl.W = W; pl.L = L;
  pl.nplanes = B * C;
  const int R = K / 2;
  pl.P = R > 1 ? R : 1;
  pl.h[0] = H; pl.w[0] = W;
  for (int l = 1; l <= L; ++l) { pl.h[l] = (pl.h[l - 1] + 1) / 2; pl.w[l] = (pl.w[l - 1] + 1) / 2; }
  // element (r, col) of sub-band s of level l sits at aoff[l] + s*apl[l] + (r+P)*astr[l] + col + P
  int off = 0;            // start of the zero gap above the next plane
  for (int l = 0; l <= L; ++l) {
    pl.astr[l] = round_up(pl.w[l] + 2 * pl.P, 4);
    pl.apl[l] = pb * (pl.h[l] + pl.P) * pl.astr[l];        // pb planes stacked, P shared zero rows between them
    if (l > 0) off += pl.P * (pl.astr[l - 1] - pl.astr[l]);   // the gap keeps the wider stride of the level above
    pl.aoff[l] = off;
    off += pl.apl[l] * (l == 0 ? 1 : 4);
  }
  off += pl.P * pl.astr[L];                                   // bottom halo of the last plane
  if (!with_grad_pyramid) {
    for (int l = 2; l <= L; ++l) {
      pl.zstr[l] = pl.w[l - 1];
      pl.zoff[l] = off;
      off += round_up(pl.zstr[l] * pl.h[l - 1], 4);
    }
  } else {
    for (int l = 0; l <= L; ++l) {
      pl.gstr[l] = round_up(pl.w[l] + 1, 4);
      pl.gpl[l] = pb * (pl.h[l] + pl.P) * pl.gstr[l];      // same row pitch as the x pyramid
      pl.goff[l] = off;
      off += pl.gpl[l] * (l == 0 ? 1 : 4);
    }
  }
  pl.plane_lds_floats = round_up(off + kLdsSlackFloats, 4);
  pl.sg_shift = log2_int(nthreads);
  pl.pb = pb;
  pl.slot_shift = log2_int(nthreads);
  pl.lds_floats = pl.plane_lds_floats;
  pl.groups_per_channel = 1;
  pl.fw_stride = (1 + 4 * L) * K * K;
  pl.vec_ok = W >= 4;
  return pl;
}

inline Plan2D make_plan2d(int B, int C, int H, int W, int K, int L, bool with_grad_pyramid, int nthreads, int pb = 1) {
  return make_plan2d_geometry(B, C, H, W, K, L, with_grad_pyramid, nthreads, pb);
}

// Time of the plane kernel on a plan's planes (pl.B of them for each of pl.C channels), up to a factor and a constant, with
// level-1 strips of `tj` and 2^sg_shift threads a plane.  A unit is what takes up whole waves: a plane, or the planes of one
// channel that a wave holds.  Each of 256 compute units has `units` of them, n at a time, and takes
//   rounds * latency of one + units * issue slots of one
// where the last round counts half.  A level-1 strip is w = 8 K^2 tj multiply-adds, for narrow strips times what their LDS reads
// add (a 5 x 5 window does 1.7, 0.9 or 0.6 multiply-adds for a float it reads); a wave by itself takes seven cycles for one, four
// SIMDs together issue one a cycle.  Levels from 2 on are single coefficients, one after the other; a pass of 2 x 4 pieces is
// 160 slots, and 600 cycles a level go to barriers and latencies.  Registers leave room for 1280 threads.
// Fitted for the pick alone to every pair on 1803 shapes (fp32, 5 to 110 pixels, K = 3 to 7, 1 to 256 images, 16 to 512 channels):
// 1 % slower than the best pair at the geometric mean.  Two simpler rules, most busy lanes (A) and fewest slots (B), both with
// up to 256 threads and more only where few planes leave that many, were 7 % and 4 % slower than the best.  On 409 shapes that the
// fit has not seen it takes 0.95 of A's time and 0.96 of B's; with K = 7 it is over a tenth slower than the faster of them on one
// shape in forty.  Forward us, A / B / now: [64,64,33,21], K = 3, two levels 21.0 / 21.5 / 18.5; [8,32,64,64], K = 5, three levels
// 14.5 / 14.6 / 13.4; [16,72,45,37], K = 7, two levels 32.8 / 26.4 / 26.6; [209,22,13,16], K = 7, three levels 27.5 / 40.2 / 27.6;
// [1,83,33,36], K = 7, one level 10.3 / 13.3 / 9.1; and the worst, [134,433,9,10], K = 7, two levels 131 / 107 / 136.
// 1500 more shapes that the fit has not seen, 449 of them fp16: 2 % slower than the best pair in both types, 0.90 of the time of the kernels
// that went with A; 40 are over 3 % slower than those, 15 over a tenth (tall or wide planes of which LDS holds two or three, rows that
// fall on the same banks), at most [113,17,43,98], K = 7, one level, 57.5 -> 70.4.  A new fit to half of them gained 0.3 % there
// and 0.15 % on the other half.
constexpr double plane_cost(const Plan2D& pl, int K, int tj, int sg_shift) {
  const int threads = 1 << sg_shift, h1 = pl.h[1], per_row = (pl.w[1] + tj - 1) / tj, rows = threads / per_row;
  const int full = h1 / rows, rest = h1 - full * rows, waves = threads > kWave ? threads / kWave : 1;
  auto waves_of = [&](int lanes) { return threads > kWave ? (lanes + kWave - 1) / kWave : lanes > 0 ? 1 : 0; };
  auto passes = [](int n, int at_once) { return (n + at_once - 1) / at_once; };
  int coarse = 0;
  for (int l = 2; l <= pl.L; ++l) coarse += passes(pl.h[l], threads / pl.w[l]);
  const int pieces = passes(h1, threads / row_lanes(pl.W));
  const double wide = 8.0 * K * K, w = wide * tj * (tj == 4 ? 1.0 : tj == 2 ? (K <= 3 ? 1.0 : K <= 5 ? 1.25 : 1.6) : K <= 3 ? 1.6 : K <= 5 ? 2.1 : 3.0);
  const double latency = 7.0 * w * passes(h1, rows) + 3.0 * wide * coarse + 600.0 * (1 + pl.L) + 160.0 * pieces;
  const double issue = w * (static_cast<double>(full) * waves_of(rows * per_row) + waves_of(rest * per_row)) + 160.0 * pieces * waves;
  const int planes = threads < kWave ? kWave / threads : 1, block = threads > 256 ? threads : 256;
  const double units = static_cast<double>(pl.C) * passes(pl.B, planes) / 256.0;
  const int by_lds = kLdsLimitBytes / (pl.plane_lds_floats * 4 * (block / threads)), by_threads = block < 1280 ? 1280 / block : 1;
  const double n = static_cast<double>(by_lds < by_threads ? by_lds : by_threads) * (block / (waves * kWave));
  return (units <= n ? 1.0 : units / n + 0.5) * latency + (units < 1.0 ? 1.0 : units) * issue / 4;
}

// Level-1 strip width and threads per plane of the plane kernel: the cheapest pair (ties: the wider strip, the fewer threads)
// of those whose rows fit the threads and whose planes, of a workgroup of 256, fit half of LDS.
constexpr void choose_plane_shape(const Plan2D& pl, int K, int* tj1, int* sg_shift) {
  double best = 0.0;
  const size_t lds = static_cast<size_t>(pl.plane_lds_floats) * 4;
  for (int tj = 4; tj >= 1; tj /= 2) {
    const int per_row = (pl.w[1] + tj - 1) / tj;
    for (int s = 4; s <= 10; ++s) {
      if ((1 << s) < row_lanes(pl.W) || (1 << s) < per_row || ((1 << s) > 16 && (1 << s) > 4 * pow2_ceil(per_row * pl.h[1]))) continue;
      if (s < 8 ? lds * (256 >> s) > kLdsLimitBytes / 2 : lds > kLdsLimitBytes) continue;
      const double cost = plane_cost(pl, K, tj, s);
      if (best == 0.0 || cost < best) { best = cost; *tj1 = tj; *sg_shift = s; }
    }
  }
}

// Completes a plan for the plane kernel: threads per plane, slots per workgroup, prefetch.
constexpr void finish_plane_plan(Plan2D* pl, int tj1, int sg_shift) {
  pl->sg_shift = sg_shift;
  const int sg = 1 << pl->sg_shift;
  pl->split[1] = row_split((pl->w[1] + tj1 - 1) / tj1, sg, pl->h[1]);
  for (int l = 2; l <= pl->L; ++l) pl->split[l] = row_split(pl->w[l], sg, pl->h[l]);
  pl->block = sg > 256 ? sg : 256;   // (two whole planes per 512-thread workgroup measured slower: lockstep phases)
  const int slots = pl->block / sg;
  pl->lds_floats = pl->plane_lds_floats * slots;
  const int ppw = sg < kWave ? kWave / sg : 1;
  pl->groups_per_channel = (pl->B + ppw - 1) / ppw;
  pl->prefetch = 0;
  pl->fuse = 1;
  if (pl->vec_ok) {
    const int gs = pow2_ceil((pl->W + 3) / 4);       // 2x4 pieces per row pair, one lane each
    const int rows_per_pass = sg / gs;
    pl->prefetch = rows_per_pass >= 1 && (pl->h[1] + rows_per_pass - 1) / rows_per_pass <= kFetchPasses;
    if (pl->prefetch && sg == pl->block && gs <= 16 && pl->L >= 2) pl->fuse = pl->L >= 3 ? 3 : 2;
  }
}

// Geometry of the plane kernel's plan: the run-time plan of the launch, or a compile-time constant for a shape
// whose rows are whole aligned vectors (the launcher checks that the two agree before it picks the constant).
struct PlaneGeoRuntime {
  static constexpr bool kStatic = false, kFold = false;
  using Fold = NoFold;
  static constexpr Plan2D plan() { return Plan2D{}; }
};
struct PlaneGeoFold : PlaneGeoRuntime {
  static constexpr bool kFold = true;
  using Fold = PlaneFold;
};
// Shapes with a compile-time plan of the plane kernel (plane2d.hip): the WTConvNeXt stages, with the pairs that are fastest
// there for many planes (few take them, too: [2,96,56,56] fp32 15.2 us, with more threads 18.4).
constexpr bool plane_shape_is_static(int K, int H, int W, int L) {
  return K == 5 && H == W && ((H == 56 && L == 3) || (H == 28 && L == 3) || (H == 14 && L == 2) || (H == 7 && L == 2));
}
constexpr void static_plane_shape(int H, int* tj1, int* sg_shift) {
  *tj1 = H >= 28 ? 4 : H == 14 ? 2 : 1;
  *sg_shift = H == 56 ? 8 : H == 28 ? 6 : H == 14 ? 5 : 4;
}
constexpr Plan2D static_plane_plan(int H, int W, int K, int L, int* tj1_out) {
  Plan2D pl = make_plan2d_geometry(1, 1, H, W, K, L, false, 256, 1);
  int tj1 = 4, sg_shift = 8;
  static_plane_shape(H, &tj1, &sg_shift);
  finish_plane_plan(&pl, tj1, sg_shift);
  if (tj1_out != nullptr) *tj1_out = tj1;
  return pl;
}

template <int H, int W, int K, int L>
struct PlaneGeoStatic {
  static constexpr bool kStatic = true, kFold = false;
  using Fold = NoFold;
  static constexpr Plan2D plan() { return static_plane_plan(H, W, K, L, nullptr); }
  static constexpr int tj1() { int t = 4; static_plane_plan(H, W, K, L, &t); return t; }
  static constexpr int mode() {
    const Plan2D p = plan();
    return (p.prefetch && p.fuse >= 2) ? 3 : p.prefetch ? 0 : p.vec_ok ? 1 : 2;
  }
};
// Whether two plans describe the same LDS layout and work split (everything but batch and channels).
inline bool same_plane_geometry(const Plan2D& a, const Plan2D& b) {
  if (a.H != b.H || a.W != b.W || a.L != b.L || a.P != b.P || a.lds_floats != b.lds_floats || a.vec_ok != b.vec_ok ||
      a.prefetch != b.prefetch || a.sg_shift != b.sg_shift || a.plane_lds_floats != b.plane_lds_floats ||
      a.fuse != b.fuse || a.block != b.block || a.fw_stride != b.fw_stride || a.fw_skip != b.fw_skip)
    return false;
  for (int l = 0; l <= a.L; ++l)
    if (a.h[l] != b.h[l] || a.w[l] != b.w[l] || a.split[l] != b.split[l] || a.aoff[l] != b.aoff[l] || a.astr[l] != b.astr[l] ||
        a.apl[l] != b.apl[l] || a.zoff[l] != b.zoff[l] || a.zstr[l] != b.zstr[l])
      return false;
  return true;
}

// Planes per iteration of the weight-gradient kernel: as many (of one channel, consecutive
// batch items, stacked vertically) as fit the LDS budget of two workgroups per CU, up to 16.
// Small planes leave most of the 512 threads idle and pay the per-iteration barriers for
// little work when taken one at a time (measured, bf16: 28x28 230 -> 197 us, 14x14 193 -> 160 us,
// 7x7 148 -> 137 us); a 56x56 plane fills the budget by itself.  The threads are dealt to the
// planes of an iteration, so planes with long rows share them with fewer others.
//
// K = 7 with two levels or more takes over 128 registers a lane, so that one workgroup runs on a CU: it may have all of the LDS.
constexpr bool wgrad_is_alone(int K, int L) { return K == 7 && L >= 2; }

constexpr int wgrad_planes_that_fit(int B, int H, int W, int K, int L) {
  int pb = B < 16 ? B : 16;
  if (pb < 1) pb = 1;
  while (pb > 1) {
    const Plan2D t = make_plan2d_geometry(B, 1, H, W, K, L, true, 512, pb);
    if (static_cast<size_t>(t.plane_lds_floats) * 4 <= (wgrad_is_alone(K, L) ? 160 : 80) * 1024 && 512 / pow2_ceil(pb) >= row_lanes(W)) break;
    --pb;
  }
  return pb;
}

// Completes a plan for the weight-gradient kernel: threads per stacked plane, prefetch.
constexpr void finish_wgrad_plan(Plan2D* pl, int K) {
  // the final reduction reuses the LDS as [8 waves][sets * K * K + 1] floats, which is more
  // than the pyramids of a single tiny plane take
  const int red_floats = round_up(8 * (wgrad_sets(pl->L) * K * K + 1), 4);
  if (pl->lds_floats < red_floats) pl->lds_floats = red_floats;
  // A wave's lanes take as many whole rows as they hold.  A power of two of lanes to each left out lanes wherever a row has not
  // just as many strips: 78x66 planes (K = 5, L = 2, 17 strips of 32 lanes) 148.3 -> 127.3 us, 45x37 (K = 7, 10 of 16) 44.5 -> 39.6,
  // 15x17 (K = 7) 93.6 -> 82.3, 40x34 229.7 -> 211.4, 70x75 (K = 3) 73.4 -> 67.9; 56x56 167.6 -> 167.7, 12x10 44.4 -> 45.3.
  for (int l = 0; l <= pl->L; ++l)
    pl->split[l] = dense_rows(l < 2 || (l < 4 && pl->w[l] >= kStripMinWidth) ? (pl->w[l] + kTJW - 1) / kTJW : pl->w[l]);
  const int slots = pow2_ceil(pl->pb);
  pl->slot_shift = log2_int(512 / slots);
  const int nps = 512 / slots;
  pl->prefetch = 0;
  pl->fuse = 1;
  if (pl->vec_ok) {
    const int gs = pow2_ceil((pl->W + 3) / 4);
    pl->prefetch = nps / gs >= pl->h[1];       // one 2x4 piece per thread covers the plane
    if (pl->prefetch && pl->pb == 1 && gs <= 16 && pl->L >= 2) pl->fuse = pl->L >= 3 ? 3 : 2;
  }
}

// Weight-gradient plan of a shape as a compile-time constant: PB planes per iteration, rows of whole aligned vectors.
template <int H, int W, int K, int L, int PB>
struct WgradGeoStatic {
  static constexpr bool kStatic = true;
  static constexpr Plan2D plan() {
    Plan2D pl = make_plan2d_geometry(PB, 1, H, W, K, L, true, 512, PB);
    finish_wgrad_plan(&pl, K);
    return pl;
  }
};
inline bool same_wgrad_geometry(const Plan2D& a, const Plan2D& b) {
  if (a.H != b.H || a.W != b.W || a.L != b.L || a.P != b.P || a.lds_floats != b.lds_floats || a.vec_ok != b.vec_ok ||
      a.prefetch != b.prefetch || a.pb != b.pb || a.slot_shift != b.slot_shift || a.fuse != b.fuse ||
      a.plane_lds_floats != b.plane_lds_floats)
    return false;
  for (int l = 0; l <= a.L; ++l)
    if (a.h[l] != b.h[l] || a.w[l] != b.w[l] || a.split[l] != b.split[l] || a.aoff[l] != b.aoff[l] || a.astr[l] != b.astr[l] ||
        a.apl[l] != b.apl[l] || a.goff[l] != b.goff[l] || a.gstr[l] != b.gstr[l] || a.gpl[l] != b.gpl[l])
      return false;
  return true;
}

// ---- 1-D ------------------------------------------------------------------------------
constexpr int kTJ1D = 4;     // level coefficients per work item in the 1-D kernels
constexpr int kTile1D = 1024;

inline Plan1D make_plan1d(int C, int N, int L, bool with_grad_pyramid, size_t elem_size,
                          const void* p0, const void* p1, const void* p2) {
  Plan1D pl = {};
  pl.C = C; pl.N = N; pl.L = L;
  const int gran = 1 << L;
  int T = round_up(N, gran);
  if (T > kTile1D) T = kTile1D;          // kTile1D is a multiple of 2^L for every L <= 5
  pl.T = T;
  pl.ntiles = (N + T - 1) / T;
  int off = 0;
  for (int l = 0; l <= L; ++l) {
    pl.tl[l] = T >> l;
    pl.apl[l] = round_up(pl.tl[l], 4);
    pl.aoff[l] = off;
    off += pl.apl[l] * (l == 0 ? 1 : 2);
  }
  if (!with_grad_pyramid) {
    for (int l = 2; l <= L; ++l) { pl.zoff[l] = off; off += round_up(pl.tl[l - 1], 4); }
  } else {
    for (int l = 0; l <= L; ++l) {
      pl.gpl[l] = round_up(pl.tl[l], kTJ1D) + kTJ1D;
      pl.goff[l] = off;
      off += pl.gpl[l] * (l == 0 ? 1 : 2);
    }
  }
  pl.lds_floats = round_up(off + kLdsSlackFloats, 4);
  const size_t row_bytes = static_cast<size_t>(N) * elem_size;
  auto aligned = [](const void* p) { return p == nullptr || (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
  pl.vec_ok = (row_bytes % 16 == 0) && aligned(p0) && aligned(p1) && aligned(p2);
  return pl;
}

// (row, tile) pairs per workgroup of the 1-D weight-gradient kernel.
inline void wgrad_chunks1d(int B, int C, int ntiles, int* per_chunk, int* nchunk) {
  const int total = B * ntiles;
  int want = (2048 + C - 1) / C;
  if (want < 1) want = 1;
  if (want > total) want = total;
  int pc = (total + want - 1) / want;
  if (pc < 1) pc = 1;
  *per_chunk = pc;
  *nchunk = (total + pc - 1) / pc;
}

// Workgroups of a persistent kernel: as many as can be resident at once.
inline int resident_workgroups(int ncu, size_t lds_bytes, int waves_per_wg, int max_waves_per_simd) {
  const int by_lds = lds_bytes ? static_cast<int>(kLdsLimitBytes / lds_bytes) : 8;
  const int by_waves = (4 * max_waves_per_simd) / waves_per_wg;
  int per_cu = by_lds < by_waves ? by_lds : by_waves;
  if (per_cu < 1) per_cu = 1;
  return ncu * per_cu;
}

}  // namespace wt
