// Launches of the plane-resident WTConv2d kernel (kernels2d.h): forward and input gradient.
#include "launch.h"
#include "kernels2d.h"

namespace wt {

// ---- 2-D dispatch over (dtype, K, level-1 strip width) -------------------------------
template <typename T, int K, int TJ1, int MODE, typename Geo = PlaneGeoRuntime>
static int run_plane2d_mode(const void* x, void* out, const float* fw, const float* fb, const Plan2D& pl,
                            const PlaneFold& fold, hipStream_t stream) {
  auto kern = wt2d_plane_kernel<T, K, TJ1, kTJC, MODE, Geo>;
  const size_t lds = static_cast<size_t>(pl.lds_floats) * sizeof(float);
  if (int e = allow_lds(kern, lds)) return e;
  const int sg = 1 << pl.sg_shift;
  const int slots = pl.block / sg;
  const int nunits = sg < kWave ? (pl.C * pl.groups_per_channel + 3) / 4 : (pl.nplanes + slots - 1) / slots;
  int nwg = compute_units() * resident_per_cu(kern, pl.block, lds);
  if (nwg > nunits) nwg = nunits;
  typename Geo::Fold arg = {};
  if constexpr (Geo::kFold) arg = fold;
  WT_LAUNCH(kern, dim3(nwg), dim3(pl.block), lds, stream, static_cast<const T*>(x), static_cast<T*>(out), fw, fb, pl, arg);
  return check_launch("wt2d_plane_kernel");
}

// Plane shapes of the WTConvNeXt stages with K = 5: geometry as a compile-time constant.  Returns 1 if the shape
// is not one of them (or the run-time plan differs, e.g. unaligned pointers), else the launch's result.
template <typename T>
static int run_plane2d_static(int K, int tj1, const void* x, void* out, const float* fw, const float* fb,
                              const Plan2D& pl, const PlaneFold& fold, hipStream_t stream) {
  if (K != 5 || pl.H != pl.W) return 1;
#define WT_TRY(H_, L_)                                                                                  \
  if (pl.H == H_ && pl.L == L_) {                                                                       \
    using G = PlaneGeoStatic<H_, H_, 5, L_>;                                                            \
    constexpr Plan2D g = G::plan();                                                                     \
    constexpr int tj = G::tj1();                                                                        \
    if (tj1 == tj && same_plane_geometry(g, pl))                                                        \
      return run_plane2d_mode<T, 5, tj, G::mode(), G>(x, out, fw, fb, pl, fold, stream);                \
    return 1;                                                                                           \
  }
  WT_TRY(56, 3) WT_TRY(28, 3) WT_TRY(14, 2) WT_TRY(7, 2)
#undef WT_TRY
  return 1;
}

template <typename T, int K, int TJ1>
static int run_plane2d(const void* x, void* out, const float* fw, const float* fb, const Plan2D& pl,
                       const PlaneFold& fold, hipStream_t stream) {
  auto by_geo = [&](auto geo) {
    using G = decltype(geo);
    if (pl.prefetch && pl.fuse >= 2) return run_plane2d_mode<T, K, TJ1, 3, G>(x, out, fw, fb, pl, fold, stream);
    if (pl.prefetch) return run_plane2d_mode<T, K, TJ1, 0, G>(x, out, fw, fb, pl, fold, stream);
    if (pl.vec_ok) return run_plane2d_mode<T, K, TJ1, 1, G>(x, out, fw, fb, pl, fold, stream);
    return run_plane2d_mode<T, K, TJ1, 2, G>(x, out, fw, fb, pl, fold, stream);
  };
  return fold.dst != nullptr ? by_geo(PlaneGeoFold{}) : by_geo(PlaneGeoRuntime{});
}

template <typename T, int K>
static int run_plane2d_tj(int tj1, const void* x, void* out, const float* fw, const float* fb, const Plan2D& pl,
                          const PlaneFold& fold, hipStream_t stream) {
  switch (tj1) {
    case 1: return run_plane2d<T, K, 1>(x, out, fw, fb, pl, fold, stream);
    case 2: return run_plane2d<T, K, 2>(x, out, fw, fb, pl, fold, stream);
    default: return run_plane2d<T, K, 4>(x, out, fw, fb, pl, fold, stream);
  }
}

template <typename T>
static int run_plane2d_k(int K, int tj1, const void* x, void* out, const float* fw, const float* fb,
                         const Plan2D& pl, const PlaneFold& fold, hipStream_t stream) {
  switch (K) {
    case 1: return run_plane2d_tj<T, 1>(tj1, x, out, fw, fb, pl, fold, stream);
    case 3: return run_plane2d_tj<T, 3>(tj1, x, out, fw, fb, pl, fold, stream);
    case 5: return run_plane2d_tj<T, 5>(tj1, x, out, fw, fb, pl, fold, stream);
    case 7: return run_plane2d_tj<T, 7>(tj1, x, out, fw, fb, pl, fold, stream);
  }
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d is not built", K);
}

int launch_plane2d(int dtype, int K, int tj1, const void* x, void* out, const float* fw, const float* fb, const Plan2D& pl,
                   const PlaneFold& fold, hipStream_t stream) {
  if (dtype != WTCONV_BF16 && fold.dst == nullptr) {     // (bf16 tensors of these shapes are on the matrix-core kernels)
    const int e = dtype == WTCONV_F32 ? run_plane2d_static<float>(K, tj1, x, out, fw, fb, pl, fold, stream)
                                      : run_plane2d_static<f16_t>(K, tj1, x, out, fw, fb, pl, fold, stream);
    if (e != 1) return e;
  }
  return WT_BY_DTYPE(dtype, run_plane2d_k<T_>(K, tj1, x, out, fw, fb, pl, fold, stream));
}

}  // namespace wt
