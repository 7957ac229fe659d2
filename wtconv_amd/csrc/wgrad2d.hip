// Launches of the plane-resident parameter-gradient kernel (kernels2d.h).
#include "launch.h"
#include "kernels2d.h"

namespace wt {

template <typename T, int K, int L, typename Geo = PlaneGeoRuntime>
static int run_wgrad2d(const void* x, const void* g, float* partial, const Plan2D& pl, int B, int bchunk,
                       int nchunk, const FinishArgs& fin, hipStream_t stream) {
  auto kern = wt2d_wgrad_kernel<T, K, L, kTJW, Geo>;
  const size_t lds = static_cast<size_t>(pl.lds_floats) * sizeof(float);
  if (int e = allow_lds(kern, lds)) return e;
  WT_LAUNCH(kern, dim3(pl.C, nchunk), dim3(512), lds, stream, static_cast<const T*>(x), static_cast<const T*>(g),
            partial, pl, B, bchunk, fin);
  return check_launch("wt2d_wgrad_kernel");
}

// Plane shapes of the WTConvNeXt stages with K = 5 at their usual planes per iteration: geometry as a compile-time
// constant.  Returns 1 if the launch is not one of them, else the launch's result.
template <typename T>
static int run_wgrad2d_static(int K, int L, const void* x, const void* g, float* partial, const Plan2D& pl, int B,
                              int bchunk, int nchunk, const FinishArgs& fin, hipStream_t stream) {
  if (K != 5 || pl.H != pl.W) return 1;
#define WT_TRY(H_, L_)                                                                                   \
  if (pl.H == H_ && L == L_) {                                                                           \
    constexpr int PB = wgrad_planes_that_fit(128, H_, H_, 5, L_);                                        \
    using G = WgradGeoStatic<H_, H_, 5, L_, PB>;                                                         \
    constexpr Plan2D gp = G::plan();                                                                     \
    if (same_wgrad_geometry(gp, pl))                                                                     \
      return run_wgrad2d<T, 5, L_, G>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);                     \
    return 1;                                                                                            \
  }
  WT_TRY(56, 3) WT_TRY(28, 3) WT_TRY(14, 2) WT_TRY(7, 2)
#undef WT_TRY
  return 1;
}

template <typename T, int K>
static int run_wgrad2d_l(int L, const void* x, const void* g, float* partial, const Plan2D& pl, int B,
                         int bchunk, int nchunk, const FinishArgs& fin, hipStream_t stream) {
  switch (L) {
    case 1: return run_wgrad2d<T, K, 1>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 2: return run_wgrad2d<T, K, 2>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 3: return run_wgrad2d<T, K, 3>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 4: return run_wgrad2d<T, K, 4>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 5: return run_wgrad2d<T, K, 5>(x, g, partial, pl, B, bchunk, nchunk, fin, stream);
  }
  return fail(WTCONV_E_ARG, "wt_levels %d", L);
}

template <typename T>
static int run_wgrad2d_k(int K, int L, const void* x, const void* g, float* partial, const Plan2D& pl, int B,
                         int bchunk, int nchunk, const FinishArgs& fin, hipStream_t stream) {
  switch (K) {
    case 1: return run_wgrad2d_l<T, 1>(L, x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 3: return run_wgrad2d_l<T, 3>(L, x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 5: return run_wgrad2d_l<T, 5>(L, x, g, partial, pl, B, bchunk, nchunk, fin, stream);
    case 7: return run_wgrad2d_l<T, 7>(L, x, g, partial, pl, B, bchunk, nchunk, fin, stream);
  }
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d is not built", K);
}

int launch_wgrad2d(int dtype, int K, int L, const void* x, const void* g, float* partial, const Plan2D& pl, int B, int bchunk,
                   int nchunk, const FinishArgs& fin, hipStream_t stream) {
  if (pl.W > kMaxWgradWidth || row_lanes(pl.W) > (1 << pl.slot_shift))      // (rows are walked whole)
    return fail(WTCONV_E_UNSUPPORTED, "rows of %d pixels are too long for the plane-resident kernels", pl.W);
  const int e = dtype == WTCONV_F32   ? run_wgrad2d_static<float>(K, L, x, g, partial, pl, B, bchunk, nchunk, fin, stream)
                : dtype == WTCONV_F16 ? run_wgrad2d_static<f16_t>(K, L, x, g, partial, pl, B, bchunk, nchunk, fin, stream)
                                      : 1;
  if (e != 1) return e;
  return WT_BY_DTYPE(dtype, run_wgrad2d_k<T_>(K, L, x, g, partial, pl, B, bchunk, nchunk, fin, stream));
}

}  // namespace wt
