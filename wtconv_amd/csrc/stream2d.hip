// Launches of the level-by-level WTConv2d kernels (kernels2d_stream.h).
#include "launch.h"
#include "kernels2d.h"
#include "kernels2d_stream.h"

namespace wt {

// `ll_only`: the level-1 detail bands are not stored (forward / input-gradient pass: its last
// synthesis level rebuilds them from the pixels; the weight-gradient pass needs them).
template <typename T>
static int stream_analysis_chain(const T* src, float* pyr, const Stream2D& sp, hipStream_t stream, bool ll_only) {
  const unsigned gy = sp.nplanes < 65535 ? sp.nplanes : 65535;
  for (int l = 1; l <= sp.L; ++l) {
    const int n = sp.h[l] * sp.w[l];
    const unsigned gx = static_cast<unsigned>((n + 255) / 256);
    if (l == 1 && ll_only) {
      WT_LAUNCH((stream_analysis_kernel<T, true>), dim3(gx, gy), dim3(256), 0, stream, src,
                static_cast<size_t>(sp.H) * sp.W, sp.H, sp.W, pyr + sp.aoff[1], sp.h[1], sp.w[1], sp.nplanes);
    } else if (l == 1) {
      WT_LAUNCH((stream_analysis_kernel<T, false>), dim3(gx, gy), dim3(256), 0, stream, src,
                static_cast<size_t>(sp.H) * sp.W, sp.H, sp.W, pyr + sp.aoff[1], sp.h[1], sp.w[1], sp.nplanes);
    } else {
      WT_LAUNCH((stream_analysis_kernel<float, false>), dim3(gx, gy), dim3(256), 0, stream,
                static_cast<const float*>(pyr + sp.aoff[l - 1]), static_cast<size_t>(4) * sp.h[l - 1] * sp.w[l - 1],
                sp.h[l - 1], sp.w[l - 1], pyr + sp.aoff[l], sp.h[l], sp.w[l], sp.nplanes);
    }
    if (int e = check_launch("stream_analysis_kernel")) return e;
  }
  return 0;
}

// `have_pyramid`: the pyramid of x is in `pyr` already (the whole backward pass shares the one of grad_out).
template <typename T, int K>
static int run_stream2d(const void* x_, void* out_, const float* fw, const float* fb, float* pyr, const Stream2D& sp,
                        hipStream_t stream, bool have_pyramid = false) {
  const T* x = static_cast<const T*>(x_);
  T* out = static_cast<T*>(out_);
  if (sp.L > 1 && !have_pyramid) {      // a single level is synthesised from the pixels alone
    if (int e = stream_analysis_chain<T>(x, pyr, sp, stream, true)) return e;
  }
  const unsigned gy = sp.nplanes < 65535 ? sp.nplanes : 65535;
  const unsigned gz = (sp.nplanes + gy - 1) / gy;
  const int NF = 1 + 4 * sp.L;
  for (int l = sp.L; l >= 1; --l) {
    const unsigned tiles = static_cast<unsigned>(((sp.h[l] + kStreamTile - 1) / kStreamTile) *
                                                 ((sp.w[l] + kStreamTileW - 1) / kStreamTileW));
    const float* zin = l < sp.L ? pyr + sp.zoff[l + 1] : nullptr;
    const bool io_ok = l > 1 || (aligned16(x) && aligned16(out));
    const int vec = (sp.w[l] % 4 == 0 && aligned16(pyr) ? 1 : 0) | (sp.w[l - 1] % 4 == 0 && io_ok ? 2 : 0);
    if (l > 1) {
      WT_LAUNCH((stream_synth_kernel<T, K, false>), dim3(tiles, gy, gz), dim3(256), 0, stream,
                static_cast<const float*>(pyr + sp.aoff[l]), sp.h[l], sp.w[l], zin, pyr + sp.zoff[l], sp.h[l - 1],
                sp.w[l - 1], static_cast<const T*>(nullptr), static_cast<T*>(nullptr), fw, fb, sp.C, NF,
                1 + 4 * (l - 1), sp.nplanes, vec);
    } else {
      WT_LAUNCH((stream_synth_kernel<T, K, true>), dim3(tiles, gy, gz), dim3(256), 0, stream,
                static_cast<const float*>(pyr + sp.aoff[1]), sp.h[1], sp.w[1], zin, static_cast<float*>(nullptr), sp.H,
                sp.W, x, out, fw, fb, sp.C, NF, 1, sp.nplanes, vec);
    }
    if (int e = check_launch("stream_synth_kernel")) return e;
  }
  return 0;
}

template <typename T>
static int run_stream2d_k(int K, const void* x, void* out, const float* fw, const float* fb, float* pyr,
                          const Stream2D& sp, hipStream_t stream, bool have_pyramid = false) {
  switch (K) {
    case 1: return run_stream2d<T, 1>(x, out, fw, fb, pyr, sp, stream, have_pyramid);
    case 3: return run_stream2d<T, 3>(x, out, fw, fb, pyr, sp, stream, have_pyramid);
    case 5: return run_stream2d<T, 5>(x, out, fw, fb, pyr, sp, stream, have_pyramid);
    case 7: return run_stream2d<T, 7>(x, out, fw, fb, pyr, sp, stream, have_pyramid);
  }
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d is not built", K);
}

// `have_g_pyramid`: the pyramid of grad_out is in `pyr_g` already (left there by the input-gradient pass of the same call).
template <typename T, int K>
static int run_stream2d_wgrad(const void* x_, const void* g_, float* partial, float* pyr_x, float* pyr_g,
                              const Stream2D& sp, int B, int nchunk, hipStream_t stream, bool have_g_pyramid = false) {
  const T* x = static_cast<const T*>(x_);
  const T* g = static_cast<const T*>(g_);
  if (int e = stream_analysis_chain<T>(x, pyr_x, sp, stream, false)) return e;
  if (!have_g_pyramid)
    if (int e = stream_analysis_chain<T>(g, pyr_g, sp, stream, false)) return e;
  const int rec = (1 + 4 * sp.L) * K * K + 1;
  const bool pyr_ok = aligned16(pyr_x) && aligned16(pyr_g);
  // chunks of a launch: at least four (batch item, tile) units per workgroup where the level has them
  auto level_chunks = [&](int h, int w) {
    const long units = static_cast<long>(B) * ((h + kStreamTile - 1) / kStreamTile) *
                       ((w + kStreamTileW - 1) / kStreamTileW);
    const long nc = units / 4;
    return static_cast<unsigned>(nc < 1 ? 1 : (nc > nchunk ? nchunk : nc));
  };
  WT_LAUNCH((stream_corr_kernel<T, K>), dim3(sp.C, level_chunks(sp.H, sp.W)), dim3(256), 0, stream, x, g,
            static_cast<size_t>(sp.H) * sp.W, static_cast<size_t>(0), sp.H, sp.W, partial, rec, 0, 1, 1, B, sp.C,
            (sp.W % 4 == 0 && aligned16(x) && aligned16(g)) ? 1 : 0, nchunk);
  if (int e = check_launch("stream_corr_kernel")) return e;
  for (int l = 1; l <= sp.L; ++l) {
    const size_t n = static_cast<size_t>(sp.h[l]) * sp.w[l];
    WT_LAUNCH((stream_corr_kernel<float, K>), dim3(sp.C * 4, level_chunks(sp.h[l], sp.w[l])), dim3(256), 0, stream,
              static_cast<const float*>(pyr_x + sp.aoff[l]), static_cast<const float*>(pyr_g + sp.aoff[l]), 4 * n, n,
              sp.h[l], sp.w[l], partial, rec, 1 + 4 * (l - 1), 4, 0, B, sp.C,
              (sp.w[l] % 4 == 0 && pyr_ok) ? 1 : 0, nchunk);
    if (int e = check_launch("stream_corr_kernel")) return e;
  }
  return 0;
}

template <typename T>
static int run_stream2d_wgrad_k(int K, const void* x, const void* g, float* partial, float* pyr_x, float* pyr_g,
                                const Stream2D& sp, int B, int nchunk, hipStream_t stream, bool have_g_pyramid = false) {
  switch (K) {
    case 1: return run_stream2d_wgrad<T, 1>(x, g, partial, pyr_x, pyr_g, sp, B, nchunk, stream, have_g_pyramid);
    case 3: return run_stream2d_wgrad<T, 3>(x, g, partial, pyr_x, pyr_g, sp, B, nchunk, stream, have_g_pyramid);
    case 5: return run_stream2d_wgrad<T, 5>(x, g, partial, pyr_x, pyr_g, sp, B, nchunk, stream, have_g_pyramid);
    case 7: return run_stream2d_wgrad<T, 7>(x, g, partial, pyr_x, pyr_g, sp, B, nchunk, stream, have_g_pyramid);
  }
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d is not built", K);
}

int launch_stream_analysis(int dtype, const void* src, float* pyr, const Stream2D& sp, hipStream_t stream, bool ll_only) {
  return WT_BY_DTYPE(dtype, stream_analysis_chain<T_>(static_cast<const T_*>(src), pyr, sp, stream, ll_only));
}

int launch_stream2d(int dtype, int K, const void* x, void* out, const float* fw, const float* fb, float* pyr, const Stream2D& sp,
                    hipStream_t stream, bool have_pyramid) {
  return WT_BY_DTYPE(dtype, run_stream2d_k<T_>(K, x, out, fw, fb, pyr, sp, stream, have_pyramid));
}

int launch_stream2d_wgrad(int dtype, int K, const void* x, const void* g, float* partial, float* pyr_x, float* pyr_g,
                          const Stream2D& sp, int B, int nchunk, hipStream_t stream, bool have_g_pyramid) {
  return WT_BY_DTYPE(dtype, run_stream2d_wgrad_k<T_>(K, x, g, partial, pyr_x, pyr_g, sp, B, nchunk, stream, have_g_pyramid));
}

}  // namespace wt
