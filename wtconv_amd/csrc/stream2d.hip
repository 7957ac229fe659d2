// Launches of the WTConv2d kernels for planes beyond LDS (kernels2d_stream.h).
#include "launch.h"
#include "kernels2d.h"
#include "kernels2d_stream.h"

namespace wt {

// The tile shape that covers a level of hl x wl coefficients with the fewest tiles (a tile costs about the same time
// whatever its shape, most of its threads being at work).
template <typename F>
static int by_stream_shape(int hl, int wl, F&& launch) {
  auto tiles = [&](int tw, int th) {
    return static_cast<long long>((wl + tw - 1) / tw) * ((hl + th - 1) / th);
  };
  const long long n64 = tiles(64, 16), n80 = tiles(80, 12), n48 = tiles(48, 20);
  if (n64 <= n80 && n64 <= n48) return launch(StreamShape<64, 16>{}, n64);
  return n80 <= n48 ? launch(StreamShape<80, 12>{}, n80) : launch(StreamShape<48, 20>{}, n48);
}

template <typename T>
static int run_stream_ll(const void* src, int hs, int ws, float* dst, int nplanes, hipStream_t stream) {
  const int hd = (hs + 1) / 2, wd = (ws + 1) / 2;
  const unsigned gy = nplanes < 65535 ? nplanes : 65535;
  const unsigned gx = static_cast<unsigned>((static_cast<long long>(hd) * ((wd + 3) / 4) + kStreamThreads - 1) / kStreamThreads);
  WT_LAUNCH(stream_ll_kernel<T>, dim3(gx, gy), dim3(kStreamThreads), 0, stream, static_cast<const T*>(src), hs, ws, dst,
            hd, wd, nplanes);
  return check_launch("stream_ll_kernel");
}

template <typename T, int K>
static int run_stream_final(const StreamStep& st, const void* x, void* out, const float* sub, const float* fw,
                            const float* fb, int fstride, int fbase, int fband, hipStream_t stream) {
  const int hl = (st.H + 1) / 2, wl = (st.W + 1) / 2;
  const int nplanes = st.B * st.C;
  const unsigned gy = nplanes < 65535 ? nplanes : 65535;
  const unsigned gz = (nplanes + gy - 1) / gy;
  return by_stream_shape(hl, wl, [&](auto shape, long long tiles) {
    using Sh = decltype(shape);
    const dim3 grid(static_cast<unsigned>(tiles), gy, gz);
    if (sub != nullptr)
      WT_LAUNCH((stream_final_kernel<T, K, Sh, true>), grid, dim3(kStreamThreads), 0, stream, static_cast<const T*>(x),
                static_cast<T*>(out), sub, st.H, st.W, hl, wl, fw, fb, st.C, fstride, fbase, fband, nplanes);
    else
      WT_LAUNCH((stream_final_kernel<T, K, Sh, false>), grid, dim3(kStreamThreads), 0, stream, static_cast<const T*>(x),
                static_cast<T*>(out), sub, st.H, st.W, hl, wl, fw, fb, st.C, fstride, fbase, fband, nplanes);
    return check_launch("stream_final_kernel");
  });
}

template <typename T, int K>
static int run_stream_corr(const StreamStep& st, const void* x_, const void* g_, float* xll, float* gll, bool bands,
                           const StreamCorrOut& outp, int nchunk, hipStream_t stream) {
  const T* x = static_cast<const T*>(x_);
  const T* g = static_cast<const T*>(g_);
  const int hl = (st.H + 1) / 2, wl = (st.W + 1) / 2;
  return by_stream_shape(hl, wl, [&](auto shape, long long) {
    using Sh = decltype(shape);
    const dim3 grid(st.C, nchunk);
    if constexpr (K <= 5) {
      if (bands) {
        WT_LAUNCH((stream_corr_kernel<T, K, Sh, true, true>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H,
                  st.W, hl, wl, st.B, st.C, outp);
        return check_launch("stream_corr_kernel");
      }
    }
    WT_LAUNCH((stream_corr_kernel<T, K, Sh, true, false>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H,
              st.W, hl, wl, st.B, st.C, outp);
    if (int e = check_launch("stream_corr_kernel")) return e;
    if constexpr (K > 5) {
      if (bands) {
        WT_LAUNCH((stream_corr_kernel<T, K, Sh, false, true>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H,
                  st.W, hl, wl, st.B, st.C, outp);
        return check_launch("stream_corr_kernel");
      }
    }
    return 0;
  });
}

#define WT_BY_K(K, CALL)                                                              \
  switch (K) {                                                                        \
    case 1: { constexpr int K_ = 1; return CALL; }                                    \
    case 3: { constexpr int K_ = 3; return CALL; }                                    \
    case 5: { constexpr int K_ = 5; return CALL; }                                    \
    case 7: { constexpr int K_ = 7; return CALL; }                                    \
  }                                                                                   \
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d is not built", K)

template <typename T>
static int run_stream_final_k(int K, const StreamStep& st, const void* x, void* out, const float* sub, const float* fw,
                              const float* fb, int fstride, int fbase, int fband, hipStream_t stream) {
  WT_BY_K(K, (run_stream_final<T, K_>(st, x, out, sub, fw, fb, fstride, fbase, fband, stream)));
}

template <typename T>
static int run_stream_corr_k(int K, const StreamStep& st, const void* x, const void* g, float* xll, float* gll, bool bands,
                             const StreamCorrOut& outp, int nchunk, hipStream_t stream) {
  WT_BY_K(K, (run_stream_corr<T, K_>(st, x, g, xll, gll, bands, outp, nchunk, stream)));
}

int launch_stream_ll(int dtype, const void* src, int hs, int ws, float* dst, int nplanes, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_stream_ll<T_>(src, hs, ws, dst, nplanes, stream));
}

int launch_stream_final(int dtype, int K, const StreamStep& st, const void* x, void* out, const float* sub, const float* fw,
                        const float* fb, int fstride, int fbase, int fband, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_stream_final_k<T_>(K, st, x, out, sub, fw, fb, fstride, fbase, fband, stream));
}

int launch_stream_corr(int dtype, int K, const StreamStep& st, const void* x, const void* g, float* xll, float* gll,
                       bool bands, const StreamCorrOut& outp, int nchunk, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_stream_corr_k<T_>(K, st, x, g, xll, gll, bands, outp, nchunk, stream));
}

}  // namespace wt
