// Launches of the WTConv2d kernels for planes beyond LDS (kernels2d_stream.h).
#include "launch.h"
#include "kernels2d.h"
#include "kernels2d_stream.h"

namespace wt {

// How a level of hl x wl coefficients goes over the lanes: the tiles that take the fewest waves.
static LaneSplit lane_tiles(int wl, int K) {
  const int HL = lane_halo(K), lanes = (wl + 1) / 2, least = HL > 0 ? 2 * HL : 1;
  LaneSplit best = {};
  double waves = 0.;
  for (int n = (lanes + kWave - 1) / kWave; n <= (lanes + 7) / 8 || best.per == 0; ++n) {
    LaneSplit s = {};
    s.own = (lanes + n - 1) / n;
    if (n > 1 && s.own < least) break;
    s.tiles = (lanes + s.own - 1) / s.own;
    s.gap = s.tiles == 2 ? HL : 0;
    s.pitch = s.own + (s.tiles > 2 ? 2 * HL : HL);
    if (s.tiles > 2) s.per = kWave / s.pitch;
    else if (s.tiles == 1) s.per = (kWave + HL) / s.pitch;
    else for (s.per = 0; (s.per + 1) * s.pitch + (s.per + 1) / 2 * s.gap <= kWave; ++s.per) {}
    if (s.per < 1) continue;
    const double w = static_cast<double>(s.tiles) / s.per;
    if (best.per == 0 || w < waves) { best = s; waves = w; }
  }
  return best;
}

// The layer's step: stretches of rows of least time, in rows of a wave: 2 R more rows count for half of them, 1.2 go to the
// start; a SIMD takes up to three waves side by side (fewer than 1.6 leave it waiting), and where they make more than a round
// the last one is a third empty.
// [8,96,160,160] fp32, K = 5, us by rows of a stretch: 20 59, 16 51, 14 47, 12 53, 10 53, 9 50, 8 52, 7 49, 5 51 (while each
// row's loads were still waited for at once; 14, which it takes, is 44 since).
static LaneSplit lane_split(int B, int C, int hl, int wl, int K) {
  constexpr int kSimds = 1024;      // 256 compute units
  const int R = K / 2;
  LaneSplit best = lane_tiles(wl, K);
  double least_time = 0.;
  for (int n = 1; n <= hl; ++n) {
    const int rows = (hl + n - 1) / n < 2 * R ? 2 * R : (hl + n - 1) / n;
    const int segs = (hl + rows - 1) / rows;
    const long long units = static_cast<long long>(B) * best.tiles * segs;
    const double per_simd = static_cast<double>(C) * ((units + best.per - 1) / best.per) / kSimds;
    const double up = static_cast<double>(static_cast<long long>(per_simd) + (per_simd > static_cast<long long>(per_simd) ? 1 : 0));
    double rounds = per_simd <= 3. ? up : per_simd + 0.35;
    if (rounds < 1.6) rounds = 1.6;
    const double time = rounds * (rows + 1. * R + 1.2);
    if (n == 1 || time < least_time) {
      least_time = time;
      best.segs = segs;
      best.rows = rows;
      best.units = static_cast<int>(units);
    }
    if (rows <= 2 * R || rows <= 4) break;
  }
  constexpr int kWavesPerBlock = kStreamThreads / kWave;
  best.blocks = (best.units + kWavesPerBlock * best.per - 1) / (kWavesPerBlock * best.per);
  return best;
}

// The correlations' step, whose nchunk workgroups a channel run side by side: the stretches whose shares of the waves are
// shortest, in rows; the 2 R rows of x before a stretch's first are loaded and transformed only and count for two.
static LaneSplit corr_split(int B, int hl, int wl, int K, int nchunk) {
  LaneSplit best = lane_tiles(wl, K);
  const long long waves = static_cast<long long>(nchunk) * (kStreamThreads / kWave);
  long long least = 0;
  for (int n = 1; n <= hl; ++n) {
    const int rows = (hl + n - 1) / n, segs = (hl + rows - 1) / rows;
    const long long units = static_cast<long long>(B) * best.tiles * segs;
    const long long groups = (units + best.per - 1) / best.per, time = (groups + waves - 1) / waves * (rows + 2);
    if (n == 1 || time < least) {
      least = time;
      best.segs = segs;
      best.rows = rows;
      best.units = static_cast<int>(units);
    }
    if (rows <= 4) break;
  }
  return best;
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
  const LaneSplit sp = lane_split(st.B, st.C, hl, wl, K);
  const long long blocks = (static_cast<long long>(st.C) * sp.blocks + 7) / 8 * 8;
  if (blocks > 0x7fffffffLL) return fail(WTCONV_E_UNSUPPORTED, "stream_final_kernel: %lld workgroups", blocks);
  const dim3 grid(static_cast<unsigned>(blocks));
  if (sub != nullptr)
    WT_LAUNCH((stream_final_kernel<T, K, true>), grid, dim3(kStreamThreads), 0, stream, static_cast<const T*>(x),
              static_cast<T*>(out), sub, st.H, st.W, hl, wl, fw, fb, st.C, fstride, fbase, fband, sp);
  else
    WT_LAUNCH((stream_final_kernel<T, K, false>), grid, dim3(kStreamThreads), 0, stream, static_cast<const T*>(x),
              static_cast<T*>(out), sub, st.H, st.W, hl, wl, fw, fb, st.C, fstride, fbase, fband, sp);
  return check_launch("stream_final_kernel");
}

template <typename T, int K>
static int run_stream_corr(const StreamStep& st, const void* x_, const void* g_, float* xll, float* gll, bool bands,
                           const StreamCorrOut& outp, int nchunk, hipStream_t stream) {
  const T* x = static_cast<const T*>(x_);
  const T* g = static_cast<const T*>(g_);
  const int hl = (st.H + 1) / 2, wl = (st.W + 1) / 2;
  const dim3 grid(st.C, nchunk);
  const LaneSplit sp = corr_split(st.B, hl, wl, K, nchunk);
  if constexpr (K <= 5) {
    if (bands) {
      WT_LAUNCH((stream_corr_kernel<T, K, true, true>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H, st.W, hl,
                wl, st.C, outp, sp);
      return check_launch("stream_corr_kernel");
    }
  }
  WT_LAUNCH((stream_corr_kernel<T, K, true, false>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H, st.W, hl, wl,
            st.C, outp, sp);
  if (int e = check_launch("stream_corr_kernel")) return e;
  if constexpr (K > 5) {
    if (bands) {
      WT_LAUNCH((stream_corr_kernel<T, K, false, true>), grid, dim3(kStreamThreads), 0, stream, x, g, xll, gll, st.H, st.W, hl,
                wl, st.C, outp, sp);
      return check_launch("stream_corr_kernel");
    }
  }
  return 0;
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
