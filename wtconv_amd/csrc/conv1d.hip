// Launches of the WTConv1d kernels (kernels1d.h: tiles of a row; kernels1d_row.h: rows in registers).
#include "launch.h"
#include "kernels1d.h"
#include "kernels1d_row.h"
#include "kernels2d.h"

namespace wt {

// Chunks of a channel's units (rows, or segments of longer rows) in a row-resident kernel: C * nchunk workgroups that all run at once (one round: a second, partly
// filled round costs as much as a full one), `per_cu` of them per CU on 256 CUs -- constants, so that workspace
// sizes do not depend on the device queried.
void row1d_chunks(int units, int C, int per_cu, int* per_chunk, int* nchunk) {
  if (per_cu < 1) per_cu = 1;
  int want = 256 * per_cu / C;
  if (want < 1) want = 1;
  if (want > units) want = units;
  const int pc = (units + want - 1) / want;
  *per_chunk = pc;
  *nchunk = (units + pc - 1) / pc;
}

// ---- 1-D dispatch -------------------------------------------------------------------
template <typename T, int K = 1>
static int run_tile1d(const void* x, void* out, const float* fw, const float* fb, const Plan1D& pl, int B,
                      hipStream_t stream) {
  auto kern = wt1d_tile_kernel<T, K, kTJ1D>;
  const size_t lds = static_cast<size_t>(pl.lds_floats) * sizeof(float);
  if (int e = allow_lds(kern, lds)) return e;
  const long long nrows = static_cast<long long>(B) * pl.C;
  if (nrows > 0x7fffffffLL) return fail(WTCONV_E_UNSUPPORTED, "batch*channels = %lld is too large", nrows);
  const unsigned gy = nrows < 65535 ? static_cast<unsigned>(nrows) : 65535u;
  const unsigned gz = static_cast<unsigned>((nrows + gy - 1) / gy);
  if (gz > 65535u) return fail(WTCONV_E_UNSUPPORTED, "batch*channels = %lld is too large", nrows);
  WT_LAUNCH(kern, dim3(pl.ntiles, gy, gz), dim3(kBlock1D), lds, stream, static_cast<const T*>(x),
            static_cast<T*>(out), fw, fb, pl, static_cast<int>(nrows));
  return check_launch("wt1d_tile_kernel");
}

template <typename T, int K, int L>
static int run_wgrad1d(const void* x, const void* g, float* partial, const Plan1D& pl, int B, int per_chunk,
                       int nchunk, hipStream_t stream) {
  auto kern = wt1d_wgrad_kernel<T, K, L, kTJ1D>;
  const size_t lds = static_cast<size_t>(pl.lds_floats) * sizeof(float);
  if (int e = allow_lds(kern, lds)) return e;
  WT_LAUNCH(kern, dim3(pl.C, nchunk), dim3(kBlock1D), lds, stream, static_cast<const T*>(x),
            static_cast<const T*>(g), partial, pl, B, per_chunk);
  return check_launch("wt1d_wgrad_kernel");
}

template <typename T, int K = 1>
static int run_wgrad1d_l(int L, const void* x, const void* g, float* partial, const Plan1D& pl, int B,
                         int per_chunk, int nchunk, hipStream_t stream) {
  switch (L) {
    case 1: return run_wgrad1d<T, K, 1>(x, g, partial, pl, B, per_chunk, nchunk, stream);
    case 2: return run_wgrad1d<T, K, 2>(x, g, partial, pl, B, per_chunk, nchunk, stream);
    case 3: return run_wgrad1d<T, K, 3>(x, g, partial, pl, B, per_chunk, nchunk, stream);
    case 4: return run_wgrad1d<T, K, 4>(x, g, partial, pl, B, per_chunk, nchunk, stream);
    case 5: return run_wgrad1d<T, K, 5>(x, g, partial, pl, B, per_chunk, nchunk, stream);
  }
  return fail(WTCONV_E_ARG, "wt_levels %d", L);
}

template <typename T, int K, int L, int S>
static int run_row1d(const void* x, void* out, const wtconv_params* params, int pdtype, int flip, const Row1D& pl,
                     int B, int block, hipStream_t stream) {
  if constexpr (row1d_built(K, L, S)) {
    auto kern = wt1d_row_kernel<T, K, L, S>;
    const size_t lds = row1d_region(K, L, S, block) * sizeof(float);
    if (int e = allow_lds(kern, lds)) return e;
    int per_chunk, nchunk;
    row1d_chunks(B * pl.nseg, pl.C, resident_per_cu(kern, block, lds), &per_chunk, &nchunk);   // (no workspace depends on this)
    if (nchunk > 65535) return fail(WTCONV_E_UNSUPPORTED, "too many batch chunks (%d)", nchunk);
    WT_LAUNCH(kern, dim3(pl.C, nchunk), dim3(block), lds, stream, static_cast<const T*>(x), static_cast<T*>(out),
              to_table(params, L), pdtype, flip, pl, B * pl.nseg, per_chunk);
    return check_launch("wt1d_row_kernel");
  } else {
    return fail(WTCONV_E_UNSUPPORTED, "row-resident 1-D kernel not built for kernel_size %d, %d levels", K, L);
  }
}

// The fused backward kernel: grad_x, the chunks' partial sums and (by the last workgroup of each channel) the
// parameter gradients.  `tickets`: C words, cleared by a launch of their own right before.
template <typename T, int K, int L, int S>
static int run_row1d_bwd(const void* x, const void* g, void* gx, float* partial, unsigned* tickets,
                         const wtconv_params* params, int pdtype, const GradTable& gt, const Row1D& pl, int B,
                         int block, int per_chunk, int nchunk, hipStream_t stream) {
  if constexpr (row1d_bwd_built(K, L, S)) {
    auto kern = wt1d_row_bwd_kernel<T, K, L, S>;
    const size_t lds = 2 * row1d_region(K, L, S, block) * sizeof(float);
    if (int e = allow_lds(kern, lds)) return e;
    WT_LAUNCH(zero_tickets_kernel, dim3((pl.C + 255) / 256), dim3(256), 0, stream, tickets, pl.C);
    if (int e = check_launch("zero_tickets_kernel")) return e;
    WT_LAUNCH(kern, dim3(pl.C, nchunk), dim3(block), lds, stream, static_cast<const T*>(x),
              static_cast<const T*>(g), static_cast<T*>(gx), partial, tickets, to_table(params, L), pdtype, gt, pl,
              B * pl.nseg, per_chunk, nchunk);
    return check_launch("wt1d_row_bwd_kernel");
  } else {
    return fail(WTCONV_E_UNSUPPORTED, "row-resident 1-D kernel not built for kernel_size %d, %d levels", K, L);
  }
}

template <typename T, int K, int L, int S>
static int run_row1d_wgrad(const void* x, const void* g, float* partial, const Row1D& pl, int B, int block,
                           int per_chunk, int nchunk, hipStream_t stream) {
  if constexpr (row1d_built(K, L, S)) {
    auto kern = wt1d_row_wgrad_kernel<T, K, L, S>;
    const size_t lds = 2 * row1d_region(K, L, S, block) * sizeof(float);
    if (int e = allow_lds(kern, lds)) return e;
    WT_LAUNCH(kern, dim3(pl.C, nchunk), dim3(block), lds, stream, static_cast<const T*>(x),
              static_cast<const T*>(g), partial, pl, B * pl.nseg, per_chunk);
    return check_launch("wt1d_row_wgrad_kernel");
  } else {
    return fail(WTCONV_E_UNSUPPORTED, "row-resident 1-D kernel not built for kernel_size %d, %d levels", K, L);
  }
}

#define WT_ROW1D_SWITCH_L(T, K, CALL)                                 \
  switch (L) {                                                        \
    case 1: return CALL(T, K, 1, row1d_samples(1));                   \
    case 2: return CALL(T, K, 2, row1d_samples(2));                   \
    case 3: return CALL(T, K, 3, row1d_samples(3));                   \
    case 4: return CALL(T, K, 4, row1d_samples(4));                   \
    case 5: return CALL(T, K, 5, row1d_samples(5));                   \
  }                                                                   \
  break;
#define WT_ROW1D_SWITCH(T, CALL)                                      \
  switch (K) {                                                        \
    case 3: WT_ROW1D_SWITCH_L(T, 3, CALL)                             \
    case 5: WT_ROW1D_SWITCH_L(T, 5, CALL)                             \
    case 7: WT_ROW1D_SWITCH_L(T, 7, CALL)                             \
  }

template <typename T>
static int run_row1d_kl(int K, int L, const void* x, void* out, const wtconv_params* params, int pdtype,
                        int flip, const Row1D& pl, int B, int block, hipStream_t stream) {
#define WT_CALL(T_, K_, L_, S_) run_row1d<T_, K_, L_, S_>(x, out, params, pdtype, flip, pl, B, block, stream)
  WT_ROW1D_SWITCH(T, WT_CALL)
#undef WT_CALL
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d / %d levels not built", K, L);
}

template <typename T>
static int run_row1d_bwd_kl(int K, int L, const void* x, const void* g, void* gx, float* partial,
                            unsigned* tickets, const wtconv_params* params, int pdtype, const GradTable& gt,
                            const Row1D& pl, int B, int block, int per_chunk, int nchunk, hipStream_t stream) {
#define WT_CALL(T_, K_, L_, S_)                                                                                 \
  run_row1d_bwd<T_, K_, L_, S_>(x, g, gx, partial, tickets, params, pdtype, gt, pl, B, block, per_chunk, nchunk, \
                                stream)
  WT_ROW1D_SWITCH(T, WT_CALL)
#undef WT_CALL
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d / %d levels not built", K, L);
}

template <typename T>
static int run_row1d_wgrad_kl(int K, int L, const void* x, const void* g, float* partial, const Row1D& pl,
                              int B, int block, int per_chunk, int nchunk, hipStream_t stream) {
#define WT_CALL(T_, K_, L_, S_) \
  run_row1d_wgrad<T_, K_, L_, S_>(x, g, partial, pl, B, block, per_chunk, nchunk, stream)
  WT_ROW1D_SWITCH(T, WT_CALL)
#undef WT_CALL
  return fail(WTCONV_E_UNSUPPORTED, "kernel_size %d / %d levels not built", K, L);
}

int launch_tile1d(int dtype, const void* x, void* out, const float* fw, const float* fb, const Plan1D& pl, int B,
                  hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_tile1d<T_>(x, out, fw, fb, pl, B, stream));
}

int launch_wgrad1d(int dtype, int L, const void* x, const void* g, float* partial, const Plan1D& pl, int B, int per_chunk,
                   int nchunk, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_wgrad1d_l<T_>(L, x, g, partial, pl, B, per_chunk, nchunk, stream));
}

int launch_row1d(int dtype, int K, int L, const void* x, void* out, const wtconv_params* params, int pdtype, int flip,
                 const Row1D& pl, int B, int block, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_row1d_kl<T_>(K, L, x, out, params, pdtype, flip, pl, B, block, stream));
}

int launch_row1d_bwd(int dtype, int K, int L, const void* x, const void* g, void* gx, float* partial, unsigned* tickets,
                     const wtconv_params* params, int pdtype, const GradTable& gt, const Row1D& pl, int B, int block,
                     int per_chunk, int nchunk, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_row1d_bwd_kl<T_>(K, L, x, g, gx, partial, tickets, params, pdtype, gt, pl, B, block, per_chunk,
                                                 nchunk, stream));
}

int launch_row1d_wgrad(int dtype, int K, int L, const void* x, const void* g, float* partial, const Row1D& pl, int B,
                       int block, int per_chunk, int nchunk, hipStream_t stream) {
  return WT_BY_DTYPE(dtype, run_row1d_wgrad_kl<T_>(K, L, x, g, partial, pl, B, block, per_chunk, nchunk, stream));
}

}  // namespace wt
