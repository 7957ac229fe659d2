// Launchers of the vector-ALU kernels, one translation unit per family (the kernels are templates over element type, kernel
// size, levels and work split: compiled side by side they take a quarter of the time).
#pragma once

#include "common.h"
#include "host_util.h"
#include "kernels1d_row.h"
#include "plan.h"
#include "wgrad_finish.h"

namespace wt {

// The element type of the activations as the template argument `T_` of a launcher call.
#define WT_BY_DTYPE(dtype, CALL)                                              \
  ((dtype) == WTCONV_F32 ? [&] { using T_ = float; return CALL; }()          \
   : (dtype) == WTCONV_BF16 ? [&] { using T_ = bf16_t; return CALL; }()      \
                            : [&] { using T_ = f16_t; return CALL; }())

inline size_t round_up64(size_t v) { return (v + 63) / 64 * 64; }
inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// plane2d.hip: the layer on planes that fit LDS.
int launch_plane2d(int dtype, int K, int tj1, const void* x, void* out, const float* fw, const float* fb, const Plan2D& pl,
                   const PlaneFold& fold, hipStream_t stream);

// wgrad2d.hip: its parameter gradients.
int launch_wgrad2d(int dtype, int K, int L, const void* x, const void* g, float* partial, const Plan2D& pl, int B, int bchunk,
                   int nchunk, const FinishArgs& fin, hipStream_t stream);

// stream2d.hip: the steps that both are made of on planes beyond LDS.
struct StreamStep { int B, C, H, W; };
struct StreamCorrOut;
int launch_stream_ll(int dtype, const void* src, int hs, int ws, float* dst, int nplanes, hipStream_t stream);
int launch_stream_final(int dtype, int K, const StreamStep& st, const void* x, void* out, const float* sub, const float* fw,
                        const float* fb, int fstride, int fbase, int fband, hipStream_t stream);
int launch_stream_corr(int dtype, int K, const StreamStep& st, const void* x, const void* g, float* xll, float* gll,
                       bool bands, const StreamCorrOut& outp, int nchunk, hipStream_t stream);

// conv1d.hip: the 1-D layer, by tiles of a row and with rows in registers.
int launch_tile1d(int dtype, const void* x, void* out, const float* fw, const float* fb, const Plan1D& pl, int B,
                  hipStream_t stream);
int launch_wgrad1d(int dtype, int L, const void* x, const void* g, float* partial, const Plan1D& pl, int B, int per_chunk,
                   int nchunk, hipStream_t stream);
int launch_row1d(int dtype, int K, int L, const void* x, void* out, const wtconv_params* params, int pdtype, int flip,
                 const Row1D& pl, int B, int block, hipStream_t stream);
int launch_row1d_bwd(int dtype, int K, int L, const void* x, const void* g, void* gx, float* partial, unsigned* tickets,
                     const wtconv_params* params, int pdtype, const GradTable& gt, const Row1D& pl, int B, int block,
                     int per_chunk, int nchunk, hipStream_t stream);
int launch_row1d_wgrad(int dtype, int K, int L, const void* x, const void* g, float* partial, const Row1D& pl, int B,
                       int block, int per_chunk, int nchunk, hipStream_t stream);
void row1d_chunks(int units, int C, int per_cu, int* per_chunk, int* nchunk);

}  // namespace wt
