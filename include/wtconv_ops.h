/*
 * wtconv_ops.h -- C ABI of libwtconv_hip.so, second part: what a WTConvNeXt does around its WTConv layers beyond the two
 * passes of wtconv_hip.h.  Conventions (error codes, dtypes, streams, caller-owned memory) are those of wtconv_hip.h;
 * this part is versioned by itself, so that programs of the layer alone keep theirs.
 */
#ifndef WTCONV_OPS_H
#define WTCONV_OPS_H

#include "wtconv_hip.h"

#ifdef __cplusplus
extern "C" {
#endif

#define WTCONV_OPS_VERSION 2

/* Version of this part in the loaded library (== WTCONV_OPS_VERSION). */
int wtconv_ops_version(void);

/* ---- the backward passes of wtconv_hip.h with the parameters' gradients in a dtype of the caller's choice (float, bfloat16 or
 * half: `dtype` of the table).  Sums are in float; the results are rounded once. */
typedef struct {
  void *base_weight, *base_bias, *base_scale;
  void* wt_weight[WTCONV_MAX_LEVELS];
  void* wt_scale[WTCONV_MAX_LEVELS];
  int dtype;
} wtconv_typed_grads;

int wtconv2d_backward_params_typed(const void* x, const void* grad_out, const wtconv_params* params,
                                   const wtconv_typed_grads* grads, int B, int C, int H, int W, int K, int levels,
                                   int dtype, int param_dtype, void* workspace, size_t workspace_bytes, void* stream);
int wtconv2d_backward_typed(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                            const wtconv_typed_grads* grads, int B, int C, int H, int W, int K, int levels, int dtype,
                            int param_dtype, void* workspace, size_t workspace_bytes, void* stream);
int wtconv1d_backward_params_typed(const void* x, const void* grad_out, const wtconv_params* params,
                                   const wtconv_typed_grads* grads, int B, int C, int N, int K, int levels, int dtype,
                                   int param_dtype, void* workspace, size_t workspace_bytes, void* stream);
int wtconv1d_backward_typed(const void* x, const void* grad_out, void* grad_x, const wtconv_params* params,
                            const wtconv_typed_grads* grads, int B, int C, int N, int K, int levels, int dtype,
                            int param_dtype, void* workspace, size_t workspace_bytes, void* stream);

/* wtconv_channel_norm_backward and wtconv_block_residual_backward likewise. */
int wtconv_channel_norm_backward_typed(const void* x, const void* dy, const void* weight, void* dx, void* dweight, void* dbias,
                                       int grad_dtype, int B, int C, int HW, float eps, int dtype, int param_dtype,
                                       int dy_nhwc, void* workspace, size_t workspace_bytes, void* stream);
int wtconv_block_residual_backward_typed(const void* dout, const void* y, const void* gamma, void* dy, void* dgamma,
                                         int grad_dtype, int B, int C, int HW, int dtype, int param_dtype, void* workspace,
                                         size_t workspace_bytes, void* stream);

/* ---- the convolutions that change resolution, with the LayerNorm beside them, for inference in bfloat16:
 *   stem != 0:  out = LayerNorm_c(conv 4x4 stride 4 (x) + bias), norm parameters of `cout` values;
 *   stem == 0:  out = conv 2x2 stride 2 (LayerNorm_c(x)) + bias, norm parameters of `C` values
 * (wtconvnext/wtconvnext.py:170-181, :294-297 of the reference).  x (B, C, H, W), out (B, cout, H / P, W / P), conv_weight
 * (cout, C, P, P); everything 16-byte aligned.  Sums and LayerNorm in float; normalised values are rounded to bfloat16
 * once, as are the results.  wtconv_patch_conv_supported says whether a size has a kernel that is faster than a library's
 * convolution with passes around it (the call takes every size with a kernel: cout in multiples of 32 for C of 96, 128, 192, 256,
 * 384 and 512, cout of 96 or 128 for a stem of up to 4 channels whose rows are multiples of 16); the workspace (16-byte aligned) takes
 * the weights in the order of the products. */
typedef struct {
  const void *conv_weight, *conv_bias;
  const void *norm_weight, *norm_bias;
} wtconv_patch_params;

int wtconv_patch_conv_supported(int stem, int B, int C, int H, int W, int cout);
size_t wtconv_patch_conv_workspace_bytes(int stem, int B, int C, int H, int W, int cout);
int wtconv_patch_conv(int stem, const void* x, void* out, const wtconv_patch_params* params, int B, int C, int H, int W,
                      int cout, float eps, int dtype, int param_dtype, void* workspace, size_t workspace_bytes,
                      void* stream);

/* ---- a block's MLP in training, bfloat16: y = fc2(gelu(fc1(x))) with x, y (pixels, C), exact (erf) GELU, fc1_weight
 * (hidden, C), fc2_weight (C, hidden) (wtconvnext/wtconvnext.py:125-136; the norm and gamma of wtconv_mlp_params are not
 * read).  Everything 16-byte aligned.  Sums and GELU in float; each result is rounded to bfloat16 once.
 * The forward call writes act = gelu(h) and, unless h is NULL, h = fc1(x), both (pixels, hidden); the backward call takes
 * them and dy = dL/dy, and writes what is not NULL of dx and the parameters' gradients (a bias gradient only together
 * with its weight's).  `want` says the same to the workspace query.  wtconv_mlp_supported: whether a
 * size has kernels that are faster than a library's products with passes between them; the calls take every size with kernels,
 * those for which the workspace query is not 0. */
typedef struct {
  void *fc1_weight, *fc1_bias, *fc2_weight, *fc2_bias;
} wtconv_mlp_grads;

#define WTCONV_MLP_DX 1
#define WTCONV_MLP_FC1 2
#define WTCONV_MLP_FC2 4

int wtconv_mlp_supported(long long pixels, int C, int hidden);
int wtconv_mlp_forward(const void* x, void* h, void* act, void* y, const wtconv_mlp_params* params, long long pixels, int C,
                       int hidden, int dtype, int param_dtype, void* stream);
size_t wtconv_mlp_backward_workspace_bytes(long long pixels, int C, int hidden, int want);
int wtconv_mlp_backward(const void* x, const void* h, const void* act, const void* dy, const wtconv_mlp_params* params,
                        void* dx, const wtconv_mlp_grads* grads, long long pixels, int C, int hidden, int dtype,
                        int param_dtype, void* workspace, size_t workspace_bytes, void* stream);

/* ---- what precedes the classifier (the head at wtconvnext/wtconvnext.py:358-369 of the reference): out (B, C) =
 * LayerNorm over the channels of the means over the pixels of x (B, C, HW), the means rounded to `dtype` as between two
 * operators.  Float or bfloat16 with parameters of either, C even and at most 2048, x aligned to four bytes.
 * wtconv_pool_norm_supported says whether one workgroup an image is the faster way. */
int wtconv_pool_norm_supported(int B, int C, int HW);
int wtconv_pool_norm(const void* x, void* out, const void* weight, const void* bias, int B, int C, int HW, float eps, int dtype,
                     int param_dtype, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* WTCONV_OPS_H */
