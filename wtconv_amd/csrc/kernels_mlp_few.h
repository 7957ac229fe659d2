// The rest of a WTConvNeXt block behind its WTConv layer (kernels_mlp.h) for few pixels, as two kernels:
//
//   hidden = gelu(W1 LayerNorm_c(x) + b1)         out = shortcut + gamma * (W2 hidden + b2)
//
// With few pixels a kernel that keeps the hidden values to itself has too few workgroups, unless each takes a share of the
// hidden units and leaves partial sums of all outputs, which are then more to move than the weights: 196 pixels of 384
// channels made 18.9 MB of them.  Two kernels need none: every workgroup has a few outputs of its own and its waves share
// the contraction.
//
// What bounds them is latency -- one launch each, a chain of loads, the meeting of the waves -- and, with more pixels, the
// weights, which every tile of 32 pixels fetches as they lie: every lane 16 bytes of another row, four times the time of whole
// lines (tiles of 16 pixels: 14.7 us instead of 11.3 at 196 pixels of 384 channels).  The hidden values are written in the
// order in which the second kernel takes them, whole lines.  Figures stand with the rule that chooses them (mlp.hip).
//
// Both ask for all they read, also what only their last lines use, before their first wait.  Against the parameters and the
// shortcut loaded where they are used, us, pixels of channels: 3136 of 96 12.5 -> 12.3, 784 of 192 11.4 -> 11.2, 300 of 256
// 12.2 -> 10.2, 196 of 384 11.4 -> 10.9, 49 of 512 14.5 -> 13.8, 49 of 768 15.7 -> 15.2, 49 of 1024 20.5 -> 19.5.
#pragma once

#include "gelu.h"
#include "matrix.h"

namespace wt {

struct FewArgs {
  const bf16_t *x, *shortcut;
  bf16_t* out;
  const bf16_t *norm_w, *norm_b;      // (C)
  const bf16_t *w1, *b1;              // (hidden, C), (hidden)
  const bf16_t *w2, *b2;              // (C, hidden), (C)
  const bf16_t* gamma;                // (C) or nullptr
  bf16_t* hid;                        // in workspace: [tile of 16 pixels][step of 32 hidden units][lane][8], as the second kernel takes them
  float eps;
  int HW, C, hidden;
  int pixels;                         // B * HW
  int vec;                            // whether four consecutive pixels share an image and an aligned 8-byte word
};

// Which image pixel p is of: floor(p / HW) through the reciprocal.  Exact for the fewer than 4096 pixels that these kernels see
// (kFewPixelChannels, mlp.hip): the error of the quotient, some 2^-23 of it, is less than the half pixel added is of an image.
// A division would be 40 instructions ahead of the first load.
__device__ __forceinline__ int image_of(int p, float per_image) { return static_cast<int>((p + 0.5f) * per_image); }

// Sums of MT fragments over KG waves, added in order by the first; in the others the call returns false.  `meet`: LDS that
// nothing else is read from.
template <int KG, int MT>
__device__ __forceinline__ bool meet_waves(mat_acc (&acc)[MT], mat_acc* meet, int group, int groups, int kg, int lane) {
  if constexpr (KG > 1) {
    auto slot = [&](int k, int m) { return ((k * groups + group) * MT + m) * 64 + lane; };
    if (kg > 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m) meet[slot(kg - 1, m)] = acc[m];
    }
    __syncthreads();
    if (kg > 0) return false;
#pragma unroll
    for (int k = 0; k < KG - 1; ++k)
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        mat_acc o = meet[slot(k, m)];
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[m][r] += o[r];
      }
  }
  return true;
}

// 16 MT pixels x 16 NG hidden units a workgroup; KG waves share the channels.
template <int C_, int MT_, int NG_, int KG_>
struct FewShape {
  static constexpr int C = C_, MT = MT_, NG = NG_, KG = KG_, kThreads = 64 * NG * KG, MP = 16 * MT;
  static constexpr int PARTS = kThreads / MP, PAIRS = C / 2 / PARTS, kPitch = C + 8, kSteps = C / 32 / KG;
  static constexpr size_t kTileBytes = MP * kPitch * 2, kSumBytes = 2 * PARTS * MP * 4;
  static constexpr size_t kMeetBytes = static_cast<size_t>(KG - 1) * NG * MT * 1024;
  static constexpr size_t kLdsBytes = (kTileBytes > kSumBytes ? kTileBytes : kSumBytes) + kMeetBytes;
  static_assert((C / 2) % PARTS == 0 && (C / 32) % KG == 0 && kTileBytes % 16 == 0 && kSumBytes % 16 == 0, "whole steps");
};

template <typename S>
__global__ void __launch_bounds__(S::kThreads) few_hidden_kernel(FewArgs a) {
  constexpr int C = S::C, MT = S::MT, PARTS = S::PARTS, PAIRS = S::PAIRS, MP = S::MP, STEPS = S::kSteps;
  WT_SHARED_FLOATS(lds);
  bf16_t* tile = reinterpret_cast<bf16_t*>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4, ng = wave % S::NG, kg = wave / S::NG;
  const int first = blockIdx.x * MP, u0 = (blockIdx.y * S::NG + ng) * 16;
  // Everything that the workgroup reads is asked for here, in the order in which it is needed; of many channels the weights
  // first and the normalisation's parameters late (768 channels, 49 pixels, the order of the others: 8.4 -> 9.5 us).
  constexpr bool kWeightsFirst = PAIRS > 16;
  uint4 wf[STEPS];
  auto load_weights = [&] {
    const bf16_t* src = a.w1 + static_cast<size_t>(u0 + n) * C + kg * STEPS * 32 + 8 * q;
#pragma unroll
    for (int s = 0; s < STEPS; ++s) wf[s] = *reinterpret_cast<const uint4*>(src + 32 * s);
  };
  if constexpr (kWeightsFirst) load_weights();
  const int px = tid % MP, part = tid / MP;
  uint16_t v_lo[PAIRS], v_hi[PAIRS];
  {
    const int p = min(first + px, a.pixels - 1), b = image_of(p, 1.f / a.HW);      // (past the end: the last pixel again, not stored)
    const bf16_t* src = a.x + static_cast<size_t>(b) * C * a.HW + (p - b * a.HW);
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const bf16_t* at = src + static_cast<uint32_t>(2 * (part + i * PARTS) * a.HW);
      v_lo[i] = at[0];
      v_hi[i] = at[a.HW];
    }
  }
  uint32_t norm_w[PAIRS], norm_b[PAIRS];
  auto load_norm = [&] {
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      norm_w[i] = *reinterpret_cast<const uint32_t*>(a.norm_w + 2 * (part + i * PARTS));
      norm_b[i] = *reinterpret_cast<const uint32_t*>(a.norm_b + 2 * (part + i * PARTS));
    }
  };
  if constexpr (!kWeightsFirst) load_norm();
  if constexpr (!kWeightsFirst) load_weights();
  const uint2 b1 = *reinterpret_cast<const uint2*>(a.b1 + u0 + 4 * q);
  if constexpr (!kWeightsFirst) WT_SCHED_FENCE();
  {
    uint32_t v[PAIRS];
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) v[i] = v_lo[i] | (static_cast<uint32_t>(v_hi[i]) << 16);
    float* sums = lds;                                              // [pass][part][pixel]
    auto meet = [&](int pass, float s) {
      sums[(pass * PARTS + part) * MP + px] = s;
      __syncthreads();
      float total = 0.f;
#pragma unroll 8
      for (int j = 0; j < PARTS; ++j) total += sums[(pass * PARTS + j) * MP + px];
      return total;
    };
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      float lo, hi;
      unpack2<bf16_t>(v[i], lo, hi);
      s += lo + hi;
    }
    const float mean = meet(0, s) * (1.f / C);
    s = 0.f;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      float lo, hi;
      unpack2<bf16_t>(v[i], lo, hi);
      s = fmaf(lo - mean, lo - mean, s);
      s = fmaf(hi - mean, hi - mean, s);
    }
    const float rstd = rsqrtf(meet(1, s) * (1.f / C) + a.eps);
    __syncthreads();                                                // the sums have been read: their place takes the tile
    if constexpr (kWeightsFirst) load_norm();
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int c = 2 * (part + i * PARTS);
      float lo, hi, w_lo, w_hi, b_lo, b_hi;
      unpack2<bf16_t>(v[i], lo, hi);
      unpack2<bf16_t>(norm_w[i], w_lo, w_hi);
      unpack2<bf16_t>(norm_b[i], b_lo, b_hi);
      *reinterpret_cast<uint32_t*>(tile + px * S::kPitch + c) =
          pack_bf16x2(fmaf((lo - mean) * rstd, w_lo, b_lo), fmaf((hi - mean) * rstd, w_hi, b_hi));
    }
  }
  __syncthreads();
  mat_acc acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = mat_acc{0.f, 0.f, 0.f, 0.f};
  const bf16_t* at = tile + n * S::kPitch + kg * STEPS * 32 + 8 * q;
#pragma unroll
  for (int s = 0; s < STEPS; ++s)
#pragma unroll
    for (int m = 0; m < MT; ++m)
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          frag_of(wf[s]), frag_of(*reinterpret_cast<const uint4*>(at + 16 * m * S::kPitch + 32 * s)), acc[m], 0, 0, 0);
  mat_acc* meet = reinterpret_cast<mat_acc*>(lds) + (S::kLdsBytes - S::kMeetBytes) / 16;
  if (!meet_waves<S::KG>(acc, meet, ng, S::NG, kg, lane)) return;
  // lane (n, q) holds hidden units u0 + 4 q + 0..3 of pixel n of each tile
  float b[4];
  unpack2<bf16_t>(b1.x, b[0], b[1]);
  unpack2<bf16_t>(b1.y, b[2], b[3]);
  const int u = (u0 & 16) + 4 * q;                                  // within the step
#pragma unroll
  for (int m = 0; m < MT; ++m)
    *reinterpret_cast<uint2*>(a.hid + (static_cast<size_t>(blockIdx.x * MT + m) * (a.hidden / 32) + u0 / 32) * 512 +
                              ((u >> 3) * 16 + n) * 8 + (u & 7)) =
        uint2{pack_bf16x2(gelu_erf(acc[m][0] + b[0]), gelu_erf(acc[m][1] + b[1])),
              pack_bf16x2(gelu_erf(acc[m][2] + b[2]), gelu_erf(acc[m][3] + b[3]))};
}

// 16 MT pixels x 16 channels a workgroup; its KG waves share the hidden units, every KG-th step of 32 each.
template <int MT, int KG>
__global__ void __launch_bounds__(64 * KG) few_out_kernel(FewArgs a) {
  constexpr int D = 6;                                              // steps in flight
  __shared__ mat_acc meet[(KG - 1) * MT * 64];
  const int tid = threadIdx.x, lane = tid & 63, kg = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int c0 = blockIdx.y * 16, steps = a.hidden / 32;
  const bf16_t* hsrc = a.hid + static_cast<size_t>(blockIdx.x * MT) * steps * 512 + 8 * lane;
  const bf16_t* wsrc = a.w2 + static_cast<size_t>(c0 + n) * a.hidden + 8 * q;
  // What the end needs is asked for now: lane (n, q) will hold pixels 4 q + 0..3 of channel n of each tile.
  const int c = c0 + n;
  float g = 1.f, b2 = 0.f;
  size_t at[MT][4];
  uint2 sc[MT];
  if (kg == 0) {
    const float per_image = 1.f / a.HW;
    if (a.gamma != nullptr) g = bf16_to_f32(a.gamma[c]);
    b2 = bf16_to_f32(a.b2[c]);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int p0 = (blockIdx.x * MT + m) * 16 + 4 * q;
      sc[m] = uint2{0u, 0u};
      if (a.vec) {
        const int b = image_of(p0, per_image);
        at[m][0] = (static_cast<size_t>(b) * a.C + c) * a.HW + (p0 - b * a.HW);
        if (p0 < a.pixels) sc[m] = *reinterpret_cast<const uint2*>(a.shortcut + at[m][0]);
      } else {
        uint32_t s[4] = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int b = image_of(p0 + r, per_image);
          at[m][r] = (static_cast<size_t>(b) * a.C + c) * a.HW + (p0 + r - b * a.HW);
          if (p0 + r < a.pixels) s[r] = a.shortcut[at[m][r]];
        }
        sc[m] = uint2{s[0] | (s[1] << 16), s[2] | (s[3] << 16)};
      }
    }
  }
  mat_acc acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = mat_acc{0.f, 0.f, 0.f, 0.f};
  for (int s0 = kg; s0 < steps; s0 += D * KG) {
    uint4 hf[D][MT], wf[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int s = min(s0 + d * KG, steps - 1);                    // (past the end: any step, not multiplied)
      wf[d] = *reinterpret_cast<const uint4*>(wsrc + 32 * s);
#pragma unroll
      for (int m = 0; m < MT; ++m) hf[d][m] = *reinterpret_cast<const uint4*>(hsrc + static_cast<size_t>(m * steps + s) * 512);
    }
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (s0 + d * KG < steps) {
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag_of(hf[d][m]), frag_of(wf[d]), acc[m], 0, 0, 0);
      }
  }
  if (!meet_waves<KG>(acc, meet, 0, 1, kg, lane)) return;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int p0 = (blockIdx.x * MT + m) * 16 + 4 * q;
    float s[4];
    unpack2<bf16_t>(sc[m].x, s[0], s[1]);
    unpack2<bf16_t>(sc[m].y, s[2], s[3]);
    if (a.vec) {
      if (p0 >= a.pixels) return;
      *reinterpret_cast<uint2*>(a.out + at[m][0]) = uint2{pack_bf16x2(fmaf(g, acc[m][0] + b2, s[0]), fmaf(g, acc[m][1] + b2, s[1])),
                                                          pack_bf16x2(fmaf(g, acc[m][2] + b2, s[2]), fmaf(g, acc[m][3] + b2, s[3]))};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (p0 + r < a.pixels) a.out[at[m][r]] = f32_to_bf16(fmaf(g, acc[m][r] + b2, s[r]));
    }
  }
}

}  // namespace wt
