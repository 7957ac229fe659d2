// The convolutions with which a WTConvNeXt changes resolution, each with the LayerNorm beside it in one matrix-core kernel, for
// inference in bfloat16:
//
//   stem         out = LayerNorm_c(conv 4 x 4, stride 4 (x) + bias)        (wtconvnext/wtconvnext.py:294-297)
//   downsample   out = conv 2 x 2, stride 2 (LayerNorm_c(x)) + bias        (:170-181)
//
// x, out are (B, C, H, W); the weights are (Cout, Cin, P, P) as nn.Conv2d keeps them.  The patches do not overlap, so both
// are products of a pixel's patch, K = Cin * P * P values in the order of the weights, with the weights' rows.
//
// What bounds them is memory, the input read once and the output written once, and, the more channels, the weights that every
// workgroup takes from the L2.  The separate passes (a norm, a library convolution between two layout changes, the bias)
// move eight to ten times as much: on 256 images of 224 x 224 they take about 230 us for the stem and 660 for the three
// downsample layers of WTConvNeXt-T, these kernels 41 (5.6 TB/s) and 201.
#pragma once

#include "matrix.h"

namespace wt {

struct PatchArgs {
  const bf16_t* x;
  bf16_t* out;
  const bf16_t *w, *bias;             // (cout, cin, P, P), (cout)
  const bf16_t *norm_w, *norm_b;
  bf16_t* frags;                      // the weights as fragments, in workspace (cout * cin * P * P)
  float eps;
  int cin, cout, H, W, HO, WO;
  int pixels;                         // B * HO * WO
  int vec;                            // whether four consecutive output pixels share an image and an aligned 8-byte word
};

// ---- downsample -----------------------------------------------------------------------------------------------------
// A workgroup takes 16 MT output pixels.  It loads the 2 x 2 patches of all channels into registers (a thread: one output
// pixel, every PARTS-th pair of channels), finds the statistics of the four input pixels in two exact passes over them,
// and leaves the normalised values in LDS as the A operand, [pixel][k] with k = 4 c + 2 ky + kx -- which is the order of
// the weights.  The weights are the B operand: each fragment is used by one wave only, so it comes straight from memory
// (the caches: they are the same for every workgroup) into that wave's registers, kAhead steps before its use.
//
// NG groups of waves share the output channels, NTW tiles of 16 each; KG groups share the contraction (their sums meet in
// LDS): with few pixels, a wave that goes through the whole of K is a chain of loads.
template <int C_, int MT_, int NG_, int KG_, int NTW_>
struct PatchShape {
  static constexpr int C = C_, MT = MT_, NG = NG_, KG = KG_, NTW = NTW_;
  static constexpr int kThreads = 64 * NG * KG, MP = 16 * MT;
  static constexpr int PARTS = kThreads / MP, PAIRS = C / 2 / PARTS;
  static constexpr int K = 4 * C, kPitch = K + 8;      // (rows 16 bytes apart modulo the banks)
  static constexpr int COUT = NG * NTW * 16;           // of a workgroup
  static constexpr bool kLaidOut = KG == 1;
  static constexpr int kSteps = K / 32 / KG;
  static constexpr int kAhead = kSteps % 6 == 0 ? 6 : 4;
  static_assert(kThreads % MP == 0 && (C / 2) % PARTS == 0 && (K / 32) % KG == 0 && kSteps % kAhead == 0, "whole steps");
  static constexpr size_t kTileBytes = static_cast<size_t>(MP) * kPitch * 2;
  static constexpr size_t kSumBytes = 2 * static_cast<size_t>(PARTS) * MP * 16;
  static constexpr size_t kMeetBytes = KG > 1 ? static_cast<size_t>(KG) * NG * NTW * MT * 1024 : 0;
  static constexpr size_t kLdsBytes = kTileBytes > kSumBytes ? (kTileBytes > kMeetBytes ? kTileBytes : kMeetBytes)
                                                             : (kSumBytes > kMeetBytes ? kSumBytes : kMeetBytes);
};

// The weights in the order in which the product takes them: tile of 16 output channels, step of 32 along K, lane, 8 values.  One
// wave a fragment.  A fragment's 16 rows lie far apart in the weights and neighbouring lanes hold different rows, so
// every lane's 16 bytes are an access of their own -- four times the time of a contiguous kilobyte, which each of hundreds of
// workgroups would pay (384 -> 768 channels, 256 images of 14 x 14: 156 us against 107 with this pass, or 80 with twice the waves that it makes worth while).
__global__ void __launch_bounds__(256) patch_weights_kernel(PatchArgs a, int K) {
  const int lane = threadIdx.x & 63, frag = blockIdx.x * 4 + (threadIdx.x >> 6), steps = K / 32;
  if (frag >= a.cout / 16 * steps) return;
  const int tile = frag / steps, step = frag - tile * steps;
  const bf16_t* src = a.w + static_cast<size_t>(16 * tile + (lane & 15)) * K + step * 32 + 8 * (lane >> 4);
  *reinterpret_cast<uint4*>(a.frags + static_cast<size_t>(frag) * 512 + 8 * lane) = *reinterpret_cast<const uint4*>(src);
}

template <typename S>
__global__ void __launch_bounds__(S::kThreads) norm_patch_kernel(PatchArgs a) {
  constexpr int C = S::C, MT = S::MT, MP = S::MP, PARTS = S::PARTS, PAIRS = S::PAIRS, NTW = S::NTW, D = S::kAhead;
  WT_SHARED_FLOATS(lds);
  bf16_t* tile = reinterpret_cast<bf16_t*>(lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int first = xcd_contiguous(blockIdx.x, gridDim.x) * MP;      // (neighbours share cache lines of the input)
  const int hwo = a.HO * a.WO;

  // ---- the patches, normalised, into LDS
  {
    const int px = tid % MP, part = tid / MP;
    const int p = min(first + px, a.pixels - 1);      // (past the end: the last pixel again, not stored)
    const int b = p / hwo, r = p - b * hwo, oy = r / a.WO, ox = r - oy * a.WO;
    const int plane = a.H * a.W;
    const bf16_t* src = a.x + static_cast<size_t>(b) * C * plane + 2 * oy * a.W + 2 * ox;
    uint32_t v[PAIRS][4];                             // channel c: rows 0 and 1 of the patch, then channel c + 1
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const bf16_t* at = src + static_cast<size_t>(2 * (part + i * PARTS)) * plane;
      v[i][0] = *reinterpret_cast<const uint32_t*>(at);
      v[i][1] = *reinterpret_cast<const uint32_t*>(at + a.W);
      v[i][2] = *reinterpret_cast<const uint32_t*>(at + plane);
      v[i][3] = *reinterpret_cast<const uint32_t*>(at + plane + a.W);
    }
    float4* sums = reinterpret_cast<float4*>(lds);    // [pass][part][pixel]: the four input pixels
    auto meet = [&](int pass, const float (&s)[4], float (&total)[4]) {
      sums[(pass * PARTS + part) * MP + px] = float4{s[0], s[1], s[2], s[3]};
      __syncthreads();
      total[0] = total[1] = total[2] = total[3] = 0.f;
#pragma unroll
      for (int j = 0; j < PARTS; ++j) {
        const float4 t = sums[(pass * PARTS + j) * MP + px];
        total[0] += t.x; total[1] += t.y; total[2] += t.z; total[3] += t.w;
      }
    };
    float s[4] = {0.f, 0.f, 0.f, 0.f}, mean[4], rstd[4];
#pragma unroll
    for (int i = 0; i < PAIRS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float lo, hi;
        unpack2<bf16_t>(v[i][j], lo, hi);
        s[2 * (j & 1)] += lo;
        s[2 * (j & 1) + 1] += hi;
      }
    meet(0, s, mean);
#pragma unroll
    for (int j = 0; j < 4; ++j) { mean[j] *= 1.f / C; s[j] = 0.f; }
#pragma unroll
    for (int i = 0; i < PAIRS; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 2 * (j & 1);
        float lo, hi;
        unpack2<bf16_t>(v[i][j], lo, hi);
        s[k] = fmaf(lo - mean[k], lo - mean[k], s[k]);
        s[k + 1] = fmaf(hi - mean[k + 1], hi - mean[k + 1], s[k + 1]);
      }
    meet(1, s, rstd);
#pragma unroll
    for (int j = 0; j < 4; ++j) rstd[j] = rsqrtf(rstd[j] * (1.f / C) + a.eps);
    __syncthreads();                                  // the sums have been read: their place takes the tile
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int c = 2 * (part + i * PARTS);
      float w[2], bb[2];
      unpack2<bf16_t>(*reinterpret_cast<const uint32_t*>(a.norm_w + c), w[0], w[1]);
      unpack2<bf16_t>(*reinterpret_cast<const uint32_t*>(a.norm_b + c), bb[0], bb[1]);
      uint32_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = 2 * (j & 1);
        float lo, hi;
        unpack2<bf16_t>(v[i][j], lo, hi);
        o[j] = pack_bf16x2(fmaf((lo - mean[k]) * rstd[k], w[j >> 1], bb[j >> 1]),
                           fmaf((hi - mean[k + 1]) * rstd[k + 1], w[j >> 1], bb[j >> 1]));
      }
      *reinterpret_cast<uint4*>(tile + px * S::kPitch + 4 * c) = uint4{o[0], o[1], o[2], o[3]};
    }
  }

  // ---- the product
  const int ng = wave % S::NG, kg = wave / S::NG;
  const int co0 = blockIdx.y * S::COUT + ng * NTW * 16;
  // (fragments in their own order when they have been laid out, rows of the weights otherwise)
  const bf16_t* wsrc = S::kLaidOut ? a.frags + (static_cast<size_t>(co0 / 16) * (S::K / 32) + kg * S::kSteps) * 512 + 8 * lane
                                   : a.w + static_cast<size_t>(co0 + n) * S::K + kg * S::kSteps * 32 + 8 * q;
  constexpr int kStep = S::kLaidOut ? 512 : 32, kTile = 16 * S::K;
  uint4 wf[D][NTW];                                   // fragments in flight
  auto fetch = [&](int step, int at) {
#pragma unroll
    for (int t = 0; t < NTW; ++t) wf[at][t] = *reinterpret_cast<const uint4*>(wsrc + t * kTile + step * kStep);
  };
#pragma unroll
  for (int d = 0; d < D; ++d) fetch(d, d);
  __syncthreads();
  mat_acc acc[MT][NTW];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NTW; ++t) acc[m][t] = mat_acc{0.f, 0.f, 0.f, 0.f};
  const bf16_t* asrc = tile + n * S::kPitch + kg * S::kSteps * 32 + 8 * q;
  for (int s0 = 0; s0 < S::kSteps; s0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      mat_frag af[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        af[m] = frag_of(*reinterpret_cast<const uint4*>(asrc + 16 * m * S::kPitch + (s0 + d) * 32));
#pragma unroll
      for (int t = 0; t < NTW; ++t)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          acc[m][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[m], frag_of(wf[d][t]), acc[m][t], 0, 0, 0);
      if (s0 + D < S::kSteps) fetch(s0 + D + d, d);
    }
  }
  if constexpr (S::KG > 1) {
    // the sums over the parts of K, added in order by the waves of the first part
    __syncthreads();
    mat_acc* meet = reinterpret_cast<mat_acc*>(lds);
    auto slot = [&](int g, int m, int t) { return (((g * S::NG + ng) * NTW + t) * MT + m) * 64 + lane; };
    if (kg > 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NTW; ++t) meet[slot(kg, m, t)] = acc[m][t];
    }
    __syncthreads();
    if (kg > 0) return;
#pragma unroll
    for (int g = 1; g < S::KG; ++g)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int t = 0; t < NTW; ++t) {
          mat_acc o = meet[slot(g, m, t)];
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[m][t][r] += o[r];
        }
  }

  // ---- lane (n, q) holds pixels 16 m + 4 q + 0..3 of channel 16 t + n
  float bias[NTW];
#pragma unroll
  for (int t = 0; t < NTW; ++t) bias[t] = bf16_to_f32(a.bias[co0 + 16 * t + n]);
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int p0 = first + 16 * m + 4 * q;
    if (a.vec) {
      if (p0 < a.pixels) {
        const int b = p0 / hwo;
        bf16_t* dst = a.out + (static_cast<size_t>(b) * a.cout + co0 + n) * hwo + (p0 - b * hwo);
#pragma unroll
        for (int t = 0; t < NTW; ++t)
          *reinterpret_cast<uint2*>(dst + static_cast<size_t>(16 * t) * hwo) =
              uint2{pack_bf16x2(acc[m][t][0] + bias[t], acc[m][t][1] + bias[t]),
                    pack_bf16x2(acc[m][t][2] + bias[t], acc[m][t][3] + bias[t])};
      }
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (p0 + r < a.pixels) {
          const int b = (p0 + r) / hwo;
          bf16_t* dst = a.out + (static_cast<size_t>(b) * a.cout + co0 + n) * hwo + (p0 + r - b * hwo);
#pragma unroll
          for (int t = 0; t < NTW; ++t) dst[static_cast<size_t>(16 * t) * hwo] = f32_to_bf16(acc[m][t][r] + bias[t]);
        }
    }
  }
}

// ---- stem -----------------------------------------------------------------------------------------------------------
// A wave takes 16 T consecutive output pixels at a time (in rows of a multiple of four) and all NT * 16 output channels: the
// weights stay in its registers as the A operand, the patches are the B operand and come straight from memory -- a lane's
// eight values of K are two rows of a patch.  Pixel T n + t is column n of product tile t, so that a lane ends up with
// T neighbouring pixels of its channels (T = 4: 16 lanes write a whole cache line); the channels of a pixel are in four
// lanes.  (Up to four input channels, K <= 64; what is missing of K is zero on both sides.)
template <int NT_, int T_>
struct StemShape {
  static constexpr int NT = NT_, T = T_, C = 16 * NT, kWaves = 4, PX = 16 * T;
  static_assert(T == 2 || T == 4, "");
};

template <typename S>
__global__ void __launch_bounds__(64 * S::kWaves, 2) patch_norm_kernel(PatchArgs a) {
  constexpr int NT = S::NT, T = S::T, C = S::C;
  __shared__ float par[3][C];                         // bias, norm weight, norm bias
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4, lane4 = lane << 2;
  for (int i = tid; i < C; i += 64 * S::kWaves) {
    par[0][i] = bf16_to_f32(a.bias[i]);
    par[1][i] = bf16_to_f32(a.norm_w[i]);
    par[2][i] = bf16_to_f32(a.norm_b[i]);
  }
  const int K = a.cin * 16;
  uint4 wf[NT][2];
#pragma unroll
  for (int j = 0; j < NT; ++j)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int k = 32 * s + 8 * q;
      wf[j][s] = k < K ? *reinterpret_cast<const uint4*>(a.w + (16 * j + n) * K + k) : uint4{0u, 0u, 0u, 0u};
    }
  __syncthreads();

  const int hwo = a.HO * a.WO, plane = a.H * a.W;
  const int groups = (a.pixels + S::PX - 1) / S::PX, step = gridDim.x * S::kWaves;
  // this lane's part of the patches of a group: pixels T n + t, input channel 2 s + q / 2, rows 2 (q % 2) and the next
  uint4 xf[2][T];
  auto fetch = [&](int g) {
    const int p = min(g * S::PX + T * n, a.pixels - T);      // (past the end: the last pixels again, not stored)
    const int b = p / hwo, r = p - b * hwo, oy = r / a.WO, ox = r - oy * a.WO;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const int c = 2 * s + (q >> 1);
      const bf16_t* src = a.x + (static_cast<size_t>(b) * a.cin + c) * plane + (4 * oy + 2 * (q & 1)) * a.W + 4 * ox;
#pragma unroll
      for (int h = 0; h < T / 2; ++h) {      // two pixels
        uint4 top = {0u, 0u, 0u, 0u}, low = {0u, 0u, 0u, 0u};
        if (c < a.cin) {
          top = *reinterpret_cast<const uint4*>(src + 8 * h);
          low = *reinterpret_cast<const uint4*>(src + a.W + 8 * h);
        }
        xf[s][2 * h] = uint4{top.x, top.y, low.x, low.y};
        xf[s][2 * h + 1] = uint4{top.z, top.w, low.z, low.w};
      }
    }
  };
  int g = xcd_contiguous(blockIdx.x, gridDim.x) * S::kWaves + wave;
  if (g < groups) fetch(g);
  for (; g < groups; g += step) {
    mat_acc acc[T][NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const mat_acc bias = *reinterpret_cast<const mat_acc*>(&par[0][16 * j + 4 * q]);
#pragma unroll
      for (int t = 0; t < T; ++t) acc[t][j] = bias;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int t = 0; t < T; ++t)
          acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(frag_of(wf[j][s]), frag_of(xf[s][t]), acc[t][j], 0, 0, 0);
    if (g + step < groups) fetch(g + step);
    float mean[T], rstd[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j) sum += (acc[t][j][0] + acc[t][j][1]) + (acc[t][j][2] + acc[t][j][3]);
      sum += wave_xor(sum, lane4, 16);
      sum += wave_xor(sum, lane4, 32);
      mean[t] = sum * (1.f / C);
      float sq = 0.f;
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) sq = fmaf(acc[t][j][r] - mean[t], acc[t][j][r] - mean[t], sq);
      sq += wave_xor(sq, lane4, 16);
      sq += wave_xor(sq, lane4, 32);
      rstd[t] = rsqrtf(sq * (1.f / C) + a.eps);
    }
    const int p = g * S::PX + T * n;
    if (p < a.pixels) {
      const int b = p / hwo;
      bf16_t* dst = a.out + (static_cast<size_t>(b) * C + 4 * q) * hwo + (p - b * hwo);
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        mat_acc w = *reinterpret_cast<const mat_acc*>(&par[1][16 * j + 4 * q]);
        mat_acc bb = *reinterpret_cast<const mat_acc*>(&par[2][16 * j + 4 * q]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float y[T];
#pragma unroll
          for (int t = 0; t < T; ++t) y[t] = fmaf((acc[t][j][r] - mean[t]) * rstd[t], w[r], bb[r]);
          bf16_t* at = dst + static_cast<size_t>(16 * j + r) * hwo;
          if constexpr (T == 4) *reinterpret_cast<uint2*>(at) = uint2{pack_bf16x2(y[0], y[1]), pack_bf16x2(y[T - 2], y[T - 1])};
          else *reinterpret_cast<uint32_t*>(at) = pack_bf16x2(y[0], y[1]);
        }
      }
    }
  }
}

}  // namespace wt
