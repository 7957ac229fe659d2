// The matrix products of a WTConvNeXt block's MLP in training, in bfloat16 with float sums, and what stands between them:
//
//   forward    h = x W1^T + b1, a = gelu(h);   y = a W2^T + b2
//   backward   dh = (dy W2) * gelu'(h);        dx = dh W1
//              dW2 = dy^T a, db2 = sum dy;     dW1 = dh^T x, db1 = sum dh
//
// (wtconvnext/wtconvnext.py:125-136 of the reference; x, y (pixels, C), h, a (pixels, hidden), W1 (hidden, C), W2 (C, hidden)).
#pragma once

#include "gelu.h"
#include "matrix.h"

namespace wt {

// ---- products along the channels: out[p][n] = sum_k pix[p][k] w[n][k], both operands contiguous along k ----------------
enum ProductEnd { kEndPlain, kEndBias, kEndGelu, kEndDerivative };

struct ProductArgs {
  const bf16_t *pix, *w;      // (M, K), (N, K)
  const bf16_t* bias;         // (N): kEndBias, kEndGelu
  bf16_t* out;                // (M, N)
  bf16_t* pre;                // (M, N): h, written by kEndGelu (unless nullptr), read by kEndDerivative
  int M, N, K;
};

// A workgroup of WM x WN waves computes BM pixels x BN outputs; BK of k at a time come straight from memory into one of
// STAGES places of LDS.
template <int BM_, int BN_, int WM_, int WN_, int BK_, int STAGES_>
struct ProductShape {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, BK = BK_, STAGES = STAGES_, kThreads = 64 * WM * WN;
  static constexpr int TM = BM / WM / 16, TN = BN / WN / 16;      // tiles of a wave
  static constexpr int G = BK / 8;                                // 16-byte granules of a row
  static constexpr int kPixBytes = BM * BK * 2, kStageBytes = (BM + BN) * BK * 2;
  static constexpr int kPixLoads = BM * G / kThreads, kLoads = (BM + BN) * G / kThreads;
  static constexpr size_t kLdsBytes = static_cast<size_t>(STAGES) * kStageBytes;
  static_assert(BM * G % kThreads == 0 && BN * G % kThreads == 0 && TN % 2 == 0 && (BK == 32 || BK == 64), "whole loads, pairs of tiles");
  static constexpr int of4(int k) { return ((k << 1) & 3) ^ ((k >> 1) * 3); }      // 0, 2, 3, 1
  // Where granule g of row r sits within its row, so that the 16 lanes that the LDS serves at a time find different banks:
  // 16 consecutive rows (pixels), rows 8a + b (+4), a, b = 0..3 (weights).
  static __device__ __forceinline__ int swz_pix(int r, int g) { return G == 8 ? g ^ ((r >> 1) & 7) : g ^ of4((r >> 2) & 3); }
  static __device__ __forceinline__ int swz_w(int r, int g) {
    return G == 8 ? g ^ (((r >> 1) & 1) | ((r >> 2) & 6)) : g ^ of4((r >> 3) & 3);
  }
};

template <typename S, int END>
__global__ void __launch_bounds__(S::kThreads, 2) product_kernel(ProductArgs a) {
  constexpr int TM = S::TM, TN = S::TN, G = S::G, BK = S::BK;
  WT_SHARED_FLOATS(product_lds);
  unsigned char* lds = reinterpret_cast<unsigned char*>(product_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4, wm = wave / S::WN, wn = wave % S::WN;
  const int ntn = a.N / S::BN, at = xcd_contiguous(blockIdx.x, gridDim.x);      // (an XCD's workgroups share pixels)
  const int m0 = at / ntn * S::BM, n0 = (at - at / ntn * ntn) * S::BN;

  // this thread's granules of a stage, as byte offsets from the tile's first one (past the last pixel: the last again)
  uint32_t src[S::kLoads];
#pragma unroll
  for (int i = 0; i < S::kLoads; ++i) {
    const int p = (i < S::kPixLoads ? i : i - S::kPixLoads) * S::kThreads + tid, r = p / G;
    src[i] = i < S::kPixLoads ? static_cast<uint32_t>(min(r, a.M - 1 - m0) * a.K + 8 * S::swz_pix(r, p % G)) * 2
                              : static_cast<uint32_t>(r * a.K + 8 * S::swz_w(r, p % G)) * 2;
  }
  const bf16_t* pix0 = a.pix + static_cast<size_t>(m0) * a.K;
  const bf16_t* w0 = a.w + static_cast<size_t>(n0) * a.K;
  const lds_addr lds0 = WT_LDS_ADDR(lds);
  auto load_stage = [&](int s, int place) {
    const lds_addr dst = WT_UNIFORM(lds0 + place * S::kStageBytes + wave * 1024);
#pragma unroll
    for (int i = 0; i < S::kLoads; ++i)
      granules_to_lds(i < S::kPixLoads ? pix0 + s * BK : w0 + s * BK, src[i], dst + i * (S::kThreads * 16));
  };

  mat_acc acc[TN][TM];
#pragma unroll
  for (int t = 0; t < TN; ++t)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[t][m] = mat_acc{0.f, 0.f, 0.f, 0.f};
  // The rows of a pair of weight tiles are dealt so that lane (n, q) ends up with outputs 8q..8q+7 of 32, from both tiles.
  const int row_pix = wm * (TM * 16) + n, row_w = wn * (TN * 16) + 8 * (n >> 2) + (n & 3);
  const int steps = a.K / BK;
#pragma unroll
  for (int s = 0; s < S::STAGES - 1; ++s)
    if (s < steps) load_stage(s, s);
  arrive_and_wait<0>();
  int place = 0, fill = S::STAGES - 1;
  for (int s = 0; s < steps; ++s) {
    const bool more = s + S::STAGES - 1 < steps;
    if (more) load_stage(s + S::STAGES - 1, fill);
    const unsigned char *pix = lds + place * S::kStageBytes, *w = pix + S::kPixBytes;
#pragma unroll
    for (int k = 0; k < BK / 32; ++k) {
      mat_frag pf[TM], wf[TN];
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        const int r = row_pix + 16 * m;
        pf[m] = *reinterpret_cast<const mat_frag*>(pix + (r * G + S::swz_pix(r, 4 * k + q)) * 16);
      }
#pragma unroll
      for (int t = 0; t < TN; ++t) {
        const int r = row_w + 32 * (t / 2) + 4 * (t & 1);
        wf[t] = *reinterpret_cast<const mat_frag*>(w + (r * G + S::swz_w(r, 4 * k + q)) * 16);
      }
#pragma unroll
      for (int t = 0; t < TN; ++t)
#pragma unroll
        for (int m = 0; m < TM; ++m) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t], pf[m], acc[t][m], 0, 0, 0);
    }
    // behind this the next stage has arrived for everybody, and this one's place is no longer read
    if (more) arrive_and_wait<(S::STAGES - 2) * S::kLoads>();
    else arrive_and_wait<0>();
    place = place + 1 == S::STAGES ? 0 : place + 1;
    fill = fill + 1 == S::STAGES ? 0 : fill + 1;
  }

#pragma unroll
  for (int t = 0; t < TN; t += 2) {
    const int col = n0 + wn * (TN * 16) + 16 * t + 8 * q;
    float bias[8];
    if constexpr (END == kEndBias || END == kEndGelu) {
      const uint4 b = *reinterpret_cast<const uint4*>(a.bias + col);
      unpack2<bf16_t>(b.x, bias[0], bias[1]);
      unpack2<bf16_t>(b.y, bias[2], bias[3]);
      unpack2<bf16_t>(b.z, bias[4], bias[5]);
      unpack2<bf16_t>(b.w, bias[6], bias[7]);
    }
#pragma unroll
    for (int m = 0; m < TM; ++m) {
      const int p = m0 + row_pix + 16 * m;
      if (p >= a.M) continue;
      const size_t to = static_cast<size_t>(p) * a.N + col;
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        v[i] = acc[t + (i >> 2)][m][i & 3];
        if constexpr (END == kEndBias || END == kEndGelu) v[i] += bias[i];
      }
      if constexpr (END == kEndGelu) {
        // (GELU of the stored value: the one that the backward pass sees)
        uint32_t h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          h[i] = pack_bf16x2(v[2 * i], v[2 * i + 1]);
          unpack2<bf16_t>(h[i], v[2 * i], v[2 * i + 1]);
          v[2 * i] = gelu_train(v[2 * i]);
          v[2 * i + 1] = gelu_train(v[2 * i + 1]);
        }
        if (a.pre != nullptr) *reinterpret_cast<uint4*>(a.pre + to) = uint4{h[0], h[1], h[2], h[3]};
      }
      if constexpr (END == kEndDerivative) {
        const uint4 h4 = *reinterpret_cast<const uint4*>(a.pre + to);
        const uint32_t h[4] = {h4.x, h4.y, h4.z, h4.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float lo, hi;
          unpack2<bf16_t>(h[i], lo, hi);
          v[2 * i] *= gelu_derivative(lo);
          v[2 * i + 1] *= gelu_derivative(hi);
        }
      }
      *reinterpret_cast<uint4*>(a.out + to) = uint4{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]),
                                                    pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])};
    }
  }
}

// (rows, cols) -> (cols, rows) of both weight matrices, which the backward products take along their other extent: W1
// (hidden, C) in blockIdx.z 0, W2 (C, hidden) in 1.  A workgroup moves 64 x 64 values.
struct TransposeArgs {
  const bf16_t* src[2];
  bf16_t* dst[2];
  int rows[2], cols[2];      // multiples of 32
};
__global__ void __launch_bounds__(256) transpose_weights_kernel(TransposeArgs a) {
  __shared__ bf16_t tile[64][66];
  const int z = blockIdx.z, rows = a.rows[z], cols = a.cols[z];
  const int tiles = (cols + 63) / 64, r0 = blockIdx.x / tiles * 64, c0 = (blockIdx.x % tiles) * 64;
  const int x = threadIdx.x & 31, y = threadIdx.x >> 5;      // two columns, one of eight rows
  for (int r = y; r < 64; r += 8)
    if (r0 + r < rows && c0 + 2 * x < cols) {
      const uint32_t v = *reinterpret_cast<const uint32_t*>(a.src[z] + static_cast<size_t>(r0 + r) * cols + c0 + 2 * x);
      tile[r][2 * x] = static_cast<bf16_t>(v);
      tile[r][2 * x + 1] = static_cast<bf16_t>(v >> 16);
    }
  __syncthreads();
  for (int c = y; c < 64; c += 8)
    if (c0 + c < cols && r0 + 2 * x < rows)
      *reinterpret_cast<uint32_t*>(a.dst[z] + static_cast<size_t>(c0 + c) * rows + r0 + 2 * x) =
          tile[2 * x][c] | (static_cast<uint32_t>(tile[2 * x + 1][c]) << 16);
}

// ---- products along the pixels: the weight gradients ---------------------------------------------------------------
// Both are sums over the pixels of an outer product of hidden and channel values: job 0 takes (a, dy) and gives dW2 and
// db2 = sum dy, job 1 (dh, x), dW1 and db1 = sum dh.  A workgroup sums BH hidden x BC channel values over a share of the
// pixels; the shares (enough to fill the chip) meet in wgrad_sum_kernel, in order.
//
// The operands lie along the pixels' rows, the matrix instructions take eight pixels of one column a lane: the tiles come
// into LDS as they lie and are read transposed (column_of_4).
struct WeightGradArgs {
  const bf16_t *hid[2], *chan[2];      // (M, hidden), (M, C) of each job
  float* partial;                      // [share][job][tile][fragment][lane] of four floats
  float* bias_partial;                 // [share][C + hidden]: db2, then db1
  bf16_t *dw[2], *db[2];               // dW2 (C, hidden), dW1 (hidden, C); db2, db1 (nullptr: not wanted)
  int M, hidden, C;
  int shares, stages;                  // shares of the pixels, of `stages` stages each
  int jobs, first_job;                 // 2, or 1 and which
};

template <int BH_, int BC_, int BK_, int STAGES_>
struct WeightGradShape {
  static constexpr int BH = BH_, BC = BC_, BK = BK_, STAGES = STAGES_;
  static constexpr int TH = BH / 32, TC = BC / 32;      // tiles of a wave, 2 x 2 waves
  static constexpr int GH = BH / 8, GC = BC / 8;        // granules of a row
  static constexpr int kHidBytes = BH * BK * 2, kStageBytes = (BH + BC) * BK * 2;
  static constexpr int kHidLoads = BK * GH / 256, kLoads = BK * (GH + GC) / 256;
  static constexpr size_t kLdsBytes = static_cast<size_t>(STAGES) * kStageBytes;
  static constexpr int kTileFloats = BH * BC;
  static_assert(BK * GH % 256 == 0 && BK * GC % 256 == 0 && BK % 32 == 0, "whole loads");
  // Where granule g of row r sits within a row of `granules`.  A fragment read takes two neighbouring granules of each of
  // the rows 8q + 0..3: those of two q at a time are put on different banks.
  static __device__ __forceinline__ int swz(int r, int g, int granules) {
    const int v = (r & 3) + ((r >> 3) & 1) * 4;
    return granules % 16 == 0 ? g ^ (2 * v) : granules % 8 == 0 ? g ^ (2 * (v >> 1)) : g ^ (2 * (v >> 2));
  }
};

template <typename S>
__global__ void __launch_bounds__(256, 2) weight_grad_kernel(WeightGradArgs a) {
  constexpr int TH = S::TH, TC = S::TC;
  WT_SHARED_FLOATS(wgrad_lds);
  unsigned char* lds = reinterpret_cast<unsigned char*>(wgrad_lds);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4, wh = wave >> 1, wc = wave & 1;
  const int tiles_h = a.hidden / S::BH, tiles_c = a.C / S::BC, tiles = tiles_h * tiles_c;
  // (the workgroups of an XCD share pixels: tile fastest)
  const int at = xcd_contiguous(blockIdx.x, gridDim.x), share = at / (tiles * a.jobs), rest = at - share * (tiles * a.jobs);
  const int job = a.first_job + rest / tiles, tile = rest % tiles, th = tile / tiles_c, tc = tile - th * tiles_c;
  const int first = share * a.stages * S::BK, left = a.M - first;      // pixels from here to the end
  const int steps = min(a.stages, (left + S::BK - 1) / S::BK);

  uint32_t src[S::kLoads];
#pragma unroll
  for (int i = 0; i < S::kLoads; ++i) {
    const bool hid = i < S::kHidLoads;
    const int g = hid ? S::GH : S::GC, p = (hid ? i : i - S::kHidLoads) * 256 + tid, r = p / g;
    src[i] = static_cast<uint32_t>(r * (hid ? a.hidden : a.C) + 8 * S::swz(r, p % g, g)) * 2;
  }
  const bf16_t* hid0 = (job ? a.hid[1] : a.hid[0]) + static_cast<size_t>(first) * a.hidden + th * S::BH;
  const bf16_t* chan0 = (job ? a.chan[1] : a.chan[0]) + static_cast<size_t>(first) * a.C + tc * S::BC;
  const lds_addr lds0 = WT_LDS_ADDR(lds);
  auto load_stage = [&](int s, int place) {
    const lds_addr dst = WT_UNIFORM(lds0 + place * S::kStageBytes + wave * 1024);
    const bf16_t *hid = hid0 + static_cast<size_t>(s) * S::BK * a.hidden, *chan = chan0 + static_cast<size_t>(s) * S::BK * a.C;
    const int rows = left - s * S::BK;
    if (rows >= S::BK) {
#pragma unroll
      for (int i = 0; i < S::kLoads; ++i) granules_to_lds(i < S::kHidLoads ? hid : chan, src[i], dst + i * 4096);
    } else {
      // rows past the last pixel: any pixel's, cleared below
#pragma unroll
      for (int i = 0; i < S::kLoads; ++i) {
        const bool h = i < S::kHidLoads;
        const int g = h ? S::GH : S::GC, p = (h ? i : i - S::kHidLoads) * 256 + tid, r = p / g;
        granules_to_lds(h ? hid : chan, r < rows ? src[i] : src[i] - static_cast<uint32_t>(r * (h ? a.hidden : a.C)) * 2, dst + i * 4096);
      }
    }
  };

  mat_acc acc[TC][TH], sums[TH > TC ? TH : TC];
#pragma unroll
  for (int c = 0; c < TC; ++c)
#pragma unroll
    for (int h = 0; h < TH; ++h) acc[c][h] = mat_acc{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < (TH > TC ? TH : TC); ++i) sums[i] = mat_acc{0.f, 0.f, 0.f, 0.f};
  // the bias gradients are products with ones, in the workgroups and waves that come first in the other extent
  const bool sum_c = job == 0 && th == 0 && wh == 0, sum_h = job == 1 && tc == 0 && wc == 0;
  const mat_frag ones = frag_of(uint4{0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u});

#pragma unroll
  for (int s = 0; s < S::STAGES - 1; ++s)
    if (s < steps) load_stage(s, s);
  arrive_and_wait<0>();
  int place = 0, fill = S::STAGES - 1;
  for (int s = 0; s < steps; ++s) {
    const bool more = s + S::STAGES - 1 < steps;
    if (more) load_stage(s + S::STAGES - 1, fill);
    unsigned char *hid = lds + place * S::kStageBytes, *chan = hid + S::kHidBytes;
    if (const int rows = left - s * S::BK; rows < S::BK) {
      for (int i = tid; i < (S::BK - rows) * (S::GH + S::GC); i += 256) {
        const int r = rows + i / (S::GH + S::GC), g = i % (S::GH + S::GC);
        *reinterpret_cast<uint4*>(g < S::GH ? hid + (r * S::GH + g) * 16 : chan + (r * S::GC + g - S::GH) * 16) = uint4{0u, 0u, 0u, 0u};
      }
      __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < S::BK / 32; ++k) {
      // lane (n, q): pixels 8q..8q+7 of column n of each tile
      auto fetch = [&](const unsigned char* tile_at, int granules, int col) {
        uint2 half[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const int r = 32 * k + 8 * q + 4 * e + (n >> 2), c = col + 4 * (n & 3);
          half[e] = column_of_4(reinterpret_cast<const bf16_t*>(tile_at + (r * granules + S::swz(r, c >> 3, granules)) * 16) + (c & 4));
        }
        return frag_of(uint4{half[0].x, half[0].y, half[1].x, half[1].y});
      };
      mat_frag hf[TH], cf[TC];
#pragma unroll
      for (int h = 0; h < TH; ++h) hf[h] = fetch(hid, S::GH, (wh * TH + h) * 16);
#pragma unroll
      for (int c = 0; c < TC; ++c) cf[c] = fetch(chan, S::GC, (wc * TC + c) * 16);
#pragma unroll
      for (int c = 0; c < TC; ++c)
#pragma unroll
        for (int h = 0; h < TH; ++h) acc[c][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hf[h], cf[c], acc[c][h], 0, 0, 0);
      if (sum_c) {
#pragma unroll
        for (int c = 0; c < TC; ++c) sums[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(cf[c], ones, sums[c], 0, 0, 0);
      }
      if (sum_h) {
#pragma unroll
        for (int h = 0; h < TH; ++h) sums[h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hf[h], ones, sums[h], 0, 0, 0);
      }
    }
    if (more) arrive_and_wait<(S::STAGES - 2) * S::kLoads>();
    else arrive_and_wait<0>();
    place = place + 1 == S::STAGES ? 0 : place + 1;
    fill = fill + 1 == S::STAGES ? 0 : fill + 1;
  }

  // lane (n, q) holds hidden units 4q..4q+3 of channel n of each fragment
  mat_acc* out = reinterpret_cast<mat_acc*>(a.partial) +
                 (static_cast<size_t>(share * a.jobs + job - a.first_job) * tiles + tile) * (S::kTileFloats / 4) + wave * (TC * TH * 64) + lane;
#pragma unroll
  for (int c = 0; c < TC; ++c)
#pragma unroll
    for (int h = 0; h < TH; ++h) out[(c * TH + h) * 64] = acc[c][h];
  // (the columns of a product with ones are all the same)
  if (n == 0) {
    float* b = a.bias_partial + static_cast<size_t>(share) * (a.C + a.hidden);
    if (sum_c) {
#pragma unroll
      for (int c = 0; c < TC; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) b[tc * S::BC + (wc * TC + c) * 16 + 4 * q + r] = sums[c][r];
    }
    if (sum_h) {
#pragma unroll
      for (int h = 0; h < TH; ++h)
#pragma unroll
        for (int r = 0; r < 4; ++r) b[a.C + th * S::BH + (wh * TH + h) * 16 + 4 * q + r] = sums[h][r];
    }
  }
}

// The shares' sums, added in order, rounded to bfloat16 once.  One thread per four values of a weight gradient (in the
// order of the records), then one per four of a bias gradient.
template <typename S>
__global__ void __launch_bounds__(256) wgrad_sum_kernel(WeightGradArgs a) {
  const int tiles_c = a.C / S::BC, tiles = a.hidden / S::BH * tiles_c;
  const int per_share = a.jobs * tiles * (S::kTileFloats / 4), i = blockIdx.x * 256 + threadIdx.x;
  if (i < per_share) {
    const float4* src = reinterpret_cast<const float4*>(a.partial) + i;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
    for (int s = 0; s < a.shares; ++s) {
      const float4 t = src[static_cast<size_t>(s) * per_share];
      v[0] += t.x; v[1] += t.y; v[2] += t.z; v[3] += t.w;
    }
    const int lane = i & 63, frag = i / 64 % (S::TC * S::TH), wave = i / (64 * S::TC * S::TH) % 4;
    const int t = i / (S::kTileFloats / 4), job = a.first_job + t / tiles, tile = t % tiles, th = tile / tiles_c, tc = tile % tiles_c;
    const int h = th * S::BH + ((wave >> 1) * S::TH + frag % S::TH) * 16 + 4 * (lane >> 4);
    const int c = tc * S::BC + ((wave & 1) * S::TC + frag / S::TH) * 16 + (lane & 15);
    if (job == 0) {
      *reinterpret_cast<uint2*>(a.dw[0] + static_cast<size_t>(c) * a.hidden + h) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r) a.dw[1][static_cast<size_t>(h + r) * a.C + c] = f32_to_bf16(v[r]);
    }
    return;
  }
  const int b = (i - per_share) * 4;      // of C + hidden
  if (b >= a.C + a.hidden) return;
  const int job = b < a.C ? 0 : 1;
  bf16_t* dst = a.db[job];
  if (dst == nullptr || job < a.first_job || job >= a.first_job + a.jobs) return;
  float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 8
  for (int s = 0; s < a.shares; ++s) {
    const float4 t = *reinterpret_cast<const float4*>(a.bias_partial + static_cast<size_t>(s) * (a.C + a.hidden) + b);
    v[0] += t.x; v[1] += t.y; v[2] += t.z; v[3] += t.w;
  }
  *reinterpret_cast<uint2*>(dst + b - (job ? a.C : 0)) = uint2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
}

}  // namespace wt
