// WTConv2d kernels for planes whose pyramid does not fit the 160 KB of LDS of a compute unit (e.g. 128x128 and larger).
//
// The layer is recursive.  With X_1 the LL band of x and everything else as in kernels2d.h (reference
// wtconv/wtconv2d.py:38-87, wtconv/util/wavelet.py:62-75),
//   layer_L(x) = base (*) x + iHaar(layer_{L-1}(X_1), w_1[LH] (*) LH_1, w_1[HL] (*) HL_1, w_1[HH] (*) HH_1)
// where layer_{L-1} has w_1[LL] for its base conv and the levels 2..L for its levels.  So a large plane is taken one
// level at a time until what is left fits LDS, and the plane-resident kernels do the rest on planes of a quarter, a
// sixteenth, ... of the pixels:
//   stream_ll_kernel       X_1 of x, a quarter of the pixels, fp32
//   (the sub-layer, by the same rule: plane-resident or another step)
//   stream_final_kernel    tiles: detail bands of level 1 from the pixels in LDS, their convs, the sub-layer's result,
//                          inverse Haar, base conv
// Parameter gradients follow the same recursion: stream_corr_kernel sums the base conv's and the detail bands' filters
// from the pixels of x and grad_out, and the sub-layer's filters are its parameter gradients on X_1 and G_1.
// Nothing of a level but its LL band goes through memory.
//
// Measured, us a training step (forward): [8,96,160,160] fp32 523 -> 380 (167 -> 118) against one launch per level and
// pass with every band in memory; [8,64,141,155] fp16, K = 7 1018 -> 556 (350 -> 156); [4,64,199,230] fp32, five levels
// 443 -> 325 (138 -> 109).
//
// Rows start at any element's address and may have any length (16-byte accesses need no more than that).
#pragma once

#include "common.h"
#include "kernels2d.h"

namespace wt {

constexpr int kStreamPad = 4;       // column halo of the LDS tiles in coefficients (>= K/2, keeps rows 16-byte aligned)
constexpr int kStreamThreads = 256;

// Four elements, or the `n` < 4 that exist, to any element address.
template <typename T>
__device__ __forceinline__ void store4_any(T* __restrict__ p, int n, const float (&v)[4]) {
  if (n >= 4) {
    if constexpr (sizeof(T) == 4)
      store_u4<4>(p, uint4{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])});
    else
      store_u2<2>(p, uint2{pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])});
  } else {
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (e < n) p[e] = from_f32<T>(v[e]);
  }
}

// `n` = pixels of the row from p on that exist, the rest reads as zero.
template <typename T>
__device__ __forceinline__ void load8_row(const T* __restrict__ p, int n, float (&v)[8]) {
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = 0.f;
  if (n >= 8) {
    float a[4], b[4];
    load4_any<T>(p, a);
    load4_any<T>(p + 4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) { v[e] = a[e]; v[4 + e] = b[e]; }
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (e < n) v[e] = to_f32<T>(p[e]);
  }
}

__device__ __forceinline__ void store4_row(float* __restrict__ p, int n, const float (&v)[4]) {
  if (n >= 4) {
    uint4 q;
    q.x = __float_as_uint(v[0]); q.y = __float_as_uint(v[1]); q.z = __float_as_uint(v[2]); q.w = __float_as_uint(v[3]);
    store_u4<4>(p, q);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (e < n) p[e] = v[e];
  }
}

// The LL band of planes: src (planes, hs, ws) -> dst (planes, hd, wd), fp32.  Reading one past an odd extent gives the
// zero padding the reference applies (wtconv2d.py:49-51).  Four coefficients a thread.
// grid = (ceil(hd * ceil(wd / 4) / 256), planes <= 65535), block = 256.
template <typename T>
__global__ void stream_ll_kernel(const T* __restrict__ src, int hs, int ws, float* __restrict__ dst, int hd, int wd,
                                 int nplanes) {
  const int wq = (wd + 3) >> 2;
  const int item = blockIdx.x * kStreamThreads + threadIdx.x;
  if (item >= hd * wq) return;
  const int i = item / wq, j = 4 * (item - i * wq);
  const size_t ssz = static_cast<size_t>(hs) * ws, dsz = static_cast<size_t>(hd) * wd;
  for (int plane = blockIdx.y; plane < nplanes; plane += gridDim.y) {
    const T* s = src + plane * ssz + static_cast<size_t>(2 * i) * ws + 2 * j;
    float a[8], b[8], o[4];
    load8_row<T>(s, ws - 2 * j, a);
    load8_row<T>(s + ws, 2 * i + 1 < hs ? ws - 2 * j : 0, b);
#pragma unroll
    for (int t = 0; t < 4; ++t) o[t] = 0.5f * ((a[2 * t] + b[2 * t]) + (a[2 * t + 1] + b[2 * t + 1]));
    store4_row(dst + plane * dsz + static_cast<size_t>(i) * wd + j, wd - j, o);
  }
}

// Window of a plane -> LDS: dst[r * WD + c] = plane[gi0 + r][gj0 + c], zero outside the plane; gj0 a multiple of 4.
// Four elements at a time; the position of a thread's next piece advances without divisions.  All loads of a thread
// are issued before the first LDS write.
template <typename T, int ROWS, int WD>
__device__ __forceinline__ void stage_window(const T* __restrict__ src, int h, int w, int gi0, int gj0,
                                             float* __restrict__ dst, int tid) {
  constexpr int W4 = WD / 4;
  constexpr int N = ROWS * W4;
  constexpr int IT = (N + kStreamThreads - 1) / kStreamThreads;
  constexpr int DR = kStreamThreads / W4, DC = kStreamThreads % W4;
  static_assert(WD % 4 == 0, "whole vectors");
  float v[IT][4];
  {
    int row = tid / W4, col = tid - row * W4;
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int gi = gi0 + row, gj = gj0 + col * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[it][e] = 0.f;
      if (row < ROWS && gi >= 0 && gi < h && gj >= 0 && gj < w) {
        const T* q = src + (static_cast<size_t>(gi) * w + gj);
        if (gj + 4 <= w) {
          load4_any<T>(q, v[it]);
        } else {
#pragma unroll
          for (int e = 0; e < 3; ++e)
            if (gj + e < w) v[it][e] = to_f32<T>(q[e]);
        }
      }
      col += DC;
      row += DR;
      if (col >= W4) { col -= W4; ++row; }
    }
  }
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int p = it * kStreamThreads + tid;
    if (p < N) {
      float4 t4;
      t4.x = v[it][0]; t4.y = v[it][1]; t4.z = v[it][2]; t4.w = v[it][3];
      reinterpret_cast<float4*>(dst)[p] = t4;
    }
  }
}

// Twelve / sixteen floats of an LDS row from a 16-byte aligned address.
template <int N>
__device__ __forceinline__ void lds_read(const float* __restrict__ p, float (&v)[N]) {
#pragma unroll
  for (int q = 0; q < N / 4; ++q) {
    const float4 t4 = reinterpret_cast<const float4*>(p)[q];
    v[4 * q] = t4.x; v[4 * q + 1] = t4.y; v[4 * q + 2] = t4.z; v[4 * q + 3] = t4.w;
  }
}

// Tile shapes: TW x TH coefficients, four adjacent ones of a row a thread.  Tiles of 64 columns left a third of the
// threads of an 80-column level (160-pixel planes) without work; the launch takes the shape that covers the level with
// the fewest tiles.
template <int TW_, int TH_>
struct StreamShape {
  static constexpr int TW = TW_, TH = TH_;
  static_assert(TW / 4 * TH <= kStreamThreads, "one thread per four coefficients");
};

// Level-1 Haar bands S0..3 of a pixel tile in LDS: coefficient (rr, cc) of the AH x AWD tile comes from pixels
// (2rr .. 2rr+1, 2cc .. 2cc+1) of the 2AH x 2AWD pixel tile.  Pixels outside the plane were staged as zeros, which is
// both the zero padding of odd sizes and the zero halo of the sub-band convs (a coefficient outside the level has all
// four pixels outside the plane).
template <int AH, int AWD, int S0>
__device__ __forceinline__ void haar_tile(const float* __restrict__ Xt, float* __restrict__ At, int tid) {
  constexpr int XWD = 2 * AWD;
  constexpr int PAIRS = AWD / 2;             // two coefficients (four pixels of each row) per step
  for (int e = tid; e < AH * PAIRS; e += kStreamThreads) {
    const int rr = e / PAIRS, cp = e - rr * PAIRS;
    const float4 top = *reinterpret_cast<const float4*>(Xt + (2 * rr) * XWD + 4 * cp);
    const float4 bot = *reinterpret_cast<const float4*>(Xt + (2 * rr + 1) * XWD + 4 * cp);
    const float a[2] = {top.x, top.z}, b[2] = {top.y, top.w}, c[2] = {bot.x, bot.z}, d[2] = {bot.y, bot.w};
    float o[4][2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const float sac = a[t] + c[t], sbd = b[t] + d[t], dac = a[t] - c[t], dbd = b[t] - d[t];
      o[0][t] = 0.5f * (sac + sbd);
      o[1][t] = 0.5f * (dac + dbd);
      o[2][t] = 0.5f * (sac - sbd);
      o[3][t] = 0.5f * (dac - dbd);
    }
#pragma unroll
    for (int s = S0; s < 4; ++s) {
      float2 t2;
      t2.x = o[s][0]; t2.y = o[s][1];
      *reinterpret_cast<float2*>(At + ((s - S0) * AH + rr) * AWD + 2 * cp) = t2;
    }
  }
}

// ---- rows over the lanes of a wave ------------------------------------------------------------------------------------
// A lane owns four pixels of a row (two coefficients) and walks down the plane; what it needs of its neighbours' rows comes
// from their registers (wave_before, wave_behind), so there is no LDS, no barrier, and a wave only ever waits for its loads.
// A unit is a stretch of rows of one tile (a column of lanes) of a plane; a wave takes `per` units of one channel side by
// side.  Lanes whose pixels lie outside the plane hold zeros, which are the zero padding of the convolutions and of odd
// extents; where two units that end at the plane's edge meet, lanes between them hold zeros as well.
struct LaneSplit {
  int tiles, own;          // tiles of a plane, lanes that each owns
  int pitch, gap;          // lanes from unit to unit; more lanes behind each second one (two tiles a plane)
  int per;                 // units of a wave
  int segs, rows;          // stretches of a tile and their rows of coefficients
  int units, blocks;       // of a channel
};

// Lanes that a lane's K x K windows reach to either side: the coefficients' reach further than the pixels'.
constexpr int lane_halo(int K) { return (K / 2 + 1) / 2; }

// v and its neighbours' values, R to either side.
template <int N, int R>
__device__ __forceinline__ void widen(const float (&v)[N], float (&w)[N + 2 * R]) {
#pragma unroll
  for (int e = 0; e < N; ++e) w[R + e] = v[e];
#pragma unroll
  for (int d = 1; d <= R; ++d) {
    float l = wave_before(v[(4 * N - d) % N]), r = wave_behind(v[(d - 1) % N]);
    if (d > N) {
      l = wave_before(l);
      r = wave_behind(r);
    }
    w[R - d] = l;
    w[R + N - 1 + d] = r;
  }
}

// Two rows of four pixels as they come from memory.
template <typename T>
struct RowPair {
  static constexpr int N = sizeof(T) == 4 ? 4 : 2;      // words of a row
  uint32_t w[2][N];

  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < N; ++k) w[0][k] = w[1][k] = 0u;
  }
  __device__ __forceinline__ void load(int row, const T* __restrict__ p) {
    if constexpr (N == 4) {
      const uint4 q = load_u4<4>(p);
      w[row][0] = q.x; w[row][1] = q.y; w[row][2] = q.z; w[row][3] = q.w;
    } else {
      const uint2 q = load_u2<2>(p);
      w[row][0] = q.x; w[row][1] = q.y;
    }
  }
  // (planes less than four pixels wide)
  __device__ __forceinline__ void load_few(int row, const T* __restrict__ p, int n) {
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < 3; ++e)
      if (e < n) v[e] = to_f32<T>(p[e]);
    if constexpr (N == 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) w[row][e] = __float_as_uint(v[e]);
    } else {
      w[row][0] = pack2<T>(v[0], v[1]);
      w[row][1] = pack2<T>(v[2], v[3]);
    }
  }
  __device__ __forceinline__ void get(int row, float (&v)[4]) const {
    if constexpr (N == 4) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = __uint_as_float(w[row][e]);
    } else {
      unpack2<T>(w[row][0], v[0], v[1]);
      unpack2<T>(w[row][1], v[2], v[3]);
    }
  }
};

// This lane's unit and place in it.
struct LaneUnit {
  int b, tile, seg;
  int j;             // its first coefficient's column
  bool have, owns;   // within the plane; owned by the unit
};
template <int HL>
__device__ __forceinline__ LaneUnit lane_unit(const LaneSplit& sp, int u0, int lane, int wl) {
  LaneUnit r;
  // with two tiles a plane the gap follows each right one
  const int first = sp.gap > 0 ? u0 & 1 : 0, pair = 2 * sp.pitch + sp.gap, l = lane + first * sp.pitch;
  int slot, q;
  if (sp.gap > 0) {
    const int p = l / pair, in = l - p * pair;
    slot = 2 * p + (in >= sp.pitch ? 1 : 0);
    q = in - (in >= sp.pitch ? sp.pitch : 0);
    slot -= first;
  } else {
    slot = lane / sp.pitch;
    q = lane - slot * sp.pitch;
  }
  const int u = u0 + slot, bs = u / sp.tiles;
  r.tile = u - bs * sp.tiles;
  r.b = bs / sp.segs;
  r.seg = bs - r.b * sp.segs;
  if (r.tile > 0 || sp.tiles > 2) q -= HL;
  r.j = 2 * (r.tile * sp.own + q);
  r.have = slot < sp.per && u < sp.units && q < sp.own + HL && r.j >= 0 && r.j < wl;
  r.owns = r.have && q >= 0 && q < sp.own;
  return r;
}

// One step of the layer.  `sub` (CARRY) = the sub-layer's result on the LL band, (planes, hl, wl); without it the LL band is
// convolved here (the last level).  A lane takes its rows of coefficients one after the other: each adds to the K rows of
// band results around it and to as many rows of pixels, which move up by one (two) as the row ends; the first K - 1 rows and
// the last, which reach beyond the stretch, skip what they would add outside it.  Coefficients are sums and differences
// without their factor 1/2 (a power of two, made up for at the inverse).
// fw[c * fstride]: the channel's folded filters; `fbase` / `fband` = offsets of the base filter and of the four sub-band
// filters, in SGPRs a filter at a time.  fb == nullptr: no bias.
// A row of coefficients at K = 5 is 350 multiply-adds of about 450 vector instructions, and [8,96,160,160] fp32 52 us (47 from
// the caches), where the memory that it moves takes 35; tiles in LDS with a thread for four coefficients took 68.
// grid = 1-D, a multiple of eight, at least C * sp.blocks; block = 256 (waves on their own).
template <typename T, int K, bool CARRY>
__global__ __launch_bounds__(kStreamThreads, K <= 5 ? 3 : 2) void stream_final_kernel(
    const T* __restrict__ x, T* __restrict__ out, const float* __restrict__ sub, int H, int W, int hl, int wl,
    const float* __restrict__ fw, const float* __restrict__ fb, int C, int fstride, int fbase, int fband, LaneSplit sp) {
  constexpr int R = K / 2, KK = K * K, S0 = CARRY ? 1 : 0, NP = 3 * R + 2;
  const int tid = threadIdx.x, lane = tid & (kWave - 1);
  const int at = xcd_contiguous(blockIdx.x, gridDim.x);      // (an XCD's workgroups share rows)
  const int ch = WT_UNIFORM(at / sp.blocks);
  const int u0 = WT_UNIFORM(((at - ch * sp.blocks) * (kStreamThreads / kWave) + (tid >> 6)) * sp.per);
  if (ch >= C || u0 >= sp.units) return;
  const LaneUnit un = lane_unit<lane_halo(K)>(sp, u0, lane, wl);
  const bool have = un.have;
  const int i0 = un.seg * sp.rows, i1 = un.owns ? min(i0 + sp.rows, hl) : i0, c0 = 2 * un.j;
  const int steps = sp.rows + 2 * R;
  const long long row0 = (static_cast<long long>(un.b) * C + ch) * H + 2 * i0;
  const T* px = x + (row0 - 2 * R) * W + (W >= 4 ? piece_start(c0, W) : c0);
  T* po = out + row0 * W + c0;
  const float* pz = CARRY ? sub + ((static_cast<long long>(un.b) * C + ch) * hl + i0) * wl + un.j : nullptr;
  wt_uniform_ptr fwc = (wt_uniform_ptr)(fw + static_cast<size_t>(ch) * fstride);
  const float bias = fb != nullptr ? fb[ch] : 0.f;
  // rows of pixels 2 (i - R) ..., and of band results i - R ..., around the row i of the step
  float P[NP][4], Y[4][K][2];
#pragma unroll
  for (int k = 0; k < NP; ++k)
#pragma unroll
    for (int e = 0; e < 4; ++e) P[k][e] = bias;
#pragma unroll
  for (int s = 0; s < 4; ++s)
#pragma unroll
    for (int k = 0; k < K; ++k) Y[s][k][0] = Y[s][k][1] = 0.f;

  // (lanes without pixels keep the zeros that they start with)
  auto fetch = [&](int t, int width, RowPair<T>& r) __attribute__((always_inline)) {
    const int i = i0 - R + t;
    const bool top = have && i >= 0 && 2 * i < H, bottom = have && i >= 0 && 2 * i + 1 < H;
    if (WT_ANY_LANE(have && !bottom)) r.clear();
    if (width >= 4) {
      if (top) r.load(0, px);
      if (bottom) r.load(1, px + width);
    } else {
      if (top) r.load_few(0, px, width - c0);
      if (bottom) r.load_few(1, px + width, width - c0);
    }
    px += 2 * width;
  };
  // Row t of the stretch: it adds to rows KLO .. KHI - 1 of the K around it.
  auto step = [&](auto klo, auto khi, auto ends, int t, const RowPair<T>& now, RowPair<T>& next) __attribute__((always_inline)) {
    constexpr int KLO = decltype(klo)::value, KHI = decltype(khi)::value;
    constexpr bool ENDS = decltype(ends)::value;      // (and a row of results ends with it)
    const int o = i0 + t - 2 * R;
    // (what follows from these is not kept over the loop: the SGPRs are for the weights)
    int at_c = c0, width = W;
    WT_LAUNDER_LANE_INT(at_c);
    WT_LAUNDER_UNIFORM(width);
    float a[4], c[4], z[2] = {0.f, 0.f};
    now.get(0, a);
    now.get(1, c);
    if (width >= 4) {
      piece_shift(a, at_c, width);
      piece_shift(c, at_c, width);
    }
    if (t + 1 < steps) fetch(t + 1, width, next);
    if constexpr (ENDS && CARRY) {
      if (o < i1) {
        if (at_c + 2 < width) {
          const uint2 v = load_u2<2>(pz);
          z[0] = __uint_as_float(v.x);
          z[1] = __uint_as_float(v.y);
        } else {
          z[0] = *pz;
        }
      }
      pz += wl;
    }
    {
      float ar[4 + 2 * R], cr[4 + 2 * R];
      widen<4, R>(a, ar);
      widen<4, R>(c, cr);
      wt_uniform_ptr w = fwc + fbase;
      WT_LAUNDER_UNIFORM(w);
#pragma unroll
      for (int k = 0; k < NP; ++k) {
        if (K > 3 && k > R && (k - R) % 2 == 0) {      // (three rows of a filter at a time)
          pin_values(P[k - 1]);
          pin_values(P[k - 2]);
          WT_SCHED_FENCE();
          WT_LAUNDER_UNIFORM(w);
        }
        const int up = 3 * R - k, low = up + 1;      // rows of the filter that the two rows of pixels meet
        const bool adds = k >= R && k / 2 >= KLO && k / 2 < KHI;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = k + 2 < NP ? P[k + 2][e] : bias;
          if (adds && up >= 0) {
#pragma unroll
            for (int kw = 0; kw < K; ++kw) v = kw == 0 ? fma_apart(w[up * K], ar[e], v) : fmaf(w[up * K + kw], ar[e + kw], v);
          }
          if (adds && low < K) {
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
              v = kw == 0 && up < 0 ? fma_apart(w[low * K], cr[e], v) : fmaf(w[low * K + kw], cr[e + kw], v);
          }
          P[k][e] = v;
        }
      }
    }
    WT_SCHED_FENCE();
#pragma unroll
    for (int s = S0; s < 4; ++s) {
      float v[2], vr[2 + 2 * R];
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float sac = a[2 * e] + c[2 * e], sbd = a[2 * e + 1] + c[2 * e + 1];
        const float dac = a[2 * e] - c[2 * e], dbd = a[2 * e + 1] - c[2 * e + 1];
        v[e] = s == 0 ? sac + sbd : s == 1 ? dac + dbd : s == 2 ? sac - sbd : dac - dbd;
      }
      widen<2, R>(v, vr);
      wt_uniform_ptr w = fwc + fband + s * KK;
      WT_LAUNDER_UNIFORM(w);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        if (K > 3 && k == (K + 1) / 2) {
#pragma unroll
          for (int d = 0; d < (K + 1) / 2; ++d) pin_values(Y[s][d]);
          WT_SCHED_FENCE();
          WT_LAUNDER_UNIFORM(w);
        }
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          float y = k + 1 < K ? Y[s][k + 1][e] : 0.f;
          if (k >= KLO && k < KHI) {
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
              y = kw == 0 ? fma_apart(w[(2 * R - k) * K], vr[e], y) : fmaf(w[(2 * R - k) * K + kw], vr[e + kw], y);
          }
          Y[s][k][e] = y;
        }
      }
      WT_SCHED_FENCE();      // (a filter at a time in SGPRs)
    }
    if constexpr (ENDS) {
      if (o < i1) {
        float r[2][4];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float y1 = Y[1][0][e];
          const float p = CARRY ? fmaf(2.f, z[e], y1) : Y[0][0][e] + y1, m = CARRY ? fmaf(2.f, z[e], -y1) : Y[0][0][e] - y1;
          const float q = Y[2][0][e] + Y[3][0][e], d = Y[2][0][e] - Y[3][0][e];
          r[0][2 * e] = fmaf(0.25f, p + q, P[0][2 * e]);
          r[0][2 * e + 1] = fmaf(0.25f, p - q, P[0][2 * e + 1]);
          r[1][2 * e] = fmaf(0.25f, m + d, P[1][2 * e]);
          r[1][2 * e + 1] = fmaf(0.25f, m - d, P[1][2 * e + 1]);
        }
        store4_any<T>(po, width - at_c, r[0]);
        if (2 * o + 1 < H) store4_any<T>(po + width, width - at_c, r[1]);
      }
      po += 2 * width;
    }
  };
  // (both ways round, so that no row moves from register to register)
  using std::false_type;
  using std::true_type;
#define WT_ROWS(n) std::integral_constant<int, (n)>{}
  RowPair<T> ra, rb;
  ra.clear();
  rb.clear();
  fetch(0, W, ra);
  if constexpr (R >= 1) {
    step(WT_ROWS(2 * R), WT_ROWS(K), false_type{}, 0, ra, rb);
    step(WT_ROWS(2 * R - 1), WT_ROWS(K), false_type{}, 1, rb, ra);
  }
  if constexpr (R >= 2) {
    step(WT_ROWS(2 * R - 2), WT_ROWS(K), false_type{}, 2, ra, rb);
    step(WT_ROWS(2 * R - 3), WT_ROWS(K), false_type{}, 3, rb, ra);
  }
  if constexpr (R >= 3) {
    step(WT_ROWS(2 * R - 4), WT_ROWS(K), false_type{}, 4, ra, rb);
    step(WT_ROWS(2 * R - 5), WT_ROWS(K), false_type{}, 5, rb, ra);
  }
  int t = 2 * R;
  for (; t + 1 < sp.rows; t += 2) {
    step(WT_ROWS(0), WT_ROWS(K), true_type{}, t, ra, rb);
    step(WT_ROWS(0), WT_ROWS(K), true_type{}, t + 1, rb, ra);
  }
  if (t < sp.rows) {
    step(WT_ROWS(0), WT_ROWS(K), true_type{}, t, ra, rb);
    ++t;
    ra = rb;
  }
  if constexpr (R >= 1) {
    step(WT_ROWS(0), WT_ROWS(2 * R), true_type{}, t, ra, rb);
    step(WT_ROWS(0), WT_ROWS(2 * R - 1), true_type{}, t + 1, rb, ra);
  }
  if constexpr (R >= 2) {
    step(WT_ROWS(0), WT_ROWS(2 * R - 2), true_type{}, t + 2, ra, rb);
    step(WT_ROWS(0), WT_ROWS(2 * R - 3), true_type{}, t + 3, rb, ra);
  }
  if constexpr (R >= 3) {
    step(WT_ROWS(0), WT_ROWS(2 * R - 4), true_type{}, t + 4, ra, rb);
    step(WT_ROWS(0), WT_ROWS(2 * R - 5), true_type{}, t + 5, rb, ra);
  }
#undef WT_ROWS
}

// Where the sums of stream_corr_kernel go: partial[(chunk * C + c) * rec + f * K*K + t].
struct StreamCorrOut {
  float* partial;
  int rec;
  int fbase;       // filter of the base conv; its detail bands' are fband .. fband + 2
  int fband;
  int with_gsum;   // the plain sum of grad_out goes to the last word of the record (the bias gradient)
};

// One step of the parameter gradients: correlation sums of x with grad_out (BASE) and of their level-1 detail bands
// (BANDS), dWt[kh][kw] = sum_{b,i,j} G[i][j] * X[i+kh-R][j+kw-R], and the LL bands of both for the sub-layer (where
// xll / gll are given; BASE only).  A workgroup takes a contiguous range of the (batch item, tile) units of a channel;
// a thread owns four coefficients (2 x 8 pixels of grad_out, in registers) and keeps the sums of all four filters, so
// that x and grad_out are read once.  K = 7 has too many sums for that (196): two launches.
// [8,96,160,160] fp32, K = 5: 82 us; a workgroup per filter over bands from memory took 43 + 65 for the same filters,
// after 26 us for writing the bands.
// grid = (C, nchunk), block = 256.
template <typename T, int K, typename Shape, bool BASE, bool BANDS>
__global__ __launch_bounds__(kStreamThreads, K <= 5 ? 3 : 2) void stream_corr_kernel(const T* __restrict__ x,
                                                                        const T* __restrict__ g,
                                                                        float* __restrict__ xll,
                                                                        float* __restrict__ gll, int H, int W, int hl,
                                                                        int wl, int B, int C, StreamCorrOut outp) {
  constexpr int R = K / 2, KK = K * K;
  constexpr int TH = Shape::TH, TW = Shape::TW, HP = kStreamPad, TJ = 4, NT = TW / TJ;
  constexpr int AH = TH + 2 * R, AWD = TW + 2 * HP;
  constexpr int XH = 2 * AH, XWD = 2 * AWD;
  constexpr int NS = (BASE ? 1 : 0) + (BANDS ? 3 : 0);
  __shared__ alignas(16) float At[BANDS ? 3 * AH * AWD : 4];
  __shared__ alignas(16) float Xt[XH * XWD];
  __shared__ float red[4][NS * KK + 1];
  const int cc = blockIdx.x, chunk = blockIdx.y, tid = threadIdx.x;
  const int r = tid / NT, c0 = (tid - r * NT) * TJ;
  const int tiles_x = (wl + TW - 1) / TW, tiles = tiles_x * ((hl + TH - 1) / TH);
  const int units = B * tiles;
  const int per = (units + static_cast<int>(gridDim.y) - 1) / static_cast<int>(gridDim.y);
  const int u_begin = chunk * per;
  const int u_end = u_begin + per < units ? u_begin + per : units;
  const size_t psz = static_cast<size_t>(H) * W, lsz = static_cast<size_t>(hl) * wl;
  float acc[NS][KK];
  float gsum = 0.f;
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int t = 0; t < KK; ++t) acc[s][t] = 0.f;
  int b = u_begin / tiles, tile = u_begin - b * tiles;
  for (int u = u_begin; u < u_end; ++u) {
    const size_t plane = static_cast<size_t>(b) * C + cc;
    const int ty = tile / tiles_x, tx = tile - ty * tiles_x;
    if (++tile == tiles) { tile = 0; ++b; }
    const int i0 = ty * TH, j0 = tx * TW;
    const int i = i0 + r, j = j0 + c0;
    const bool own = r < TH && i < hl && j < wl;
    float gv[2][2 * TJ];
#pragma unroll
    for (int dr = 0; dr < 2; ++dr)
      load8_row<T>(g + plane * psz + static_cast<size_t>(2 * i + dr) * W + 2 * j,
                   own && 2 * i + dr < H ? W - 2 * j : 0, gv[dr]);
    stage_window<T, XH, XWD>(x + plane * psz, H, W, 2 * (i0 - R), 2 * (j0 - HP), Xt, tid);
    __syncthreads();
    if constexpr (BANDS) {
      haar_tile<AH, AWD, 1>(Xt, At, tid);
      __syncthreads();
    }
    if (own) {
      if constexpr (BASE) {
#pragma unroll
        for (int e = 0; e < 2 * TJ; ++e) gsum += gv[0][e] + gv[1][e];
        if (gll != nullptr) {
          float ll[TJ];
#pragma unroll
          for (int t = 0; t < TJ; ++t) ll[t] = 0.5f * ((gv[0][2 * t] + gv[1][2 * t]) + (gv[0][2 * t + 1] + gv[1][2 * t + 1]));
          store4_row(gll + plane * lsz + static_cast<size_t>(i) * wl + j, wl - j, ll);
        }
        if (xll != nullptr) {
          float a[8], c[8], ll[TJ];
          lds_read<8>(Xt + (2 * (r + R)) * XWD + 2 * (c0 + HP), a);
          lds_read<8>(Xt + (2 * (r + R) + 1) * XWD + 2 * (c0 + HP), c);
#pragma unroll
          for (int t = 0; t < TJ; ++t) ll[t] = 0.5f * ((a[2 * t] + c[2 * t]) + (a[2 * t + 1] + c[2 * t + 1]));
          store4_row(xll + plane * lsz + static_cast<size_t>(i) * wl + j, wl - j, ll);
        }
#pragma unroll
        for (int xr = 0; xr < K + 1; ++xr) {
          float v[16];
          lds_read<16>(Xt + (2 * r + xr + R) * XWD + 2 * c0 + HP, v);
#pragma unroll
          for (int dr = 0; dr < 2; ++dr) {
            const int kh = xr - dr;
            if (kh < 0 || kh >= K) continue;
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
#pragma unroll
              for (int e = 0; e < 2 * TJ; ++e)
                acc[0][kh * K + kw] = fmaf(gv[dr][e], v[e + kw - R + HP], acc[0][kh * K + kw]);
          }
          if (xr & 1) {
            pin_values(acc[0]);
            WT_CHUNK_FENCE();
          }
        }
      }
      if constexpr (BANDS) {
#pragma unroll
        for (int s = 1; s < 4; ++s) {
          constexpr int A0 = BASE ? 0 : -1;
          float gb[TJ];
#pragma unroll
          for (int t = 0; t < TJ; ++t) {
            const float sac = gv[0][2 * t] + gv[1][2 * t], sbd = gv[0][2 * t + 1] + gv[1][2 * t + 1];
            const float dac = gv[0][2 * t] - gv[1][2 * t], dbd = gv[0][2 * t + 1] - gv[1][2 * t + 1];
            gb[t] = 0.5f * (s == 1 ? dac + dbd : s == 2 ? sac - sbd : dac - dbd);
          }
#pragma unroll
          for (int kh = 0; kh < K; ++kh) {
            float v[12];
            lds_read<12>(At + ((s - 1) * AH + r + kh) * AWD + c0, v);
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
#pragma unroll
              for (int t = 0; t < TJ; ++t)
                acc[A0 + s][kh * K + kw] = fmaf(gb[t], v[t + kw - R + HP], acc[A0 + s][kh * K + kw]);
          }
          pin_values(acc[A0 + s]);
          WT_CHUNK_FENCE();
        }
      }
    }
    __syncthreads();
  }
  const int wave = tid >> 6, lane = tid & (kWave - 1);
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int t = 0; t < KK; ++t) {
      const float v = wave_sum(acc[s][t]);
      if (lane == 0) red[wave][s * KK + t] = v;
    }
  {
    const float v = wave_sum(gsum);
    if (lane == 0) red[wave][NS * KK] = v;
  }
  __syncthreads();
  float* dst = outp.partial + (static_cast<size_t>(chunk) * C + cc) * outp.rec;
  for (int o = tid; o <= NS * KK; o += kStreamThreads) {
    const float v = (red[0][o] + red[1][o]) + (red[2][o] + red[3][o]);
    const int s = o / KK, t = o - s * KK;
    if (s == NS) {
      if (BASE && outp.with_gsum) dst[outp.rec - 1] = v;
    } else {
      const int f = BASE && s == 0 ? outp.fbase : outp.fband + s - (BASE ? 1 : 0);
      dst[f * KK + t] = v;
    }
  }
}

}  // namespace wt
