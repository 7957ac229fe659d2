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
//   stream_final_kernel    detail bands of level 1, their convs, the sub-layer's result, inverse Haar, base conv
// Parameter gradients follow the same recursion: stream_corr_kernel sums the base conv's and the detail bands' filters
// from the pixels of x and grad_out, and the sub-layer's filters are its parameter gradients on X_1 and G_1.
// Nothing of a level but its LL band goes through memory.
//
// Measured, us a training step: [8,96,160,160] fp32 523 with a launch per level and pass and every band in memory, 366 with
// tiles of a step in LDS, 310 with rows over the lanes of a wave.
//
// Rows start at any element's address and may have any length (16-byte accesses need no more than that).
#pragma once

#include "common.h"
#include "kernels2d.h"

namespace wt {

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

// A lane's rows 2 i and 2 i + 1 of a plane of H rows, from p on (`lanes`: whether it has any there).  The loads are the last
// thing that happens to r until take_rows, whatever the width: a value that one of several paths may have written is moved
// where they meet, and waited for there.  (A path of its own for narrow planes cost both kernels below each load's latency: 50
// and 72 us, 44 and 63 without, at [8,96,160,160] fp32, K = 5.)
// Rows of less than four pixels are read on into the next ones, the tensor's last up to three pixels early: `left` = rows from
// the first one to the tensor's end.
__device__ __forceinline__ int narrow_back(long long left, int width) {
  return left * width < 4 ? 4 - static_cast<int>(left) * width : 0;
}
template <typename T>
__device__ __forceinline__ void fetch_rows(bool lanes, int i, int H, const T* __restrict__ p, int width, long long left,
                                           RowPair<T>& r) {
  const bool in = lanes && i >= 0;
  int b0 = 0, b1 = 0;
  if (width < 4) {
    b0 = narrow_back(left, width);
    b1 = narrow_back(left - 1, width);
  }
  if (in && 2 * i < H) r.load(0, p - b0);
  if (in && 2 * i + 1 < H) r.load(1, p + (width - b1));
}
// The values, zero outside the plane; lanes that never load hold the zeros that they start with.
template <typename T>
__device__ __forceinline__ void take_rows(const RowPair<T>& r, bool lanes, int i, int H, int c0, int width, long long left,
                                          float (&a)[4], float (&c)[4]) {
  r.get(0, a);
  r.get(1, c);
  if (width >= 4) {
    piece_shift(a, c0, width);
    piece_shift(c, c0, width);
  } else {
    const int b0 = narrow_back(left, width), b1 = narrow_back(left - 1, width);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float va = 0.f, vc = 0.f;
#pragma unroll
      for (int d = 0; e + d < 4; ++d) {
        if (d == b0) va = a[e + d];
        if (d == b1) vc = c[e + d];
      }
      a[e] = e < width ? va : 0.f;
      c[e] = e < width ? vc : 0.f;
    }
  }
  const bool top = i >= 0 && 2 * i < H, bottom = i >= 0 && 2 * i + 1 < H;
  if (WT_ANY_LANE(lanes && !bottom)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      a[e] = top ? a[e] : 0.f;
      c[e] = bottom ? c[e] : 0.f;
    }
  }
}

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
// A row of coefficients at K = 5 is 350 multiply-adds of about 450 vector instructions, and [8,96,160,160] fp32 44 us, where
// the memory that it moves takes 35; tiles in LDS with a thread for four coefficients took 68.
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

  const long long rows_end = W < 4 ? static_cast<long long>(sp.units / (sp.tiles * sp.segs)) * C * H : 0;
  auto fetch = [&](int t, int width, RowPair<T>& r) WT_INLINE_LAMBDA {
    fetch_rows<T>(have, i0 - R + t, H, px, width, rows_end - row0 + 2 * (R - t), r);
    px += 2 * width;
  };
  // Row t of the stretch: it adds to rows KLO .. KHI - 1 of the K around it.
  auto step = [&](auto klo, auto khi, auto ends, int t, const RowPair<T>& now, RowPair<T>& next) WT_INLINE_LAMBDA {
    constexpr int KLO = decltype(klo)::value, KHI = decltype(khi)::value;
    constexpr bool ENDS = decltype(ends)::value;      // (and a row of results ends with it)
    const int o = i0 + t - 2 * R;
    // (what follows from these is not kept over the loop: the SGPRs are for the weights)
    int at_c = c0, width = W;
    WT_LAUNDER_LANE_INT(at_c);
    WT_LAUNDER_UNIFORM(width);
    float a[4], c[4], z[2] = {0.f, 0.f};
    take_rows<T>(now, have, i0 - R + t, H, at_c, width, rows_end - row0 + 2 * (R - t), a, c);
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
// xll / gll are given; BASE only).  Rows over the lanes of a wave, as above: a lane walks down its rows of grad_out, keeps the
// rows of x and of its bands around them in registers (a ring, whose place follows from the row: the loop is unrolled over a
// round of it) and the sums of all four filters, so that x and grad_out are read once and every multiply-add is one of the
// sums'.  K = 7 has too many sums for that (196): two launches.
// A wave takes every `waves`-th group of `per` units of its channel, an even number apart: a lane beside its unit's own ones
// is beside them in all its groups, and its sums (an infinity of x times the zero of no grad_out) are left out at the end.
// Coefficients are sums and differences without their factor 1/2, products take the 1/4 at the end.
// A row at K = 5 is 350 multiply-adds, 84 moves from the neighbours and some 90 others, and two waves fit a SIMD (229
// registers).  [8,96,160,160] fp32: 63 us, of which the issue of its instructions is 43; tiles in LDS with a thread for four
// coefficients took 81, two thirds of it LDS reads and their bank conflicts.
// grid = (C, nchunk), block = 256 (waves on their own until their sums meet).
template <typename T, int K, bool BASE, bool BANDS>
__global__ __launch_bounds__(kStreamThreads, 2) void stream_corr_kernel(const T* __restrict__ x, const T* __restrict__ g,
                                                                        float* __restrict__ xll, float* __restrict__ gll,
                                                                        int H, int W, int hl, int wl, int C,
                                                                        StreamCorrOut outp, LaneSplit sp) {
  constexpr int R = K / 2, KK = K * K, HP = (R + 1) / 2;
  constexpr int LEAD = BANDS ? R : HP, P = 2 * LEAD + 1;      // rows of x ahead of grad_out's; rows of the ring
  constexpr int NS = (BASE ? 1 : 0) + (BANDS ? 3 : 0), A0 = BASE ? 1 : 0;
  constexpr int NR = (NS * KK + 4) / 4 * 4;                    // the sums and grad_out's own, in fours
  __shared__ float red[kStreamThreads / kWave][NR];
  const int ch = blockIdx.x, chunk = blockIdx.y, tid = threadIdx.x, lane = tid & (kWave - 1);
  const int wave = WT_UNIFORM(tid >> 6), waves = static_cast<int>(gridDim.y) * (kStreamThreads / kWave);
  float acc[NS][KK], gsum = 0.f;
  const long long rows_end = W < 4 ? static_cast<long long>(sp.units / (sp.tiles * sp.segs)) * C * H : 0;
  bool keep = false;
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int t = 0; t < KK; ++t) acc[s][t] = 0.f;

  for (int u0 = (chunk * (kStreamThreads / kWave) + wave) * sp.per; u0 < sp.units; u0 += waves * sp.per) {
    const LaneUnit un = lane_unit<lane_halo(K)>(sp, u0, lane, wl);
    const bool have = un.have, owns = un.owns;
    keep = keep || owns;
    const int i0 = un.seg * sp.rows, i1 = owns ? min(i0 + sp.rows, hl) : i0, c0 = 2 * un.j;
    const long long plane = static_cast<long long>(un.b) * C + ch;
    const int cl = W >= 4 ? piece_start(c0, W) : c0;
    const T* px = x + (plane * H + 2 * (i0 - LEAD)) * W + cl;
    const T* pg = g + (plane * H + 2 * i0) * W + cl;
    long long pl = (plane * hl + i0) * wl + un.j;
    float X[BASE ? P : 1][2][4], Z[BANDS ? P : 1][3][2];
    RowPair<T> rx, rg;
    rx.clear();
    rg.clear();
    // (row i of the coefficients')
    auto left = [&](int i) WT_INLINE_LAMBDA { return rows_end - (plane * H + 2 * i); };
    auto detail = [](const float (&a)[4], const float (&c)[4], float (&z)[3][2]) WT_INLINE_LAMBDA {
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float sac = a[2 * e] + c[2 * e], sbd = a[2 * e + 1] + c[2 * e + 1];
        const float dac = a[2 * e] - c[2 * e], dbd = a[2 * e + 1] - c[2 * e + 1];
        z[0][e] = dac + dbd;
        z[1][e] = sac - sbd;
        z[2][e] = dac - dbd;
      }
    };
    auto put = [&](auto slot, int i, int width, const RowPair<T>& r) WT_INLINE_LAMBDA {      // row i of x, which has come
      constexpr int S = decltype(slot)::value;
      float a[4], c[4];
      take_rows<T>(r, have, i, H, c0, width, left(i), a, c);
      if constexpr (BASE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          X[S][0][e] = a[e];
          X[S][1][e] = c[e];
        }
      }
      if constexpr (BANDS) detail(a, c, Z[S]);
    };
    // Row t of the stretch, t % P == PH: rows t .. t + P - 1 of x from the stretch's first one are in places PH, PH + 1, ...
    auto step = [&](auto phase, int t) WT_INLINE_LAMBDA {
      constexpr int PH = decltype(phase)::value;
      const int o = i0 + t;
      int width = W;
      WT_LAUNDER_UNIFORM(width);
      put(std::integral_constant<int, (PH + P - 1) % P>{}, o + LEAD, width, rx);
      float gv[2][4];
      take_rows<T>(rg, owns, o < i1 ? o : hl, H, c0, width, left(o), gv[0], gv[1]);
      px += 2 * width;
      pg += 2 * width;
      if (t + 1 < sp.rows) {
        fetch_rows<T>(have, o + LEAD + 1, H, px, width, left(o + LEAD + 1), rx);
        fetch_rows<T>(owns && o + 1 < i1, o + 1, H, pg, width, left(o + 1), rg);
      }
      if (WT_ANY_LANE(have && o >= hl)) {      // (no row of grad_out meets the rows of x that are left)
        const bool past = o >= hl;
#pragma unroll
        for (int k = 0; k < P; ++k) {
          if constexpr (BASE) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              X[k][0][e] = past ? 0.f : X[k][0][e];
              X[k][1][e] = past ? 0.f : X[k][1][e];
            }
          }
          if constexpr (BANDS) {
#pragma unroll
            for (int s = 0; s < 3; ++s) {
              Z[k][s][0] = past ? 0.f : Z[k][s][0];
              Z[k][s][1] = past ? 0.f : Z[k][s][1];
            }
          }
        }
      }
      if constexpr (BASE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) gsum += gv[0][e] + gv[1][e];
        auto ll = [&](float* __restrict__ dst, const float (&a)[4], const float (&c)[4]) WT_INLINE_LAMBDA {
          const float v0 = 0.5f * ((a[0] + c[0]) + (a[1] + c[1])), v1 = 0.5f * ((a[2] + c[2]) + (a[3] + c[3]));
          if (un.j + 1 < wl) store_u2<2>(dst + pl, uint2{__float_as_uint(v0), __float_as_uint(v1)});
          else dst[pl] = v0;
        };
        if (xll != nullptr && o < i1) ll(xll, X[(PH + LEAD) % P][0], X[(PH + LEAD) % P][1]);
        if (gll != nullptr && o < i1) ll(gll, gv[0], gv[1]);
        pl += wl;
        WT_SCHED_FENCE();
#pragma unroll
        for (int xr = 0; xr < K + 1; ++xr) {      // row 2 o + xr - R of pixels
          const int q = xr - R + 2 * HP;          // (from the first of the ring's middle 2 HP + 1 pairs)
          float v[4 + 2 * R];
          widen<4, R>(X[(PH + LEAD - HP + q / 2) % P][q & 1], v);
#pragma unroll
          for (int dr = 0; dr < 2; ++dr) {
            const int kh = xr - dr;
            if (kh < 0 || kh >= K) continue;
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
#pragma unroll
              for (int e = 0; e < 4; ++e) acc[0][kh * K + kw] = fmaf(v[e + kw], gv[dr][e], acc[0][kh * K + kw]);
          }
          if (xr & 1) {
            pin_values(acc[0]);
            WT_SCHED_FENCE();
          }
        }
      }
      if constexpr (BANDS) {
        float gz[3][2];
        detail(gv[0], gv[1], gz);
#pragma unroll
        for (int s = 0; s < 3; ++s) {
#pragma unroll
          for (int kh = 0; kh < K; ++kh) {
            float v[2 + 2 * R];
            widen<2, R>(Z[(PH + kh) % P][s], v);
#pragma unroll
            for (int kw = 0; kw < K; ++kw)
#pragma unroll
              for (int e = 0; e < 2; ++e) acc[A0 + s][kh * K + kw] = fmaf(v[e + kw], gz[s][e], acc[A0 + s][kh * K + kw]);
          }
          pin_values(acc[A0 + s]);
          WT_SCHED_FENCE();
        }
      }
    };
    // (all the rows before the first one at once)
    auto fill = [&](auto... q) WT_INLINE_LAMBDA {
      RowPair<T> r[sizeof...(q)];
      (r[decltype(q)::value].clear(), ...);
      (fetch_rows<T>(have, i0 - LEAD + decltype(q)::value, H, px + 2LL * decltype(q)::value * W, W,
                     left(i0 - LEAD + decltype(q)::value), r[decltype(q)::value]), ...);
      px += 2LL * LEAD * 2 * W;
      fetch_rows<T>(have, i0 + LEAD, H, px, W, left(i0 + LEAD), rx);
      fetch_rows<T>(owns, i0, H, pg, W, left(i0), rg);
      (put(q, i0 - LEAD + decltype(q)::value, W, r[decltype(q)::value]), ...);
    };
    auto round = [&](int t, auto... ph) WT_INLINE_LAMBDA {
      (void)(... && (t + decltype(ph)::value < sp.rows ? (step(ph, t + decltype(ph)::value), true) : false));
    };
#define WT_PH(n) std::integral_constant<int, (n)>{}
    if constexpr (LEAD == 1) fill(WT_PH(0), WT_PH(1));
    if constexpr (LEAD == 2) fill(WT_PH(0), WT_PH(1), WT_PH(2), WT_PH(3));
    if constexpr (LEAD == 3) fill(WT_PH(0), WT_PH(1), WT_PH(2), WT_PH(3), WT_PH(4), WT_PH(5));
    if constexpr (LEAD == 0) {
      fetch_rows<T>(have, i0, H, px, W, left(i0), rx);
      fetch_rows<T>(owns, i0, H, pg, W, left(i0), rg);
    }
    for (int t = 0; t < sp.rows; t += P) {
      if constexpr (P == 1) round(t, WT_PH(0));
      if constexpr (P == 3) round(t, WT_PH(0), WT_PH(1), WT_PH(2));
      if constexpr (P == 5) round(t, WT_PH(0), WT_PH(1), WT_PH(2), WT_PH(3), WT_PH(4));
      if constexpr (P == 7) round(t, WT_PH(0), WT_PH(1), WT_PH(2), WT_PH(3), WT_PH(4), WT_PH(5), WT_PH(6));
    }
#undef WT_PH
  }
  {
    float sums[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) sums[i] = !keep ? 0.f : i < NS * KK ? acc[i < NS * KK ? i / KK : 0][i % KK] : i == NS * KK ? gsum : 0.f;
    wave_sums<NR>(sums, lane, red[wave]);
  }
  __syncthreads();
  float* dst = outp.partial + (static_cast<size_t>(chunk) * C + ch) * outp.rec;
  for (int o = tid; o <= NS * KK; o += kStreamThreads) {
    const float v = (red[0][o] + red[1][o]) + (red[2][o] + red[3][o]);
    const int s = o / KK, t = o - s * KK;
    if (s == NS) {
      if (BASE && outp.with_gsum) dst[outp.rec - 1] = v;
    } else {
      const int f = s < A0 ? outp.fbase : outp.fband + s - A0;
      dst[f * KK + t] = s < A0 ? v : 0.25f * v;
    }
  }
}

}  // namespace wt
