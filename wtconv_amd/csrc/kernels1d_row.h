// Row-resident WTConv1d kernels for gfx950.
//
// One workgroup owns a (b, c) row, or a segment of a longer one; every lane owns S consecutive samples and keeps
// them, their complete Haar pyramid and the outputs in registers.  S is a multiple of 2^L, so
// the analysis and synthesis butterflies never leave the lane.  The K-tap conv of a level
// needs R = K/2 coefficients from beyond either end of the lane's array: each lane publishes
// the edge entries of each of its arrays in LDS once per row, and reads its neighbours'
// (on the coarsest levels, where a lane holds fewer than R coefficients, from up to R lanes
// away).  LDS is otherwise used only to turn coalesced 16-byte HBM accesses into the
// lane-contiguous register layout and back (slot stride = odd number of 16-byte units:
// conflict-free both ways).  Three workgroup barriers per row instead of one per pyramid
// level and phase.
//
// Maths as in kernels1d.h (reference wtconv/wtconv1d.py:38-82, wtconv/util/wavelet.py:6-20,
// 46-59).  Samples past the end of the row are staged as zeros, which gives the 'same'
// padding of every level and the zero padding of odd lengths at once.
//
// A workgroup works on rows of ONE channel (grid = channels x batch chunks), and folds that
// channel's parameters itself when it starts (gamma * w, taps reversed for the input gradient):
// one entry per lane, read back as wave-uniform values -- no fold launch, no folded table in
// HBM.  The backward pass is one kernel: the row of x and the row of grad_out are read once and
// give grad_x and the running sums of the parameter gradients; the workgroup that finishes a
// channel last (a ticket per channel) sums the chunks' partial sums in chunk order and writes
// the channel's parameter gradients.
#pragma once

#include "common.h"
#include "kernels1d.h"
#include "wgrad_finish.h"

namespace wt {

// Samples per lane S: a multiple of 2^L (the pyramid of a lane is local) and of 8 (16-byte vectors of either
// dtype): 16 up to four levels (half the registers per lane of 32: more waves in flight, which is what these
// latency-bound kernels need), 32 for five.
constexpr int kRow1dMaxLanes = 256;      // threads per workgroup
constexpr int row1d_samples(int L) { return L <= 4 ? 16 : 32; }
constexpr bool row1d_built(int K, int L, int S) { return K >= 3 && S == row1d_samples(L); }

// Edge entries a lane publishes of an array of n entries: the first and last R, or all of
// them when there are fewer than 2R.
constexpr int row1d_pub(int n, int R) { return n < 2 * R ? n : 2 * R; }
// Entries of array `a` (0: the samples; 1 + 2(l-1) + s: level l, sub-band s).
constexpr int row1d_len(int S, int a) { return a == 0 ? S : S >> (1 + (a - 1) / 2); }
// Offset of array `a` inside a lane's published edges.
constexpr int row1d_edge_off(int K, int S, int a) {
  int off = 0;
  for (int i = 0; i < a; ++i) off += row1d_pub(row1d_len(S, i), K / 2);
  return off;
}

// Floats of LDS per lane: the lane's S samples (plus a pad that makes the stride an odd
// number of 16-byte units) or its published edges, whichever is larger.
constexpr int row1d_slot(int K, int L, int S) {
  const int halo = row1d_edge_off(K, S, 1 + 2 * L);
  int f = S + 4 > halo ? S + 4 : halo;
  f = (f + 3) / 4 * 4;
  if ((f / 4) % 2 == 0) f += 4;
  return f;
}

// Zero slots on either side of a region's `block` lane slots: a lane reads the edges of up to ceil(R / n) lanes
// away (n = entries per lane at the coarsest level), and beyond either end of the row those reads land here --
// no condition, no branch around the read, every edge at a constant offset from the lane's own slot.
constexpr int row1d_guard(int K, int L, int S) {
  const int nmin = S >> L;
  const int R = K / 2;
  return nmin < 1 ? R : (R + nmin - 1) / nmin;
}
// Floats of one region (guards included) for a workgroup of `block` lanes.
constexpr size_t row1d_region(int K, int L, int S, int block) {
  return static_cast<size_t>(block + 2 * row1d_guard(K, L, S)) * row1d_slot(K, L, S);
}

// A row longer than a workgroup is cut into `nseg` segments of `use` lanes each.  A segment is staged with `hal` more
// lanes on either side, whose samples give the convolutions of its own lanes their neighbours (the pyramid of a lane
// is local, so nothing reaches further than row1d_guard lanes); what the halo lanes compute themselves is dropped: their
// outputs are not stored, their sums not added up.  Rows that fit the workgroup are one segment without halo.
struct Row1D {
  int C, N;
  int nl;        // lanes that hold samples of a segment, halo included
  int hal, use, nseg;
  __device__ __forceinline__ bool own(int lane) const { return lane >= hal && lane < hal + use; }
};

// The (batch item, segment) units of a channel, one after the other.
struct RowUnit {
  int b, seg;
  __device__ __forceinline__ RowUnit(int unit, const Row1D& pl) : b(unit / pl.nseg), seg(unit - b * pl.nseg) {}
  __device__ __forceinline__ void next(const Row1D& pl) {
    if (++seg == pl.nseg) { seg = 0; ++b; }
  }
  // the sample that the segment's first lane holds first (negative in the halo of a row's first segment)
  __device__ __forceinline__ int first(const Row1D& pl, int S) const { return WT_UNIFORM((seg * pl.use - pl.hal) * S); }
  template <typename T>
  __device__ __forceinline__ T* row(T* base, const Row1D& pl, int c) const {
    return base + (static_cast<size_t>(WT_UNIFORM(b)) * pl.C + c) * pl.N;
  }
};

// HBM row -> LDS slots (slot of lane j = samples [p0 + j*S, p0 + (j+1)*S), zeros outside the row), in two steps
// so that the loads of the next row can be in flight while the current one is computed:
// row1d_fetch issues every 16-byte load of the thread at once (at most S / EV of them, since
// the workgroup has at least as many threads as lanes that hold samples), row1d_commit
// converts and writes them to the slots.  The vectors are those of the row, whatever its address: rows of odd length
// start anywhere, and a 16-byte load at an element's alignment costs one cache line more per wave, where loads of
// single elements are eight times as many (rows of 20011 bfloat16 samples).  The elements behind the last whole
// vector are loaded one each by the first lanes.
// STREAM: the loads are marked non-temporal (measured: pays in the whole-backward kernel, which reads two rows per
// row it writes, not in the forward kernel).
template <typename T, int S>
struct RowFetch {
  static constexpr int EV = 16 / sizeof(T);
  static constexpr int NQ = S / EV;
  uint4 q[NQ];
  float tail;

  template <bool STREAM = false>
  __device__ __forceinline__ void fetch(const T* __restrict__ row, int p0, int N, int tid, int nth) {
    const unsigned nvec = static_cast<unsigned>(N / EV * EV);
#pragma unroll
    for (int u = 0; u < NQ; ++u) {
      const unsigned p = static_cast<unsigned>(p0) + (tid + u * nth) * EV;      // (a negative sample is a large one)
      q[u].x = 0u; q[u].y = 0u; q[u].z = 0u; q[u].w = 0u;
      if (p < nvec) {
        if constexpr (STREAM) q[u] = load_stream_u4<sizeof(T)>(row + p);
        else q[u] = load_u4<sizeof(T)>(row + p);
      }
    }
    if (N % EV != 0) tail = tid < N % EV ? to_f32<T>(row[nvec + tid]) : 0.f;
  }

  template <int SLOT>
  __device__ __forceinline__ void commit(float* __restrict__ lds, int p0, int N, int nl, int tid, int nth) const;
};

template <int S, int SLOT, int EV>
__device__ __forceinline__ void row1d_put(float* __restrict__ lds, int p, const float (&vals)[EV]) {
  const int owner = p / S;               // S is a multiple of EV: one owner per vector
  float* dst = lds + owner * SLOT + (p - owner * S);
#pragma unroll
  for (int g = 0; g < EV / 4; ++g) {
    float4 w4;
    w4.x = vals[4 * g]; w4.y = vals[4 * g + 1]; w4.z = vals[4 * g + 2]; w4.w = vals[4 * g + 3];
    reinterpret_cast<float4*>(dst)[g] = w4;
  }
}

template <typename T>
__device__ __forceinline__ void row1d_unpack(const uint4& q, float (&vals)[16 / sizeof(T)]) {
  if constexpr (sizeof(T) == 4) {
    vals[0] = __uint_as_float(q.x); vals[1] = __uint_as_float(q.y);
    vals[2] = __uint_as_float(q.z); vals[3] = __uint_as_float(q.w);
  } else {
    const uint32_t qq[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      unpack2<T>(qq[k], vals[2 * k], vals[2 * k + 1]);
    }
  }
}

template <typename T, int S>
template <int SLOT>
__device__ __forceinline__ void RowFetch<T, S>::commit(float* __restrict__ lds, int p0, int N, int nl, int tid,
                                                       int nth) const {
  const int total = nl * S, nvec = N / EV * EV;
  const int split = N % EV != 0 ? nvec - p0 : -1;      // the vector that the tail's elements take the place of
#pragma unroll
  for (int u = 0; u < NQ; ++u) {
    const int p = (tid + u * nth) * EV;
    if (p < total && p != split) {
      float vals[EV];
      row1d_unpack<T>(q[u], vals);
      row1d_put<S, SLOT, EV>(lds, p, vals);
    }
  }
  if (split >= 0 && split < total && tid < EV) {
    const int owner = split / S;
    lds[owner * SLOT + (split - owner * S) + tid] = tail;
  }
}

// Fetch and commit of two rows (x and grad_out) in one call, at most four vectors of each at a time:
// bounded register use for the kernel that holds many running sums, and the loads of both
// rows share their HBM latency.
template <typename T, int S, int SLOT>
__device__ __forceinline__ void row1d_stage_pair(const T* __restrict__ row0, const T* __restrict__ row1,
                                                 float* __restrict__ lds0, float* __restrict__ lds1, int p0, int N,
                                                 int nl, int tid, int nth) {
  constexpr int EV = 16 / sizeof(T);
  constexpr int U = S / EV < 4 ? S / EV : 4;
  const int total = nl * S, nvec = N / EV * EV;
  const int split = N % EV != 0 ? nvec - p0 : -1;
  float t0 = 0.f, t1 = 0.f;
  if (split >= 0 && tid < N % EV) {
    t0 = to_f32<T>(row0[nvec + tid]);
    t1 = to_f32<T>(row1[nvec + tid]);
  }
  for (int v0 = tid; v0 * EV < total; v0 += U * nth) {
    uint4 q0[U], q1[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned p = static_cast<unsigned>(p0) + (v0 + u * nth) * EV;
      q0[u].x = 0u; q0[u].y = 0u; q0[u].z = 0u; q0[u].w = 0u;
      q1[u] = q0[u];
      if (p < static_cast<unsigned>(nvec)) {
        q0[u] = load_u4<sizeof(T)>(row0 + p);
        q1[u] = load_u4<sizeof(T)>(row1 + p);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = (v0 + u * nth) * EV;
      if (p < total && p != split) {
        float vals[EV];
        row1d_unpack<T>(q0[u], vals);
        row1d_put<S, SLOT, EV>(lds0, p, vals);
        row1d_unpack<T>(q1[u], vals);
        row1d_put<S, SLOT, EV>(lds1, p, vals);
      }
    }
  }
  if (split >= 0 && split < total && tid < EV) {
    const int owner = split / S, at = owner * SLOT + (split - owner * S) + tid;
    lds0[at] = t0;
    lds1[at] = t1;
  }
}

// LDS slots of a segment's own lanes -> HBM row (entries past N are dropped).  p0: sample of the slot of lane 0.
template <typename T, int S, int SLOT>
__device__ __forceinline__ void row1d_unstage(T* __restrict__ row, const float* __restrict__ lds, int p0,
                                              const Row1D& pl, int tid, int nth) {
  constexpr int EV = 16 / sizeof(T);
  const int first = p0 + pl.hal * S, N = pl.N;
  const int end = N - first < pl.use * S ? N - first : pl.use * S;
  const float* own = lds + pl.hal * SLOT;
  for (int v = tid; v * EV < end; v += nth) {
    const int lp = v * EV, p = first + lp;
    const int owner = lp / S;
    const float* src = own + owner * SLOT + (lp - owner * S);
    float vals[EV];
#pragma unroll
    for (int g = 0; g < EV / 4; ++g) {
      const float4 r4 = reinterpret_cast<const float4*>(src)[g];
      vals[4 * g] = r4.x; vals[4 * g + 1] = r4.y; vals[4 * g + 2] = r4.z; vals[4 * g + 3] = r4.w;
    }
    if (lp + EV <= N - first) {
      uint4 q;
      if constexpr (sizeof(T) == 4) {
        q.x = __float_as_uint(vals[0]); q.y = __float_as_uint(vals[1]);
        q.z = __float_as_uint(vals[2]); q.w = __float_as_uint(vals[3]);
      } else {
        uint32_t qq[4];
#pragma unroll
        for (int k = 0; k < 4; ++k)
          qq[k] = pack2<T>(vals[2 * k], vals[2 * k + 1]);
        q.x = qq[0]; q.y = qq[1]; q.z = qq[2]; q.w = qq[3];
      }
      store_stream_u4<sizeof(T)>(row + p, q);       // written once, read by another kernel: non-temporal
    } else {
#pragma unroll
      for (int k = 0; k < EV; ++k)
        if (lp + k < N - first) row[p + k] = from_f32<T>(vals[k]);
    }
  }
}

// Zeroes the guard slots of the `nregion` regions that start at `lds` (once per workgroup: nothing else writes them).
template <int K, int L, int S>
__device__ __forceinline__ void row1d_zero_guards(float* __restrict__ lds, int nregion, int tid, int nth) {
  constexpr int SLOT = row1d_slot(K, L, S), G = row1d_guard(K, L, S);
  const int rfl = (nth + 2 * G) * SLOT;
  for (int r = 0; r < nregion; ++r)
    for (int i = tid; i < 2 * G * SLOT; i += nth) {
      const int off = i < G * SLOT ? i : rfl - 2 * G * SLOT + i;
      lds[r * rfl + off] = 0.f;
    }
}

template <int S>
__device__ __forceinline__ void row1d_read_slot(const float* __restrict__ slot, float (&v)[S]) {
#pragma unroll
  for (int g = 0; g < S / 4; ++g) {
    const float4 r4 = reinterpret_cast<const float4*>(slot)[g];
    v[4 * g] = r4.x; v[4 * g + 1] = r4.y; v[4 * g + 2] = r4.z; v[4 * g + 3] = r4.w;
  }
}

template <int S>
__device__ __forceinline__ void row1d_write_slot(float* __restrict__ slot, const float (&v)[S]) {
#pragma unroll
  for (int g = 0; g < S / 4; ++g) {
    float4 w4;
    w4.x = v[4 * g]; w4.y = v[4 * g + 1]; w4.z = v[4 * g + 2]; w4.w = v[4 * g + 3];
    reinterpret_cast<float4*>(slot)[g] = w4;
  }
}

// Scaling.  The butterflies here are sums and differences without their 1/sqrt(2): level l's coefficients are
// 2^(l/2) times the orthonormal ones of wtconv/util/wavelet.py:46-59.  The folded weights of level l carry 2^-l
// (row1d_fold), which makes every level's reconstruction come out exactly scaled -- each inverse butterfly and each
// repeat of a coarse value owes 2^(-1/2), l of them in all -- and the correlation sums of level l (two pyramids, each
// 2^(l/2) up) are brought back by 2^-l when they leave the registers (row1d_store_partial).  Only powers of two are
// moved, which is exact; the 2 n multiplications per level and pass, and their roundings, are gone.
// The lane's pyramid: level l (1-based) has S >> l low-pass and as many high-pass entries.
template <int S, int L>
struct RowPyramid {
  float lo[L][S / 2];
  float hi[L][S / 2];
};

template <int S, int L>
__device__ __forceinline__ void row1d_analysis(const float (&x)[S], RowPyramid<S, L>& py) {
#pragma unroll
  for (int l = 0; l < L; ++l) {
#pragma unroll
    for (int q = 0; q < (S >> (l + 1)); ++q) {
      const float e = l == 0 ? x[2 * q] : py.lo[l > 0 ? l - 1 : 0][2 * q];
      const float o = l == 0 ? x[2 * q + 1] : py.lo[l > 0 ? l - 1 : 0][2 * q + 1];
      py.lo[l][q] = e + o;
      py.hi[l][q] = e - o;
    }
  }
}

// Publishes the edge entries of array number A (n entries) in the lane's slot.
template <int K, int S, int A, int NA>
__device__ __forceinline__ void row1d_publish(float* __restrict__ slot, const float (&arr)[NA]) {
  constexpr int R = K / 2, n = row1d_len(S, A), OFF = row1d_edge_off(K, S, A);
  static_assert(n <= NA, "array shorter than its level");
  if constexpr (n < 2 * R) {
#pragma unroll
    for (int d = 0; d < n; ++d) slot[OFF + d] = arr[d];
  } else {
#pragma unroll
    for (int d = 0; d < R; ++d) {
      slot[OFF + d] = arr[d];
      slot[OFF + R + d] = arr[n - R + d];
    }
  }
}

template <int K, int S, int L, int l>
__device__ __forceinline__ void row1d_publish_levels(float* __restrict__ slot, const RowPyramid<S, L>& py) {
  if constexpr (l <= L) {
    row1d_publish<K, S, 1 + 2 * (l - 1)>(slot, py.lo[l - 1]);
    row1d_publish<K, S, 2 + 2 * (l - 1)>(slot, py.hi[l - 1]);
    row1d_publish_levels<K, S, L, l + 1>(slot, py);
  }
}

// ext = [R entries to the left | the lane's n entries | R entries to the right] of array A;
// the neighbours' entries come from the slots of the lanes that own them (one or, on coarse
// levels with n < R, several lanes away); beyond either end of the workgroup those are the
// region's zero guard slots.
template <int K, int S, int SLOT, int A, int NA>
__device__ __forceinline__ void row1d_extend(const float* __restrict__ region, int tid, int nth,
                                             const float (&arr)[NA],
                                             float (&ext)[row1d_len(S, A) + 2 * (K / 2)]) {
  (void)nth;
  constexpr int R = K / 2, n = row1d_len(S, A), OFF = row1d_edge_off(K, S, A);
  const float* own = region + tid * SLOT;
#pragma unroll
  for (int d = 0; d < R; ++d) {
    {                                              // entry -R + d
      const int e = R - d;                         // distance to the left of entry 0
      const int o = (e + n - 1) / n;               // lanes to the left
      const int loc = o * n - e;                   // its index in that lane's array
      const int pos = n < 2 * R ? loc : R + loc - (n - R);
      ext[d] = own[-o * SLOT + OFF + pos];
    }
    {                                              // entry n + d
      const int o = (n + d) / n;
      const int loc = (n + d) - o * n;
      ext[R + n + d] = own[o * SLOT + OFF + loc];
    }
  }
#pragma unroll
  for (int q = 0; q < n; ++q) ext[R + q] = arr[q];
}

// The edges of every array of a lane's neighbours, fetched in one go (all the LDS reads of a row are in flight together
// and waited for once): v[A][0..R) the R entries to the left of the lane's array A, v[A][R..2R) the R to its right.
template <int K, int L>
struct RowEdges { float v[1 + 2 * L][2 * (K / 2) > 0 ? 2 * (K / 2) : 1]; };

template <int K, int S, int SLOT, int L, int A>
__device__ __forceinline__ void row1d_load_edges_from(const float* __restrict__ own, RowEdges<K, L>& ed) {
  if constexpr (A <= 2 * L) {
    constexpr int R = K / 2, n = row1d_len(S, A), OFF = row1d_edge_off(K, S, A);
#pragma unroll
    for (int d = 0; d < R; ++d) {
      {
        const int e = R - d, o = (e + n - 1) / n, loc = o * n - e;
        const int pos = n < 2 * R ? loc : R + loc - (n - R);
        ed.v[A][d] = own[-o * SLOT + OFF + pos];
      }
      {
        const int o = (n + d) / n, loc = (n + d) - o * n;
        ed.v[A][R + d] = own[o * SLOT + OFF + loc];
      }
    }
    row1d_load_edges_from<K, S, SLOT, L, A + 1>(own, ed);
  }
}

template <int K, int S, int SLOT, int L>
__device__ __forceinline__ void row1d_load_edges(const float* __restrict__ region, int tid, RowEdges<K, L>& ed) {
  row1d_load_edges_from<K, S, SLOT, L, 0>(region + tid * SLOT, ed);
}

// ext of array A from edges fetched earlier
template <int K, int S, int L, int A, int NA>
__device__ __forceinline__ void row1d_extend_with(const RowEdges<K, L>& ed, const float (&arr)[NA],
                                                  float (&ext)[row1d_len(S, A) + 2 * (K / 2)]) {
  constexpr int R = K / 2, n = row1d_len(S, A);
#pragma unroll
  for (int d = 0; d < R; ++d) { ext[d] = ed.v[A][d]; ext[R + n + d] = ed.v[A][R + d]; }
#pragma unroll
  for (int q = 0; q < n; ++q) ext[R + q] = arr[q];
}

// Folded parameters of one channel: entry f * K + k = gamma[f] * w[f][k] (k reversed when flip != 0), f = 0 base
// conv, f = 1 + 2 (l - 1) + s level l sub-band s.  The same products as fold_params_kernel forms.
template <int K, int L>
using RowWeights = LaneTable<(1 + 2 * L) * K>;

template <int K, int L>
__device__ __forceinline__ void row1d_fold(const ParamTable& p, int pdtype, int c, int flip, RowWeights<K, L>& tab) {
  tab.fill([&](int i) {
    const int f = i / K, t = i - f * K;
    const int ts = flip ? K - 1 - t : t;
    float v = 0.f;
    if (f == 0) v = load_param(p.base_weight, pdtype, c * K + ts) * load_param(p.base_scale, pdtype, c);
#pragma unroll
    for (int l = 0; l < L; ++l) {
      if (f >= 1 + 2 * l && f < 3 + 2 * l) {
        const int ch = c * 2 + (f - 1 - 2 * l);
        v = load_param(p.wt_weight[l], pdtype, ch * K + ts) * load_param(p.wt_scale[l], pdtype, ch) *
            (1.f / static_cast<float>(2 << l));          // 2^-(level): see "Scaling"
      }
    }
    return v;
  });
}

// y += (filter F of the channel) (*) ext
template <int K, int L, int F, int n>
__device__ __forceinline__ void row1d_conv(const float (&ext)[n + K - 1], const RowWeights<K, L>& w, float (&y)[n]) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float wv = w.get(F * K + k);
#pragma unroll
    for (int q = 0; q < n; ++q) y[q] = fmaf(wv, ext[q + k], y[q]);
  }
}

// Synthesis from level l (1-based) down to level 1: `zc` holds Z_{l+1} (n_l entries) on
// entry when l < L; the level-1 reconstruction is added into `out`.
template <int K, int S, int SLOT, int L, int l>
__device__ __forceinline__ void row1d_synth(const RowPyramid<S, L>& py, const float* __restrict__ region, int tid,
                                            int nth, const RowWeights<K, L>& fwc, float (&zc)[S / 2], float (&out)[S]) {
  if constexpr (l >= 1) {
    constexpr int R = K / 2;
    constexpr int n = S >> l;
    float ylo[n], yhi[n];
#pragma unroll
    for (int q = 0; q < n; ++q) { ylo[q] = l < L ? zc[q] : 0.f; yhi[q] = 0.f; }
    {
      float ext[n + 2 * R];
      row1d_extend<K, S, SLOT, 1 + 2 * (l - 1)>(region, tid, nth, py.lo[l - 1], ext);
      row1d_conv<K, L, 1 + 2 * (l - 1), n>(ext, fwc, ylo);
    }
    {
      float ext[n + 2 * R];
      row1d_extend<K, S, SLOT, 2 + 2 * (l - 1)>(region, tid, nth, py.hi[l - 1], ext);
      row1d_conv<K, L, 2 + 2 * (l - 1), n>(ext, fwc, yhi);
    }
    if constexpr (l > 1) {
#pragma unroll
      for (int q = 0; q < n; ++q) {
        zc[2 * q] = ylo[q] + yhi[q];       // ylo[q] was read from zc[q] before: q <= 2q
        zc[2 * q + 1] = ylo[q] - yhi[q];
      }
    } else {
#pragma unroll
      for (int q = 0; q < n; ++q) {
        out[2 * q] += ylo[q] + yhi[q];
        out[2 * q + 1] += ylo[q] - yhi[q];
      }
    }
    row1d_synth<K, S, SLOT, L, l - 1>(py, region, tid, nth, fwc, zc, out);
  }
}

// sum_q g[q] * ext[q + k] for the K taps of one filter
template <int K, int n, int NG>
__device__ __forceinline__ void row1d_corr(const float (&ext)[n + K - 1], const float (&g)[NG], float (&acc)[K]) {
#pragma unroll
  for (int q = 0; q < n; ++q)
#pragma unroll
    for (int k = 0; k < K; ++k) acc[k] = fmaf(g[q], ext[q + k], acc[k]);
}

// Levels l..L of the parameter-gradient sums; `gprev` = low-pass of grad_out at level l-1
// (2n entries), analysed one level at a time so that only one level of it is live.
template <int K, int S, int SLOT, int L, int l>
__device__ __forceinline__ void row1d_wgrad_levels(const RowPyramid<S, L>& py, const float* __restrict__ region,
                                                   int tid, int nth, const float (&gprev)[(S >> (l - 1))],
                                                   float (&acc)[1 + 2 * L][K]) {
  constexpr int R = K / 2;
  constexpr int n = S >> l;
  float glo[n], ghi[n];
#pragma unroll
  for (int q = 0; q < n; ++q) {
    glo[q] = gprev[2 * q] + gprev[2 * q + 1];
    ghi[q] = gprev[2 * q] - gprev[2 * q + 1];
  }
  {
    float ext[n + 2 * R];
    row1d_extend<K, S, SLOT, 1 + 2 * (l - 1)>(region, tid, nth, py.lo[l - 1], ext);
    row1d_corr<K, n>(ext, glo, acc[1 + 2 * (l - 1)]);
  }
  {
    float ext[n + 2 * R];
    row1d_extend<K, S, SLOT, 2 + 2 * (l - 1)>(region, tid, nth, py.hi[l - 1], ext);
    row1d_corr<K, n>(ext, ghi, acc[2 + 2 * (l - 1)]);
  }
  if constexpr (l < L) row1d_wgrad_levels<K, S, SLOT, L, l + 1>(py, region, tid, nth, glo, acc);
}

// The per-chunk record of a workgroup's running sums: cross-lane sums, then cross-wave through `red`
// ([waves][NRED] floats of LDS, idle by now), into partial[chunk][c][NF * K + 1].  The sums of lanes that are not `own` are
// left out here and not by a grad_out of zero: a sample in reach of them may be infinite.
template <int K, int NF, bool SHARED = false>
__device__ __forceinline__ void row1d_store_partial(const float (&acc)[NF][K], float gsum, bool own,
                                                    float* __restrict__ red, float* __restrict__ dst, int tid, int nth) {
  constexpr int NRED = NF * K + 1;
  const int wave = tid >> 6, lane = tid & (kWave - 1);
  float sums[(NRED + 3) / 4 * 4] = {};
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int k = 0; k < K; ++k)
      // the sums of level l were formed from coefficients 2^(l/2) times the orthonormal ones on either side
      sums[f * K + k] = (own ? acc[f][k] : 0.f) * (f == 0 ? 1.f : 1.f / static_cast<float>(2 << ((f - 1) / 2)));
  sums[NRED - 1] = own ? gsum : 0.f;
  wave_sums<(NRED + 3) / 4 * 4, NRED>(sums, lane, red + wave * NRED);
  WT_LDS_BARRIER();
  const int nwaves = nth >> 6;
  for (int o = tid; o < NRED; o += nth) {
    float v = 0.f;
    for (int wv = 0; wv < nwaves; ++wv) v += red[wv * NRED + o];
    if constexpr (SHARED) store_shared_f32(dst + o, v);
    else dst[o] = v;
  }
}

// Fused backward kernel, before the barrier: level l of a lane's pyramid from level l - 1 (`prev`), its edges
// published at once; only the low-pass of the current level stays live (the levels are formed again, one at a time,
// after the barrier: two operations per coefficient, against sixty registers for a whole pyramid).
template <int K, int S, int L, int l>
__device__ __forceinline__ void row1d_publish_chain(float* __restrict__ slot, const float (&prev)[(S >> (l - 1))]) {
  constexpr int n = S >> l;
  float lo[n], hi[n];
#pragma unroll
  for (int q = 0; q < n; ++q) {
    lo[q] = prev[2 * q] + prev[2 * q + 1];
    hi[q] = prev[2 * q] - prev[2 * q + 1];
  }
  row1d_publish<K, S, 1 + 2 * (l - 1)>(slot, lo);
  row1d_publish<K, S, 2 + 2 * (l - 1)>(slot, hi);
  if constexpr (l < L) row1d_publish_chain<K, S, L, l + 1>(slot, lo);
}

// Fused backward kernel, after the barrier: levels l..L of both halves of the backward pass, walking from the
// finest level down.  `xprev` / `gprev` = low-pass of x / grad_out at level l - 1.  Per level: the four coefficient
// arrays; the correlation sums of x's with grad_out's; the level's contribution to grad_x.  That contribution is
// added to the samples directly: the inverse transform is linear, and a reconstruction with zero detail below level
// l is the level-l result repeated 2^(l-1) times and scaled by 2^(-(l-1)/2), so the levels need not be visited
// coarsest first and no level's coefficients outlive its visit.
template <int K, int S, int SLOT, int L, int l>
__device__ __forceinline__ void row1d_bwd_levels(const float* __restrict__ xregion, const float* __restrict__ gregion,
                                                 int tid, int nth, const RowWeights<K, L>& fwc,
                                                 const float (&xprev)[(S >> (l - 1))],
                                                 const float (&gprev)[(S >> (l - 1))], float (&acc)[1 + 2 * L][K],
                                                 float (&o)[S]) {
  constexpr int R = K / 2;
  constexpr int n = S >> l;
  constexpr int A = 1 + 2 * (l - 1);
  float xlo[n], glo[n], ylo[n], yhi[n];
#pragma unroll
  for (int q = 0; q < n; ++q) { ylo[q] = 0.f; yhi[q] = 0.f; }
  {
    float xhi[n], ghi[n];
#pragma unroll
    for (int q = 0; q < n; ++q) {
      xlo[q] = xprev[2 * q] + xprev[2 * q + 1];
      xhi[q] = xprev[2 * q] - xprev[2 * q + 1];
      glo[q] = gprev[2 * q] + gprev[2 * q + 1];
      ghi[q] = gprev[2 * q] - gprev[2 * q + 1];
    }
    {
      float ext[n + 2 * R];
      row1d_extend<K, S, SLOT, A + 1>(xregion, tid, nth, xhi, ext);
      row1d_corr<K, n>(ext, ghi, acc[A + 1]);
    }
    {
      float ext[n + 2 * R];
      row1d_extend<K, S, SLOT, A + 1>(gregion, tid, nth, ghi, ext);
      row1d_conv<K, L, A + 1, n>(ext, fwc, yhi);
    }
    pin_values(yhi);
    WT_CHUNK_FENCE();      // (the edge reads of the next part stay below: one part's edges live at a time)
  }
  {
    float ext[n + 2 * R];
    row1d_extend<K, S, SLOT, A>(xregion, tid, nth, xlo, ext);
    row1d_corr<K, n>(ext, glo, acc[A]);
  }
  {
    float ext[n + 2 * R];
    row1d_extend<K, S, SLOT, A>(gregion, tid, nth, glo, ext);
    row1d_conv<K, L, A, n>(ext, fwc, ylo);
  }
  // (one inverse butterfly and l - 1 repeats: no factor left, see "Scaling" above)
  constexpr int REP = 1 << (l - 1);
#pragma unroll
  for (int q = 0; q < n; ++q) {
    const float ev = ylo[q] + yhi[q], od = ylo[q] - yhi[q];
#pragma unroll
    for (int r = 0; r < REP; ++r) {
      o[(2 * q) * REP + r] += ev;
      o[(2 * q + 1) * REP + r] += od;
    }
  }
  pin_values(o);
  WT_CHUNK_FENCE();
  if constexpr (l < L) row1d_bwd_levels<K, S, SLOT, L, l + 1>(xregion, gregion, tid, nth, fwc, xlo, glo, acc, o);
}

// The forward / input-gradient kernel's walk over the levels, finest first, on the same terms: per level the two
// coefficient arrays, their convolutions, and the level's contribution added to the samples directly.
template <int K, int S, int SLOT, int L, int l>
__device__ __forceinline__ void row1d_fwd_levels(const RowEdges<K, L>& ed, const RowWeights<K, L>& fwc,
                                                 const float (&xprev)[(S >> (l - 1))], float (&o)[S]) {
  constexpr int R = K / 2;
  constexpr int n = S >> l;
  constexpr int A = 1 + 2 * (l - 1);
  float xlo[n], ylo[n], yhi[n];
#pragma unroll
  for (int q = 0; q < n; ++q) { ylo[q] = 0.f; yhi[q] = 0.f; }
  {
    float xhi[n];
#pragma unroll
    for (int q = 0; q < n; ++q) {
      xlo[q] = xprev[2 * q] + xprev[2 * q + 1];
      xhi[q] = xprev[2 * q] - xprev[2 * q + 1];
    }
    float ext[n + 2 * R];
    row1d_extend_with<K, S, L, A + 1>(ed, xhi, ext);
    row1d_conv<K, L, A + 1, n>(ext, fwc, yhi);
  }
  {
    float ext[n + 2 * R];
    row1d_extend_with<K, S, L, A>(ed, xlo, ext);
    row1d_conv<K, L, A, n>(ext, fwc, ylo);
  }
  constexpr int REP = 1 << (l - 1);
#pragma unroll
  for (int q = 0; q < n; ++q) {
    const float ev = ylo[q] + yhi[q], od = ylo[q] - yhi[q];
#pragma unroll
    for (int r = 0; r < REP; ++r) {
      o[(2 * q) * REP + r] += ev;
      o[(2 * q + 1) * REP + r] += od;
    }
  }
  if constexpr (l < L) row1d_fwd_levels<K, S, SLOT, L, l + 1>(ed, fwc, xlo, o);
}

// Forward / input-gradient kernel.  grid = (channels, chunks of units), block = lanes (multiple of 64,
// >= Row1D::nl), dynamic LDS = one slot region (row1d_region floats).  A workgroup walks the units (segments of
// rows (b, c)) of its chunk; the next row is fetched into registers while the current one is computed and
// committed to the slots once the current outputs have left them.  One region instead of two alternating
// ones: half the LDS per workgroup, i.e. twice the workgroups per CU, which pays more here than the two
// barriers per row it costs.  flip != 0: the input gradient (taps reversed, no bias).
//
// Measured, forward us (training step us), tiles of 1024 samples in LDS (kernels1d.h) -> this kernel in segments:
// [8,48,20011] bfloat16, K = 7, five levels 46.3 -> 21.8 (172 -> 75); [8,16,39000] float32, K = 5, four levels
// 28.4 -> 9.5.  Short rows: [256,64,100] float32, three levels 37.1 -> 17.2, although a wave's lanes are mostly idle.
template <typename T, int K, int L, int S>
__global__ __launch_bounds__(kRow1dMaxLanes, 2) void wt1d_row_kernel(const T* __restrict__ x, T* __restrict__ out,
                                                                   const ParamTable prm, int pdtype, int flip,
                                                                   Row1D pl, int units, int per_chunk) {
  WT_SHARED_FLOATS(lds);
  constexpr int R = K / 2;
  constexpr int SLOT = row1d_slot(K, L, S);
  const int tid = threadIdx.x, nth = blockDim.x;
  const int c = blockIdx.x;
  const int u_begin = static_cast<int>(blockIdx.y) * per_chunk;
  const int u_end = u_begin + per_chunk < units ? u_begin + per_chunk : units;
  constexpr int G = row1d_guard(K, L, S);
  float* cur = lds + G * SLOT;                      // (the region points at the slot of lane 0, behind its left guard)
  row1d_zero_guards<K, L, S>(lds, 1, tid, nth);

  RowFetch<T, S> rf;
  RowUnit at(u_begin, pl);
  if (u_begin < u_end) rf.fetch(at.row(x, pl, c), at.first(pl, S), pl.N, tid, nth);
  RowWeights<K, L> fwc;                 // (its parameter loads share the latency of the first row's)
  row1d_fold<K, L>(prm, pdtype, c, flip, fwc);
  const float bias = (!flip && prm.base_bias != nullptr)
                         ? load_param(prm.base_bias, pdtype, c) * load_param(prm.base_scale, pdtype, c) : 0.f;
  if (u_begin < u_end) rf.template commit<SLOT>(cur, at.first(pl, S), pl.N, pl.nl, tid, nth);
  WT_LDS_BARRIER();
  for (int u = u_begin; u < u_end; ++u) {
    const bool more = u + 1 < u_end;
    RowUnit nx = at;
    nx.next(pl);
    float* slot = cur + tid * SLOT;
    float xs[S];
    if (tid < pl.nl) {
      row1d_read_slot<S>(slot, xs);
    } else {
#pragma unroll
      for (int e = 0; e < S; ++e) xs[e] = 0.f;
    }
    if (more) rf.fetch(nx.row(x, pl, c), nx.first(pl, S), pl.N, tid, nth);
    // the slot held this lane's samples only: it can take the lane's edges right away
    row1d_publish<K, S, 0>(slot, xs);
    row1d_publish_chain<K, S, L, 1>(slot, xs);
    WT_LDS_BARRIER();
    pin_values(xs);              // (the levels are formed again below, one at a time, not kept across the barrier)

    RowEdges<K, L> ed;
    row1d_load_edges<K, S, SLOT, L>(cur, tid, ed);
    float o[S];
    {
#pragma unroll
      for (int e = 0; e < S; ++e) o[e] = bias;
      float ext[S + 2 * R];
      row1d_extend_with<K, S, L, 0>(ed, xs, ext);
      row1d_conv<K, L, 0, S>(ext, fwc, o);
    }
    row1d_fwd_levels<K, S, SLOT, L, 1>(ed, fwc, xs, o);
    WT_LDS_BARRIER();            // every neighbour has read this lane's edges
    row1d_write_slot<S>(slot, o);
    WT_LDS_BARRIER();
    row1d_unstage<T, S, SLOT>(at.row(out, pl, c), cur, at.first(pl, S), pl, tid, nth);
    WT_LDS_BARRIER();            // the outputs have left the slots
    if (more) rf.template commit<SLOT>(cur, nx.first(pl, S), pl.N, pl.nl, tid, nth);
    at = nx;
    WT_LDS_BARRIER();
  }
}

// Parameter gradients, first stage.  grid = (C, nchunk), block = lanes, dynamic LDS =
// 2 * block * SLOT floats (x slots, then grad_out slots).  A workgroup walks `per_chunk` units
// of one channel; every lane keeps K sums per filter in registers.  Output layout as the
// tiled kernel: partial[chunk][c][(1 + 2L) * K + 1].
template <typename T, int K, int L, int S>
__global__ __launch_bounds__(kRow1dMaxLanes, 2) void wt1d_row_wgrad_kernel(const T* __restrict__ x,
                                                                         const T* __restrict__ g,
                                                                         float* __restrict__ partial, Row1D pl,
                                                                         int units, int per_chunk) {
  WT_SHARED_FLOATS(lds);
  constexpr int R = K / 2;
  constexpr int SLOT = row1d_slot(K, L, S);
  constexpr int NF = 1 + 2 * L;
  const int c = blockIdx.x;
  const int chunk = blockIdx.y;
  const int tid = threadIdx.x, nth = blockDim.x;
  constexpr int G = row1d_guard(K, L, S);
  float* xlds = lds + G * SLOT;                     // (regions point at the slot of lane 0, behind their left guard)
  float* glds = xlds + (nth + 2 * G) * SLOT;
  float* slot = xlds + tid * SLOT;
  const float* gslot = glds + tid * SLOT;
  row1d_zero_guards<K, L, S>(lds, 2, tid, nth);

  float acc[NF][K];
  float gsum = 0.f;
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int k = 0; k < K; ++k) acc[f][k] = 0.f;

  const int u_end = (chunk + 1) * per_chunk < units ? (chunk + 1) * per_chunk : units;
  RowUnit at(chunk * per_chunk, pl);
  for (int u = chunk * per_chunk; u < u_end; ++u, at.next(pl)) {
    row1d_stage_pair<T, S, SLOT>(at.row(x, pl, c), at.row(g, pl, c), xlds, glds, at.first(pl, S), pl.N, pl.nl, tid, nth);
    WT_LDS_BARRIER();
    float xs[S], gs[S];
#pragma unroll
    for (int q = 0; q < S; ++q) { xs[q] = 0.f; gs[q] = 0.f; }
    if (tid < pl.nl) {
      row1d_read_slot<S>(slot, xs);
      row1d_read_slot<S>(gslot, gs);
    }
    RowPyramid<S, L> py;
    row1d_analysis<S, L>(xs, py);
    row1d_publish<K, S, 0>(slot, xs);
    row1d_publish_levels<K, S, L, 1>(slot, py);
    WT_LDS_BARRIER();
    {
      float ext[S + 2 * R];
      row1d_extend<K, S, SLOT, 0>(xlds, tid, nth, xs, ext);
      row1d_corr<K, S>(ext, gs, acc[0]);
#pragma unroll
      for (int q = 0; q < S; ++q) gsum += gs[q];
    }
    row1d_wgrad_levels<K, S, SLOT, L, 1>(py, xlds, tid, nth, gs, acc);
    WT_LDS_BARRIER();            // the next row's staging overwrites the edges read above
  }

  constexpr int NRED = NF * K + 1;
  row1d_store_partial<K, NF>(acc, gsum, pl.own(tid), lds, partial + (static_cast<size_t>(chunk) * pl.C + c) * NRED, tid, nth);
}

// (K, L) pairs the fused backward kernel is built for: its (1 + 2L) * K + 1 running sums per lane must leave room for
// the rest in 256 registers (beyond 50 sums, 45 with 32 samples per lane, the compiler spills; those pairs run the
// backward pass as two kernels).
constexpr bool row1d_bwd_built(int K, int L, int S) {
  return row1d_built(K, L, S) && (1 + 2 * L) * K <= (S == 16 ? 50 : 45);
}

// The whole backward pass of a row-resident shape in one kernel.  grid = (C, nchunk), block = lanes, dynamic LDS =
// 2 * block * SLOT floats (x slots, then grad_out slots, which also stage grad_x on its way out).  Per row: x and
// grad_out are read once; grad_x = the layer applied to grad_out with reversed taps and no bias; the correlation
// sums of x's pyramid with grad_out's go into (1 + 2L) * K + 1 running sums per lane.  After its rows a workgroup
// stores its record of sums and draws its channel's ticket; the last one of a channel runs the second stage
// (wgrad_finish_channel) for it and leaves the ticket zero.  `tickets`: C words, zero at launch.
template <typename T, int K, int L, int S>
__global__ __launch_bounds__(kRow1dMaxLanes, 2) void wt1d_row_bwd_kernel(const T* __restrict__ x,
                                                                          const T* __restrict__ g,
                                                                          T* __restrict__ gx,
                                                                          float* __restrict__ partial,
                                                                          unsigned* __restrict__ tickets,
                                                                          const ParamTable prm, int pdtype,
                                                                          const GradTable gt, Row1D pl, int units,
                                                                          int per_chunk, int nchunk) {
  WT_SHARED_FLOATS(lds);
  constexpr int R = K / 2;
  constexpr int SLOT = row1d_slot(K, L, S);
  constexpr int NF = 1 + 2 * L;
  const int c = blockIdx.x;
  const int chunk = blockIdx.y;
  const int tid = threadIdx.x, nth = blockDim.x;
  constexpr int G = row1d_guard(K, L, S);
  float* xlds = lds + G * SLOT;                     // (regions point at the slot of lane 0, behind their left guard)
  float* glds = xlds + (nth + 2 * G) * SLOT;
  float* xslot = xlds + tid * SLOT;
  float* gslot = glds + tid * SLOT;
  row1d_zero_guards<K, L, S>(lds, 2, tid, nth);

  RowWeights<K, L> fwc;
  row1d_fold<K, L>(prm, pdtype, c, 1, fwc);

  float acc[NF][K];
  float gsum = 0.f;
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int k = 0; k < K; ++k) acc[f][k] = 0.f;

  const int u_first = chunk * per_chunk;
  const int u_end = u_first + per_chunk < units ? u_first + per_chunk : units;
  // with 16 samples per lane, the rows are fetched one unit ahead into registers; with 32 the registers for that are
  // not there, and they are staged as the loop reaches them
  constexpr bool kAhead = S <= 16;
  RowFetch<T, kAhead ? S : 8> rx, rg;
  RowUnit at(u_first, pl);
  if constexpr (kAhead) {
    if (u_first < u_end) {
      const int p0 = at.first(pl, S);
      rx.template fetch<true>(at.row(x, pl, c), p0, pl.N, tid, nth);
      rg.template fetch<true>(at.row(g, pl, c), p0, pl.N, tid, nth);
      rx.template commit<SLOT>(xlds, p0, pl.N, pl.nl, tid, nth);
      rg.template commit<SLOT>(glds, p0, pl.N, pl.nl, tid, nth);
    }
  }
  for (int u = u_first; u < u_end; ++u) {
    const bool more = u + 1 < u_end;
    RowUnit nx = at;
    nx.next(pl);
    if constexpr (!kAhead)
      row1d_stage_pair<T, S, SLOT>(at.row(x, pl, c), at.row(g, pl, c), xlds, glds, at.first(pl, S), pl.N, pl.nl, tid, nth);
    WT_LDS_BARRIER();
    float xs[S], gs[S];
    if (tid < pl.nl) {
      row1d_read_slot<S>(xslot, xs);
      row1d_read_slot<S>(gslot, gs);
    } else {
#pragma unroll
      for (int q = 0; q < S; ++q) { xs[q] = 0.f; gs[q] = 0.f; }
    }
    if constexpr (kAhead) {
      if (more) {
        rx.template fetch<true>(nx.row(x, pl, c), nx.first(pl, S), pl.N, tid, nth);
        rg.template fetch<true>(nx.row(g, pl, c), nx.first(pl, S), pl.N, tid, nth);
      }
    }
    row1d_publish<K, S, 0>(xslot, xs);
    row1d_publish<K, S, 0>(gslot, gs);
    row1d_publish_chain<K, S, L, 1>(xslot, xs);
    row1d_publish_chain<K, S, L, 1>(gslot, gs);
    WT_LDS_BARRIER();
    // (opaque from here on: otherwise the compiler keeps the coefficients it formed for the edges above alive across
    // the barrier instead of forming them again level by level)
    pin_values(xs);
    pin_values(gs);
    // base conv: its correlation sums, and its share of grad_x (the layer on grad_out with the reversed taps)
    float o[S];
#pragma unroll
    for (int e = 0; e < S; ++e) o[e] = 0.f;
    {
      float ext[S + 2 * R];
      row1d_extend<K, S, SLOT, 0>(xlds, tid, nth, xs, ext);
      row1d_corr<K, S>(ext, gs, acc[0]);
#pragma unroll
      for (int q = 0; q < S; ++q) gsum += gs[q];
    }
    {
      float ext[S + 2 * R];
      row1d_extend<K, S, SLOT, 0>(glds, tid, nth, gs, ext);
      row1d_conv<K, L, 0, S>(ext, fwc, o);
    }
    pin_values(o);
    WT_CHUNK_FENCE();
    row1d_bwd_levels<K, S, SLOT, L, 1>(xlds, glds, tid, nth, fwc, xs, gs, acc, o);
    WT_LDS_BARRIER();            // every neighbour has read this lane's edges
    row1d_write_slot<S>(gslot, o);
    WT_LDS_BARRIER();
    row1d_unstage<T, S, SLOT>(at.row(gx, pl, c), glds, at.first(pl, S), pl, tid, nth);
    WT_LDS_BARRIER();            // the next unit's staging overwrites the slots read above
    if constexpr (kAhead) {
      if (more) {
        rx.template commit<SLOT>(xlds, nx.first(pl, S), pl.N, pl.nl, tid, nth);
        rg.template commit<SLOT>(glds, nx.first(pl, S), pl.N, pl.nl, tid, nth);
      }
    }
    at = nx;
  }

  constexpr int NRED = NF * K + 1;
  row1d_store_partial<K, NF, true>(acc, gsum, pl.own(tid), lds, partial + (static_cast<size_t>(chunk) * pl.C + c) * NRED, tid, nth);
  unsigned* flag = reinterpret_cast<unsigned*>(lds + (nth >> 6) * NRED);
  if (workgroup_is_last(tickets + c, static_cast<unsigned>(nchunk), flag)) {
    wgrad_finish_channel<true>(partial, nchunk, prm, pdtype, gt, pl.C, c, 2, L, K, lds);
    if (tid == 0) tickets[c] = 0u;
  }
}

}  // namespace wt
