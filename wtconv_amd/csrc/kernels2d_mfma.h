// WTConv2d on the matrix cores of gfx950: plane-resident kernel for kernel sizes up to 5.
//
// Same layer maths as kernels2d.h (reference wtconv/wtconv2d.py:38-82), different arithmetic:
// every depthwise K x K convolution of the layer (base conv and the four sub-bands of every
// level) runs as v_mfma_f32_16x16x32_bf16 products.  A 4 x 4 block of outputs depends on an
// 8 x 8 patch of inputs (K <= 5), so for 16 blocks of one filter
//     D[16 outputs of a block][16 blocks] = Wt[16 outputs][64 patch elements] * Patch[64][16 blocks]
// is two MFMAs (patch rows 0-3 and 4-7).  Wt is the filter laid out as a Toeplitz matrix
// (39 % non-zero), kept in the compact form that the lanes pick their
// fragment from.  Lane (n = lane % 16, q = lane / 16) supplies row q (+4) of block n's patch
// -- 8 consecutive bf16 of an LDS row -- and receives four outputs of block n: its row q at the coarse levels, a square or
// a lattice of it in the pixels and at level 1 (see the kernel).
//
// What bounds it: LDS (busy 63 % of a 56 x 56 launch, 24 % on bank conflicts), vector code (44 %: commit with two levels of
// analysis, synthesis) and the two barriers of a unit, at four waves a SIMD for want of registers (the constant plans spill one to
// four of 128, the run-time plan more); the matrix cores are busy an eighth of the time.  us per launch, before level 1 and base
// convolution met in registers (with the base convolution through LDS as fp32, levels 3 and up behind a barrier each and one table
// entry a lane in the fold) -> now: [128,96,56,56], three levels 56.5 -> 49.6; [256,96,56,56], five 161 -> 141; [128,192,28,28]
// 36.1 -> 31.7; [256,384,14,14] 47.3 -> 36.6; [128,768,7,7] 21.3 -> 15.5; a single image of 14 x 14 x 384 12.0 -> 7.2;
// 250 drawn shapes 0.87 at the geometric mean, from 0.64 to 1.06 (two over 1.05: single images of few channels and two levels,
// 8.5 -> 9.0; [34,36], whose fifteen block rows make eight tiles for four waves, 20.9 -> 21.2).
//
// Activations live in LDS as bf16 planes with a zero halo of 2.  bf16 tensors take one plane
// per buffer (NS = 1).  fp32 tensors are split into NS = 3 bf16 planes (v = h0 + h1 + h2
// exactly, 24 mantissa bits) and the folded weights likewise; the six products of total
// order <= 2 are accumulated in fp32, which leaves an error below that of an fp32 FMA chain.
// The Haar butterflies run unnormalised in fp32 (the factors 1/2 of analysis and synthesis
// are folded into the weights as 4^-level), coefficients are rounded (or split) to bf16 when
// they are written to LDS, accumulators, the partial reconstructions Z_l and the raw LL chain
// stay fp32.
#pragma once

#include "common.h"

namespace wt {

constexpr int kFragEntries = 21;     // 5 kernel rows x 4 column shifts, then one all-zero entry
constexpr int kTapRow = 12;          // elements of a filter row with the zeros around it
constexpr int kMfmaBlock = 256;
constexpr int kDivShift = 20;        // magic reciprocals: exact for dividends < 4096, divisors <= 256

struct MPlan {
  int B, C, H, W, L;
  int pb, upc, nunits;               // planes (one channel, consecutive batch items) per unit; units per channel; total
  int bq, br;                        // B = upc * bq + br: the first br units of a channel take bq + 1 batch items, the rest bq
  int nfilt;                         // 1 + 4 L
  int h[kMaxLevels + 1], w[kMaxLevels + 1];        // extent of level l (0 = pixels)
  int nbr[kMaxLevels + 1], nbc[kMaxLevels + 1];    // 4x4 blocks per plane: rows, columns
  int bpp[kMaxLevels + 1], nblk[kMaxLevels + 1];   // blocks per plane, per unit
  unsigned mg_bpp0, mg_nbc0;                                 // reciprocals of bpp[0], nbc[0]
  unsigned mg_hw[kMaxLevels + 1], mg_w[kMaxLevels + 1];      // reciprocals of h*w, w
  // MFMA tiles: 16 blocks = TR block-rows x TC block-columns, TC = 2^tcs >= nbc; the block-rows of
  // the stacked planes of a unit are numbered R = p * nbr + bi
  int tcs[kMaxLevels + 1], nrow[kMaxLevels + 1], ntile[kMaxLevels + 1];
  int rtoff[kMaxLevels + 1];         // byte offset of the block-row table of level l >= 1
  int pitch[kMaxLevels + 1];         // LDS row pitch of a level-l plane in bf16 elements (multiple of 4)
  int prows[kMaxLevels + 1];         // LDS rows from one stacked plane to the next: 4 nbr + 2
  int aoff[kMaxLevels + 1];          // byte offset of (slot 0, row -2, column -2) of sub-band 0, split 0
  int asub[kMaxLevels + 1];          // bytes from one plane stack to the next (sub-bands, then splits)
  int zoff[kMaxLevels + 2], zpitch[kMaxLevels + 2], zpl[kMaxLevels + 2];   // fp32 Z_l, l = 2..L
  int lloff[kMaxLevels + 1], llpl[kMaxLevels + 1];                         // fp32 raw LL of level l, 2 <= l < L
  int toff;                          // byte offset of the fragment table of the current channel: the base filter, then
  int tskip;                         // the others but this many (those of level 1, where they live in registers)
  int taps, tap_rows;                // byte offset of the folded filters as rows of taps; rows, the last one of zeros
  int behind;                        // planes that hold what the last rows' loads take along: (4 nbr - H) W + 3 elements
  int uq, ur;                        // units of a workgroup: uq, ur of them one more
  int lds_bytes;
};

// ------------------------------------------------------------------------------ planning
// Reciprocal for fast_div(): exact for every dividend in [0, maxv], or the shape is refused.
constexpr bool make_magic(int d, int maxv, unsigned* magic) {
  if (d < 1 || maxv >= 4096) return false;
  const unsigned m = ((1u << kDivShift) + d - 1) / d;
  if (m >= (1u << 24)) return false;
  for (int v = 0; v <= maxv; ++v)
    if (static_cast<int>((static_cast<unsigned long long>(v) * m) >> kDivShift) != v / d) return false;
  *magic = m;
  return true;
}

// Everything of a plan that depends on the plane shape, the levels, the split count and the
// planes per unit only (not on batch or channels); false if the kernel cannot index the shape.
// constexpr: the kernels of the common shapes take it as a compile-time constant.
constexpr bool make_mplan_geometry(int H, int W, int L, int NS, int pb, MPlan* out) {
  auto cdiv = [](int a, int b) { return (a + b - 1) / b; };
  auto rup = [](int v, int m) { return (v + m - 1) / m * m; };
  MPlan pl = {};
  pl.H = H; pl.W = W; pl.L = L;
  pl.pb = pb;
  pl.nfilt = 1 + 4 * L;
  pl.h[0] = H; pl.w[0] = W;
  for (int l = 1; l <= L; ++l) { pl.h[l] = (pl.h[l - 1] + 1) / 2; pl.w[l] = (pl.w[l - 1] + 1) / 2; }
  int off = 0;
  pl.toff = off;
  pl.tskip = NS == 1 ? 4 : 0;        // one split plane: level 1 stays in registers
  off += NS * (pl.nfilt - pl.tskip) * kFragEntries * 16;
  for (int l = 0; l <= L; ++l) {
    pl.nbr[l] = cdiv(pl.h[l], 4);
    pl.nbc[l] = cdiv(pl.w[l], 4);
    pl.bpp[l] = pl.nbr[l] * pl.nbc[l];
    pl.nblk[l] = pb * pl.bpp[l];
    pl.pitch[l] = 4 * pl.nbc[l] + 4;
    pl.prows[l] = 4 * pl.nbr[l] + 2;
    if (l == 0) {
      if (!make_magic(pl.bpp[0], pl.nblk[0] + kMfmaBlock * 4, &pl.mg_bpp0)) return false;
      if (!make_magic(pl.nbc[0], pl.bpp[0], &pl.mg_nbc0)) return false;
    }
    pl.tcs[l] = 0;
    while ((1 << pl.tcs[l]) < pl.nbc[l]) ++pl.tcs[l];
    if (pl.tcs[l] > 4) return false;                 // planes wider than 64 are not tiled
    pl.nrow[l] = pb * pl.nbr[l];
    pl.ntile[l] = cdiv(pl.nrow[l], 16 >> pl.tcs[l]);
    if (pb * pl.prows[l] + 8 >= 4096 || pb > 255 || pl.nbr[l] >= 4096) return false;   // block-row table fields
    if (l >= 3) {
      if (!make_magic(pl.h[l] * pl.w[l], pb * pl.h[l] * pl.w[l] + kMfmaBlock, &pl.mg_hw[l])) return false;
      if (!make_magic(pl.w[l], pl.h[l] * pl.w[l], &pl.mg_w[l])) return false;
    }
    pl.aoff[l] = off;
    pl.asub[l] = rup((pb * pl.prows[l] + 2) * pl.pitch[l] * 2, 16);
    off += pl.asub[l] * NS * (l == 0 ? 1 : 4);
    if (off > (1 << 20)) return false;
  }
  pl.behind = cdiv((4 * pl.nbr[0] - H) * W + 3, H * W);
  pl.tap_rows = NS * pl.nfilt * 5 + 1;
  pl.taps = off;
  off += rup(pl.tap_rows * kTapRow * 2 + 4, 16);
  for (int l = 2; l <= L; ++l) {
    pl.zpitch[l] = 4 * pl.nbc[l - 1];
    pl.zpl[l] = 4 * pl.nbr[l - 1] * pl.zpitch[l];
    pl.zoff[l] = off;
    off += pb * pl.zpl[l] * 4;
    if (off > (1 << 20)) return false;
  }
  for (int l = 2; l < L; ++l) {
    pl.llpl[l] = pl.h[l] * pl.w[l];
    pl.lloff[l] = off;
    off += rup(pb * pl.llpl[l] * 4, 16);
  }
  for (int l = 1; l <= L; ++l) {
    pl.rtoff[l] = off;
    off += rup(pl.nrow[l] * 4, 16);
  }
  off += 256;      // lanes beyond a plane's last block column read a few elements past its rows
  pl.lds_bytes = rup(off, 16);
  *out = pl;
  return true;
}

// Where a kernel takes the shape-dependent part of its plan from: the kernel argument, or a
// compile-time constant (every LDS offset then folds into the instructions).
struct GeoRuntime {
  static constexpr bool kStatic = false;
  static constexpr int kL = 0;
};
template <int H, int W, int L, int PB>
struct GeoStatic {
  static constexpr bool kStatic = true;
  static constexpr int kL = L;
  template <int NS> static constexpr MPlan plan() {
    MPlan p = {};
    make_mplan_geometry(H, W, L, NS, PB, &p);
    return p;
  }
};

// f(l) for l = LO..L (upwards) / L..LO (downwards).  With a static geometry the calls are
// separate instantiations with a constant level, so that every per-level plan field folds; a
// level that is only known at run time would force the constant plan into scratch memory.
template <typename Geo, int LO, typename F>
__device__ __forceinline__ void levels_up(int L, F&& f) {
  if constexpr (Geo::kStatic) {
    using std::integral_constant;
    if constexpr (LO <= 0) f(integral_constant<int, 0>{});
    if constexpr (LO <= 1 && Geo::kL >= 1) f(integral_constant<int, 1>{});
    if constexpr (LO <= 2 && Geo::kL >= 2) f(integral_constant<int, 2>{});
    if constexpr (LO <= 3 && Geo::kL >= 3) f(integral_constant<int, 3>{});
    if constexpr (LO <= 4 && Geo::kL >= 4) f(integral_constant<int, 4>{});
    if constexpr (LO <= 5 && Geo::kL >= 5) f(integral_constant<int, 5>{});
  } else {
#pragma unroll 1
    for (int l = LO; l <= L; ++l) f(l);
  }
}
template <typename Geo, int LO, typename F>
__device__ __forceinline__ void levels_down(int L, F&& f) {
  if constexpr (Geo::kStatic) {
    using std::integral_constant;
    if constexpr (LO <= 5 && Geo::kL >= 5) f(integral_constant<int, 5>{});
    if constexpr (LO <= 4 && Geo::kL >= 4) f(integral_constant<int, 4>{});
    if constexpr (LO <= 3 && Geo::kL >= 3) f(integral_constant<int, 3>{});
    if constexpr (LO <= 2 && Geo::kL >= 2) f(integral_constant<int, 2>{});
    if constexpr (LO <= 1 && Geo::kL >= 1) f(integral_constant<int, 1>{});
  } else {
#pragma unroll 1
    for (int l = L; l >= LO; --l) f(l);
  }
}

// -------------------------------------------------------------------------------- helpers
struct Frag { uint32_t d[4]; };      // 8 bf16
struct Acc { float v[4]; };

__device__ __forceinline__ void mfma_bf16(const Frag& a, const Frag& b, Acc& c) {
#ifdef WT_EMULATE
  uint16_t ua[8], ub[8];
  for (int i = 0; i < 4; ++i) {
    ua[2 * i] = static_cast<uint16_t>(a.d[i]); ua[2 * i + 1] = static_cast<uint16_t>(a.d[i] >> 16);
    ub[2 * i] = static_cast<uint16_t>(b.d[i]); ub[2 * i + 1] = static_cast<uint16_t>(b.d[i] >> 16);
  }
  ::emu::mfma_16x16x32_bf16(ua, ub, c.v);
#else
  typedef __bf16 wt_bf16x8 __attribute__((ext_vector_type(8)));
  typedef float wt_f32x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t wt_u32x4 __attribute__((ext_vector_type(4)));
  const wt_u32x4 au = {a.d[0], a.d[1], a.d[2], a.d[3]}, bu = {b.d[0], b.d[1], b.d[2], b.d[3]};
  wt_f32x4 cv = {c.v[0], c.v[1], c.v[2], c.v[3]};
  cv = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(wt_bf16x8, au), __builtin_bit_cast(wt_bf16x8, bu),
                                               cv, 0, 0, 0);
  c.v[0] = cv[0]; c.v[1] = cv[1]; c.v[2] = cv[2]; c.v[3] = cv[3];
#endif
}

// Orders the LDS traffic of one wave inside code that only some waves of the workgroup run.
#ifdef WT_EMULATE
#define WT_WAVE_SYNC_DIVERGENT() ::emu::wave_barrier()
#else
#define WT_WAVE_SYNC_DIVERGENT() WT_WAVE_LDS_SYNC()
#endif

template <typename V> __device__ __forceinline__ V lds_ld(const char* lds, int off) {
  return *reinterpret_cast<const V*>(lds + off);
}
template <typename V> __device__ __forceinline__ void lds_st(char* lds, int off, V v) {
  *reinterpret_cast<V*>(lds + off) = v;
}

// 8 consecutive bf16 at an 8-byte aligned LDS offset
__device__ __forceinline__ Frag lds_frag8(const char* lds, int off) {
  const uint2 lo = lds_ld<uint2>(lds, off), hi = lds_ld<uint2>(lds, off + 8);
  Frag f; f.d[0] = lo.x; f.d[1] = lo.y; f.d[2] = hi.x; f.d[3] = hi.y;
  return f;
}
// ... at a 16-byte aligned offset (fragment table)
__device__ __forceinline__ Frag lds_frag16(const char* lds, int off) {
  const uint4 v = lds_ld<uint4>(lds, off);
  Frag f; f.d[0] = v.x; f.d[1] = v.y; f.d[2] = v.z; f.d[3] = v.w;
  return f;
}

__device__ __forceinline__ int fast_div(int v, unsigned magic) {
#ifdef WT_EMULATE
  return static_cast<int>((static_cast<uint64_t>(static_cast<unsigned>(v)) * magic) >> kDivShift);
#else
  return static_cast<int>(__umul24(static_cast<unsigned>(v), magic) >> kDivShift);
#endif
}

// Two floats -> NS words of two bf16 each whose sum is the pair (exactly, for NS = 3).
template <int NS>
__device__ __forceinline__ void split_pair(float lo, float hi, uint32_t (&w)[NS]) {
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    w[j] = pack_bf16x2(lo, hi);
    if (j + 1 < NS) {
      lo -= __uint_as_float(w[j] << 16);
      hi -= __uint_as_float(w[j] & 0xffff0000u);
    }
  }
}

// ------------------------------------------------------------------ pixel blocks in registers
template <typename T> struct PixRow;
template <> struct PixRow<float> { float4 v; };
template <> struct PixRow<bf16_t> { uint2 v; };
// Rows of bf16 planes that are not whole aligned vectors still move as one 8-byte access per row of a block: global
// memory takes unaligned accesses (the compiler itself emits one dwordx2 for an 8-byte copy from a 2-byte aligned
// address).  Columns past the row end come along and are cleared before use; nothing is computed on the loaded
// words before the commit, so all the loads of a block stay in flight.
__device__ __forceinline__ void pix_load4u(uint2& v, const bf16_t* p) { __builtin_memcpy(&v, p, 8); }
// words that keep the valid columns of a block row: bits 4..7 of `cmask` say which of its four columns exist
__device__ __forceinline__ uint2 pix_col_mask(unsigned cmask) {
  uint2 m;
  m.x = ((cmask & 16u) ? 0x0000ffffu : 0u) | ((cmask & 32u) ? 0xffff0000u : 0u);
  m.y = ((cmask & 64u) ? 0x0000ffffu : 0u) | ((cmask & 128u) ? 0xffff0000u : 0u);
  return m;
}

__device__ __forceinline__ void pix_zero(PixRow<float>& r) { r.v.x = r.v.y = r.v.z = r.v.w = 0.f; }
__device__ __forceinline__ void pix_zero(PixRow<bf16_t>& r) { r.v.x = r.v.y = 0u; }
__device__ __forceinline__ void pix_load4(PixRow<float>& r, const float* p) { r.v = *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ void pix_load4(PixRow<bf16_t>& r, const bf16_t* p) { r.v = *reinterpret_cast<const uint2*>(p); }
__device__ __forceinline__ void pix_set(PixRow<float>& r, int i, float v) {
  if (i == 0) r.v.x = v; else if (i == 1) r.v.y = v; else if (i == 2) r.v.z = v; else r.v.w = v;
}
__device__ __forceinline__ void pix_set(PixRow<bf16_t>& r, int i, bf16_t v) {
  const uint32_t u = static_cast<uint32_t>(v) << ((i & 1) * 16);
  if (i < 2) r.v.x |= u; else r.v.y |= u;
}
// the four bf16 of a row as two packed words
__device__ __forceinline__ uint2 pix_words(const PixRow<bf16_t>& r) { return r.v; }
__device__ __forceinline__ uint2 pix_words(const PixRow<float>&) { uint2 w; w.x = w.y = 0u; return w; }   // (never taken)
__device__ __forceinline__ void pix_get(const PixRow<float>& r, float (&f)[4]) {
  f[0] = r.v.x; f[1] = r.v.y; f[2] = r.v.z; f[3] = r.v.w;
}
__device__ __forceinline__ void pix_get(const PixRow<bf16_t>& r, float (&f)[4]) {
  f[0] = __uint_as_float(r.v.x << 16); f[1] = __uint_as_float(r.v.x & 0xffff0000u);
  f[2] = __uint_as_float(r.v.y << 16); f[3] = __uint_as_float(r.v.y & 0xffff0000u);
}

// Block-row table entry: LDS row of the block-row's first patch row | plane slot << 12 | block-row in the plane << 20.
__device__ __forceinline__ unsigned rowtab_entry(int rowidx, int p, int bi) {
  return static_cast<unsigned>(rowidx) | (static_cast<unsigned>(p) << 12) | (static_cast<unsigned>(bi) << 20);
}

template <int NS>
__device__ __forceinline__ void load_b(const char* lds, int boff, int bsplit, int row4, Frag (&bt)[NS], Frag (&bb)[NS]) {
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    bt[j] = lds_frag8(lds, boff + j * bsplit);
    bb[j] = lds_frag8(lds, boff + j * bsplit + row4);
  }
}

// Toeplitz fragments of one filter: `tab` = byte offset of the filter's table in split 0.
template <int NS>
__device__ __forceinline__ void load_a(const char* lds, int tab, int tsplit, int ent_top, int ent_bot,
                                       Frag (&at)[NS], Frag (&ab)[NS]) {
#pragma unroll
  for (int j = 0; j < NS; ++j) {
    at[j] = lds_frag16(lds, tab + j * tsplit + ent_top * 16);
    ab[j] = lds_frag16(lds, tab + j * tsplit + ent_bot * 16);
  }
}

// acc += Wt * Patch over both patch halves: all split products of total order < NS, smallest terms first.
template <int NS>
__device__ __forceinline__ void mma_tile(const Frag (&at)[NS], const Frag (&ab)[NS], const Frag (&bt)[NS],
                                         const Frag (&bb)[NS], Acc& acc) {
#pragma unroll
  for (int order = NS - 1; order >= 0; --order)
#pragma unroll
    for (int js = 0; js <= order; ++js) {
      const int jw = order - js;
      mfma_bf16(at[jw], bt[js], acc);
      mfma_bf16(ab[jw], bb[js], acc);
    }
}

// Inverse Haar butterfly (unnormalised) of four coefficients per sub-band: two rows of 8.
__device__ __forceinline__ void synth_rows(const Acc (&a)[4], float (&top)[8], float (&bot)[8]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float s1 = a[0].v[j] + a[1].v[j], d1 = a[0].v[j] - a[1].v[j];
    const float s2 = a[2].v[j] + a[3].v[j], d2 = a[2].v[j] - a[3].v[j];
    top[2 * j] = s1 + s2; top[2 * j + 1] = s1 - s2;
    bot[2 * j] = d1 + d2; bot[2 * j + 1] = d1 - d2;
  }
}

// Lane's share of tile T at one level: which block (plane slot p, block-row bi, block-column tc)
// and where its patch row q starts.
struct TileLane {
  int boff, p, bi, tc;
  bool valid;
};
__device__ __forceinline__ TileLane tile_lane(const char* lds, int T, int n, int q, int tcs, int nrow, int nbc,
                                              int rtoff, int aoff, int pitch_bytes) {
  TileLane t;
  t.tc = n & ((1 << tcs) - 1);
  const int R = (T << (4 - tcs)) + (n >> tcs);
  t.valid = R < nrow && t.tc < nbc;
  const unsigned e = lds_ld<uint32_t>(lds, rtoff + 4 * (R < nrow ? R : nrow - 1));
  t.p = static_cast<int>((e >> 12) & 0xffu);
  t.bi = static_cast<int>(e >> 20);
  t.boff = aoff + imul(static_cast<int>(e & 0xfffu) + q, pitch_bytes) + 8 * t.tc;
  return t;
}

// ------------------------------------------------------------------------------ the kernel
// Grid: persistent workgroups, each takes a contiguous range of units (pb planes of one
// channel).  NBL: 4x4 pixel blocks a thread loads per unit.  VEC: plane rows are whole,
// aligned 4-element vectors.  RES: the Toeplitz fragments of level 1 stay in registers while the channel does not change.
//
// A wave computes its 8 x 8 pixels of a level-1 block whole: the four sub-bands' convolutions of the 4 x 4 coefficients and
// the base convolution of the four pixel blocks above them.  The output rows of the products are dealt so that a lane's
// results of both meet: accumulator 4 q + v of a sub-band is coefficient (2 (v / 2) + q / 2, 2 (v % 2) + q % 2), and of the
// base convolution of block v pixel (2 (q / 2) + i, 2 (q % 2) + j) of it -- the 2 x 2 pixels that the inverse Haar
// transform makes of that coefficient.  The base convolution therefore never passes through LDS (as fp32 it took a third of
// a 56 x 56 plane's LDS), and nothing but Z_2 has to be waited for between the convolutions and the stores.
template <typename T, int NS, int NBL, bool VEC, bool RES, typename Geo>
__global__ void __launch_bounds__(kMfmaBlock, NS == 1 ? 4 : 2)      // waves per SIMD the register budget must allow
wt2d_mfma_kernel(const T* __restrict__ x, T* __restrict__ out, const ParamTable prm, int pdtype, int K, int flip,
                 int use_bias, const MPlan plarg, unsigned* __restrict__ zero_words, int nzero) {
  // the plan: shape-dependent fields from the compile-time constant where there is one
  const MPlan pl = [&]() {
    if constexpr (Geo::kStatic) {
      constexpr MPlan g = Geo::template plan<NS>();
      MPlan p = g;
      p.B = plarg.B; p.C = plarg.C; p.upc = plarg.upc; p.nunits = plarg.nunits; p.bq = plarg.bq; p.br = plarg.br;
      p.uq = plarg.uq; p.ur = plarg.ur;
      return p;
    } else {
      return plarg;
    }
  }();
  WT_SHARED_FLOATS(ldsf);
  char* lds = reinterpret_cast<char*>(ldsf);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4;
  const int L = pl.L, H = pl.H, W = pl.W;
  const int HW = H * W;
  // every 4x4 pixel block that exists is whole
  const bool whole = Geo::kStatic && H % 4 == 0 && W % 4 == 0;
  // the channel tickets of a parameter-gradient pass that follows on the stream
  if (blockIdx.x == 0)
    for (int i = tid; i < nzero; i += kMfmaBlock) zero_words[i] = 0u;

  // Toeplitz fragment entries of this lane for patch row q (+4) and output (row r, column c) of a block
  auto entry_top = [&](int r, int c) { return q - r >= 0 ? (q - r) * 4 + c : 20; };
  auto entry_bot = [&](int r, int c) { return q - r <= 0 ? (4 + q - r) * 4 + c : 20; };
  // coarse levels: output n of a block in rows; level 1 and base conv as said above
  const int ent_top = entry_top(n >> 2, n & 3), ent_bot = entry_bot(n >> 2, n & 3);
  const int r1 = 2 * ((n >> 1) & 1) + (n >> 3), c1 = 2 * (n & 1) + ((n >> 2) & 1);
  const int ent1_top = entry_top(r1, c1), ent1_bot = entry_bot(r1, c1);
  const int r0 = 2 * (n >> 3) + ((n >> 1) & 1), c0 = 2 * ((n >> 2) & 1) + (n & 1);
  const int ent0_top = entry_top(r0, c0), ent0_bot = entry_bot(r0, c0);
  const int tsplit = (pl.nfilt - pl.tskip) * kFragEntries * 16;      // bytes between the split tables in LDS

  // ---- per-thread constants of the commit role: which 4x4 pixel blocks this thread owns
  int c_goff[NBL], c_x0[NBL], c_a1[NBL], c_a2[NBL], c_ll[NBL], c_p[NBL];
  unsigned c_mask[NBL];      // bits 0-3: rows inside the plane; bits 4-7: columns inside; bit 8: block exists
#pragma unroll
  for (int i = 0; i < NBL; ++i) {
    const int g = tid + kMfmaBlock * i;
    const bool act = g < pl.nblk[0];
    const int gg = act ? g : 0;
    const int p = fast_div(gg, pl.mg_bpp0);
    const int rem = gg - imul(p, pl.bpp[0]);
    const int bi = fast_div(rem, pl.mg_nbc0);
    const int bj = rem - imul(bi, pl.nbc[0]);
    unsigned m = act ? 0x100u : 0u;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (4 * bi + r < H) m |= 1u << r;
      if (4 * bj + r < W) m |= 16u << r;
    }
    c_mask[i] = m;
    c_p[i] = p;
    c_goff[i] = p * pl.C * HW + 4 * bi * W + 4 * bj;
    c_x0[i] = pl.aoff[0] + ((p * pl.prows[0] + 4 * bi + 2) * pl.pitch[0] + 4 * bj + 2) * 2;
    c_a1[i] = pl.aoff[1] + ((p * pl.prows[1] + 2 * bi + 2) * pl.pitch[1] + 2 * bj + 2) * 2;
    c_a2[i] = L >= 2 ? pl.aoff[2] + ((p * pl.prows[2] + bi + 2) * pl.pitch[2] + bj + 2) * 2 : 0;
    c_ll[i] = L >= 3 ? pl.lloff[2] + (p * pl.llpl[2] + bi * pl.w[2] + bj) * 4 : 0;
  }
  // plan fields of the two finest levels, used in every unit
  const int asub0 = pl.asub[0], asub1 = pl.asub[1], asub2 = pl.asub[2];
  const int pitchB0 = pl.pitch[0] * 2, pitchB1 = pl.pitch[1] * 2;
  const int aoff0 = pl.aoff[0], aoff1 = pl.aoff[1], prows0 = pl.prows[0];
  const int tcs1 = pl.tcs[1], nrow1 = pl.nrow[1], nbc1 = pl.nbc[1], rtoff1 = pl.rtoff[1];
  const int zoff2 = pl.zoff[2], zpitch2 = pl.zpitch[2], zpl2 = pl.zpl[2];
  const int toff = pl.toff, upc = pl.upc, C = pl.C, B = pl.B;

  const int G = gridDim.x;
  const int wg = xcd_contiguous(blockIdx.x, G);
  // The workgroups with a unit more are the first to be dispatched, and so the first few of each XCD's and on different CUs.  With
  // the first ranges longer instead, the first XCDs had twice the work of the last: us [30,48,57,64], two levels 18.4 -> 15.8,
  // [256,264,8,6], one level 18.9 -> 15.6, [256,384,14,14], three levels 38.9 -> 36.3; 614 drawn shapes 0.99, one in eight over 5 %
  // faster, two over 5 % slower, at most 9 %.  (Spread evenly over the ranges they meet on one CU: [256,33,16,18] 16.3 -> 20.6.)
  const int xcds = (G & 7) == 0 ? 3 : 0, xcd = blockIdx.x & ((1 << xcds) - 1), nth = blockIdx.x >> xcds;
  const int longer = (pl.ur + (1 << xcds) - 1 - xcd) >> xcds;                              // of this XCD, and of those before it
  const int before = xcd * (pl.ur >> xcds) + min(xcd, pl.ur & ((1 << xcds) - 1));
  const int u_begin = wg * pl.uq + before + min(nth, longer);
  const int u_end = u_begin + pl.uq + (nth < longer ? 1 : 0);

  // A unit's channel, its number among the channel's units, and the batch items it takes: the batch is spread evenly over
  // the units of a channel, at most pb items each, all units within one plane of each other (a short last unit would leave
  // the workgroups that get it with less work than the rest).
  struct Unit { int c, ub; };
  auto first_item = [&](const Unit& u) { return u.ub * pl.bq + (u.ub < pl.br ? u.ub : pl.br); };
  auto items = [&](const Unit& u) { return pl.bq + (u.ub < pl.br ? 1 : 0); };
  // tiles of level l that hold blocks of the first np planes: a batch smaller than pb does not pay for planes that do not
  // exist.  (Where a constant plan makes a tile a wave or less of it, the constant: 56x56 planes 194 -> 153 us.)
  auto tiles_of = [&](int np, int l) {
    if (Geo::kStatic && (pl.pb == 1 || pl.ntile[l] <= (l == 1 ? 4 : 1))) return pl.ntile[l];
    return (np * pl.nbr[l] + (16 >> pl.tcs[l]) - 1) >> (4 - pl.tcs[l]);
  };

  // ---- a channel's filters, folded: gamma * w * 4^-level, rotated by 180 degrees when flip != 0, embedded in 5 x 5.  They
  // come from memory one tap a lane, all of them in flight at once (one entry of the fragment table a lane, which wants up
  // to five taps and a scale, took a single unit's workgroup 9000 of its 22 000 cycles), and go to LDS as rows of twelve
  // bf16: three zeros, five taps, four zeros.  A fragment entry is eight neighbours of such a row.
  // Two waves take a level (0: the base filter, and its bias), so that its tables are addressed through scalar registers.
  constexpr int kTapItems = ((Geo::kStatic ? Geo::kL : kMaxLevels) + 2) / 2;
  uint32_t tap_w[kTapItems], tap_s[kTapItems];
  struct Tap { int s, row, col; };
  auto tap_of = [&](int r) {
    Tap t;
    t.s = r / 25;
    const int e = r - t.s * 25;
    t.row = e / 5;
    t.col = e - t.row * 5;
    return t;
  };
  auto load_taps = [&](int c) {
    int r = tid & 127;
    WT_LAUNDER_LANE_INT(r);      // (nothing that follows from it is kept for the next channel)
    const Tap t = tap_of(r);
    const int o = 2 - K / 2, ih = t.row - o, iw = t.col - o, in = ih * K + iw;
    const bool inside = ih >= 0 && ih < K && iw >= 0 && iw < K;
    const int tap = flip ? K * K - 1 - in : in;
#pragma unroll
    for (int k = 0; k < kTapItems; ++k) {
      const int l = (wave >> 1) + 2 * k;
      tap_w[k] = tap_s[k] = 0u;
      if (l > L) continue;
      const void *w = l > 0 ? prm.wt_weight[l - 1] : prm.base_weight, *g = l > 0 ? prm.wt_scale[l - 1] : prm.base_scale;
      const int ch = l > 0 ? 4 * c + t.s : c;
      if (inside && t.s < (l > 0 ? 4 : 1)) {
        if (pdtype == WTCONV_F32) {
          tap_w[k] = static_cast<const uint32_t*>(w)[ch * K * K + tap];
          tap_s[k] = static_cast<const uint32_t*>(g)[ch];
        } else {
          tap_w[k] = static_cast<const uint16_t*>(w)[ch * K * K + tap];
          tap_s[k] = static_cast<const uint16_t*>(g)[ch];
        }
      } else if (l == 0 && r == 25 && use_bias && prm.base_bias != nullptr) {
        if (pdtype == WTCONV_F32) {
          tap_w[k] = static_cast<const uint32_t*>(prm.base_bias)[c];
          tap_s[k] = static_cast<const uint32_t*>(g)[c];
        } else {
          tap_w[k] = static_cast<const uint16_t*>(prm.base_bias)[c];
          tap_s[k] = static_cast<const uint16_t*>(g)[c];
        }
      }
    }
  };
  auto store_taps = [&] {
    int r = tid & 127;
    WT_LAUNDER_LANE_INT(r);
    const Tap t = tap_of(r);
#pragma unroll
    for (int k = 0; k < kTapItems; ++k) {
      const int l = (wave >> 1) + 2 * k;
      if (l > L) continue;
      float v = __uint_as_float(tap_w[k]), scale = __uint_as_float(tap_s[k]);
      if (pdtype == WTCONV_F16) {
        v = f16_bits_to_f32(static_cast<uint16_t>(tap_w[k]));
        scale = f16_bits_to_f32(static_cast<uint16_t>(tap_s[k]));
      } else if (pdtype == WTCONV_BF16) {
        v = bf16_to_f32(static_cast<bf16_t>(tap_w[k]));
        scale = bf16_to_f32(static_cast<bf16_t>(tap_s[k]));
      }
      v *= ldexpf(scale, -2 * l);
      if (t.s < (l > 0 ? 4 : 1)) {
        const int f = l > 0 ? 4 * l - 3 + t.s : 0;
#pragma unroll
        for (int js = 0; js < NS; ++js) {
          const bf16_t h = f32_to_bf16(v);
          lds_st<bf16_t>(lds, pl.taps + (((js * pl.nfilt + f) * 5 + t.row) * kTapRow + 3 + t.col) * 2, h);
          v -= bf16_to_f32(h);
        }
      } else if (l == 0 && r == 25) {
        lds_st<float>(lds, pl.taps + pl.tap_rows * kTapRow * 2, v);
      }
    }
  };
  // entry e = 4 kh + cs of filter f: row kh, shifted right by cs in a window of eight; entry 20 is zero (a row of zeros)
  auto entry_of = [&](int js, int f, int e) {
    const int row = e < 20 ? (js * pl.nfilt + f) * 5 + (e >> 2) : pl.tap_rows - 1, at = 3 - (e & 3);
    const int o = pl.taps + row * (kTapRow * 2) + (at & 2) * 2;
    uint32_t d[5];
#pragma unroll
    for (int j = 0; j < 5; ++j) d[j] = lds_ld<uint32_t>(lds, o + 4 * j);
    Frag fr;
#pragma unroll
    for (int j = 0; j < 4; ++j) fr.d[j] = at & 1 ? (d[j] >> 16 | d[j + 1] << 16) : d[j];
    return fr;
  };

  PixRow<T> pf[NBL][4];
  // 16-bit planes whose rows are not whole vectors move as one unaligned 8-byte load a row, all four rows of a block: what
  // comes along from past the row or the plane is cleared at the commit.  The planes at the tensor's end that do not have
  // that much behind them (pl.behind) go element by element.
  constexpr bool kOver = !VEC && sizeof(T) == 2;
  auto fetch = [&](const Unit& u) {
    const int b0 = first_item(u), np = items(u);
    const T* base = x + (static_cast<size_t>(b0) * C + u.c) * HW;
    const bool at_end = (B - b0 - np) * C + (C - 1 - u.c) < pl.behind;
#pragma unroll
    for (int i = 0; i < NBL; ++i) {
      // (a plane that does not exist keeps what an earlier one left: its results are not stored)
      if (!(c_mask[i] & 0x100u) || c_p[i] >= np) continue;
      // (a uniform base and a 32-bit offset in bytes, which a 16-bit unit's elements fit, not added up ahead of the loop)
      int goff = c_goff[i];
      WT_LAUNDER_LANE_INT(goff);
      const T* from = sizeof(T) == 2 ? reinterpret_cast<const T*>(reinterpret_cast<const char*>(base) + static_cast<size_t>(static_cast<uint32_t>(goff) * 2))
                                     : base + goff;
      if constexpr (kOver) {
        if (!at_end) {
#pragma unroll
          for (int r = 0; r < 4; ++r) pix_load4u(pf[i][r].v, from + r * W);
          continue;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (!whole) pix_zero(pf[i][r]);
        if (whole || (c_mask[i] >> r & 1u)) {
          const T* src = from + r * W;
          if constexpr (VEC) {
            pix_load4(pf[i][r], src);      // (a block's first column exists, and with it the other three)
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (c_mask[i] >> (4 + e) & 1u) pix_set(pf[i][r], e, src[e]);
          }
        }
      }
    }
  };
#pragma unroll
  for (int i = 0; i < NBL; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) pix_zero(pf[i][r]);
  Unit nxt;
  nxt.c = u_begin / upc;
  nxt.ub = u_begin - nxt.c * upc;
  if (u_begin < u_end) fetch(nxt);
  load_taps(nxt.c);

  // ---- while they are on their way: halos, and the block-row tables
  for (int o = tid * 16; o < pl.lds_bytes; o += kMfmaBlock * 16) {
    uint4 z; z.x = z.y = z.z = z.w = 0u;
    lds_st<uint4>(lds, o, z);
  }
  WT_LDS_BARRIER();
  levels_up<Geo, 1>(L, [&](auto lc) {
    const int l = lc;
    const float per_plane = 1.f / static_cast<float>(pl.nbr[l]);
    for (int R = tid; R < pl.nrow[l]; R += kMfmaBlock) {
      const int p = static_cast<int>((R + 0.5f) * per_plane), bi = R - p * pl.nbr[l];      // (whole below 500 block rows a plane)
      lds_st<uint32_t>(lds, pl.rtoff[l] + 4 * R, rowtab_entry(p * pl.prows[l] + 4 * bi, p, bi));
    }
  });

  // ---- level-1 tiles: where a lane finds its block's patches and Z_2, and where its results go
  struct Tile {
    int b1, b0, z2;      // LDS offsets: patch row q of the block's sub-band 0, of its pixels, Z_2 of its first coefficient
    int p, to, y, x;     // plane slot; element offset of row y = 8 bi + q, column x = 8 tc in the unit's output
    bool valid;
  };
  auto tile_of = [&](int t) {
    Tile o;
    int n = lane & 15, q = lane >> 4;
    if constexpr (!Geo::kStatic) {
      WT_LAUNDER_LANE_INT(n);
      WT_LAUNDER_LANE_INT(q);
    }
    const int tc = n & ((1 << tcs1) - 1);
    const int R = (t << (4 - tcs1)) + (n >> tcs1);
    o.valid = R < nrow1 && tc < nbc1;
    const unsigned e = lds_ld<uint32_t>(lds, rtoff1 + 4 * (R < nrow1 ? R : nrow1 - 1));
    o.p = static_cast<int>((e >> 12) & 0xffu);
    const int bi = static_cast<int>(e >> 20);
    o.b1 = aoff1 + imul(static_cast<int>(e & 0xfffu) + q, pitchB1) + 8 * tc;
    o.b0 = aoff0 + imul(imul(o.p, prows0) + 8 * bi + q, pitchB0) + 16 * tc;
    o.z2 = zoff2 + (imul(o.p, zpl2) + imul(4 * bi + (q >> 1), zpitch2) + 4 * tc + (q & 1)) * 4;
    o.y = 8 * bi + q;
    o.x = 8 * tc;
    o.to = o.p * C * HW + o.y * W + o.x;
    return o;
  };

  constexpr int NR = RES ? NS : 1;
  Frag ra1t[4][NR], ra1b[4][NR];     // resident fragments (RES only)
  float bias = 0.f;
  // the base convolution of the four pixel blocks and the sub-band convolutions of a tile
  auto convolve = [&](const Tile& tl, Acc (&base)[4], Acc (&band)[4]) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      base[v].v[0] = base[v].v[1] = base[v].v[2] = base[v].v[3] = bias;
      band[v].v[0] = band[v].v[1] = band[v].v[2] = band[v].v[3] = 0.f;
    }
    {
      uint2 w[NS][3][3];      // patch rows q, q + 4, q + 8: twelve columns each
#pragma unroll
      for (int js = 0; js < NS; ++js)
#pragma unroll
        for (int r = 0; r < 3; ++r)
#pragma unroll
          for (int k = 0; k < 3; ++k) w[js][r][k] = lds_ld<uint2>(lds, tl.b0 + js * asub0 + 4 * r * pitchB0 + 8 * k);
      Frag at[NS], ab[NS];
      load_a<NS>(lds, toff, tsplit, ent0_top, ent0_bot, at, ab);
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        Frag bt[NS], bb[NS];
#pragma unroll
        for (int js = 0; js < NS; ++js) {
          const uint2 a = w[js][v >> 1][v & 1], b = w[js][v >> 1][(v & 1) + 1];
          const uint2 c = w[js][(v >> 1) + 1][v & 1], d = w[js][(v >> 1) + 1][(v & 1) + 1];
          bt[js].d[0] = a.x; bt[js].d[1] = a.y; bt[js].d[2] = b.x; bt[js].d[3] = b.y;
          bb[js].d[0] = c.x; bb[js].d[1] = c.y; bb[js].d[2] = d.x; bb[js].d[3] = d.y;
        }
        mma_tile<NS>(at, ab, bt, bb, base[v]);
      }
    }
    WT_SCHED_FENCE();      // (all of a tile's reads at once would not fit the registers)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      Frag bt[NS], bb[NS];
      load_b<NS>(lds, tl.b1 + s * asub1, 4 * asub1, 4 * pitchB1, bt, bb);
      if constexpr (RES) {
        mma_tile<NS>(ra1t[s], ra1b[s], bt, bb, band[s]);
      } else {
        Frag at[NS], ab[NS];
        load_a<NS>(lds, toff + (1 + s - pl.tskip) * kFragEntries * 16, tsplit, ent1_top, ent1_bot, at, ab);
        mma_tile<NS>(at, ab, bt, bb, band[s]);
      }
      if (s == 1) WT_SCHED_FENCE();
    }
  };
  // Z_2, the inverse Haar transform, the sum with the base convolution, and the way to memory
  auto finish = [&](const Tile& tl, Acc (&base)[4], Acc (&band)[4], T* obase, int np, bool wait) {
    if (L >= 2) {
#pragma unroll
      for (int v = 0; v < 4; ++v) band[0].v[v] += lds_ld<float>(lds, tl.z2 + (2 * (v >> 1) * zpitch2 + 2 * (v & 1)) * 4);
    }
    float row[2][8];      // pixel rows y and y + 4, after the exchange
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const float s1 = band[0].v[v] + band[1].v[v], d1 = band[0].v[v] - band[1].v[v];
      const float s2 = band[2].v[v] + band[3].v[v], d2 = band[2].v[v] - band[3].v[v];
      // a lane has 2 x 2 pixels of each block, the lane 16 further (or back) the ones beside them: after the exchange the
      // first has the upper row of four, the second the lower one
      if constexpr (sizeof(T) == 2) {
        uint32_t up = pack_bf16x2(s1 + s2 + base[v].v[0], s1 - s2 + base[v].v[1]);
        uint32_t lo = pack_bf16x2(d1 + d2 + base[v].v[2], d1 - d2 + base[v].v[3]);
        swap_rows16(up, lo);
        row[v >> 1][2 * (v & 1)] = __uint_as_float(up);
        row[v >> 1][2 * (v & 1) + 1] = __uint_as_float(lo);
      } else {
        uint32_t up[2] = {__float_as_uint(s1 + s2 + base[v].v[0]), __float_as_uint(s1 - s2 + base[v].v[1])};
        uint32_t lo[2] = {__float_as_uint(d1 + d2 + base[v].v[2]), __float_as_uint(d1 - d2 + base[v].v[3])};
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          swap_rows16(up[j], lo[j]);
          row[v >> 1][4 * (v & 1) + j] = __uint_as_float(up[j]);
          row[v >> 1][4 * (v & 1) + 2 + j] = __uint_as_float(lo[j]);
        }
      }
    }
    // the prefetch of the next unit has had this tile's convolutions to land; waiting for it here, ahead of
    // the first store, lets the stores drain behind the next unit's work instead of being waited for at its commit
    if (wait) WT_WAIT_VMEM();
    if (!tl.valid || tl.p >= np) return;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      if (tl.y + 4 * half >= H) continue;
      int to = tl.to;
      WT_LAUNDER_LANE_INT(to);      // (not added to the tensor's address ahead of the loop)
      T* dst = sizeof(T) == 2 ? reinterpret_cast<T*>(reinterpret_cast<char*>(obase) + static_cast<size_t>(static_cast<uint32_t>(to) * 2)) + 4 * half * W
                              : obase + to + 4 * half * W;
      const int left = W - tl.x;      // columns of the row from here on
      if constexpr (sizeof(T) == 2) {
        const uint32_t d[4] = {__float_as_uint(row[half][0]), __float_as_uint(row[half][1]),
                               __float_as_uint(row[half][2]), __float_as_uint(row[half][3])};
        if ((Geo::kStatic && W % 8 == 0) || left >= 8) {
          __builtin_memcpy(dst, d, 16);
        } else {
          // 4, 2 and 1 of them
          if (left & 4) __builtin_memcpy(dst, d, 8);
          if constexpr (!VEC) {
            const uint32_t two = left & 4 ? d[2] : d[0], one = left & 4 ? (left & 2 ? d[3] : d[2]) : (left & 2 ? d[1] : d[0]);
            if (left & 2) __builtin_memcpy(dst + (left & 4), &two, 4);
            if (left & 1) dst[left & 6] = static_cast<T>(one);
          }
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; e += 4) {
          if (VEC) {
            if (e < left) {
              float4 o4; o4.x = row[half][e]; o4.y = row[half][e + 1]; o4.z = row[half][e + 2]; o4.w = row[half][e + 3];
              *reinterpret_cast<float4*>(dst + e) = o4;
            }
          } else {
#pragma unroll
            for (int k = e; k < e + 4; ++k)
              if (k < left) dst[k] = from_f32<T>(row[half][k]);
          }
        }
      }
    }
  };
  // the fragment table and the resident fragments from the loaded taps
  auto take_channel = [&] {
    store_taps();
    WT_LDS_BARRIER();      // (in the first unit the block-row tables, too)
    int first = tid;
    WT_LAUNDER_LANE_INT(first);
    for (int i = first; i < (pl.nfilt - pl.tskip) * kFragEntries; i += kMfmaBlock) {
      const int slot = i / kFragEntries, e = i - slot * kFragEntries;
#pragma unroll
      for (int j = 0; j < NS; ++j) {
        const Frag fr = entry_of(j, slot > 0 ? slot + pl.tskip : 0, e);
        uint4 v; v.x = fr.d[0]; v.y = fr.d[1]; v.z = fr.d[2]; v.w = fr.d[3];
        lds_st<uint4>(lds, toff + j * tsplit + i * 16, v);
      }
    }
    if constexpr (RES) {
      int top = ent1_top, bot = ent1_bot;
      WT_LAUNDER_LANE_INT(top);
      WT_LAUNDER_LANE_INT(bot);
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        ra1t[s][0] = entry_of(0, 1 + s, top);
        ra1b[s][0] = entry_of(0, 1 + s, bot);
        WT_SCHED_FENCE();
      }
    }
    bias = lds_ld<float>(lds, pl.taps + pl.tap_rows * kTapRow * 2);
  };
  take_channel();
  Tile own = {};
  if constexpr (Geo::kStatic) own = tile_of(wave < pl.ntile[1] ? wave : 0);      // a wave's first tile, the same in every unit
  int cur_c = nxt.c;
#pragma unroll 1
  for (int u = u_begin; u < u_end; ++u) {
    const Unit un = nxt;
    const int c = un.c, b0 = first_item(un), np = items(un), ntile1 = tiles_of(np, 1);
    if (++nxt.ub == upc) { nxt.ub = 0; ++nxt.c; }
    if (c != cur_c) {      // (every read of the old filters lies behind a barrier)
      load_taps(c);
      take_channel();
      cur_c = c;
    }

    // ---- commit: pixels -> level-0 planes; analysis levels 1 and 2 from registers
#pragma unroll
    for (int i = 0; i < NBL; ++i) {
      if (!(c_mask[i] & 0x100u)) continue;
      int x0 = c_x0[i], a1 = c_a1[i], a2 = c_a2[i];
      WT_LAUNDER_LANE_INT(x0);      // (the sums with the plan's fields below are not kept from unit to unit)
      WT_LAUNDER_LANE_INT(a1);
      WT_LAUNDER_LANE_INT(a2);
      float v[4][4];
      if constexpr (kOver) {      // clear what came along from past the row and the plane
        const uint2 m = pix_col_mask(c_mask[i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool row = c_mask[i] >> r & 1u;
          pf[i][r].v.x &= row ? m.x : 0u;
          pf[i][r].v.y &= row ? m.y : 0u;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) pix_get(pf[i][r], v[r]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        uint32_t w0[NS], w1[NS];
        if constexpr (NS == 1 && sizeof(T) == 2) {
          const uint2 w = pix_words(pf[i][r]);      // the values are bf16 already
          w0[0] = w.x;
          w1[0] = w.y;
        } else {
          split_pair<NS>(v[r][0], v[r][1], w0);
          split_pair<NS>(v[r][2], v[r][3], w1);
        }
#pragma unroll
        for (int j = 0; j < NS; ++j) {
          const int o = x0 + j * asub0 + r * pitchB0;
          lds_st<uint32_t>(lds, o, w0[j]);
          lds_st<uint32_t>(lds, o + 4, w1[j]);
        }
      }
      float ll1[2][2];
#pragma unroll
      for (int i2 = 0; i2 < 2; ++i2) {
        float cf[4][2];
#pragma unroll
        for (int j2 = 0; j2 < 2; ++j2) {
          const float a = v[2 * i2][2 * j2], b = v[2 * i2][2 * j2 + 1];
          const float cc = v[2 * i2 + 1][2 * j2], d = v[2 * i2 + 1][2 * j2 + 1];
          const float s1 = a + b, d1 = a - b, s2 = cc + d, d2 = cc - d;
          cf[0][j2] = s1 + s2; cf[1][j2] = s1 - s2; cf[2][j2] = d1 + d2; cf[3][j2] = d1 - d2;
        }
        ll1[i2][0] = cf[0][0]; ll1[i2][1] = cf[0][1];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          uint32_t w[NS];
          split_pair<NS>(cf[s][0], cf[s][1], w);
#pragma unroll
          for (int j = 0; j < NS; ++j)
            lds_st<uint32_t>(lds, a1 + (j * 4 + s) * asub1 + i2 * pitchB1, w[j]);
        }
      }
      if (L >= 2) {
        const float a = ll1[0][0], b = ll1[0][1], cc = ll1[1][0], d = ll1[1][1];
        const float s1 = a + b, d1 = a - b, s2 = cc + d, d2 = cc - d;
        const float cf[4] = {s1 + s2, s1 - s2, d1 + d2, d1 - d2};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          uint32_t w[NS];
          split_pair<NS>(cf[s], 0.f, w);
#pragma unroll
          for (int j = 0; j < NS; ++j)
            lds_st<uint16_t>(lds, a2 + (j * 4 + s) * asub2, static_cast<uint16_t>(w[j]));
        }
        if (L >= 3) lds_st<float>(lds, c_ll[i], cf[0]);
      }
    }
    if (u + 1 < u_end) fetch(nxt);
    WT_LDS_BARRIER();

    // ---- the last wave: levels L..2 on its own (the others wait for this chain at the barrier)
    if (L >= 2 && wave == 3) {
      WT_WAVE_PRIORITY(3);
      // (lane numbers that the compiler cannot see through: it would keep every address below in registers from unit to unit)
      int n = lane & 15, q = lane >> 4, lane_ = lane;
      WT_LAUNDER_LANE_INT(n);
      WT_LAUNDER_LANE_INT(q);
      WT_LAUNDER_LANE_INT(lane_);
      // analysis levels 3..L from the raw LL of the level above (fp32 in LDS)
      levels_up<Geo, 3>(L, [&](auto lc) {
        const int l = lc;
        const int hl = pl.h[l], wl = pl.w[l], npos = (Geo::kStatic && pl.pb == 1 ? 1 : np) * hl * wl;
        for (int idx = lane_; idx < npos; idx += 64) {
          const int p = fast_div(idx, pl.mg_hw[l]);
          const int rem = idx - imul(p, hl * wl);
          const int i = fast_div(rem, pl.mg_w[l]);
          const int j = rem - imul(i, wl);
          const int hs = pl.h[l - 1], wsrc = pl.w[l - 1];
          const int so = pl.lloff[l - 1] + (imul(p, pl.llpl[l - 1]) + imul(2 * i, wsrc) + 2 * j) * 4;
          const bool r1 = 2 * i + 1 < hs, c1 = 2 * j + 1 < wsrc;
          const float a = lds_ld<float>(lds, so);
          const float b = c1 ? lds_ld<float>(lds, so + 4) : 0.f;
          const float cc = r1 ? lds_ld<float>(lds, so + wsrc * 4) : 0.f;
          const float d = (r1 && c1) ? lds_ld<float>(lds, so + wsrc * 4 + 4) : 0.f;
          const float s1 = a + b, d1 = a - b, s2 = cc + d, d2 = cc - d;
          const float cf[4] = {s1 + s2, s1 - s2, d1 + d2, d1 - d2};
          const int ao = pl.aoff[l] + (imul(imul(p, pl.prows[l]) + i + 2, pl.pitch[l]) + j + 2) * 2;
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            uint32_t w[NS];
            split_pair<NS>(cf[s], 0.f, w);
#pragma unroll
            for (int js = 0; js < NS; ++js)
              lds_st<uint16_t>(lds, ao + (js * 4 + s) * pl.asub[l], static_cast<uint16_t>(w[js]));
          }
          if (l < L) lds_st<float>(lds, pl.lloff[l] + (imul(p, pl.llpl[l]) + imul(i, wl) + j) * 4, cf[0]);
        }
        WT_WAVE_SYNC_DIVERGENT();
      });
      // convolutions and inverse Haar transforms -> Z_l
      levels_down<Geo, 2>(L, [&](auto lc) {
        const int l = lc;
        const int ntile = tiles_of(np, l);
        const int pitchB = pl.pitch[l] * 2, asub = pl.asub[l];
        const int zo_in = pl.zoff[l + 1], zp_in = pl.zpitch[l + 1], zpl_in = pl.zpl[l + 1];
        const int zo = pl.zoff[l], zp = pl.zpitch[l], zpl_o = pl.zpl[l], zrows = 4 * pl.nbr[l - 1];
        const int tab = toff + (1 + 4 * (l - 1) - pl.tskip) * kFragEntries * 16;
#pragma unroll 1
        for (int t = 0; t < ntile; ++t) {
          const TileLane tl = tile_lane(lds, t, n, q, pl.tcs[l], pl.nrow[l], pl.nbc[l], pl.rtoff[l], pl.aoff[l], pitchB);
          Acc acc[4];
#pragma unroll
          for (int s = 0; s < 4; ++s) acc[s].v[0] = acc[s].v[1] = acc[s].v[2] = acc[s].v[3] = 0.f;
          if (l < L) {
            const float4 z = lds_ld<float4>(lds, zo_in + (imul(tl.p, zpl_in) + imul(4 * tl.bi + q, zp_in) + 4 * tl.tc) * 4);
            acc[0].v[0] = z.x; acc[0].v[1] = z.y; acc[0].v[2] = z.z; acc[0].v[3] = z.w;
          }
#pragma unroll
          for (int s2 = 0; s2 < 4; s2 += 2) {      // (the LDS reads of all four sub-bands at once would not fit the registers)
            Frag at[2][NS], ab[2][NS], bt[2][NS], bb[2][NS];
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              load_b<NS>(lds, tl.boff + (s2 + k) * asub, 4 * asub, 4 * pitchB, bt[k], bb[k]);
              load_a<NS>(lds, tab + (s2 + k) * kFragEntries * 16, tsplit, ent_top, ent_bot, at[k], ab[k]);
            }
#pragma unroll
            for (int k = 0; k < 2; ++k) mma_tile<NS>(at[k], ab[k], bt[k], bb[k], acc[s2 + k]);
            WT_SCHED_FENCE();
          }
          float top[8], bot[8];
          synth_rows(acc, top, bot);
          const int y = 2 * (4 * tl.bi + q), xx = 8 * tl.tc;
          if (tl.valid) {
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              if (xx + 4 * half < zp) {
                const int o = zo + (imul(tl.p, zpl_o) + imul(y, zp) + xx + 4 * half) * 4;
                float4 a, b;
                a.x = top[4 * half]; a.y = top[4 * half + 1]; a.z = top[4 * half + 2]; a.w = top[4 * half + 3];
                b.x = bot[4 * half]; b.y = bot[4 * half + 1]; b.z = bot[4 * half + 2]; b.w = bot[4 * half + 3];
                if (y < zrows) lds_st<float4>(lds, o, a);
                if (y + 1 < zrows) lds_st<float4>(lds, o + zp * 4, b);
              }
            }
          }
        }
        WT_WAVE_SYNC_DIVERGENT();
      });
      WT_WAVE_PRIORITY(0);
    }
    // ---- level 1 and base conv: each wave's first tile up to the barrier, which Z_2 is waited for at
    Acc base[4], band[4];
    T* obase = out + (static_cast<size_t>(b0) * C + c) * HW;
    if (wave < ntile1) {
      if constexpr (!Geo::kStatic) own = tile_of(wave);      // (the run-time plan's fields leave no registers to keep it in)
      convolve(own, base, band);
    }
    WT_LDS_BARRIER();
    if (wave < ntile1) finish(own, base, band, obase, np, true);
    if (ntile1 > 4) {
#pragma unroll 1
      for (int t = wave + 4; t < ntile1; t += 4) {
        const Tile tl = tile_of(t);
        convolve(tl, base, band);
        finish(tl, base, band, obase, np, false);
      }
      WT_LDS_BARRIER();      // the next unit's commit overwrites what these tiles read
    }
    // (With one tile a wave nothing but Z_2 is read behind the barrier above, and Z_2 is written next behind the barrier
    // that follows the next commit.)
  }
}

}  // namespace wt
