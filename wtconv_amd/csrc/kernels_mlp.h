// The rest of a WTConvNeXt block behind its WTConv layer as one matrix-core kernel, for inference in bfloat16:
//
//   out = shortcut + gamma * (W2 gelu(W1 LayerNorm_c(x) + b1) + b2)
//
// (wtconvnext/wtconvnext.py:125-140: permute, norm, mlp, permute, layer scale, shortcut).  x, shortcut and out are
// (B, C, HW), W1 is (hidden, C), W2 is (C, hidden) as nn.Linear keeps them.
//
// What bounds the unfused passes is memory: the hidden activations are 4x the block's, written by fc1, read and written
// by GELU, read by fc2 -- at 56 x 56 that is 2.5 GB a block against 0.46 GB for everything else.  Here they never leave
// the registers of the wave that computes them:
//
//   * a wave owns 16 * NT pixels for the whole kernel: their normalised channels (the B operand of the first product,
//     C / 32 * NT fragments) and their C / 16 * NT output tiles stay in registers;
//   * the hidden units go by in groups of 32.  A product tile leaves hidden units 4q..4q+3 of pixel n in lane (n, q); the
//     rows of W1 are dealt to the two tiles of a group so that the lane ends up with hidden units 8q..8q+7, which is
//     exactly the B fragment that the second product wants: GELU, rounding and packing happen in place, no exchange;
//   * the weights are the A operands.  They are the same for every wave, so they come through LDS, in slices of HC hidden
//     units, straight from memory into a ring of stages: while one is multiplied, the next ones are on their way, and a
//     wave waits only for the loads of the next one.
//
// LayerNorm needs all channels of a pixel and the wave has them: the statistics are two exact passes over its registers.
//
// What bounds it: with few channels the vector pipe (busy 91 % of the time at C = 96, most of it GELU, which costs 59 us of
// 226 there, 33 of 175 at C = 192, 24 of 175 at C = 384), with many nothing alone: at C = 384 the vector pipe is busy a third of
// the time, LDS 29 % and the matrix cores 27 %; the pixels' way in and out with LayerNorm is 30 % of a tile's time, and 392 tiles
// are 1.53 rounds of the compute units.  Two pixel tiles a wave and one wave a SIMD there (accumulators in accumulation
// registers, half the LDS reads) took 205: a lone wave issues half as often.  Smaller tiles for the last round gave nothing
// (a SIMD with two waves takes as long as all with two) and 192 channels 1 % less.
// Measured at batch 256, us a block, the passes it replaces (norm, fc1, GELU, fc2, residual) -> this kernel: 56 x 56 x 96
// 917 -> 222 (530 TFLOP/s), 28 x 28 x 192 455 -> 168, 14 x 14 x 384 295 -> 171 (690 TFLOP/s); 56 x 56 x 128 1059 -> 342,
// 28 x 28 x 256 609 -> 338.  (228, 173, 179, 352 and 349 with a stage's loads in one piece, the first one's behind LayerNorm
// and a clamp in GELU.)
#pragma once

#include "gelu.h"
#include "matrix.h"

namespace wt {

struct MlpArgs {
  const bf16_t* x;
  const bf16_t* shortcut;
  bf16_t* out;
  const bf16_t *norm_w, *norm_b;      // (C)
  const bf16_t *w1, *b1;              // (hidden, C), (hidden)
  const bf16_t *w2, *b2;              // (C, hidden), (C)
  const bf16_t* gamma;                // (C) or nullptr
  float* partial;                     // (splits, C, pixels padded to a tile) when splits > 1
  float eps;
  int HW, hidden;
  int pixels;                         // B * HW
  int padded;                         // pixels rounded up to whole tiles
  int splits;
  int vec;                            // pixels moved at once: 8, 4 or 1 (they share an image and an aligned word)
};

// C channels, NT pixel tiles a wave, WAVES waves a workgroup, at least PER_SIMD waves a SIMD, slices of HC hidden units,
// RING stages in LDS.
template <int C_, int NT_, int WAVES_, int PER_SIMD_, int HC_, int RING_>
struct MlpShape {
  static constexpr int C = C_, NT = NT_, WAVES = WAVES_, PER_SIMD = PER_SIMD_, HC = HC_, RING = RING_;
  static constexpr int kThreads = 64 * WAVES;
  static constexpr int PX = WAVES * 16 * NT;                // pixels of a workgroup
  static constexpr int G1 = C / 8, G2 = HC / 8;             // 16-byte granules of a row of a W1 / W2 slice
  static constexpr int kGranules = HC * G1;                 // of a slice, either kind (= C * G2)
  static constexpr int kLoads = (kGranules + kThreads - 1) / kThreads;      // per thread and slice, at most
  static constexpr int kSliceBytes = kGranules * 16;
  static constexpr int kStageBytes = 2 * kSliceBytes;       // W1's slice i and W2's slice i - 1
  static_assert(C % 32 == 0 && kGranules % 64 == 0, "slices are loaded by whole waves");
  // The pixels of the workgroup pass through LDS on the way in and out, [channel][pixel] with a padding that puts the
  // rows 8q apart on different banks.  (The memory is the ring's.  On the way in they lie at its end, behind W1's first
  // slice, which is on its way meanwhile; on the way out all slices are done with.)
  static constexpr int kPitch = PX + 4;
  static constexpr int kTileBytes = C * kPitch * 2;
  static_assert(RING == 3, "see the pipeline");
  static constexpr int kRegionBytes = RING * kStageBytes > kTileBytes ? RING * kStageBytes : kTileBytes;
  static constexpr int kTileAt = kRegionBytes - kTileBytes / 16 * 16 - 16;
  static_assert(kTileAt >= kSliceBytes, "W1's first slice lies before the pixels");
  static constexpr size_t lds_bytes(int hidden_here) { return kRegionBytes + 4 * static_cast<size_t>(hidden_here); }

  // Where granule g of row r sits within its row.  The LDS serves a 16-byte read in four goes of 16 lanes -- lanes 0-3,
  // 12-15 and 20-27 (then 4-11, 16-19, 28-31, and both again in the upper half) -- and has 16 granules of banks: these
  // permutations put the 16 granules of a go on different ones.  (Measured: 570 against 300 bytes per ns and CU.)
  static constexpr int of4(int k) { return ((k << 1) & 3) ^ ((k >> 1) * 3); }      // 0, 2, 3, 1
  static __device__ __forceinline__ int swz1(int r, int g) {          // rows r = 8a + b (+4), a, b = 0..3
    if constexpr (G1 % 16 == 0) return g ^ ((r & 3) | ((r >> 1) & 12));
    else if constexpr (G1 % 8 == 0) return g ^ (((r >> 1) & 1) | ((r >> 2) & 6));
    else return g ^ of4((r >> 3) & 3);
  }
  static __device__ __forceinline__ int swz2(int r, int g) {          // 16 consecutive rows
    if constexpr (G2 == 8) return g ^ ((r >> 1) & 7);
    else return g ^ of4((r >> 2) & 3);
  }
};

// ROOM: there are HC floats of LDS behind the bias (which S::lds_bytes does not count).
template <typename S, bool ROOM>
__global__ void __launch_bounds__(S::kThreads, S::PER_SIMD)
block_mlp_kernel(MlpArgs a) {
  constexpr int C = S::C, NT = S::NT, HC = S::HC, KS = C / 32, MT = C / 16, RING = S::RING;
  WT_SHARED_FLOATS(mlp_lds_floats);
  unsigned char* mlp_lds = reinterpret_cast<unsigned char*>(mlp_lds_floats);
  float* bias_lds = reinterpret_cast<float*>(mlp_lds + S::kRegionBytes);
  const int tid = threadIdx.x, lane = tid & 63, wave = WT_UNIFORM(tid >> 6);
  const int n = lane & 15, q = lane >> 4;

  // ---- the slices of this workgroup: hidden units [h0, h1)
  const int nslice = a.hidden / HC;
  const int per = (nslice + a.splits - 1) / a.splits;
  const int s_begin = blockIdx.y * per, s_end = min(nslice, s_begin + per);
  const int h0 = s_begin * HC, nsl = s_end - s_begin;

  // this thread's granules in a slice, as byte offsets from the slice's first one
  uint32_t src1[S::kLoads], src2[S::kLoads];
#pragma unroll
  for (int i = 0; i < S::kLoads; ++i) {
    const int p = i * S::kThreads + tid;
    const int r1 = p / S::G1, g1 = S::swz1(r1, p - r1 * S::G1);      // (the permutation is its own inverse)
    src1[i] = static_cast<uint32_t>(r1 * C + g1 * 8) * 2;
    const int r2 = p / S::G2, g2 = S::swz2(r2, p - r2 * S::G2);
    src2[i] = static_cast<uint32_t>(r2 * a.hidden + g2 * 8) * 2;
  }
  const lds_addr lds0 = WT_LDS_ADDR(mlp_lds);
  auto holds = [&](int k) { return (k + 1) * S::kThreads <= S::kGranules || k * S::kThreads + wave * 64 < S::kGranules; };
  // stage i of the ring: W1's slice i and W2's slice i - 1, as far as they exist (slices counted from s_begin); its loads
  // k = 0 .. 2 kLoads
  auto load_piece = [&](int i, int at, int k) {
    const lds_addr dst = WT_UNIFORM(lds0 + at * S::kStageBytes + wave * 1024);
    if (k < S::kLoads) {
      if (i < nsl && holds(k)) granules_to_lds(a.w1 + static_cast<size_t>(h0 + i * HC) * C, src1[k], dst + k * (S::kThreads * 16));
    } else if (i > 0 && i <= nsl && holds(k - S::kLoads)) {
      granules_to_lds(a.w2 + (h0 + (i - 1) * HC), src2[k - S::kLoads], dst + S::kSliceBytes + (k - S::kLoads) * (S::kThreads * 16));
    }
  };
  auto load_stage = [&](int i, int at) {
#pragma unroll
    for (int k = 0; k < 2 * S::kLoads; ++k) load_piece(i, at, k);
  };
  for (int i = tid; i < nsl * HC; i += S::kThreads) bias_lds[i] = bf16_to_f32(a.b1[h0 + i]);

  // ---- the pixels, into LDS.  This thread's group of them, and the channels it moves: row, row + rows, ...
  load_stage(0, 0);
  bf16_t* tile = reinterpret_cast<bf16_t*>(mlp_lds + S::kTileAt);
  auto for_pixels = [&](auto vec, auto&& load, auto&& use) {      // load(offset in memory), use(value, channel, offset, offset in the tile)
    constexpr int V = decltype(vec)::value, groups = S::PX / V, rows = S::kThreads / groups, iters = C / rows;
    constexpr int U = iters % 12 == 0 ? 12 : (iters % 8 == 0 ? 8 : 6);      // in flight at once
    static_assert(iters % U == 0, "whole batches");
    const int g = tid % groups, row = tid / groups, p = blockIdx.x * S::PX + g * V;
    if (p >= a.pixels) return;
    const int b = p / a.HW;
    const size_t from = static_cast<size_t>(b) * C * a.HW + (p - b * a.HW);
    for (int c0 = row; c0 < C; c0 += rows * U) {
      decltype(load(from)) v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) v[u] = load(from + static_cast<uint32_t>((c0 + u * rows) * a.HW));
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int c = c0 + u * rows;
        use(v[u], c, from + static_cast<uint32_t>(c * a.HW), c * S::kPitch + g * V);
      }
    }
  };
  using std::integral_constant;
  if (a.vec == 8) {
    for_pixels(integral_constant<int, 8>{}, [&](size_t at) { return *reinterpret_cast<const uint4*>(a.x + at); },
               [&](const uint4& v, int, size_t, int dst) {
                 *reinterpret_cast<uint2*>(tile + dst) = uint2{v.x, v.y};
                 *reinterpret_cast<uint2*>(tile + dst + 4) = uint2{v.z, v.w};
               });
  } else if (a.vec == 4) {
    for_pixels(integral_constant<int, 4>{}, [&](size_t at) { return *reinterpret_cast<const uint2*>(a.x + at); },
               [&](const uint2& v, int, size_t, int dst) { *reinterpret_cast<uint2*>(tile + dst) = v; });
  } else {
    for_pixels(integral_constant<int, 1>{}, [&](size_t at) { return a.x[at]; },
               [&](bf16_t v, int, size_t, int dst) { tile[dst] = v; });
  }
  __syncthreads();

  // ---- LayerNorm over the channels, in place in what becomes the B fragments of the first product.  (Pixels past the
  // end hold whatever the LDS held; a column of a product depends on its own pixel alone, and they are not stored.)
  const int p_lane = wave * (16 * NT) + NT * n;      // this lane's first pixel within the tile
  uint32_t xf[NT][KS][4];                            // channels 32 s + 8 q + 2 j and + 1
  {
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bf16_t* src = tile + (32 * s + 8 * q + 2 * j) * S::kPitch + p_lane;
        if constexpr (NT == 2) {      // two pixels of a channel in one word
          const uint32_t lo = *reinterpret_cast<const uint32_t*>(src);
          const uint32_t hi = *reinterpret_cast<const uint32_t*>(src + S::kPitch);
          xf[0][s][j] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
          xf[NT - 1][s][j] = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        } else {
          xf[0][s][j] = src[0] | (static_cast<uint32_t>(src[S::kPitch]) << 16);
        }
        WT_LAUNDER_LANE_INT(xf[0][s][j]);      // (packed here, not kept in halves)
        WT_LAUNDER_LANE_INT(xf[NT - 1][s][j]);
      }
    auto over_channels = [&](float v) {      // sum over the four lanes that share the pixels
      const int lane4 = lane << 2;
      v += wave_xor(v, lane4, 16);
      v += wave_xor(v, lane4, 32);
      return v;
    };
    // (each pass unpacks anew: the values kept as floats from one to the next would not fit the registers)
    auto opaque = [&](int t) {
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) WT_LAUNDER_LANE_INT(xf[t][s][j]);
    };
    float mean[NT], rstd[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float sum = 0.f;
      opaque(t);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float lo, hi;
          unpack2<bf16_t>(xf[t][s][j], lo, hi);
          sum += lo + hi;
        }
      mean[t] = over_channels(sum) * (1.f / C);
      float sq = 0.f;
      opaque(t);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float lo, hi;
          unpack2<bf16_t>(xf[t][s][j], lo, hi);
          sq = fmaf(lo - mean[t], lo - mean[t], sq);
          sq = fmaf(hi - mean[t], hi - mean[t], sq);
        }
      rstd[t] = rsqrtf(over_channels(sq) * (1.f / C) + a.eps);
      opaque(t);
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const uint4 w4 = *reinterpret_cast<const uint4*>(a.norm_w + 32 * s + 8 * q);
      const uint4 b4 = *reinterpret_cast<const uint4*>(a.norm_b + 32 * s + 8 * q);
      const uint32_t ww[4] = {w4.x, w4.y, w4.z, w4.w}, bb[4] = {b4.x, b4.y, b4.z, b4.w};
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float lo, hi, w_lo, w_hi, b_lo, b_hi;
          unpack2<bf16_t>(xf[t][s][j], lo, hi);
          unpack2<bf16_t>(ww[j], w_lo, w_hi);
          unpack2<bf16_t>(bb[j], b_lo, b_hi);
          xf[t][s][j] = pack_bf16x2(fmaf((lo - mean[t]) * rstd[t], w_lo, b_lo), fmaf((hi - mean[t]) * rstd[t], w_hi, b_hi));
          WT_LAUNDER_LANE_INT(xf[t][s][j]);
        }
      if (s % 2 == 1) WT_CHUNK_FENCE();
    }
  }
  WT_WAIT_VMEM();       // (the first slice)
  __syncthreads();      // the tile has been read: the ring may be filled

  load_stage(1, 1);
  load_stage(2, 2);
  auto frag = [](const uint32_t (&v)[4]) { return frag_of(uint4{v[0], v[1], v[2], v[3]}); };

  mat_acc acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[m][t] = mat_acc{0.f, 0.f, 0.f, 0.f};

  // this lane's part of the fragment addresses (bytes): its row, and the granule of each step in it (the permutations
  // do not depend on what is added to the row below)
  const int row1 = 8 * (n >> 2) + (n & 3);
  const int at1 = row1 * S::G1 * 16, at2 = n * S::G2 * 16;
  int go1[KS], go2[HC / 32];
#pragma unroll
  for (int s = 0; s < KS; ++s) go1[s] = S::swz1(row1, 4 * s + q) * 16;
#pragma unroll
  for (int g = 0; g < HC / 32; ++g) go2[g] = S::swz2(n, 4 * g + q) * 16;

  // ---- the slices, in a software pipeline: iteration i multiplies W1's slice i while the vector pipe is at the GELU of
  // slice i - 1, and then W2's slice i - 1.  The one barrier of an iteration is in its middle: behind it stage i + 1 has
  // arrived for everybody and stage i - 1 is no longer read, so its place takes stage i + 2; the reads of the next
  // iteration start before this one ends.
  constexpr int NG = HC / 32, N1 = NG * KS * 2, N2 = NG * MT, kAhead = N1 % 4 == 0 && N2 % 4 == 0 ? 4 : 3, PACKS = NG * NT * 4;
  static_assert(N1 % kAhead == 0 && N2 % kAhead == 0, "the fragments in flight keep their places");
  mat_acc h[NG][2][NT], hn[NG][2][NT];            // slice i - 1 and slice i before GELU
  mat_frag w[kAhead];                             // fragments in flight
  uint32_t hf[NG][NT][4];                         // slice i - 1 behind GELU
  const unsigned char* stage = mlp_lds;           // this iteration's
  int fill = 2;                                   // where stage i + 2 goes
  auto fetch1 = [&](const unsigned char* st, int j) {
    return *reinterpret_cast<const mat_frag*>(st + at1 + go1[j / 2 % KS] + (32 * (j / (2 * KS)) + 4 * (j & 1)) * S::G1 * 16);
  };
  auto fetch2 = [&](const unsigned char* st, int j) {
    return *reinterpret_cast<const mat_frag*>(st + S::kSliceBytes + at2 + go2[j % NG] + 16 * (j / NG) * S::G2 * 16);
  };
  auto start = [&](const unsigned char* st, int i) {      // first reads of iteration i
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const mat_acc b = *reinterpret_cast<const mat_acc*>(bias_lds + i * HC + 32 * g + 8 * q + 4 * m);
#pragma unroll
        for (int t = 0; t < NT; ++t) hn[g][m][t] = b;
      }
  };
  auto activate = [&](int k) {
    const int g = k / (NT * 4), t = k / 4 % NT, m = k / 2 % 2, r = k % 2 * 2;
    hf[g][t][2 * m + k % 2] = pack_bf16x2(gelu_erf(h[g][m][t][r]), gelu_erf(h[g][m][t][r + 1]));
  };
  auto middle = [&] {
    asm volatile("" ::: "memory");
    WT_WAIT_VMEM();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto after = [&](const unsigned char* st) { return st == mlp_lds + 2 * S::kStageBytes ? mlp_lds : st + S::kStageBytes; };
  // A product step is one fragment read (kAhead steps before it is used) and its NT products; the GELU of a pair of values
  // goes between two steps of the first product.  The fences keep this order: left to itself the compiler puts every read
  // right in front of its use and all vector work in one piece.
  auto first_product = [&](auto with_gelu, auto then_second) {
#pragma unroll
    for (int j = 0; j < N1; ++j) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        mat_acc& d = hn[j / (2 * KS)][j & 1][t];
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j % kAhead], frag(xf[t][j / 2 % KS]), d, 0, 0, 0);
      }
      if (j + kAhead < N1) w[j % kAhead] = fetch1(stage, j + kAhead);
      else if (decltype(then_second)::value) w[j % kAhead] = fetch2(stage, j + kAhead - N1);
      if (decltype(with_gelu)::value) {
#pragma unroll
        for (int k = j * PACKS / N1; k < (j + 1) * PACKS / N1; ++k) activate(k);
      }
      WT_SCHED_FENCE();
    }
  };
  // (`load`: the stage whose loads are issued on the way)
  auto second_product = [&](const unsigned char* next, int ahead, int load, auto then_first) {
#pragma unroll
    for (int j = 0; j < N2; ++j) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        mat_acc& d = acc[j / NG][t];
        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[j % kAhead], frag(hf[j % NG][t]), d, 0, 0, 0);
      }
      if (j + kAhead < N2) w[j % kAhead] = fetch2(stage, j + kAhead);
      else if (decltype(then_first)::value) {
        if (j + kAhead == N2) start(next, ahead);
        w[j % kAhead] = fetch1(next, j + kAhead - N2);
      }
      if (decltype(then_first)::value) {
#pragma unroll
        for (int k = 0; k < 2 * S::kLoads; ++k)
          if (k * N2 / (2 * S::kLoads) == j) load_piece(load, fill, k);
      }
      WT_SCHED_FENCE();
    }
    fill = fill == 2 ? 0 : fill + 1;
  };
  auto keep = [&] {
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int m = 0; m < 2; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t) h[g][m][t] = hn[g][m][t];
  };
  using std::true_type;
  using std::false_type;
  // slice 0 through W1
  start(stage, 0);
#pragma unroll
  for (int j = 0; j < kAhead; ++j) w[j] = fetch1(stage, j);
  first_product(false_type{}, false_type{});
  middle();
  fill = 0;
  stage = after(stage);
  keep();
  if (nsl > 1) {
    start(stage, 1);
#pragma unroll
    for (int j = 0; j < kAhead; ++j) w[j] = fetch1(stage, j);
  }
  for (int i = 1; i < nsl; ++i) {
    // the slice whose bias is read ahead: one that does not exist, of whatever the LDS holds there, or, without room for
    // that, the last one again (which costs 1 to 3 %: 384 channels 190 -> 192 us, 96 channels 222 -> 229)
    const int ahead = ROOM || i + 1 < nsl ? i + 1 : i;
    first_product(true_type{}, true_type{});
    middle();
    keep();
    const unsigned char* next = after(stage);
    second_product(next, ahead, i + 2, true_type{});      // (behind the last slice the reads ahead are of a stage nobody fills: unused)
    stage = next;
  }
  // the last slice through W2
#pragma unroll
  for (int k = 0; k < PACKS; ++k) activate(k);
#pragma unroll
  for (int j = 0; j < kAhead; ++j) w[j] = fetch2(stage, j);
  second_product(stage, nsl, 0, false_type{});
  __syncthreads();

  // ---- lane (n, q) holds channels 16 m + 4 q + 0..3 of its pixels
  tile = reinterpret_cast<bf16_t*>(mlp_lds);
  if (a.splits > 1) {
    float* part = a.partial + static_cast<size_t>(blockIdx.y) * C * a.padded + blockIdx.x * S::PX + p_lane;
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int t = 0; t < NT; ++t) part[static_cast<size_t>(16 * m + 4 * q + r) * a.padded + t] = acc[m][t][r];
    return;
  }
  // The result of the second product goes back through LDS, rounded to bfloat16 as nn.Linear leaves it, and meets the
  // layer scale and the shortcut on the way out.
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const uint2 b2 = *reinterpret_cast<const uint2*>(a.b2 + 16 * m + 4 * q);
    float bias[4];
    unpack2<bf16_t>(b2.x, bias[0], bias[1]);
    unpack2<bf16_t>(b2.y, bias[2], bias[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bf16_t* dst = tile + (16 * m + 4 * q + r) * S::kPitch + p_lane;
      if constexpr (NT == 2) *reinterpret_cast<uint32_t*>(dst) = pack_bf16x2(acc[m][0][r] + bias[r], acc[m][NT - 1][r] + bias[r]);
      else *dst = f32_to_bf16(acc[m][0][r] + bias[r]);
    }
  }
  __syncthreads();
  auto scale = [&](int c) { return a.gamma != nullptr ? bf16_to_f32(a.gamma[c]) : 1.f; };
  auto finish2 = [](uint32_t y, uint32_t s, float g) {
    float y0, y1, s0, s1;
    unpack2<bf16_t>(y, y0, y1);
    unpack2<bf16_t>(s, s0, s1);
    return pack_bf16x2(fmaf(g, y0, s0), fmaf(g, y1, s1));
  };
  if (a.vec == 8) {
    for_pixels(integral_constant<int, 8>{}, [&](size_t at) { return *reinterpret_cast<const uint4*>(a.shortcut + at); },
               [&](const uint4& s, int c, size_t at, int src) {
                 const uint2 y0 = *reinterpret_cast<const uint2*>(tile + src), y1 = *reinterpret_cast<const uint2*>(tile + src + 4);
                 const float g = scale(c);
                 *reinterpret_cast<uint4*>(a.out + at) =
                     uint4{finish2(y0.x, s.x, g), finish2(y0.y, s.y, g), finish2(y1.x, s.z, g), finish2(y1.y, s.w, g)};
               });
  } else if (a.vec == 4) {
    for_pixels(integral_constant<int, 4>{}, [&](size_t at) { return *reinterpret_cast<const uint2*>(a.shortcut + at); },
               [&](const uint2& s, int c, size_t at, int src) {
                 const uint2 y = *reinterpret_cast<const uint2*>(tile + src);
                 const float g = scale(c);
                 *reinterpret_cast<uint2*>(a.out + at) = uint2{finish2(y.x, s.x, g), finish2(y.y, s.y, g)};
               });
  } else {
    for_pixels(integral_constant<int, 1>{}, [&](size_t at) { return a.shortcut[at]; },
               [&](bf16_t s, int c, size_t at, int src) {
                 a.out[at] = f32_to_bf16(fmaf(scale(c), bf16_to_f32(tile[src]), bf16_to_f32(s)));
               });
  }
}

// The sums over the hidden units of `splits` workgroups, added in order, and the end of the block.  One thread per
// channel and pixel; grid (ceil(pixels / 256), C).
__global__ void __launch_bounds__(256) block_mlp_combine_kernel(MlpArgs a, int C) {
  const int p = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
  if (p >= a.pixels) return;
  const float* part = a.partial + static_cast<size_t>(c) * a.padded + p;
  float v = 0.f;
#pragma unroll 16
  for (int s = 0; s < a.splits; ++s) v += part[static_cast<size_t>(s) * C * a.padded];
  const int b = p / a.HW;
  const size_t at = (static_cast<size_t>(b) * C + c) * a.HW + (p - b * a.HW);
  const float g = a.gamma != nullptr ? bf16_to_f32(a.gamma[c]) : 1.f;
  a.out[at] = f32_to_bf16(fmaf(g, v + bf16_to_f32(a.b2[c]), bf16_to_f32(a.shortcut[at])));
}

}  // namespace wt
