// Matrix-core types and the loads that go straight from memory into LDS, shared by the kernels around the WTConv layer.
#pragma once

#include "common.h"

namespace wt {

#ifdef WT_EMULATE
typedef ::emu::bf16x8 mat_frag;
typedef ::emu::f32x4 mat_acc;
typedef unsigned char* lds_addr;
#define WT_LDS_ADDR(p) (p)
#else
typedef __bf16 mat_frag __attribute__((ext_vector_type(8)));
typedef float mat_acc __attribute__((ext_vector_type(4)));
typedef uint32_t lds_addr;
#define WT_LDS_ADDR(p) \
  static_cast<uint32_t>(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) unsigned char*)(p)))
#endif

__device__ __forceinline__ mat_frag frag_of(const uint4& v) { return __builtin_bit_cast(mat_frag, v); }

// 64 granules of 16 bytes straight from memory (a uniform base and a byte offset per lane) into LDS: lane i's go to
// dst + 16 i.  (Issued as one instruction; the caller counts it in vmcnt.)
__device__ __forceinline__ void granules_to_lds(const void* base, uint32_t offset, lds_addr lds_dst) {
#ifdef WT_EMULATE
  memcpy(lds_dst + 16 * (threadIdx.x & (kWave - 1)), static_cast<const unsigned char*>(base) + offset, 16);
#else
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_dst), "v"(offset), "s"(base)
               : "memory", "m0");
#endif
}

// Four values of one column of a row-major tile of 16-bit values in LDS: the 16 lanes that share lane / 16 each name four
// neighbouring values, lane i those of row i / 4 of four and of the columns 4 (i % 4) ... of sixteen; lane i gets column i,
// rows 0 to 3.  (ds_read_b64_tr_b16.)
__device__ __forceinline__ uint2 column_of_4(const bf16_t* p) {
#ifdef WT_EMULATE
  return ::emu::column_of_4(p);
#else
  typedef short four __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) four*)(p)));
#endif
}

// Waits until at most N of this wave's loads are on their way and its LDS reads have arrived, then for the workgroup.
template <int N>
__device__ __forceinline__ void arrive_and_wait() {
#ifdef WT_EMULATE
  __syncthreads();
#else
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
#endif
}

}  // namespace wt
