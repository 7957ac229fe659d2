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

}  // namespace wt
