// Device helpers shared by the attention kernels (forward, backward).
#pragma once

#include "common.h"

namespace pdh {

// v_mfma_f32_16x16x32: lane l holds A[l % 16][8 (l / 16) + j] and
// B[8 (l / 16) + j][l % 16], j = 0..7, and receives D[4 (l / 16) + i][l % 16].
template <typename T>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c);

template <>
__device__ __forceinline__ f32x4 mfma16<__hip_bfloat16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                 0, 0);
}

template <>
__device__ __forceinline__ f32x4 mfma16<_Float16>(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0,
                                                0);
}

// ------------------------------------------------ LDS staging for key tiles
//
// Key/value tiles are copied HBM -> LDS by direct buffer loads (no VGPR round
// trip): one buffer_load_dwordx4 ... lds writes 16 bytes per lane to
// M0 + 16 * lane, i.e. 1 KB contiguous per wave. Rows are D * 2 bytes with no
// padding; instead, the 16-byte slot that holds chunk c of row r is
// c ^ swz(r), each kernel choosing swz so that its operand reads hit
// distinct banks.

// (dma16 and wait_vmcnt0: dev.h)

// 4 bytes per lane, buffer -> LDS (lane i's dword lands at lds + 4 i).
__device__ __forceinline__ void dma4(rsrc_t r, unsigned char* lds, uint32_t voff, uint32_t soff) {
  // the low 32 bits of a generic LDS address are its LDS offset (no address-space cast needed)
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(reinterpret_cast<uintptr_t>(lds)));
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(m0), "v"(voff), "s"(r), "s"(soff)
               : "memory", "m0");
#pragma clang diagnostic pop
}

// (ds_read_tr16: dev.h)

}  // namespace pdh
