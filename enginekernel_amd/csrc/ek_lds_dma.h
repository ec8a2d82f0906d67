// Direct global-to-LDS loads (LDS-DMA) and the operand types of the kernels
// that feed matrix products from LDS tiles (ek_prefill.hip, ek_gemm.hip).
//
// A load brings 16 bytes per lane to the LDS bytes from m0 on, lane after
// lane, and is counted by the vector memory counter alone; nothing the
// compiler sees depends on it, so a counted wait and a barrier come before its
// bytes are read. The compiler's own builtin would wait for every load in
// flight before any LDS read, which leaves no stages ahead, so these are
// written out. Its hazard pass does not look into them: the load may read m0
// from one wait state after the scalar write on, hence the s_nop (1 x 16000 tokens
// of attention 1.890 ms without it, 1.889 with). m0 is a reserved register that cannot be named
// as clobbered; a kernel that includes this has no other use of it.
#pragma once

#include <stdint.h>

#include "ek_common.h"

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) u32x4_t lds_u32x4_t;
typedef __attribute__((address_space(3))) char lds_char_t;

// Rows of CH 16-byte chunks: row r's are permuted by an xor with this, so that rows
// which share banks differ in it (conflict-free reads of a chunk column). For r0 a
// multiple of 64 / CH, a load's rows, lds_xor(r0 + i) = lds_xor(r0) ^ lds_xor(i).
template <int CH>
__device__ __forceinline__ constexpr int lds_xor(int r) { return (r / (16 / CH)) & (CH - 1); }

// from base + voff
__device__ __forceinline__ void lds_dma16(uint32_t lds, const char* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory");
}

// the same, non-temporal: bytes that one workgroup reads once
__device__ __forceinline__ void lds_dma16_nt(uint32_t lds, const char* base, uint32_t voff) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds), "v"(voff), "s"(base) : "memory");
}

// from a 64-bit address per lane
__device__ __forceinline__ void lds_dma16_addr(uint32_t lds, const char* addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(addr) : "memory");
}
