// Device helpers shared by the prompt GEMM kernels (gemm.hip, gemm_small.hip).
#pragma once

#include "common.hpp"

namespace prg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Two f32 -> packed bf16 pair, round to nearest even (v_cvt_pk_bf16_f32).
__device__ inline uint32_t pack_bf16(float lo, float hi) {
  const bf16x2 v = {static_cast<__bf16>(lo), static_cast<__bf16>(hi)};
  return __builtin_bit_cast(uint32_t, v);
}

// One Q4 word (8 nibbles, nibble j = column j) -> 8 bf16(s*q + b) in column
// order. s*q is exact in f32 (8-bit by 4-bit significands), so the fma rounds
// once, exactly like the reference's separate multiply and add.
__device__ inline uint4 dequant_word(uint32_t w, float s, float b) {
  uint32_t lo = w & 0x0F0F0F0Fu;         // columns 0, 2, 4, 6 in bytes 0..3
  uint32_t hi = (w >> 4) & 0x0F0F0F0Fu;  // columns 1, 3, 5, 7
  // Hide the masks from the optimiser so each byte converts with one
  // v_cvt_f32_ubyteN instead of a bit-field extract plus a convert.
  asm("" : "+v"(lo), "+v"(hi));
  uint4 r;
  r.x = pack_bf16(fmaf(s, static_cast<float>(lo & 0xffu), b), fmaf(s, static_cast<float>(hi & 0xffu), b));
  r.y = pack_bf16(fmaf(s, static_cast<float>((lo >> 8) & 0xffu), b), fmaf(s, static_cast<float>((hi >> 8) & 0xffu), b));
  r.z = pack_bf16(fmaf(s, static_cast<float>((lo >> 16) & 0xffu), b), fmaf(s, static_cast<float>((hi >> 16) & 0xffu), b));
  r.w = pack_bf16(fmaf(s, static_cast<float>(lo >> 24), b), fmaf(s, static_cast<float>(hi >> 24), b));
  return r;
}

constexpr uint32_t kBufferWord3 = 0x00020000;  // raw buffer descriptor, 32-bit data format

__device__ inline __amdgpu_buffer_rsrc_t buffer_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, kBufferWord3);
}

constexpr uint32_t kLdsBytes = 160 * 1024;

// One direct-to-LDS load: 16 bytes per lane at LDS address m0 + 16 * lane.
// m0 is written only here; nothing else in the kernel reads it (no indirect
// register indexing or GWS / ordered-count operations).
__device__ inline void lds_load16(__amdgpu_buffer_rsrc_t r, uint32_t lds_addr, uint32_t voff, uint32_t soff) {
  asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
               :
               : "s"(lds_addr), "v"(voff), "s"(r), "s"(soff)
               : "memory", "m0");
}
// s_waitcnt with vmcnt <= n and the other counters left alone (gfx9 encoding:
// vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8).
#define PRG_WAIT_VMCNT(n) \
  __builtin_amdgcn_s_waitcnt(((n) & 15) | (7 << 4) | (15 << 8) | ((((n) >> 4) & 3) << 14))

}  // namespace prg
