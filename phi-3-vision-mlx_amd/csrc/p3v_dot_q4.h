// 8 repacked 4-bit weights . 8 bf16 activations: shared by k_gemv3_q4 (p3v_gemv_q4.hip, which documents the layout) and the
// o_proj half of k_attn_decode128_o4 (p3v_attention.hip), which must repeat the GEMV's arithmetic bit for bit.
#pragma once
#include "p3v_common.h"

typedef __bf16 q4_pair_t __attribute__((ext_vector_type(2)));
typedef __bf16 q4_oct_t __attribute__((ext_vector_type(8)));

// 8 weights (one repacked dword) . 8 activations -> += sum_k x_k (128 + q_k)
__device__ __forceinline__ float dot8_q4(uint32_t r, u32x4_t x, float acc) {
  const q4_oct_t xv = __builtin_bit_cast(q4_oct_t, x);
  // v_and_or_b32 takes no literal: with the constants written out hipcc makes an and and an or of each (15 instead of 11 instructions
  // per dword).  One scalar and one vector register may be read, so that is where they are put.
  uint32_t mask = 0x000F000Fu, magic = 0x43004300u;
  asm("" : "+s"(mask), "+v"(magic));
  const uint32_t p0 = (r & mask) | magic, p1 = ((r >> 4) & mask) | magic;
  const uint32_t p2 = ((r >> 8) & mask) | magic, p3 = ((r >> 12) & mask) | magic;
  // (each dword goes through an asm no-op before it is viewed as a bf16 pair: hipcc 7.2 folds such bit_casts, see dot8)
  uint32_t q0 = p0, q1 = p1, q2 = p2, q3 = p3;
  asm("" : "+v"(q0), "+v"(q1), "+v"(q2), "+v"(q3));
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(q4_pair_t, q0), __builtin_shufflevector(xv, xv, 0, 1), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(q4_pair_t, q1), __builtin_shufflevector(xv, xv, 2, 3), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(q4_pair_t, q2), __builtin_shufflevector(xv, xv, 4, 5), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(q4_pair_t, q3), __builtin_shufflevector(xv, xv, 6, 7), acc, false);
  return acc;
}

// += the sum of 8 activations (the pair of ones goes through a register: as a constant hipcc may encode it as an inline 1.0, which is one bf16 only)
__device__ __forceinline__ float sum8_q4(u32x4_t x, float acc) {
  const q4_oct_t xv = __builtin_bit_cast(q4_oct_t, x);
  uint32_t ones = 0x3F803F80u;
  asm("" : "+v"(ones));
  const q4_pair_t o = __builtin_bit_cast(q4_pair_t, ones);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(xv, xv, 0, 1), o, acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(xv, xv, 2, 3), o, acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(xv, xv, 4, 5), o, acc, false);
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(xv, xv, 6, 7), o, acc, false);
}

// one 16-weight piece of a row: acc + scale sum_k x_k q_k + bias X, X = sum_k x_k (the - 128 X of the pairs 128 + q opens the chain)
__device__ __forceinline__ float piece_q4(uint32_t w0, uint32_t w1, uint32_t sb, u32x4_t xa, u32x4_t xb, float X, float acc) {
  const float S = dot8_q4(w1, xb, dot8_q4(w0, xa, -128.f * X));
  return fmaf(bf16lo(sb), S, fmaf(bf16hi(sb), X, acc));
}
