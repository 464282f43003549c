// Tiles of the matrix-core attention kernels (attention_mfma.hip,
// attention_f32.hip): 64 positions x D bf16 in LDS as plain rows of D + 8, and
// the operands v_mfma_f32_32x32x16_bf16 takes from them.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ uint32_t pack2(float a, float b) {
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
// x = part 0 + part 1 + part 2 in bf16, two values a word (8 bits each, rounded
// to nearest: what is left is at most 2^-27 of x, or 2^-134, half of bf16's
// least subnormal, which the matrix cores keep).
__device__ __forceinline__ void split2(float u, float v, uint32_t& w0, uint32_t& w1, uint32_t& w2) {
  w0 = pack2(u, v);
  u -= __uint_as_float(w0 << 16), v -= __uint_as_float(w0 & 0xffff0000u);
  w1 = pack2(u, v);
  u -= __uint_as_float(w1 << 16), v -= __uint_as_float(w1 & 0xffff0000u);
  w2 = pack2(u, v);
}
// The same (of anything but -0), exactly from 2^-94 on, and every part of x's sign
// and not 0: each is the top 8 bits of the number next to what is left towards
// 0, and the last all of it.  An infinity among the values that x multiplies, or in
// x, then gives what it gives with x itself; nearest parts, which are 0 or of both
// signs, would make it NaN.
__device__ __forceinline__ void split2_towards0(float u, float v, uint32_t& w0, uint32_t& w1, uint32_t& w2) {
  auto next = [](float x) { return __builtin_elementwise_sub_sat(__float_as_uint(x), 1u); };
  auto high = [](uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); };
  uint32_t a = next(u), b = next(v);
  w0 = high(a, b);
  u -= __uint_as_float(a & 0xffff0000u), v -= __uint_as_float(b & 0xffff0000u);
  a = next(u), b = next(v);
  w1 = high(a, b);
  u -= __uint_as_float(a & 0xffff0000u), v -= __uint_as_float(b & 0xffff0000u);
  w2 = high(__float_as_uint(u), __float_as_uint(v));
}
// The value lane l ^ 32 holds.
__device__ __forceinline__ float other_half(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(threadIdx.x % 64 < 32 ? r[1] : r[0]);
}
__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

// A operand from a tile (rows of D + 8 bf16), M along its rows: rows
// r0 + lane % 32, k = columns 16 ks + 8 (lane / 32) + (0..7).
template <int D>
__device__ __forceinline__ bf16x8 frag_rows(const uint16_t* t, int r0, int ks) {
  const int lane = threadIdx.x % 64;
  return *reinterpret_cast<const bf16x8*>(t + (r0 + lane % 32) * (D + 8) + 16 * ks + 8 * (lane / 32));
}

// A operand from a tile, M along its columns: m = column d0 + lane % 32, k
// = the 16 rows of step ks in the order the accumulator's registers give the
// B operand (k-slot 8 h + e <-> row 16 ks + 8 (e / 4) + 4 h + e % 4, h =
// lane / 32).  ds_read_b64_tr_b16 hands lane i of each 16 element i % 4 of
// the 8-byte pieces addressed by lanes 4 k + i / 4; lane j here addresses row
// base + j / 4, columns dgrp + 4 (j % 4) + (0..3), so lane i receives rows
// base + (0..3) of column dgrp + i; two reads cover the eight rows.
template <int D>
__device__ __forceinline__ bf16x8 frag_tr(const uint16_t* t, int d0, int ks) {
  const int lane = threadIdx.x % 64, j = lane % 16;
  const int col = d0 + 16 * ((lane / 16) % 2) + 4 * (j % 4);
  const int row = 16 * ks + 4 * (lane / 32) + j / 4;
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + row * (D + 8) + col));
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(t + (row + 8) * (D + 8) + col));
  const s16x8 w = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, w);
}

}  // namespace
