// Matrix-core helpers: 16x16x32 bf16 products and transposed LDS reads.
#pragma once
#include "common.h"

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

__device__ __forceinline__ f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
      __builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
      0);
}

// An operand whose 8 elements lie in 8 successive LDS rows: 16 lanes
// address a 4 x 16 block (lane i: row i / 4, columns 4 (i % 4) ..) and
// each gets one of its columns; the second block is ``down`` further.
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
__device__ __forceinline__ u32x4 load_columns(const unsigned short* p,
                                              int down) {
  const uint2 a = __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
  const uint2 b = __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + down)));
  return u32x4{a.x, a.y, b.x, b.y};
}

// The same of bytes: lane i addresses 8 of row i / 2 (columns 8 (i % 2) ..) of
// 8 rows of 16, and gets its column of all of them.
typedef __attribute__((ext_vector_type(2))) int s32x2;
typedef __attribute__((address_space(3))) s32x2 lds_s32x2;
__device__ __forceinline__ uint2 load_byte_columns(const char* p) {
  return __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_s32x2*)p));
}

// what bf16 holds of four numbers
__device__ __forceinline__ f32x4 rounded(f32x4 v) {
  const unsigned a = to_bf16x2(v[0], v[1]), b = to_bf16x2(v[2], v[3]);
  return f32x4{__uint_as_float(a << 16), __uint_as_float(a & 0xffff0000u),
               __uint_as_float(b << 16), __uint_as_float(b & 0xffff0000u)};
}

// two floats as sums of bf16 numbers, hi + lo
__device__ __forceinline__ void split2(float a, float b, unsigned& hi,
                                       unsigned& lo) {
  hi = to_bf16x2(a, b);
  lo = to_bf16x2(a - __uint_as_float(hi << 16),
                 b - __uint_as_float(hi & 0xffff0000u));
}

// ... and of three, which hold all of a float's 24 bits
__device__ __forceinline__ void split3(float a, float b, unsigned& hi,
                                       unsigned& mid, unsigned& lo) {
  hi = to_bf16x2(a, b);
  split2(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xffff0000u),
         mid, lo);
}

__device__ __forceinline__ void split_into(float a, float b,
                                           unsigned (&parts)[2]) {
  split2(a, b, parts[0], parts[1]);
}
__device__ __forceinline__ void split_into(float a, float b,
                                           unsigned (&parts)[3]) {
  split3(a, b, parts[0], parts[1], parts[2]);
}

#define LOG2E 1.4426950408889634f
