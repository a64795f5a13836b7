// What the kernels that stream a prompt's rows through the bf16 matrix cores share.
#pragma once
#include "common.hpp"

namespace lrqk {

typedef float gd_floatx16 __attribute__((ext_vector_type(16)));
typedef __bf16 gd_bf16x8 __attribute__((ext_vector_type(8)));
// 16 bytes of rows on their way to LDS (a native vector: arrays of the uint4 struct that are filled under a condition
// end up in scratch memory, with a wait behind every load)
typedef uint32_t gd_u32x4 __attribute__((ext_vector_type(4)));
typedef float gd_floatx4 __attribute__((ext_vector_type(4)));
typedef short gd_v4s __attribute__((ext_vector_type(4)));
typedef gd_v4s __attribute__((address_space(3))) * gd_lds_v4s;

// C tile of a 32x32 matrix product: lane l, element v -> row (the column is l % 32)
__device__ __forceinline__ int gd_mfma_row(int lane, int v) { return ((v >> 2) << 3) + ((lane >> 5) << 2) + (v & 3); }

// the row of lane 0 in element v; the upper half of a wave is 4 rows further
__device__ __forceinline__ constexpr int gd_mfma_row0(int v) { return ((v >> 2) << 3) + (v & 3); }

// Rows of a group are addressed by 32-bit byte offsets from the group's first row, an address that the whole wave
// shares (its wave's number made uniform by gd_wave): the load takes a scalar base and one register.  A 64-bit product
// per row and lane costs 16 cycles: 48 of them were a third of a step's vector instructions in the kernels that sum over
// the rows (32 heads of 32K bf16 rows, rank 32: K side's sums 64 -> 57 us, A_K 50 -> 46 us; three prompts of 2531 rows of
// 64: 19.2 -> 16.7 us; 16K rows at rank 64, A_K 38.6 -> 33.6 us).
__device__ __forceinline__ int gd_wave() { return __builtin_amdgcn_readfirstlane(wave_id()); }
template <typename V>
__device__ __forceinline__ V gd_at(const void* base, uint32_t bytes) {
  return *reinterpret_cast<const V*>((const char*)base + bytes);
}
// element `col` of row min(row, last) of a group of rows of r floats (r < 2^22)
__device__ __forceinline__ float gd_factor(const float* base, int row, int last, int r, int col) {
  return gd_at<float>(base, __umul24((uint32_t)min(row, last), 4u * (uint32_t)r) + 4u * (uint32_t)col);
}

// An fp32 number as the exact sum of three bf16 numbers (8 + 8 + 8 mantissa bits, by truncation), as the upper halves
// of fp32 bit patterns
__device__ __forceinline__ void gd_split3(float x, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
  hi = __float_as_uint(x) & 0xffff0000u;
  const float r1 = x - __uint_as_float(hi);  // exact
  mid = __float_as_uint(r1) & 0xffff0000u;
  const float r2 = r1 - __uint_as_float(mid);  // exact, at most 8 significant bits
  lo = __float_as_uint(r2) & 0xffff0000u;
}
__device__ __forceinline__ uint32_t gd_pack2(uint32_t a, uint32_t b) { return (a >> 16) | (b & 0xffff0000u); }

// the three pieces of eight fp32 numbers as operands of a 32x32x16 product
__device__ __forceinline__ void gd_split3x8(const float (&x)[8], gd_bf16x8 (&p)[3]) {
  uint32_t pc[3][8];
#pragma unroll
  for (int q = 0; q < 8; ++q) gd_split3(x[q], pc[0][q], pc[1][q], pc[2][q]);
#pragma unroll
  for (int k = 0; k < 3; ++k)
    p[k] = __builtin_bit_cast(gd_bf16x8, make_uint4(gd_pack2(pc[k][0], pc[k][1]), gd_pack2(pc[k][2], pc[k][3]),
                                                    gd_pack2(pc[k][4], pc[k][5]), gd_pack2(pc[k][6], pc[k][7])));
}

// A factor to its output's type.  bf16 by the conversion instruction: to nearest even like st_f32, whose test for NaN
// is a branch per value in the kernels that write whole factors.
__device__ __forceinline__ void gd_store(float* p, int64_t i, float v) { p[i] = v; }
__device__ __forceinline__ void gd_store(bf16_t* p, int64_t i, float v) { p[i].v = __builtin_bit_cast(uint16_t, (__bf16)v); }

// The first `rows` rows (32, or fewer at the end of a head) of a C tile to rows of r factors from `base` on.
template <typename OUT>
__device__ __forceinline__ void gd_store_tile(OUT* base, const gd_floatx16& c, int rows, int col, int half, int r) {
  if (col >= r) return;
  const uint32_t at = (uint32_t)(4 * half * r + col) * (uint32_t)sizeof(OUT);
  if (rows >= 32) {  // (wave-uniform)
#pragma unroll
    for (int v = 0; v < 16; ++v) gd_store((OUT*)((char*)(base + gd_mfma_row0(v) * r) + at), 0, c[v]);
  } else {
#pragma unroll
    for (int v = 0; v < 16; ++v)
      if (gd_mfma_row0(v) + 4 * half < rows) gd_store((OUT*)((char*)(base + gd_mfma_row0(v) * r) + at), 0, c[v]);
  }
}

}  // namespace lrqk
