// Products on the bf16 matrix cores at float32 accuracy, for the SSD scan.
//
// A float32 value is the sum of three bf16 values: its rounding to bf16, that
// of what is left, and that of what is left then (8 + 8 + 8 significand bits;
// the last step is exact). An f16 value is the sum of two, a bf16 value of
// one. A product of two such sums keeps the terms down to 2^-18 of the whole
// (piece numbers i + j <= 2); the terms left out are below 2^-26, under
// float32's own rounding, and every term is accumulated in float32. Six
// v_mfma_f32_16x16x32_bf16 replace the eight v_mfma_f32_16x16x4_f32 of a
// float32 product over 32 terms at half the cycles each, three where one side
// is stored in bf16, one where both are: 2.7, 5.3 and 16 times the rate.
// An infinite float32 operand splits into inf, NaN, NaN: products of infinities
// are NaN where the float32 unit gives inf or NaN.
#pragma once

#include "mcpu_common.h"

namespace mcpu {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T> constexpr int kPieces = sizeof(T) == 4 ? 3 : (std::is_same_v<T, bf16> ? 1 : 2);

// Two floats into NP pairs of bf16 (element 0 in the low half).
template <int NP> __device__ __forceinline__ void split2(float a, float b, uint32_t (&o)[NP]) {
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    o[i] = pack_bf16x2(a, b);
    if (i + 1 < NP) {
      a -= __builtin_bit_cast(float, o[i] << 16);
      b -= __builtin_bit_cast(float, o[i] & 0xffff0000u);
    }
  }
}
template <int NP> __device__ __forceinline__ void split4(const float (&v)[4], uint2 (&o)[NP]) {
  uint32_t lo[NP], hi[NP];
  split2<NP>(v[0], v[1], lo);
  split2<NP>(v[2], v[3], hi);
#pragma unroll
  for (int i = 0; i < NP; ++i) o[i] = make_uint2(lo[i], hi[i]);
}

// A lane's part of an operand of one v_mfma_f32_16x16x32_bf16: eight terms of
// its row (A) or column (B) l % 16, NP pieces each. Which eight of the 32 terms
// a lane (its quarter l / 16) holds is free as long as A and B agree.
template <int NP> struct Frag { u32x4 u[NP]; };

template <int NP> __device__ __forceinline__ Frag<NP> split8(const float (&v)[8]) {
  Frag<NP> f;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    uint32_t o[NP];
    split2<NP>(v[2 * k], v[2 * k + 1], o);
#pragma unroll
    for (int i = 0; i < NP; ++i) f.u[i][k] = o[i];
  }
  return f;
}

// c + A B over 32 terms, the small products first.
template <int NA, int NB>
__device__ __forceinline__ v4f mma32(const Frag<NA>& a, const Frag<NB>& b, v4f c) {
#pragma unroll
  for (int order = 2; order >= 0; --order)
#pragma unroll
    for (int i = 0; i < NA; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j)
        if (i + j == order)
          c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.u[i]),
                                                      __builtin_bit_cast(bf16x8, b.u[j]), c, 0, 0, 0);
  return c;
}

// LDS tiles of bf16 pieces: piece i of element (row, col) at i * plane + row *
// ld + col, in rows of 64 or 128 columns padded by 16 bytes, so that the 16
// rows a wave reads at a time fall on different banks.
constexpr int kLdP = 64 + 8;     // rows of up to 64 columns
constexpr int kLdN = 128 + 8;    // rows of up to 128 columns
constexpr int kPlaneP = 64 * kLdP;
constexpr int kPlaneN = 64 * kLdN;

// Terms along the row: lane (r, q) takes columns 8 q .. 8 q + 8 of row r of
// the 16-row, 32-column block at s.
template <int NP>
__device__ __forceinline__ Frag<NP> frag_row(const uint16_t* s, int ld, int plane) {
  const int lane = threadIdx.x & 63;
  const uint16_t* p = s + (lane & 15) * ld + 8 * (lane >> 4);
  Frag<NP> f;
#pragma unroll
  for (int i = 0; i < NP; ++i) f.u[i] = *reinterpret_cast<const u32x4*>(p + i * plane);
  return f;
}

// Terms along the column: lane (r, q) takes rows 4 q .. 4 q + 4 and 16 + 4 q ..
// 16 + 4 q + 4 of column r of the 32-row, 16-column block at s. These are the
// rows a lane holds of two stacked 16 x 16 products, so such a product, split in
// registers, is the matching other operand. ds_read_b64_tr_b16 transposes
// within 16 lanes: lane i reads four columns 4 (i % 4) of row i / 4 and gets
// column i of the four rows.
__device__ __forceinline__ uint2 lds_tr4(const uint16_t* p) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_bit_cast(
      uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(p)));
}
template <int NP>
__device__ __forceinline__ Frag<NP> frag_col(const uint16_t* s, int ld, int plane) {
  const int lane = threadIdx.x & 63, i16 = lane & 15, q = lane >> 4;
  const uint16_t* p = s + (4 * q + (i16 >> 2)) * ld + 4 * (i16 & 3);
  Frag<NP> f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const uint2 a = lds_tr4(p + i * plane), b = lds_tr4(p + i * plane + 16 * ld);
    f.u[i] = u32x4{a.x, a.y, b.x, b.y};
  }
  return f;
}

// Terms along the row in frag_col's order: columns 4 q .. 4 q + 4 and 16 + 4 q ..
// 16 + 4 q + 4 of row r.
template <int NP>
__device__ __forceinline__ Frag<NP> frag_row_as_col(const uint16_t* s, int ld, int plane) {
  const int lane = threadIdx.x & 63;
  const uint16_t* p = s + (lane & 15) * ld + 4 * (lane >> 4);
  Frag<NP> f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const uint2 a = *reinterpret_cast<const uint2*>(p + i * plane);
    const uint2 b = *reinterpret_cast<const uint2*>(p + i * plane + 16);
    f.u[i] = u32x4{a.x, a.y, b.x, b.y};
  }
  return f;
}

// The same eight terms of two stacked products' registers (rows 4 q + e of
// tiles lo and hi).
template <int NP> __device__ __forceinline__ Frag<NP> frag_acc(const v4f& lo, const v4f& hi) {
  const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return split8<NP>(v);
}

// Eight consecutive elements from memory (16-byte aligned), zero unless ok.
template <typename T> __device__ __forceinline__ Frag<kPieces<T>> frag_mem(const T* src, bool ok) {
  Frag<kPieces<T>> f;
  if constexpr (std::is_same_v<T, bf16>) {
    f.u[0] = ok ? *reinterpret_cast<const u32x4*>(src) : u32x4{0, 0, 0, 0};
  } else {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.f;
    if (ok) {
      ld4_elem<T>(src, 0, v);
      ld4_elem<T>(src, 4, v + 4);
    }
    f = split8<kPieces<T>>(v);
  }
  return f;
}

}  // namespace mcpu
