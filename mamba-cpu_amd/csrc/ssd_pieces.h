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
// The split is that of bf16x3 products, Henry, Tang and Heinecke, "Leveraging
// the bfloat16 Artificial Intelligence Datatype For Higher-Precision
// Computations", ARITH 2019.
// The split holds a value to 2^-24 of itself, or to 2^-134 where that is more
// (below about 2^-110 the last pieces are bf16 subnormals).
// A product in pieces of an infinite factor is NaN: infinity times the other's
// pieces, of which some are zero or of the other sign. So is one of a finite value
// above the largest bf16, whose first piece is infinite. No result that such a
// factor enters is finite, and where a workgroup ends with one that is not, it
// does its work again in float32 (spoil).
#pragma once

#include <type_traits>

#include "mcpu_common.h"

namespace mcpu {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <typename T> constexpr int kPieces = sizeof(T) == 4 ? 3 : (std::is_same_v<T, bf16> ? 1 : 2);

// Two floats into NP pairs of bf16 (element 0 in the low half). F32: of three pieces
// the first is held to the largest bf16, so that their sum is every finite value;
// an infinity is then that, infinity, NaN (in two pieces infinity, NaN; whole_of).
template <int NP, bool F32 = false> __device__ __forceinline__ void split2(float a, float b, uint32_t (&o)[NP]) {
  const float most = __builtin_bit_cast(float, 0x7f7f0000u);
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    if (F32 && NP == 3 && i == 0)
      o[i] = pack_bf16x2(__builtin_amdgcn_fmed3f(a, -most, most), __builtin_amdgcn_fmed3f(b, -most, most));
    else
      o[i] = pack_bf16x2(a, b);
    if (i + 1 < NP) {
      a -= __builtin_bit_cast(float, o[i] << 16);
      b -= __builtin_bit_cast(float, o[i] & 0xffff0000u);
    }
  }
}
template <int NP, bool F32 = false>
__device__ __forceinline__ void split4(const float (&v)[4], uint2 (&o)[NP]) {
  uint32_t lo[NP], hi[NP];
  split2<NP, F32>(v[0], v[1], lo);
  split2<NP, F32>(v[2], v[3], hi);
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

// Element e of a lane's eight, its pieces put back together (here, not ahead of a
// loop that the pieces do not change in: registers).
template <int NP> __device__ __forceinline__ float whole_of(const Frag<NP>& f, int e) {
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    uint32_t u = f.u[i][e >> 1];
    asm volatile("" : "+v"(u));
    const float w = __builtin_bit_cast(float, e & 1 ? u & 0xffff0000u : u << 16);
    if (i == 0) v = w;
    else if (i + 1 < NP || w == w) v += w;   // the last piece of an infinity is NaN
  }
  return v;
}

// c + A B over 32 terms: in pieces, the small products first, or with F32 on the
// float32 unit (term 4 k + q of its step e is element e of quarter q, in A and B
// alike).
template <bool F32 = false, int NA, int NB>
__device__ __forceinline__ v4f mma32(const Frag<NA>& a, const Frag<NB>& b, v4f c) {
  if constexpr (F32) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(whole_of(a, e), whole_of(b, e), c, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);  // one term of each lane at a time: registers
    }
  } else {
#pragma unroll
    for (int order = 2; order >= 0; --order)
#pragma unroll
      for (int i = 0; i < NA; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          if (i + j == order)
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a.u[i]),
                                                        __builtin_bit_cast(bf16x8, b.u[j]), c, 0, 0, 0);
  }
  return c;
}

// Waits for the matrix cores' last results. The compiler does so by itself, but
// where the products sit under conditions it counts along the longest way to their
// use, and a tile whose successors were skipped would be read before it is written.
template <int NT> __device__ __forceinline__ void mma_wait(v4f (&acc)[NT]) {
  static_assert(NT == 4 || NT == 2, "tiles");
  if constexpr (NT == 4) asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]), "+v"(acc[2]), "+v"(acc[3]));
  else asm volatile("s_nop 15" : "+v"(acc[0]), "+v"(acc[1]));
}

// sum + 0 v: no longer 0 once a v was not finite.
__device__ __forceinline__ float spoil(float sum, float v) { return fmaf(v, 0.f, sum); }

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
