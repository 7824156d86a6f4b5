// MFMA fragment helpers shared by the gather-GEMM-scatter kernels.
#pragma once

#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>

#include "fgms_internal.h"

namespace fgms {

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float4v __attribute__((ext_vector_type(4)));
typedef float float16v __attribute__((ext_vector_type(16)));
typedef int int4v __attribute__((ext_vector_type(4)));

template <typename T> struct Elem;
template <> struct Elem<__half> { static constexpr int per_chunk = 8; };
template <> struct Elem<float> { static constexpr int per_chunk = 4; };

template <typename T>
__device__ __forceinline__ void mma(float16v &acc, const int4v &a, const int4v &b) {
  if constexpr (sizeof(T) == 2) {
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8, a),
                                                 __builtin_bit_cast(half8, b), acc, 0, 0, 0);
  } else {
    const float4v fa = __builtin_bit_cast(float4v, a), fb = __builtin_bit_cast(float4v, b);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[0], fb[0], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[1], fb[1], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[2], fb[2], acc, 0, 0, 0);
    acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[3], fb[3], acc, 0, 0, 0);
  }
}

__device__ __forceinline__ float swap_with_neighbour(float v) {
  // lane ^ 1 inside each quad: quad_perm [1, 0, 3, 2]
  return __builtin_bit_cast(
      float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, true));
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef int int2v __attribute__((ext_vector_type(2)));

// Four fp32 values as P bf16 parts each, largest first, packed as they go to LDS.  P = 2: x = hi + lo + O(2^-17 x).
// P = 3: x = h + m + l exactly -- h is x cut off after 8 bits (which no finite value overflows), m the rest rounded to 8,
// and what is left of it fits 8.  (Published as a way to fp32 results on narrower matrix units: Henry, Tang, Heinecke, "Leveraging the
// bfloat16 artificial intelligence datatype for higher-precision computations", ARITH 2019.)
// P = 3: `lost` is set if a value's last part is not zero and below 2^-126, where bf16 numbers may end before its last bit does
// (values below 2^-102).  (Asked of that part and not of x, which would stay in registers for it: the least size met instead took
// 35 more of them in the weight gradient's loop, 64 x 64 over 200 k voxels 202 us, this 181, neither 174.)
template <int P>
__device__ __forceinline__ void split_parts(const float4v &x, int2v (&part)[P], bool &lost) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float float2v __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    float2v r = {x[2 * q], x[2 * q + 1]};
    if constexpr (P == 3) {
      const float x0 = r[0], x1 = r[1];      // (a bit cast of a vector's element takes element 0)
      const unsigned a = __builtin_bit_cast(unsigned, x0), b = __builtin_bit_cast(unsigned, x1);
      part[0][q] = (int)__builtin_amdgcn_perm(b, a, 0x07060302u);      // the upper halves of a, b
      r[0] -= __builtin_bit_cast(float, a & 0xffff0000u);
      r[1] -= __builtin_bit_cast(float, b & 0xffff0000u);
    } else {
      const int h = __builtin_bit_cast(int, __builtin_convertvector(r, bf16x2));
      part[0][q] = h;
      // (an infinite or NaN value stays in hi alone)
      const float h0 = __builtin_bit_cast(float, h << 16), h1 = __builtin_bit_cast(float, h & (int)0xffff0000);
      r[0] = __builtin_fabsf(h0) < __builtin_inff() ? r[0] - h0 : 0.f;
      r[1] = __builtin_fabsf(h1) < __builtin_inff() ? r[1] - h1 : 0.f;
    }
    const int m = __builtin_bit_cast(int, __builtin_convertvector(r, bf16x2));
    part[1][q] = m;
    if constexpr (P == 3) {
      r[0] -= __builtin_bit_cast(float, m << 16);
      r[1] -= __builtin_bit_cast(float, m & (int)0xffff0000);
      part[2][q] = __builtin_bit_cast(int, __builtin_convertvector(r, bf16x2));
      lost |= __builtin_amdgcn_classf(r[0], 0x90) | __builtin_amdgcn_classf(r[1], 0x90);      // (subnormal, of either sign)
    }
  }
}

// acc += a x b for operands of P parts, the small products first.  P = 2: all but lo x lo.  P = 3: all but l x l, which is
// below 2^-30 of the product, so that a single product is rounded once, as by fp32 arithmetic (without m x l and l x m, which
// reach 1.7 x 2^-23 of it, its error was up to 3.9 x 2^-24).  The small ones have an accumulator of their own, `low`, to be added
// at the end: the big one is then rounded once per 16 products.
template <int P>
__device__ __forceinline__ void mma_parts(float16v &acc, float16v &low, const bf16x8 (&a)[P], const bf16x8 (&b)[P]) {
#pragma unroll
  for (int rank = P == 3 ? 3 : 1; rank >= 0; --rank)
#pragma unroll
    for (int i = P - 1; i >= 0; --i) {
      if (i > rank || rank - i >= P) continue;
      float16v &to = P == 3 && rank > 0 ? low : acc;
      to = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[rank - i], to, 0, 0, 0);
    }
}

// Re-lays the weights into per-lane MFMA fragment order in the stream's
// workspace (see pack_weights_kernel) and returns the packed buffer.
int pack_weights_any(const GmsArgs &a, int S, const void **packed);
int num_cus();

}  // namespace fgms
