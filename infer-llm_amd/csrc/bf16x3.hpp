// bf16x3.hpp — a float as three bf16 numbers that add up to it exactly, and
// the products of two such sums on bf16 MFMAs (gemm_bf16x3.hip,
// attn_bf16x3.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

namespace ikv::pieces {

typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// f(std::integral_constant<int, i>) for i = 0 .. N-1, in order.
template <int N, int I = 0, class F>
__device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

// 8 floats x = p[0] + p[1] + p[2]: each piece the bf16 nearest to what the
// ones before it leave (8 + 8 + 8 bits; both residues are exact floats, the
// last fits bf16 as it stands). Exact for |x| from 2^-109 up to bf16's largest
// and for many smaller ones (bf16 values and all whose last bit is 2^-133 or
// above; the MFMAs keep denormals). What the last piece drops of a smaller x
// is in the low halfs of `lost` (see any_lost); a larger, infinite or NaN x
// leaves a NaN among the pieces.
struct Pieces {
  bf16x8 p[3];
};
constexpr int kSplitOps = 48;  // VALU instructions of split8, as scheduled (it has 49)

__device__ __forceinline__ void split2(float a, float b, unsigned &h, unsigned &m, unsigned &l,
                                       unsigned &lost) {
  h = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{a, b}, bf16x2));
  const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xffff0000u);
  m = __builtin_bit_cast(unsigned, __builtin_convertvector(floatx2{ra, rb}, bf16x2));
  const float sa = ra - __uint_as_float(m << 16), sb = rb - __uint_as_float(m & 0xffff0000u);
  l = __builtin_amdgcn_perm(__float_as_uint(sb), __float_as_uint(sa), 0x07060302u);
  lost |= __float_as_uint(sa) | __float_as_uint(sb);
}
// PIN: what is dropped is collected with the last piece, so that the third
// residues need no registers past it (GEMM loops; one chain through `lost` for
// all splits was 2% slower there, and straight-line code schedules better
// without).
template <bool PIN>
__device__ __forceinline__ Pieces split8(floatx4 u, floatx4 v, unsigned &lost) {
  uintx4 q[3];
  unsigned t = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    unsigned h, m, l;
    if (e < 2)
      split2(u[2 * e], u[2 * e + 1], h, m, l, t);
    else
      split2(v[2 * e - 4], v[2 * e - 3], h, m, l, t);
    q[0][e] = h;
    q[1][e] = m;
    q[2][e] = l;
  }
  lost |= t;
  if constexpr (PIN) asm("" : "+v"(q[2][3]), "+v"(lost));
  return Pieces{{__builtin_bit_cast(bf16x8, q[0]), __builtin_bit_cast(bf16x8, q[1]),
                 __builtin_bit_cast(bf16x8, q[2])}};
}

// Whether any of the wave's splits dropped bits (a NaN may count, too).
__device__ __forceinline__ bool any_lost(unsigned lost) {
  return __builtin_amdgcn_ballot_w64((lost & 0xffffu) != 0) != 0;
}

// The six products formed, small ones first (pieces of A, of B).
constexpr int kPieceA[6] = {2, 0, 1, 1, 0, 0}, kPieceB[6] = {0, 2, 1, 0, 1, 0};

}  // namespace ikv::pieces
