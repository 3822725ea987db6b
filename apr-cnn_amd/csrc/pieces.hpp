// fp32 values as sums of three bfloat16 pieces (see conv_split.hip).
#pragma once
#include "conv_common.hpp"

namespace aprnet {

typedef unsigned uintx2s __attribute__((ext_vector_type(2)));
typedef unsigned uintx4s __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2s __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8s __attribute__((ext_vector_type(8)));

constexpr int SP_CIB = 4;                      // channels of a group that is split and staged at a time

// two fp32 numbers -> their bfloat16 roundings, the first in the low half (v_cvt_pk_bf16_f32)
__device__ __forceinline__ unsigned split_round(float a, float b) {
    const bf16x2s h = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(unsigned, h);
}
__device__ __forceinline__ float split_lo(unsigned p) { return __builtin_bit_cast(float, p << 16); }
__device__ __forceinline__ float split_hi(unsigned p) { return __builtin_bit_cast(float, p & 0xffff0000u); }

// What is split lies SPLIT_SCALE times higher than the caller's values (the copies and the packed weights), the results are brought
// down again: the last bit of any fp32 number, 2^-149 at the least, then is one that a bfloat16 number can hold (2^-133).
constexpr float SPLIT_SCALE = 65536.f, SPLIT_UNSCALE = 1.f / (SPLIT_SCALE * SPLIT_SCALE);

// two fp32 numbers -> three words with their pieces
__device__ __forceinline__ void split_pair(float a, float b, unsigned& p1, unsigned& p2, unsigned& p3) {
    p1 = split_round(a, b);
    const float ra = a - split_lo(p1), rb = b - split_hi(p1);
    p2 = split_round(ra, rb);
    p3 = split_round(ra - split_lo(p2), rb - split_hi(p2));
}

// Bytes from a plane of `ld` fp32 values to the one `planes` further on, for the scalar offset of a buffer load, which is an unsigned 32-bit
// number: a signed product overflows from 2^31 bytes on, two planes of 2^28 values or seven of 77 million.
__host__ __device__ constexpr int plane_offset(int planes, int64_t ld) { return (int)(4u * (unsigned)planes * (unsigned)ld); }
// the largest ones that the rules of the two kernels let through: eight planes of fewer than 2^27 values, four of fewer than 2^28
static_assert((unsigned)plane_offset(7, (1 << 27) - 1) == 3758096356u && (unsigned)plane_offset(3, (1 << 28) - 1) == 3221225460u, "wraps nowhere");

}  // namespace aprnet
