// chunk_common.h — float32 operands on the bfloat16 matrix cores, for the chunked recurrences (chunk_scan.hip, gla_scan.hip).
#pragma once
#include "hybrid_common.h"

namespace chronos {
namespace hy {

__device__ __forceinline__ f32x4 mfma_16x16x32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x = h + m + l exactly: each term the bfloat16 nearest to what is left (the second remainder has 8 bits at most)
struct Terms {
    bf16x8 h, m, l;
};
__device__ __forceinline__ Terms split3(const float (&x)[8]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 t[3];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float a = x[2 * i], b = x[2 * i + 1];
#pragma unroll
        for (int k = 0; k < 3; ++k) t[k][i] = round_pair(a, b);
    }
    return {__builtin_bit_cast(bf16x8, t[0]), __builtin_bit_cast(bf16x8, t[1]), __builtin_bit_cast(bf16x8, t[2])};
}
__device__ __forceinline__ bf16x8 join8(bf16x4 a, bf16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// Where piece c (16 bytes) of row r of a tile with CPR pieces per row lies: c ^ spread<CPR>(r).  16 rows at the same c, and
// 4 rows at 4 neighbouring c, fall on different banks.  Depends on r % 16 only.
template <int CPR> __device__ __forceinline__ int spread(int r) {
    if constexpr (CPR >= 16) return ((r & 3) << 2) | ((r >> 2) & 3);
    else if constexpr (CPR == 8) return ((r & 2) << 1) | ((r >> 2) & 3);
    else if constexpr (CPR == 4) return (r >> 2) & 3;
    else return 0;
}

// a * b of two float32 operands in matrix layout (4 elements per lane, k = 4 g + e), as the six leading products of their terms:
// the other three are below 2^-26 of the result.  The two halves of a 32-deep instruction hold two of the six.
struct Terms4 {
    bf16x4 h, m, l;
};
__device__ __forceinline__ Terms4 split3(const f32x4& x) {
    const float v[8] = {x[0], x[1], x[2], x[3], 0.f, 0.f, 0.f, 0.f};
    const Terms t = split3(v);
    return {__builtin_shufflevector(t.h, t.h, 0, 1, 2, 3), __builtin_shufflevector(t.m, t.m, 0, 1, 2, 3), __builtin_shufflevector(t.l, t.l, 0, 1, 2, 3)};
}
__device__ __forceinline__ f32x4 mul_low(const Terms4& a, const Terms4& b, f32x4 c) {
    c = mfma_16x16x32(join8(a.m, a.h), join8(b.m, b.l), c);
    return mfma_16x16x32(join8(a.h, a.l), join8(b.m, b.h), c);
}
__device__ __forceinline__ f32x4 mul_high(const Terms4& a, const Terms4& b, f32x4 c) { return mfma_16x16x32(join8(a.h, a.m), join8(b.h, b.h), c); }

}  // namespace hy
}  // namespace chronos
