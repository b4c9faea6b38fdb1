// rowdot_tile.h — 16 TT tokens by 16 NT output rows of h w^T in float32 sums, for projections to a few rows (hybrid_elementwise.hip) and routers (moe.hip).
#pragma once
#include "hybrid_common.h"

namespace chronos {
namespace hy {

// A workgroup of NWV waves, which split d (% 64 == 0): tokens from t0 on, output rows from n0 on; put(token, row, sum + bias) by one lane each, no barrier behind
template <int TT, int NT, int NWV, typename Put>
__device__ __forceinline__ void rowdot_tile(const uint16_t* __restrict__ h, const uint16_t* __restrict__ w, const float* __restrict__ bias, int64_t t0, int n0,
                                            int rows, int d, int n, f32x4 (&red)[NWV][TT * NT][64], Put&& put) {
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ln = lane & 15, g = lane >> 4;
    const uint16_t *hp[TT], *wp[NT];   // rows past the end repeat the last one and are not stored
#pragma unroll
    for (int i = 0; i < TT; ++i) hp[i] = h + min(t0 + 16 * i + ln, (int64_t)rows - 1) * d + 8 * g;
#pragma unroll
    for (int j = 0; j < NT; ++j) wp[j] = w + (int64_t)min(n0 + 16 * j + ln, n - 1) * d + 8 * g;
    f32x4 sum[TT][NT];
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) sum[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    constexpr int P = TT * NT == 1 ? 4 : 2;   // 64-element steps in flight
    for (int k0 = wv * 64; k0 < d; k0 += P * NWV * 64) {
        bf16x8 a[2 * P][TT], b[2 * P][NT];
#pragma unroll
        for (int u = 0; u < 2 * P; ++u) {
            const int k = k0 + (u >> 1) * NWV * 64 + (u & 1) * 32;
            if (k < d) {
#pragma unroll
                for (int i = 0; i < TT; ++i) a[u][i] = *reinterpret_cast<const bf16x8*>(hp[i] + k);
#pragma unroll
                for (int j = 0; j < NT; ++j) b[u][j] = *reinterpret_cast<const bf16x8*>(wp[j] + k);
            } else {
#pragma unroll
                for (int i = 0; i < TT; ++i) a[u][i] = bf16x8{};
#pragma unroll
                for (int j = 0; j < NT; ++j) b[u][j] = bf16x8{};
            }
        }
        // chains of four products at most, added up apart: the longer a chain, the more roundings at the size of its sum
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                f32x4 acc[P / 2];
#pragma unroll
                for (int q = 0; q < P / 2; ++q) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int u = 0; u < 2 * P; ++u) acc[u / 4] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][i], b[u][j], acc[u / 4], 0, 0, 0);
#pragma unroll
                for (int q = 1; q < P / 2; ++q) acc[0] += acc[q];
                sum[i][j] += acc[0];
            }
    }
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) red[wv][i * NT + j][lane] = sum[i][j];
    __syncthreads();
    for (int p = wv; p < TT * NT; p += NWV) {   // element r of a tile: token 4 g + r, output row ln
        f32x4 part[NWV];
#pragma unroll
        for (int u = 0; u < NWV; ++u) part[u] = red[u][p][lane];
#pragma unroll
        for (int o = NWV / 2; o > 0; o >>= 1)
#pragma unroll
            for (int u = 0; u < o; ++u) part[u] += part[u + o];
        const f32x4 v = part[0];
        const int r = n0 + 16 * (p % NT) + ln;
        const int64_t t = t0 + 16 * (p / NT) + 4 * g;
        if (r < n) {
            const float bv = bias != nullptr ? bias[r] : 0.f;
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (t + e < rows) put(t + e, r, v[e] + bv);
        }
    }
}

}  // namespace hy
}  // namespace chronos
