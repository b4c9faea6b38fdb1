// moe_tile.h — where the pieces of the 256 x 256 expert tile lie in memory (moe_grouped.hip); plain arithmetic, which a host test walks.
#pragma once
#include <cstdint>

#ifdef __HIPCC__
#define CHRONOS_HD __host__ __device__ __forceinline__
#else
#define CHRONOS_HD inline
#endif

namespace chronos {
namespace hy {

// Byte offset in one expert's matrix [N, K] (bfloat16, below 2 GiB) of what a lane loads for piece i (0 .. 3) of 32 rows (group wave = 0 .. 7), k-step 0;
// step kt lies 128 kt bytes further.  The piece holds 8 rows of 128 bytes, permuted by 16-byte pieces.  Rows past the end (a last tile may
// hold 128) repeat the last one: a buffer descriptor's range check need not see the scalar part of an address, and nothing is read
// past the matrix this way.  Their products are not stored.
CHRONOS_HD uint32_t moe_weight_offset(int tn, int wave, int i, int lane, int N, int K) {
    const int in = lane >> 3, row = tn * 256 + 32 * wave + 8 * i + in;
    return ((uint32_t)(row < N ? row : N - 1) * (uint32_t)K + (uint32_t)(((lane & 7) ^ in) * 8)) * 2;
}

}  // namespace hy
}  // namespace chronos
