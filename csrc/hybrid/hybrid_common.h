// hybrid_common.h — helpers shared by the hybrid-decoder kernels (csrc/hybrid/*.hip).
//
// Every kernel is instantiated for two activation element types: bfloat16 travelling as raw 16-bit words
// (uint16_t, as in csrc/kernels) and float.  Whatever the activation type, residual stream, norms, recurrent state,
// gates, router and attention scores are float.
#pragma once
#include "chronos_act.h"
#include "chronos_hip.h"

namespace chronos {
namespace hy {

template <typename T> __device__ __forceinline__ float ld(const T* p);
template <> __device__ __forceinline__ float ld<float>(const float* p) { return *p; }
template <> __device__ __forceinline__ float ld<uint16_t>(const uint16_t* p) { return bf2f(*p); }
template <typename T> __device__ __forceinline__ void st(T* p, float v);
template <> __device__ __forceinline__ void st<float>(float* p, float v) { *p = v; }
template <> __device__ __forceinline__ void st<uint16_t>(uint16_t* p, float v) { *p = f2bf(v); }

// round a float through the activation type (what a value stored and read back would be)
template <typename T> __device__ __forceinline__ float rnd(float v);
template <> __device__ __forceinline__ float rnd<float>(float v) { return v; }
template <> __device__ __forceinline__ float rnd<uint16_t>(float v) { return bf2f(f2bf(v)); }

// log(sigmoid(z)) without overflow on either side
__device__ __forceinline__ float logsigmoidf_(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// 8 neighbouring activations, 16-byte aligned for bfloat16
__device__ __forceinline__ void ld8(const uint16_t* p, float (&v)[8]) {
    const uint4 r = *reinterpret_cast<const uint4*>(p);
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
__device__ __forceinline__ void st8(uint16_t* p, const float (&v)[8]) {
    u16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = f2bf(v[i]);
    *reinterpret_cast<u16x8*>(p) = o;
}
// 8 neighbouring floats, 16-byte aligned
__device__ __forceinline__ void ld8f(const float* p, float (&v)[8]) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) { v[i] = a[i]; v[4 + i] = b[i]; }
}
__device__ __forceinline__ void st8f(float* p, const float (&v)[8]) {
    *reinterpret_cast<f32x4*>(p) = f32x4{v[0], v[1], v[2], v[3]};
    *reinterpret_cast<f32x4*>(p + 4) = f32x4{v[4], v[5], v[6], v[7]};
}

// Transposing LDS read (gfx950): the 16 lanes of a lane group name the 8-byte pieces of a 4 x 16 matrix of 16-bit
// elements, row by row (lane l: row l / 4, columns 4 (l % 4) ..), and lane l receives column l, its 4 rows in order.
// Rows may lie anywhere.  A row-major tile thus serves as either operand of a matrix product.
__device__ __forceinline__ bf16x4 lds_read_tr4(const void* p) {
    typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}

__device__ __forceinline__ f32x4 mfma_16x16x16(bf16x4 a, bf16x4 b, f32x4 c) {
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}

// One 1 KiB piece from memory straight into LDS: lane l's 16 bytes from its own address to LDS offset lds + 16 l (lds the
// same in all lanes).  Inline asm, so that the compiler does not wait for it before every LDS read; the kernel waits with
// dma_wait() in front of the barrier that hands the piece over.
__device__ __forceinline__ void dma_1k(const void* src, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(src), "s"(lds) : "memory");
}
__device__ __forceinline__ void dma_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// All but the PW pieces of each of the AHEAD newest tiles, or of the `left` that are still to come, have landed
template <int PW, int AHEAD> __device__ __forceinline__ void dma_wait_for(int left) {
    static_assert(PW * AHEAD < 64, "counted waits");
    if constexpr (AHEAD > 0) {
        if (left >= AHEAD) {
            __builtin_amdgcn_s_waitcnt(((PW * AHEAD) & 0xF) | (0x7 << 4) | (0xF << 8) | (((PW * AHEAD) >> 4) << 14));
            asm volatile("" ::: "memory");
        } else {
            dma_wait_for<PW, AHEAD - 1>(left);
        }
    } else {
        dma_wait();
    }
}
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
    typedef __attribute__((address_space(3))) const void* lds_ptr;
    return (uint32_t)(uintptr_t)(lds_ptr)p;
}
// Piece j of a tile of rows: an LDS image of row-major rows, each CPR chunks of 16 bytes of which the last is padding
// (it spreads the rows over the banks; like the chunks past the row's n real ones it receives a copy of the last real
// one).  rows: element offset factor of each row of the tile; width: elements per row in memory.
// KT > 0: the tile has KT rows; chunks past them (a tile's last piece may hold some) repeat its last row.
template <int CPR, int KT = 0> __device__ __forceinline__ void dma_rows(const uint16_t* src, const int* rows, int width, int n, int j,
                                                            uint32_t lds, int lane) {
    const int i = j * 64 + lane, at = i / CPR, ch = i - at * CPR, row = KT > 0 ? min(at, KT - 1) : at;
    dma_1k(src + (int64_t)rows[row] * width + min(ch, n - 1) * 8, __builtin_amdgcn_readfirstlane(lds + j * 1024));
}

// bfloat16 of a (lower half) and b, and what the rounding leaves of them.  Taken apart as a word: the compiler would convert each a second
// time, alone, to have it back as a float.
__device__ __forceinline__ uint32_t round_pair(float& a, float& b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const uint32_t u = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{a, b}), bf16x2));
    a -= __uint_as_float(u << 16);
    b -= __uint_as_float(u & 0xffff0000u);
    return u;
}

// forms of the recurrences with one decay per head and token (chunk_scan.hip)
enum { kScanPlain = 0, kScanMlstm = 1, kScanDelta = 2 };

// host: every pointer (nullptr too) on a 16-byte boundary
template <typename... P> inline bool aligned16(P... p) { return ((reinterpret_cast<uintptr_t>(p) | ...) & 15) == 0; }

}  // namespace hy
}  // namespace chronos
