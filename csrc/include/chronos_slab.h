// chronos_slab.h — the main loop of the 256 x 256 bf16 tile (4 waves, one per SIMD, 128 x 128 outputs each; K in 64-deep slabs),
// shared by the projection GEMM (gemm_lg.hip) and the grouped expert GEMM (moe_grouped.hip).
#pragma once
#include "chronos_hip.h"

#include <type_traits>
#include <utility>

namespace chronos {

template <int N>
__device__ __forceinline__ void lg_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt range");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}

// raw workgroup barrier nothing is scheduled across
__device__ __forceinline__ void lg_bar() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

typedef int lg_i32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ lg_i32x4 lg_rsrc(const void* base, int bytes) {
    const uint64_t b = (uint64_t)base;
    return lg_i32x4{(int)(uint32_t)b, (int)(uint32_t)(b >> 32), bytes, 0x00020000};
}
// One 1 KiB LDS-DMA piece in two halves, with an MFMA between them for the wait state.  One wave per SIMD has issue slots for three
// instructions beside a 16-cycle MFMA: a third one per piece measured 80 of a slab's 2300 cycles.
template <int OFF>
__device__ __forceinline__ void lg_dma_dst(uint32_t lds) {
    asm volatile("s_add_u32 m0, %0, %1" ::"s"(lds), "n"(OFF) : "memory", "scc");
}
__device__ __forceinline__ void lg_dma_go(const void* base, int bytes, uint32_t voff, int soff) {
    asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(voff), "s"(lg_rsrc(base, bytes)), "s"(soff) : "memory");
}

// f(std::integral_constant<int, I>{}) for every I of the sequence, in order (a compile-time unrolled loop)
template <typename F, int... Is>
__device__ __forceinline__ void lg_static_for(F&& f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}

// Square order (slab_loop<true>): k-step 0 of a slab in growing-square order — MFMA (s, t) as soon as fa[s] and fb[t] can
// have landed — with the set-0 reads alternating fa[0], fb[0], fb[1], fa[1], fb[2], fa[2], ...: the slab head's first
// k MFMAs need ~2 sqrt(k) of the 16 reads issued at the end of the previous slab instead of k + 1, so fewer of them
// wait on the tail of that read burst
constexpr int hb_isqrt(int v) {
    int n = 0;
    while ((n + 1) * (n + 1) <= v) ++n;
    return n;
}
constexpr int hb_sq_s(int ii) { return ii - hb_isqrt(ii) * hb_isqrt(ii) < hb_isqrt(ii) ? ii - hb_isqrt(ii) * hb_isqrt(ii) : hb_isqrt(ii); }
constexpr int hb_sq_t(int ii) {
    return ii - hb_isqrt(ii) * hb_isqrt(ii) < hb_isqrt(ii) ? hb_isqrt(ii) : ii - hb_isqrt(ii) * hb_isqrt(ii) - hb_isqrt(ii);
}
// set-0 read r of the alternating order: W (fa) or x (fb) block index; r = 0 -> fa[0], 1 -> fb[0], 2 n -> fb[n],
// 2 n + 1 -> fa[n]
constexpr bool hb_sq_isw(int r) { return r == 0 || (r >= 2 && (r & 1)); }
constexpr int hb_sq_blk(int r) { return r < 2 ? 0 : r / 2; }
// the DMA piece issued before MFMA slot i (-1: none): n pieces spread evenly over slots [rel, end)
constexpr int hb_piece(int i, int rel, int end, int n) {
    for (int p = 0; p < n; ++p)
        if (rel + p * (end - rel) / n == i) return p;
    return -1;
}
// read r of a group of n reads spread evenly over slots [from, to): is it due at slot i?  (first one due at i, or -1; several may
// share a slot when the group is denser than the slots: hb_due_n of them, consecutive)
constexpr int hb_due(int i, int from, int to, int n) {
    for (int r = 0; r < n; ++r)
        if (from + r * (to - from) / n == i) return r;
    return -1;
}
constexpr int hb_due_n(int i, int from, int to, int n) {
    int c = 0;
    for (int r = 0; r < n; ++r) c += from + r * (to - from) / n == i;
    return c;
}

// The loop over NS slabs.  A slab keeps its LDS buffer only until its second k-step's fragments are in registers, so the two
// buffers hold nearly two slabs in flight.  Slab j (in buffer j % 2), slot i of 128 MFMAs (k-step i / 64), issue order pinned:
//   [0, RD1)     : the 16 fragment reads of slab j, k-step 1 (set 1)
//   REL          : lgkmcnt(0) + barrier: every wave holds both k-steps of slab j, its buffer is free
//   [REL, PEND)  : the wave's 16 LDS-DMA pieces of slab j+2, evenly, x then W
//   LAND         : vmcnt(16) (this wave's pieces of slab j+1, issued one slab ago, have landed; those of slab j+2 stay
//                  in flight) + barrier: slab j+1 is readable
//   [LAND, RD0)  : the 16 fragment reads of slab j+1, k-step 0 (set 0)
// What was measured, us at 8192^3 / 5952 x 4096 x 14336 / 1024 x 128256 x 4096: the pieces want to be spread over all the
// slots that the dependences leave: over 32 slots 820 / 643 / 891, 48 788 / 617 / 856, 64 751 / 584 / 819, 88 729 / 559 / 797
// (with three more instructions a piece than now; REL from 20 to 56 and LAND from 96 to 112 matter little); a piece as
// two instructions on either side of an MFMA instead of three before it: 698 / 559 / 764.
// Called with slab 0 landed and its set 0 read (or on its way) and slab 1's 16 pieces per wave in flight.  rbw / rbx: the lane's
// address of block 0 of each operand by buffer and k-step; roww(b): byte offset of W block b behind block 0; x block b lies
// 2048 b behind.  advance(j): once per slab, before its pieces (of slab j + 2, or of whatever lies in bounds past the last slab, which
// nobody reads); dst(buffer, piece): sets M0; go(piece): issues the load.
template <bool SQ, class Dst, class Go, class Adv, class RowW>
__device__ __forceinline__ void slab_loop(f32x4 (&acc)[8][8], bf16x8 (&fa0)[8], bf16x8 (&fb0)[8], bf16x8 (&fa1)[8], bf16x8 (&fb1)[8],
                                          const unsigned char* (&rbw)[2][2], const unsigned char* (&rbx)[2][2], int NS, const Dst& dst,
                                          const Go& go, const Adv& advance, RowW) {
    constexpr int RD1 = 16, REL = 20, PEND = 108, LAND = 112, RD0 = 128;
    static_assert(RD1 < REL && REL + 16 <= PEND && PEND <= LAND && RD0 <= 128, "slab schedule");
    auto half = [&](auto PC, int j) {
        constexpr int P = decltype(PC)::value;  // slab j lives in buffer P, slab j+1 in 1 - P
        advance(j);
        auto slot = [&](auto IC) {
            constexpr int i = decltype(IC)::value;
            if constexpr (i == REL) {
                __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), visible to hipcc's wait bookkeeping
                lg_bar();
            }
            if constexpr (i == LAND) {
                lg_vmcnt<16>();
                lg_bar();
            }
            constexpr int piece = hb_piece(i, REL, PEND, 16);
            if constexpr (piece >= 0) dst(PC, std::integral_constant<int, piece>{});
            constexpr int ii = i % 64;
            constexpr bool sq = SQ && i < 64;  // (k-step 0 only: k-step 1's reads land early)
            constexpr int s = sq ? hb_sq_s(ii) : ii / 8, t = sq ? hb_sq_t(ii) : ii % 8;
            if constexpr (i < 64)
                acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa0[s], fb0[t], acc[s][t], 0, 0, 0);
            else
                acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa1[s], fb1[t], acc[s][t], 0, 0, 0);
            if constexpr (piece >= 0) go(std::integral_constant<int, piece>{});
            auto read = [&](auto RC, int p, int kk, bf16x8 (&fa)[8], bf16x8 (&fb)[8]) {
                constexpr int r = decltype(RC)::value;
                // square order: fa0, fb0, fb1, fa1, fb2, fa2, ...; else fa[0], fb[0..7], fa[1..7]
                constexpr bool isw = SQ ? hb_sq_isw(r) : r == 0 || r > 8;
                constexpr int b = SQ ? hb_sq_blk(r) : r == 0 ? 0 : r <= 8 ? r - 1 : r - 8;
                if constexpr (isw) fa[b] = *reinterpret_cast<const bf16x8*>(rbw[p][kk] + RowW{}(b));
                else fb[b] = *reinterpret_cast<const bf16x8*>(rbx[p][kk] + 2048 * b);
            };
            constexpr int r1 = hb_due(i, 0, RD1, 16), r0 = hb_due(i, LAND, RD0, 16);
            static_assert(hb_due_n(i, 0, RD1, 16) <= 1 && hb_due_n(i, LAND, RD0, 16) <= 1, "one read a slot");
            if constexpr (r1 >= 0) read(std::integral_constant<int, r1>{}, P, 1, fa1, fb1);
            if constexpr (r0 >= 0) read(std::integral_constant<int, r0>{}, 1 - P, 0, fa0, fb0);
            __builtin_amdgcn_sched_barrier(0);
        };
        lg_static_for(slot, std::make_integer_sequence<int, 128>{});
    };
    for (int j = 0; j < NS; j += 2) {
        half(std::integral_constant<int, 0>{}, j);
        if (j + 1 < NS) half(std::integral_constant<int, 1>{}, j + 1);
    }
}

}  // namespace chronos
