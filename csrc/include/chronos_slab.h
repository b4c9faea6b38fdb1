// chronos_slab.h — tiles of 256 W rows by 256 (or 128) x rows in bfloat16: 4 waves, one per SIMD, 128 x 128 (128 x 64) outputs each, K in
// 64-deep slabs.  The slab step, and the loop of a workgroup over its tiles; shared by the projections (gemm_slab.hip, gemm_lg.hip) and
// the grouped expert products (moe_grouped.hip).
#pragma once
#include "chronos_hip.h"

#include <type_traits>
#include <utility>

namespace chronos {

typedef __attribute__((address_space(3))) const void* lg_lds_cptr;

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

// Square order (slab_step<8, true>): k-step 0 of a slab in growing-square order — MFMA (s, t) as soon as fa[s] and fb[t] can
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

// One slab.  Its LDS buffer is kept only until its second k-step's fragments are in registers, so the two buffers hold nearly two
// slabs in flight.  Slab j, slot i of 16 NM MFMAs (k-step i / (8 NM)), issue order pinned:
//   [0, RD1)     : the 8 + NM fragment reads of slab j, k-step 1 (set 1), from cw / cx
//   REL          : lgkmcnt(0) + barrier: every wave holds both k-steps of slab j, its buffer is free
//   [REL, PEND)  : the wave's 8 + NM LDS-DMA pieces of slab j+2 into that buffer, evenly, x then W: dst(piece) sets M0, go(piece)
//                  issues the load
//   LAND         : vmcnt(8 + NM) (this wave's pieces of slab j+1, issued one slab ago, have landed; those of slab j+2 stay
//                  in flight) + barrier: slab j+1 is readable
//   [LAND, end)  : the 8 + NM fragment reads of slab j+1, k-step 0 (set 0), from nw / nx
// W block b lies RowW{}(b) bytes behind block 0, x block b 2048 b.
// What was measured, us at 8192^3 / 5952 x 4096 x 14336 / 1024 x 128256 x 4096: the pieces want to be spread over all the
// slots that the dependences leave: over 32 slots 820 / 643 / 891, 48 788 / 617 / 856, 64 751 / 584 / 819, 88 729 / 559 / 797
// (with three more instructions a piece than now; REL from 20 to 56 and LAND from 96 to 112 matter little); a piece as
// two instructions on either side of an MFMA instead of three before it: 698 / 559 / 764.
template <int NM, bool SQ, class RowW, class Dst, class Go>
__device__ __forceinline__ void slab_step(f32x4 (&acc)[8][NM], bf16x8 (&fa0)[8], bf16x8 (&fb0)[NM], bf16x8 (&fa1)[8], bf16x8 (&fb1)[NM],
                                          const unsigned char* cw, const unsigned char* cx, const unsigned char* nw,
                                          const unsigned char* nx, const Dst& dst, const Go& go) {
    static_assert(NM >= 4 && NM <= 8 && (NM == 8 || !SQ), "tile");
    constexpr int NF = 8 + NM, END = 16 * NM, RD1 = NF, REL = NM == 8 ? 20 : NM + 10, LAND = END - NF, PEND = NM == 8 ? 108 : LAND;
    static_assert(RD1 < REL && REL + NF <= PEND && PEND <= LAND, "slab schedule");
    auto read = [&](auto RC, const unsigned char* w, const unsigned char* x, bf16x8 (&fa)[8], bf16x8 (&fb)[NM]) {
        constexpr int r = decltype(RC)::value;
        // square order: fa0, fb0, fb1, fa1, fb2, fa2, ...; else fa[0], fb[0..NM-1], fa[1..7]
        constexpr bool isw = SQ ? hb_sq_isw(r) : r == 0 || r > NM;
        constexpr int b = SQ ? hb_sq_blk(r) : r == 0 ? 0 : r <= NM ? r - 1 : r - NM;
        if constexpr (isw) fa[b] = *reinterpret_cast<const bf16x8*>(w + RowW{}(b));
        else fb[b] = *reinterpret_cast<const bf16x8*>(x + 2048 * b);
    };
    auto slot = [&](auto IC) {
        constexpr int i = decltype(IC)::value;
        if constexpr (i == REL) {
            __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), visible to hipcc's wait bookkeeping
            lg_bar();
        }
        if constexpr (i == LAND) {
            lg_vmcnt<NF>();
            lg_bar();
        }
        constexpr int piece = hb_piece(i, REL, PEND, NF);
        if constexpr (piece >= 0) dst(std::integral_constant<int, piece>{});
        constexpr int ii = i % (8 * NM);
        constexpr bool sq = SQ && i < 8 * NM;  // (k-step 0 only: k-step 1's reads land early)
        constexpr int s = sq ? hb_sq_s(ii) : ii / NM, t = sq ? hb_sq_t(ii) : ii % NM;
        if constexpr (i < 8 * NM)
            acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa0[s], fb0[t], acc[s][t], 0, 0, 0);
        else
            acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa1[s], fb1[t], acc[s][t], 0, 0, 0);
        if constexpr (piece >= 0) go(std::integral_constant<int, piece>{});
        if constexpr (i < RD1) read(IC, cw, cx, fa1, fb1);
        if constexpr (i >= LAND) read(std::integral_constant<int, i - LAND>{}, nw, nx, fa0, fb0);
        __builtin_amdgcn_sched_barrier(0);
    };
    lg_static_for(slot, std::make_integer_sequence<int, END>{});
}

// The accumulators live in AGPRs across a slab loop: pinned at both ends, so that an epilogue's use of VGPRs cannot make the register
// allocator move them inside the loop.
template <int NM> __device__ __forceinline__ void slab_pin(f32x4 (&acc)[8][NM]) {
#pragma unroll
    for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int t = 0; t < NM; ++t) asm volatile("" : "+a"(acc[s][t]));
}

// ---- a workgroup's tiles ----------------------------------------------------------------------------------------------
constexpr int kSlabCUs = 256, kSlabImg = 256 * 128, kSlabStage = 2 * kSlabImg, kSlabRows = 2 * kSlabStage;
constexpr int kSlabLds = kSlabRows + 4 * 4096;   // two buffers and the epilogue's rows, 4 KiB a wave

// T tiles of 256 x 256 on 256 CUs: whole rounds of them and, where at most half of the CUs would have a tile in the last round, that
// round's tiles as two halves of 128 x rows each, so that all CUs share it (a half takes 0.59 of a tile's time: it reads the W rows for
// half as many products).  tail: that many further tiles, numbered from T on, are one half each (slab_tail).
__host__ __device__ inline void slab_split(int T, int tail, int& full, int& half) {
    const int r = T % kSlabCUs;
    half = tail > 0 || r <= kSlabCUs / 2 ? 2 * r + tail : 0;
    full = half ? T - r : T;
}
// A launch of nt tiles along the W rows whose last x tile has at most 128 rows: nt if all that whole rounds of the full tiles leave fits one
// round of halves when these last tiles count as one each, else 0 (they are tiles like the others).  585 x 11264 x 2048, 220 halves
// instead of 132 tiles: 41.7 -> 31.4 us; 1100 x 7168 x 2048 39.9 -> 30.0; 350 x 20480 x 2048 (240 halves) 36.9.
// (S: times that the tiles are walked, over slices of K)
__host__ __device__ inline int slab_tail(int M, int nt, int S) {
    const int r = M % 256;
    return r > 0 && r <= 128 && (int64_t)nt * S <= kSlabCUs &&
                   2 * (int)((int64_t)(M / 256) * nt * S % kSlabCUs) + nt * S <= kSlabCUs ? nt * S : 0;
}
__host__ __device__ inline int slab_grid(int T, int tail) {
    int full, half;
    slab_split(T, tail, full, half);
    return full >= kSlabCUs ? kSlabCUs : full > half ? full : half;
}

template <bool PAIR> struct SlabRow {   // byte offset of the wave's W block b; PAIR: gate rows 0 .. 127 of the image, their up rows 128 on
    constexpr int operator()(int b) const { return 128 * (!PAIR || b < 4 ? 16 * b : 128 + 16 * (b - 4)); }
};

struct SlabFirst {   // all tiles start with slab 0
    __device__ __forceinline__ int operator()(int) const { return 0; }
};

// The tiles of one workgroup, one after the other without a pause of the slab pipeline: the pieces that a tile's last two slabs issue are
// those of the next tile's first two, which land while this tile's results are stored.  Tile v of the launch goes to workgroup
// v % gridDim.x (gridDim.x = slab_grid(T, tail)); xcd_remap gives neighbouring tiles to the same XCD.
// NMX < 8: tiles of 256 W rows by 32 NMX x rows, all alike (T of them, no tail).
//   off(NM, tile, m, wv, xv, wb): byte offsets of the lane's rows of slab 0 (x rows from row m of the tile on) and the W matrix
//   turn(tile): the slab that a tile starts with, asked once off was for the same tile; it takes them round from there
//   rows(NM, tile, m): called before a tile's first slab, for what its epilogue needs of its rows
//   epi(NM, tile, m, acc): store the results (rows: the wave's 4 KiB of LDS)
template <bool PAIR, int NMX = 8, class Off, class Rows, class Epi, class Turn = SlabFirst>
__device__ __forceinline__ void slab_run(unsigned char* smem, int T, int tail, int NS, const void* x, int xbytes, int wbytes, const Off& off,
                                         const Rows& rows, const Epi& epi, const Turn& turn = {}) {
    constexpr bool TURN = !std::is_same_v<Turn, SlabFirst>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave >> 1, wm = wave & 1, ln = lane & 15, g = lane >> 4, G = gridDim.x;
    const int ch0 = (g ^ (ln & 7)) * 16, ch1 = ((4 + g) ^ (ln & 7)) * 16;   // (16-row blocks: the swizzle depends on ln only)
    const unsigned char* const iw = smem + ((PAIR ? 64 : 128) * wn + ln) * 128;
    const uint32_t lds = (uint32_t)(uintptr_t)(lg_lds_cptr)smem;
    using Row = SlabRow<PAIR>;
    uint32_t wv[8];
    const void* wb;
    auto walk = [&](auto NMC, int first, int count, auto tile_of, auto m_of) {
        constexpr int NM = decltype(NMC)::value;
        const unsigned char* const ix = smem + kSlabImg + (16 * NM * wm + ln) * 128;
        const uint32_t ldw = lds + wave * 8192, ldx = lds + kSlabImg + wave * (1024 * NM);
        uint32_t xv[NM], nwv[8], nxv[NM];
        const void* nwb = nullptr;
        int v = first, dv = v, dj = 0;   // the tile in work; tile and slab (its number in the tile's order) whose pieces are issued
        int t0 = 0;                      // TURN: that tile's first
        auto next = [&]() {
            if (++dj < NS) return;
            if (dv + G >= count) { dj = NS - 1; return; }   // (nobody reads these)
            dv += G;
            dj = 0;
            if constexpr (TURN) t0 = __builtin_amdgcn_readfirstlane(turn(tile_of(dv)));   // (not sooner: what off asked memory for comes behind the pieces)
            wb = nwb;
#pragma unroll
            for (int i = 0; i < 8; ++i) wv[i] = nwv[i];
#pragma unroll
            for (int i = 0; i < NM; ++i) xv[i] = nxv[i];
            if (NS == 1 && dv + G < count) off(NMC, tile_of(dv + G), m_of(dv + G), nwv, nxv, nwb);   // (the next slab is the next tile's)
        };
        auto at = [&]() {   // where that slab lies in a row, bytes (an offset that went along with dj cost 35 moves a slab, 4 %)
            const int j = TURN ? dj + t0 : dj;
            return (TURN && j >= NS ? j - NS : j) * 128;
        };
        uint32_t pw = ldw, px = ldx;   // where the pieces of the slab in work go
        auto dst = [&](auto IC) {
            constexpr int p = decltype(IC)::value;
            lg_dma_dst<1024 * (p < NM ? p : p - NM)>(p < NM ? px : pw);
        };
        auto go = [&](auto IC) {
            constexpr int p = decltype(IC)::value;
            if constexpr (p < NM) lg_dma_go(x, xbytes, xv[p], at());
            else lg_dma_go(wb, wbytes, wv[p - NM], at());
        };
        auto all = [&](auto IC) {
            dst(IC);
            asm volatile("s_nop 0");
            go(IC);
        };
        auto after = [&](int u) {   // offsets of tile u
            if (u < count) off(NMC, tile_of(u), m_of(u), nwv, nxv, nwb);
        };
        off(NMC, tile_of(v), m_of(v), wv, xv, wb);
        if constexpr (TURN) t0 = __builtin_amdgcn_readfirstlane(turn(tile_of(v)));
        lg_static_for(all, std::make_integer_sequence<int, 8 + NM>{});
        after(v + G);
        next();
        pw += kSlabStage;
        px += kSlabStage;
        lg_static_for(all, std::make_integer_sequence<int, 8 + NM>{});
        rows(NMC, tile_of(v), m_of(v));
        f32x4 acc[8][NM];
#pragma unroll
        for (int s = 0; s < 8; ++s)
#pragma unroll
            for (int t = 0; t < NM; ++t) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        bf16x8 fa0[8], fb0[NM], fa1[8], fb1[NM];
        lg_vmcnt<8 + NM>();
        lg_bar();
        constexpr bool SQ = NM == 8;
#pragma unroll
        for (int r = 0; r < 8 + NM; ++r) {   // (the order of the slabs' own reads)
            const bool isw = SQ ? hb_sq_isw(r) : r == 0 || r > NM;
            const int b = SQ ? hb_sq_blk(r) : r == 0 ? 0 : r <= NM ? r - 1 : r - NM;
            if (isw) fa0[b] = *reinterpret_cast<const bf16x8*>(iw + ch0 + Row{}(b));
            else fb0[b] = *reinterpret_cast<const bf16x8*>(ix + ch0 + 2048 * b);
        }
        int par = 0;   // byte offset of the buffer of the slab in work
        for (;;) {
            slab_pin(acc);
            for (int j = 0; j < NS; ++j) {
                next();
                pw = ldw + par;
                px = ldx + par;
                const int oth = kSlabStage - par;
                slab_step<NM, SQ, Row>(acc, fa0, fb0, fa1, fb1, iw + ch1 + par, ix + ch1 + par, iw + ch0 + oth, ix + ch0 + oth, dst, go);
                par = oth;
            }
            slab_pin(acc);
            const int u = v + G;
            epi(NMC, tile_of(v), m_of(v), acc);
            if (u >= count) break;
            rows(NMC, tile_of(u), m_of(u));
            if (NS > 1) after(u + G);   // (with one slab a tile next() is a tile further already)
            v = u;
        }
        // the last pieces have landed and the last reads are done everywhere before the buffers are filled anew or given back
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        lg_bar();
    };
    const int b = blockIdx.x;
    if constexpr (NMX < 8) {
        walk(std::integral_constant<int, NMX>{}, b, T, [&](int v) { return xcd_remap(v, T); }, [](int) { return 0; });
        return;
    }
    int full, half;
    slab_split(T, tail, full, half);
    if (b < full)
        walk(std::integral_constant<int, 8>{}, b, full, [&](int v) { return xcd_remap(v, full); }, [](int) { return 0; });
    const int pairs = half - tail;   // halves that are two of a tile
    if (b < half)
        walk(std::integral_constant<int, 4>{}, b, half,
             [&](int v) {
                 const int h = xcd_remap(v, half);
                 return h < pairs ? full + h / 2 : T + h - pairs;
             },
             [&](int v) {
                 const int h = xcd_remap(v, half);
                 return h < pairs ? (h & 1) * 128 : 0;
             });
}

}  // namespace chronos
