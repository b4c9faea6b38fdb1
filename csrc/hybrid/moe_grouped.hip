// moe_grouped.hip — the experts of a mixture-of-experts layer as two grouped MFMA GEMMs (bfloat16), for any number of
// tokens: every expert's weights are streamed once per tile of its tokens, never once per token.
//
//   align     (count and place kernels, or for few items the up GEMM itself) counts the (token, choice) items of every expert with weights, gives each expert a
//             run of whole tiles in a sorted row space, and writes row -> item (or -1 for padding), item -> row
//             and the tile -> expert table.  Everything stays on the device: the GEMM grids are sized for the worst
//             case (items / tile + experts tiles) and surplus workgroups leave at once, so the host never learns the
//             routing and the step captures into a graph.
//   up GEMM   Z[row, :] = act(h[token(row), :] W_up[e]^T): the x operand's rows are GATHERED by token through the
//             per-lane LDS-DMA source addresses; activation in the epilogue.
//   down GEMM Y[row, :] = Z[row, :] W_down[e]^T.
//   combine   out[t, :] = sum_k weight[t, k] * Y[row(t, k), :]  (+ weight * h[t, :] for an identity expert), summed
//             in the order of k in float.  A row's sums over d and F have one order, whatever the tile's size and however many items there are
//             (moe_turn), so the result does not depend on what else is in the batch.
//
// Gated experts (act = gated unit): the up GEMM runs over W_gu [E, 2F, d] whose rows are PERMUTED at weight-packing
// time (moe_glu_row_order) so that every 128-row tile holds 64 gate rows and their 64 up rows in the accumulator
// positions of the same lane; the epilogue combines them and writes 64 columns of Z [rows, F] per tile.
//
// The tile loop is an LDS-DMA ring (16x16x32 bf16 MFMAs, XOR-swizzled images, one barrier per k-step with a counted vmcnt) at
// two tile sizes, below, and for experts with many tokens the projections' slab walk (chronos_slab.h).  Needs d % 128 == 0 and F % 128 == 0.
#include "hybrid_common.h"
#include "chronos_lds.h"
#include "chronos_slab.h"
#include "moe_tile.h"

namespace chronos {
namespace hy {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(1))) void* gbl_ptr_t;

// A tile: TM rows (tokens) by TN weight rows, k taken 64 at a time (whole 128-byte lines: rows of half lines reach a CU at a
// third of the rate) through a ring of ST stages; waves as 2 (weight rows) x WX (tokens).
//   256 x 256, two stages (128 KB), 4 waves of 128 x 128 outputs (moe_gemm256_kernel): experts with many tokens; half the bytes
//    per product of
//   128 x 128, two stages (64 KB: two workgroups per CU, one multiplies while the other waits), 4 waves of 64 x 64
//    64 x 128, three stages (72 KB: two workgroups per CU): experts with some tokens, whose time is the weights' (320 tokens of 4096, 32 experts of 2048,
//    top 4: 265 -> 230 us against two stages of 128 rows)
//    32 x 128, four stages (80 KB: two workgroups per CU, the weights of three k-steps in flight in each): few tokens
template <int TM> struct Tile {
    static constexpr int TN = 128, ST = TM == 32 ? 4 : TM == 64 ? 3 : 2, WX = 2, WAVES = 4;
    static constexpr int W = TN * 128, X = TM * 128;                                     // bytes of the two images of a stage
    static constexpr int WP = W / 1024 / WAVES, XP = X / 1024 / WAVES;                   // 1 KiB pieces per wave and stage
    static constexpr int NS = TN / 32, NM = TM / 16 / WX;                                // 16-row blocks per wave
    static constexpr int lds = ST * (W + X);
};

template <int N>
__device__ __forceinline__ void wait_vm() {
    __builtin_amdgcn_s_waitcnt((N & 0xF) | (0x7 << 4) | (0xF << 8) | ((N >> 4) << 14));
}
constexpr int kActGlu = 2;

// 16-byte piece c of image row r lies at c ^ (r & 7): 16 rows at the same c fall on different banks
__device__ __forceinline__ bf16x8 frag(const unsigned char* img, int row, int chunk) {
    return *reinterpret_cast<const bf16x8*>(img + row * 128 + ((chunk ^ (row & 7)) << 4));
}

// meta layout (int32): [0] tiles used | [1 .. 1+maxTiles) tile -> expert | then row -> item [maxTiles * TM] |
// then item -> row [items] | then items per workgroup and expert [workgroups, E]
constexpr int kAlignItems = 2048;   // items per workgroup

// Ranks of items [lo, hi) within their experts, into rank_of (-1: nobody's item), and the experts' counts into cnt (LDS).
// The lanes of a wave with the same expert find each other by the bits of its number (one ballot per bit) and the first of them
// moves the expert's counter for all: one LDS atomic per wave and expert.
__device__ __forceinline__ void moe_rank(const int32_t* __restrict__ idx, int lo, int hi, int E, int* cnt, int32_t* __restrict__ rank_of) {
    const int lane = threadIdx.x & 63;
    for (int e = threadIdx.x; e < E; e += blockDim.x) cnt[e] = 0;
    __syncthreads();
    int bits = 0;
    while ((1 << bits) < E) ++bits;
    for (int i0 = lo + threadIdx.x - lane; i0 < hi; i0 += blockDim.x) {   // (whole waves: the ballots take all lanes)
        const int i = i0 + lane, e = i < hi ? idx[i] : -1;
        const bool ok = e >= 0 && e < E;
        unsigned long long same = __ballot(ok);
        for (int k = 0; k < bits; ++k) {
            const unsigned long long one = __ballot((e >> k) & 1);
            same &= ((e >> k) & 1) ? one : ~one;
        }
        const int first = ok ? __ffsll(same) - 1 : lane, rank = __popcll(same & ((1ull << lane) - 1));
        int base = 0;
        if (ok && lane == first) base = atomicAdd(&cnt[e], __popcll(same));
        base = __shfl(base, first, 64);
        if (i < hi) rank_of[i] = ok ? base + rank : -1;
    }
    __syncthreads();
}

__global__ void __launch_bounds__(1024) moe_count_kernel(const int32_t* __restrict__ idx, int items, int E, int32_t* __restrict__ counts,
                                                         int32_t* __restrict__ item_row) {
    __shared__ int cnt[256];
    const int lo = blockIdx.x * kAlignItems;
    moe_rank(idx, lo, min(lo + kAlignItems, items), E, cnt, item_row);
    for (int e = threadIdx.x; e < E; e += blockDim.x) counts[blockIdx.x * E + e] = cnt[e];
}

// Gives every expert a run of whole tiles and every item its row.  One workgroup ranks its items itself; of several each places
// the items that it counted in moe_count_kernel (32768 items: 10 us in two launches of 16 workgroups; one workgroup took 38).
// Which row of its expert's run an item takes does not matter: every row is computed on its own and found again through
// item -> row, so the result is the same for any order.
__global__ void __launch_bounds__(1024) moe_place_kernel(const int32_t* __restrict__ idx, int items, int E, int TM, int maxTiles,
                                                         int32_t* __restrict__ meta) {
    __shared__ int cnt[256], before[256], start[257];
    int32_t* tile_e = meta + 1;
    int32_t* row_item = tile_e + maxTiles;
    int32_t* item_row = row_item + maxTiles * TM;
    const int32_t* counts = item_row + items;
    const int tid = threadIdx.x, wg = blockIdx.x, nwg = gridDim.x;
    const int lo = wg * kAlignItems, hi = nwg == 1 ? items : min(lo + kAlignItems, items);
    if (nwg == 1) {
        moe_rank(idx, lo, hi, E, cnt, item_row);
        if (tid < E) before[tid] = 0;
    } else if (tid < E) {
        int sum = 0, mine = 0;
        for (int g = 0; g < nwg; ++g) {
            if (g == wg) mine = sum;
            sum += counts[g * E + tid];
        }
        cnt[tid] = sum;
        before[tid] = mine;
    }
    __syncthreads();
    if (tid < 64) {   // first tile of every expert: a running sum over the experts, four per lane
        int n[4], sum = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            n[j] = 4 * tid + j < E ? (cnt[4 * tid + j] + TM - 1) / TM : 0;
            sum += n[j];
        }
        int to = sum;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(to, o, 64);
            if (tid >= o) to += v;
        }
        int at = to - sum;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            start[4 * tid + j] = at;
            at += n[j];
        }
        if (tid == 63) {
            start[256] = at;
            if (wg == 0) meta[0] = at;
        }
    }
    __syncthreads();
    // an expert's tiles, and the rows behind its last item: an expert per wave (one workgroup that took them in turn: 32 experts
    // of 256 items 10.8 us, now 4.8)
    const int lane = tid & 63, waves = blockDim.x >> 6;
    for (int e = wg * waves + (tid >> 6); e < E; e += nwg * waves) {
        for (int j = start[e] + lane; j < start[e + 1]; j += 64) tile_e[j] = e;
        for (int r = start[e] * TM + cnt[e] + lane; r < start[e + 1] * TM; r += 64) row_item[r] = -1;
    }
    for (int i = lo + tid; i < hi; i += blockDim.x) {
        const int e = idx[i], k = item_row[i];
        if (k >= 0) {
            const int r = start[e] * TM + before[e] + k;
            row_item[r] = i;
            item_row[i] = r;
        }
    }
}

// Placing inside the first product of few items: every workgroup of 256 threads finds its tile's expert and items for itself (one that
// takes the first rows of a tile's expert leaves them in meta for the launches behind it), so there is no launch in front of it.  Items keep their order
// within an expert, so all workgroups agree.  Returns whether there is such a tile; rows: its TM items (-1: padding).
// With the combining's loads in one go (below), us for the whole feed-forward: 8 experts of 1024 by 512, 1 to 64 tokens 20 -> 17.5; 16 of 2048 by
// 1024 (gated), 1 and 64 tokens 28.0 -> 24.8, 42.7 -> 39.3; 32 of 4096 by 2048, 1 and 64 tokens 47.4 -> 42.2, 237 -> 230.
constexpr int kPlaceItems = 512, kPlaceE = 64;
struct PlaceLds {
    int cnt[kPlaceItems / 64][kPlaceE];   // items of every run of 64 by expert
    int start[kPlaceE + 1], expert;
};
template <int TM>
__device__ __forceinline__ bool moe_place_tile(const int32_t* __restrict__ idx, int items, int E, int tile, bool writes, bool first, int maxTiles,
                                               int32_t* __restrict__ meta, PlaceLds& p, int* rows) {
    constexpr int RUNS = kPlaceItems / 64;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < RUNS * kPlaceE; i += 256) (&p.cnt[0][0])[i] = 0;
    if (tid < TM) rows[tid] = -1;
    int e[RUNS / 4], k[RUNS / 4];   // of the thread's items: expert, and rank within the run
#pragma unroll
    for (int j = 0; j < RUNS / 4; ++j) {
        const int i = (wave + 4 * j) * 64 + lane;
        const int v = i < items ? idx[i] : -1;
        e[j] = v >= 0 && v < E ? v : -1;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < RUNS / 4; ++j) {
        unsigned long long same = __ballot(e[j] >= 0);
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const unsigned long long one = __ballot((e[j] >> b) & 1);
            same &= ((e[j] >> b) & 1) ? one : ~one;
        }
        k[j] = __popcll(same & ((1ull << lane) - 1));
        if (e[j] >= 0 && k[j] == 0) p.cnt[wave + 4 * j][e[j]] = __popcll(same);
    }
    __syncthreads();
    if (wave == 0) {   // running sums: over the runs, then over the experts' tiles
        int sum = 0;
#pragma unroll
        for (int r = 0; r < RUNS; ++r) {
            const int n = p.cnt[r][lane];
            p.cnt[r][lane] = sum;
            sum += n;
        }
        const int n = (sum + TM - 1) / TM;
        int to = n;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int v = __shfl_up(to, o, 64);
            if (lane >= o) to += v;
        }
        p.start[lane] = to - n;
        if (lane == 63) p.start[kPlaceE] = to;
        if (tile >= to - n && tile < to) p.expert = lane;
        if (lane == 63 && first) meta[0] = to;
    }
    __syncthreads();
    const bool there = tile < p.start[kPlaceE];
    const int mine = there ? p.expert : -1, lo = there ? (tile - p.start[mine]) * TM : 0;
    int32_t* const row_item = meta + 1 + maxTiles;
    int32_t* const item_row = row_item + maxTiles * TM;
#pragma unroll
    for (int j = 0; j < RUNS / 4; ++j) {
        const int i = (wave + 4 * j) * 64 + lane;
        if (i >= items) continue;
        const int r = e[j] >= 0 ? p.cnt[wave + 4 * j][e[j]] + k[j] - lo : -1;
        if (there && e[j] == mine && r >= 0 && r < TM) {
            rows[r] = i;
            if (writes) item_row[i] = tile * TM + r;
        }
        if (first && e[j] < 0) item_row[i] = -1;
    }
    __syncthreads();
    if (there && writes) {
        if (tid == 0) meta[1 + tile] = mine;
        if (tid < TM) row_item[tile * TM + tid] = rows[tid];
    }
    return there;
}

// The k-step that tiles over an expert's weight rows 256 tn256 .. start with where they are turned; they take the steps round from there.  It follows from the weights
// alone and is the same for tiles of all sizes, so that a token's result does not depend on the batch.  All from the first, the
// workgroups read the same columns of weight rows that lie a power of two apart, lines that share few of the memory's channels.  The whole feed-forward, weights
// cold, us, from the first step -> turned: 32 experts of 4096 x 2048, top 4, GELU, 2 tokens 64 -> 56, 6 133 -> 112, 64 211 -> 171, 300 (64-row tiles) 224 -> 199, 450
// and 1000 (128-row tiles) 280 -> 221, 366 -> 338, 1600, 2500 and 8192 (256) 353 -> 295, 507 -> 472, 1131 -> 1092; gated, 4 tokens 129 -> 113, 64 298 -> 251, 450 333 ->
// 306, 2500 680 -> 648; 128 of 2048 x 1024, top 8, 4 tokens 66 -> 59, 128 196 -> 182, 2000 348 -> 336; 64 gated of 2048 x 1408, top 6, 8192 tokens 862 -> 870.
// 2 steps per 256 rows and 9 per expert: of nine pairs the best in sum (4 and 9: 64 tokens 171, 1000 345, of 256-row tiles 2500 521 where this took 493; 16 and 9:
// 172, 345, 514; 1 and 5: 174, 341, 512); 8 and 1, which give many tiles of neighbouring experts the same step, are as slow as none (64 tokens 208).
__device__ __forceinline__ int moe_turn(int e, int tn256, int KT) { return (2 * tn256 + 9 * e) % KT; }

// The wave's outputs: NS x NM accumulator tiles of 16 weight rows by 16 tokens, from weight row n0 and token row m0 on (item: the items of the lane's
// tokens, -1: padding, not stored).  Lane l
// holds D[n = 4 (l >> 4) + i][m = l & 15] of each = y[m][n .. n + 3].
template <int ACT, int NS, int NM>
__device__ __forceinline__ void moe_store(const f32x4 (&acc)[NS][NM], uint16_t* __restrict__ y, const int (&item)[NM],
                                          int m0, int n0, int N, int lane, float limit, float slope, float shift) {
#pragma unroll
    for (int t = 0; t < NM; ++t) {
        const int m = m0 + 16 * t + (lane & 15);
        if (item[t] < 0) continue;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int row = n0 + 16 * s;   // first weight row of the block
            u16x4 o;
            if constexpr (ACT == kActGlu) {
                // every 64 rows: blocks 0 and 1 are gate rows, 2 and 3 the up rows of the same outputs
                if (s & 2) continue;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float a = fminf(bf2f(f2bf(acc[s][t][i])), limit);
                    const float u = fminf(fmaxf(bf2f(f2bf(acc[s | 2][t][i])), -limit), limit);
                    o[i] = f2bf(a * sigmoid_act<uint16_t>(slope * a) * (u + shift));
                }
                const int n = (row >> 6) * 32 + (row & 31) + 4 * (lane >> 4);
                *reinterpret_cast<u16x4*>(y + (int64_t)m * (N / 2) + n) = o;
            } else {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = acc[s][t][i];
                    if constexpr (ACT >= 0) v = act_apply(bf2f(f2bf(v)), ACT);
                    o[i] = f2bf(v);
                }
                *reinterpret_cast<u16x4*>(y + (int64_t)m * N + row + 4 * (lane >> 4)) = o;
            }
        }
    }
}

// The tiles there are go to the XCDs in contiguous runs (their L2s then share rows of x and w); a launch of small tiles is
// bound by the weights' bytes and spreads them over all.
// ONCE: the weights' DMA is marked as read once (nt), which memory itself gives faster and which leaves nothing behind for a next call.
template <int TM, bool GATHER, int ACT, bool PLACE, bool ONCE>
__global__ void __launch_bounds__(256, 2) moe_gemm_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w,
                                                          uint16_t* __restrict__ y, int32_t* __restrict__ meta,
                                                          int maxTiles, int top, int N, int K, float limit, float slope,
                                                          float shift, const int32_t* __restrict__ idx, int items, int E, bool turned) {
    using C = Tile<TM>;
    constexpr int ST = C::ST, BK = 64;
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int nt = N / C::TN;
    int tile, tn, e;
    const int32_t* row_item;
    if constexpr (PLACE) {   // (TM == 32)
        tile = blockIdx.x / nt;
        tn = blockIdx.x - tile * nt;
        PlaceLds& place = *reinterpret_cast<PlaceLds*>(smem);   // (in the ring's memory: two workgroups' rings fill the CU's)
        int* const own = reinterpret_cast<int*>(smem + sizeof(PlaceLds));
        if (!moe_place_tile<TM>(idx, items, E, tile, tn == 0, blockIdx.x == 0, maxTiles, meta, place, own)) return;
        e = place.expert;
        row_item = own - tile * TM;
    } else {
        const int used = meta[0];
        if ((int)blockIdx.x >= used * nt) return;
        const int id = TM == 128 ? xcd_remap(blockIdx.x, used * nt) : (int)blockIdx.x;
        tile = id / nt;
        tn = id - tile * nt;
        e = meta[1 + tile];
        row_item = meta + 1 + maxTiles;
    }
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int m0 = tile * TM;
    const uint16_t* we = w + (int64_t)e * N * K;
    const uint16_t* wsrc[C::WP];
    const uint16_t* xsrc[C::XP];
#pragma unroll
    for (int i = 0; i < C::WP; ++i) {
        const int r = 8 * (C::WP * wave + i) + (lane >> 3), c = (lane & 7) ^ (r & 7);
        wsrc[i] = we + (int64_t)(tn * C::TN + r) * K + c * 8;
    }
#pragma unroll
    for (int i = 0; i < C::XP; ++i) {
        const int r = 8 * (C::XP * wave + i) + (lane >> 3), c = (lane & 7) ^ (r & 7);
        int64_t xr = m0 + r;
        if constexpr (GATHER) {
            const int it = row_item[m0 + r];
            xr = it < 0 ? 0 : it / top;  // padding rows read token 0 and are never stored
        }
        xsrc[i] = x + xr * K + c * 8;
    }
    const int wn = wave / C::WX, wm = wave % C::WX;
    int item[C::NM];   // of the lane's outputs
    auto items_of = [&]() {
#pragma unroll
        for (int t = 0; t < C::NM; ++t) item[t] = row_item[m0 + 16 * (C::NM * wm + t) + (lane & 15)];
    };
    if constexpr (PLACE) {
        items_of();
        __syncthreads();   // the ring's memory is read
    }
    const int KT = K / BK, turn = turned ? moe_turn(e, tn / 2, KT) : 0;
    auto issue = [&](int kt) {
        unsigned char* st = smem + (kt % ST) * (C::W + C::X);
        kt += turn;
        kt -= kt >= KT ? KT : 0;
#pragma unroll
        for (int i = 0; i < C::WP; ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(wsrc[i] + kt * BK), (lds_ptr_t)(st + (C::WP * wave + i) * 1024), 16, 0, ONCE ? 2 : 0);
#pragma unroll
        for (int i = 0; i < C::XP; ++i)
            __builtin_amdgcn_global_load_lds((gbl_ptr_t)(xsrc[i] + kt * BK), (lds_ptr_t)(st + C::W + (C::XP * wave + i) * 1024), 16, 0, 0);
    };
    f32x4 acc[C::NS][C::NM];
#pragma unroll
    for (int s = 0; s < C::NS; ++s)
#pragma unroll
        for (int t = 0; t < C::NM; ++t) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < ST - 1; ++p)
        if (p < KT) issue(p);
    for (int kt = 0; kt < KT; ++kt) {
        if (kt + ST - 2 < KT) wait_vm<(C::WP + C::XP) * (ST - 2)>();
        else wait_vm<0>();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (kt + ST - 1 < KT) issue(kt + ST - 1);
        const unsigned char* wimg = smem + (kt % ST) * (C::W + C::X);
        const unsigned char* ximg = wimg + C::W;
#pragma unroll
        for (int h = 0; h < BK / 32; ++h) {
            const int chunk = h * 4 + (lane >> 4);
            bf16x8 a[C::NS], b[C::NM];
#pragma unroll
            for (int t = 0; t < C::NM; ++t) b[t] = frag(ximg, 16 * (C::NM * wm + t) + (lane & 15), chunk);
#pragma unroll
            for (int s = 0; s < C::NS; ++s) a[s] = frag(wimg, C::TN / 2 * wn + 16 * s + (lane & 15), chunk);
#pragma unroll
            for (int s = 0; s < C::NS; ++s)
#pragma unroll
                for (int t = 0; t < C::NM; ++t)
                    acc[s][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[s], b[t], acc[s][t], 0, 0, 0);
        }
    }
    if constexpr (!PLACE) items_of();
    moe_store<ACT, C::NS, C::NM>(acc, y, item, m0 + 16 * C::NM * wm, tn * C::TN + C::TN / 2 * wn, N, lane, limit, slope, shift);
}

// The 256 x 256 tile (x and one expert's weights below 4 and 2 GiB; weight rows past the end repeat the last one): a workgroup per CU walks
// its tiles on the slab loop of chronos_slab.h.  Bound by the matrix cores and the padding of every expert's last tile.
// Results through the wave's 4 KiB of LDS, 16 rows at a time, so that a store instruction writes whole lines: 16 lanes a row (8 for a
// gated unit's 64 columns); registers as in moe_store, row r's 16-byte piece c at c ^ (r % pieces).
// TURNED (moe_turn): instances of their own (asked at run time, 16 gated experts of 2048 x 1024, 8192 tokens: 415 -> 436).
template <bool GATHER, int ACT, bool TURNED>
__global__ void __launch_bounds__(256, 1) moe_gemm256_kernel(const uint16_t* __restrict__ x, uint32_t xbytes,
                                                             const uint16_t* __restrict__ w, uint16_t* __restrict__ y,
                                                             const int32_t* __restrict__ meta, int maxTiles, int top, int N,
                                                             int K, float limit, float slope, float shift) {
    constexpr bool GLU = ACT == kActGlu;
    constexpr int RBY = GLU ? 128 : 256, NCH = RBY / 16, RPS = 64 / NCH, NK = 16 / RPS;   // bytes and pieces per row, rows per store
    extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
    const int nt = (N + 255) / 256;
    const int32_t* row_item = meta + 1 + maxTiles;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wn = wave >> 1, wm = wave & 1, in = lane >> 3, pc = (lane & 7) ^ in;
    int expert = 0;   // of the last tile that off was asked for
    auto off = [&](auto NMC, int id, int m, uint32_t (&wv)[8], auto& xv, const void*& wb) {
        constexpr int NM = decltype(NMC)::value;
        const int tile = id / nt, tn = id - tile * nt;
        expert = meta[1 + tile];
        wb = w + (int64_t)__builtin_amdgcn_readfirstlane(expert) * N * K;
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[i] = moe_weight_offset(tn, 2 * wave + (i >> 2), i & 3, lane, N, K);
#pragma unroll
        for (int i = 0; i < NM; ++i) {
            uint32_t xr = tile * 256 + m + 8 * (NM * wave + i) + in;
            if constexpr (GATHER) {
                const int it = row_item[xr];
                xr = it < 0 ? 0 : it / top;  // padding rows read token 0 and are never stored
            }
            xv[i] = (xr * (uint32_t)K + pc * 8) * 2;
        }
    };
    unsigned char* const stg = smem + kSlabRows + wave * 4096;
    const int c = lane % NCH, rr = lane / NCH;
    auto epi = [&](auto NMC, int id, int m, auto& acc) {
        constexpr int NM = decltype(NMC)::value;
        const int tile = id / nt, tn = id - tile * nt, m0 = tile * 256 + m + 16 * NM * wm;
        const int ld = GLU ? N / 2 : N, n = (tn * 256 + 128 * wn) / (GLU ? 2 : 1) + 8 * c;
#pragma unroll
        for (int t = 0; t < NM; ++t) {
            int it[NK];
#pragma unroll
            for (int k = 0; k < NK; ++k) it[k] = row_item[m0 + 16 * t + RPS * k + rr];
            const int r = lane & 15;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                if (GLU && (s & 2)) continue;
                const int col = GLU ? 32 * (s >> 2) + 16 * (s & 1) + 4 * (lane >> 4) : 16 * s + 4 * (lane >> 4);
                u16x4 o;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    float v = acc[s][t][i];
                    if constexpr (GLU) {
                        // every 64 rows: blocks 0 and 1 are gate rows, 2 and 3 the up rows of the same outputs
                        const float a = fminf(bf2f(f2bf(v)), limit);
                        const float u = fminf(fmaxf(bf2f(f2bf(acc[s | 2][t][i])), -limit), limit);
                        v = a * sigmoid_act<uint16_t>(slope * a) * (u + shift);
                    } else if constexpr (ACT >= 0) {
                        v = act_apply(bf2f(f2bf(v)), ACT);
                    }
                    o[i] = f2bf(v);
                }
                *reinterpret_cast<u16x4*>(stg + r * RBY + (((col >> 3) ^ (r % NCH)) << 4) + ((col >> 2) & 1) * 8) = o;
            }
#pragma unroll
            for (int s = 0; s < 8; ++s) acc[s][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            u16x8 v[NK];
#pragma unroll
            for (int k = 0; k < NK; ++k) {   // (a wave's LDS operations complete in order)
                const int q = RPS * k + rr;
                v[k] = *reinterpret_cast<const u16x8*>(stg + q * RBY + ((c ^ (q % NCH)) << 4));
            }
#pragma unroll
            for (int k = 0; k < NK; ++k)
                if (it[k] >= 0 && n < ld)   // (the last tile along N may be half)
                    *reinterpret_cast<u16x8*>(y + (int64_t)(m0 + 16 * t + RPS * k + rr) * ld + n) = v[k];
        }
    };
    auto run = [&](const auto& turn) {
        slab_run<false>(smem, meta[0] * nt, 0, K / 64, x, (int)xbytes, (int)((uint32_t)N * K * 2), off, [](auto, int, int) {}, epi, turn);
    };
    if constexpr (TURNED) run([&](int id) { return moe_turn(__builtin_amdgcn_readfirstlane(expert), id % nt, K / 64); });
    else run(SlabFirst{});
}

// An index of E and above is an identity expert (its output is the token itself) where the experts' layer has such
// (identity), else, like a negative one, nobody's: it adds nothing.
__global__ void __launch_bounds__(256) moe_combine_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ yrows,
                                                          const int32_t* __restrict__ idx, const float* __restrict__ wt,
                                                          const int32_t* __restrict__ item_row, uint16_t* __restrict__ out,
                                                          int d, int top, int E, int identity) {
    const int64_t t = blockIdx.x;
    const int c = (blockIdx.y * 256 + threadIdx.x) * 8;
    if (c >= d) return;
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    constexpr int U = 4;   // choices whose numbers, then rows, are under way together (one after the other: 6.7 us for 64 tokens of 4096)
    for (int k0 = 0; k0 < top; k0 += U) {
        int e[U], r[U];
        float g[U];
        u16x8 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = t * top + min(k0 + u, top - 1);
            e[u] = idx[i];
            r[u] = item_row[i];
            g[u] = wt[i];
        }
#pragma unroll
        for (int u = 0; u < U; ++u)   // (a choice that is nobody's reads the token's own row and adds nothing)
            v[u] = *reinterpret_cast<const u16x8*>(r[u] < 0 ? h + t * d + c : yrows + (int64_t)r[u] * d + c);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (k0 + u >= top || (r[u] < 0 && !(identity && e[u] >= E))) continue;
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] += g[u] * bf2f(v[u][j]);
        }
    }
    u16x8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f2bf(acc[j]);
    *reinterpret_cast<u16x8*>(out + t * d + c) = o;
}

}  // namespace hy

// Rows per tile.  32 where experts see few tokens on average, so that a tile's padding rows cost little and the launch streams weights with more of
// them in flight; 64 above; 256, whose loop is the fastest per product, where most tiles fill (192 tokens per expert, 384 of narrow ones) and the smaller
// product has a tile for a quarter of the CUs; else 128.  up: rows of an expert's first matrix.  The fewer workgroups a tile per expert and 128 of
// the smaller product's columns makes (wide), the further the smaller tiles go, whose number fills the CUs.  us at 32 / 64 / 128 rows, GELU:
// 8 experts of 1024 by 512 (wide 32), top 2, 128 tokens (32 items per expert) 20 / 28 / 33, 320 24 / 28 / 35, 1000 - / 32 / 39, 1400 - / 36 / 42; 16 of
// 2048 by 1408 (176), top 4, 96 tokens 39 / 48 / 58, 160 60 / 49 / 61, 256 68 / 56 / 66, 400 - / 72 / 67; 32 of 4096 by 2048 (512), top 4, 160 218 / 230 /
// 266, 200 248 / 231 / 269, 400 259 / 231 / 279, 600 310 / 286 / 288, 800 - / 299 / 291; with expert e chosen in proportion to 1 / e 200 tokens 230 / 233 / 339,
// 400 274 / 253 / 348, 600 324 / 299 / 348, 1400 - / 438 / 405.  Beyond 56 items an expert takes two tiles of 64, and where the two products'
// tile columns (cols) then make more than two rounds of 512 workgroups 128 rows are faster, evenly chosen: 16 gated of 2048 by 1408, 64 and 80 items 75 for
// 90, 78 for 97; 64 of 1024 by 512, 80 items 57 for 70; 32 gated of 4096 by 2048, 64 items 340 for 364; unevenly chosen ones lose by it there (64 gated of 2048 by
// 1024, choice as 1 / e, 64 items 243 for 217).  Over 17 shapes of experts, gated and not, 21 numbers of items, even and as 1 / e: 2.5 % behind the best of the three on
// average, 1.09 times as fast as 32 rows to 16 items and 128 beyond, 27 of 1428 slower than that by more than 3 %, the worst by 22 % (64 gated of 1024 by 512, 52 items).
// profiles/moe_tiles.json, which tests/test_measured_rules.py replays.  128 against 256, on gated
// experts, us at 32 / 128 / 256 rows: 16 experts of 2048 by 1024, 512
// tokens 81 / 66 / 62, 2048 tokens 248 / 154 / 150, 8192 tokens 870 / 516 / 407; 32 experts of 4096 by 1536 with 512 tokens 329 / 282 / 323,
// 1536 tokens 606 / 424 / 352, 8192 tokens 2640 / 1610 / 1180; 8 experts of 1024 by 512 with 1024 tokens (2 each) 39 / 35 / 39, 8192 tokens
// 140 / 98 / 100.  (A skewed choice fills more tiles: at 128 tokens per expert of 16 256 rows win by 6 %,
// but with expert e chosen in proportion to 1 / e they lose 27 %, 84 for 66 us; from 192 on they win there too, but for experts of at most four
// tiles across: 64 of 1024 by 512 at 192 tokens each 84 / 77, skewed 88 / 103, at 256 113 / 118, skewed 117 / 118, at 384 153 / 130, skewed 160 / 131:
// those take 256 rows from 384 on.)  32, 128 and 256 rows at 55 sizes, and at 40 skewed: profiles/prompt_form_rules.json.
int hy_moe_tile(int items, int E, int d, int F, int up) {
    const int64_t G4 = (int64_t)1 << 32, rows = (int64_t)items + 256 * E;
    const bool fits = rows * (d > F ? d : F) * 2 < G4 && (int64_t)up * d * 2 < G4 / 2;   // 32-bit offsets
    const int least = up < d ? up : d;
    const int64_t big = (int64_t)(items / 256) * least / 256;
    const int64_t wide = (int64_t)E * (least / 128);
    if (items <= (wide <= 64 ? 72 : wide < 384 ? 32 : 20) * E) return 32;
    const int64_t cols = wide + (int64_t)E * ((up < d ? d : up) / 128);
    if (items <= (wide <= 64 ? 320 : cols > 512 ? 56 : wide < 384 ? 88 : 72) * E) return 64;
    return items < (least <= 1024 ? 384 : 192) * E || big < 64 || !fits ? 128 : 256;
}
int hy_moe_max_tiles(int items, int E, int tm) {
    const int n = items / tm + E;   // an expert's last tile may hold a single item
    return n < items ? n : items;
}
static int moe_align_wgs(int items) { return items <= 2 * hy::kAlignItems ? 1 : (items + hy::kAlignItems - 1) / hy::kAlignItems; }
int64_t hy_moe_meta_ints(int items, int E, int tm) {
    const int64_t n = hy_moe_max_tiles(items, E, tm);
    return 1 + n + n * tm + items + (int64_t)moe_align_wgs(items) * E;
}

// Weights of the experts chosen (one product's, at most) from which their reads are marked as read once: what the memory-side cache holds.  Below
// it a decoder of few layers finds them there again.  The whole feed-forward, us, plain -> marked: GELU 4096 wide, 32 experts of 2048, top 4:
// 4 tokens (268 MB each product) 101 -> 89, 16 204 -> 181, 64 (512 MB) 238 -> 210, 128 239 -> 212, 400 253 -> 231, but 2 tokens 54 -> 62; 2048 wide, 16
// gated experts of 1024 (134 MB), 64 tokens 42 -> 48.  And only while nearly every expert has one tile: with more the next tile reads them again from
// memory (32 rows of a tile, 320 tokens: 249 -> 304; 64 rows, 600 tokens: 286 -> 326; tiles of 128 rows gain 3 % at best and lose 25 % at 1400 tokens).
constexpr int64_t kOnceBytes = 256 << 20;

template <int TM, bool GATHER, int ACT, bool PLACE = false>
static void moe_gemm(const uint16_t* x, int64_t rows, const uint16_t* w, uint16_t* y, int32_t* meta, int maxTiles, int top, int N, int K,
                     float limit, float slope, float shift, hipStream_t s, const int32_t* idx = nullptr, int items = 0, int E = 0) {
    // weights that come from memory, all experts' and not the chosen ones', whose number is the batch's (below, out of a cache: 2 to 4 % slower turned, 16
    // gated experts of 2048 x 1024 39.5 -> 40.7; few chosen of large ones: no slower, one token of 128 x 2048 x 1024 32.7, of 32 x 4096 x 2048 52 -> 51)
    const bool turned = (int64_t)E * N * K * 2 >= kOnceBytes;
    if constexpr (TM == 256) {
        auto go = [&](auto kern) {
            kern<<<kSlabCUs, 256, kSlabLds, s>>>(x, (uint32_t)(rows * K * 2), w, y, meta, maxTiles, top, N, K, limit, slope, shift);
        };
        lds_limit<hy::moe_gemm256_kernel<GATHER, ACT, true>>(kSlabLds);
        lds_limit<hy::moe_gemm256_kernel<GATHER, ACT, false>>(kSlabLds);
        if (turned) go(hy::moe_gemm256_kernel<GATHER, ACT, true>);
        else go(hy::moe_gemm256_kernel<GATHER, ACT, false>);
    } else {
        constexpr int lds = hy::Tile<TM>::lds;
        const bool large = std::min<int64_t>(items, E) * N * K * 2 >= kOnceBytes;
        auto go = [&](auto kern) {
            kern<<<maxTiles * (N / hy::Tile<TM>::TN), 256, lds, s>>>(x, w, y, meta, maxTiles, top, N, K, limit, slope, shift, idx, items, E, turned);
        };
        if constexpr (TM <= 64)
            if (large && items <= (TM == 32 ? 20 : 52) * E) {
                lds_limit<hy::moe_gemm_kernel<TM, GATHER, ACT, PLACE, true>>(lds);
                return go(hy::moe_gemm_kernel<TM, GATHER, ACT, PLACE, true>);
            }
        lds_limit<hy::moe_gemm_kernel<TM, GATHER, ACT, PLACE, false>>(lds);
        go(hy::moe_gemm_kernel<TM, GATHER, ACT, PLACE, false>);
    }
}

// meta: int32 [hy_moe_meta_ints]; z: bf16 [maxTiles * tile, F]; yrows: bf16 [maxTiles * tile, d]
// (tile: hy_moe_tile).  ACT kActGlu: w_up holds 2F rows in the tile order of moe_glu_row_order.
template <int TM, int ACT>
static void moe_grouped(const uint16_t* h, const int32_t* idx, const float* wt, const uint16_t* w_up, const uint16_t* w_down,
                        uint16_t* out, int32_t* meta, uint16_t* z, uint16_t* yrows, int T, int d, int F, int E, int top,
                        float limit, float slope, float shift, hipStream_t s) {
    const int items = T * top, maxTiles = hy_moe_max_tiles(items, E, TM);
    const int nwg = moe_align_wgs(items);
    int32_t* item_row = meta + 1 + maxTiles + maxTiles * TM;
    const int up = ACT == hy::kActGlu ? 2 * F : F;
    bool placed = false;
    if constexpr (TM == 32)
        if (items <= hy::kPlaceItems && E <= hy::kPlaceE) {
            moe_gemm<TM, true, ACT, true>(h, T, w_up, z, meta, maxTiles, top, up, d, limit, slope, shift, s, idx, items, E);
            placed = true;
        }
    if (!placed) {
        if (nwg > 1) hy::moe_count_kernel<<<nwg, 1024, 0, s>>>(idx, items, E, item_row + items, item_row);
        hy::moe_place_kernel<<<nwg, 1024, 0, s>>>(idx, items, E, TM, maxTiles, meta);
        moe_gemm<TM, true, ACT>(h, T, w_up, z, meta, maxTiles, top, up, d, limit, slope, shift, s, nullptr, items, E);
    }
    moe_gemm<TM, false, -1>(z, (int64_t)maxTiles * TM, w_down, yrows, meta, maxTiles, top, d, F, 0.f, 0.f, 0.f, s, nullptr, items, E);
    hy::moe_combine_kernel<<<dim3(T, (d + 2047) / 2048), 256, 0, s>>>(h, yrows, idx, wt, item_row, out, d, top, E, ACT != hy::kActGlu);
}

// no expert chosen: the sum of nothing
static void moe_no_choice(const uint16_t* h, uint16_t* out, int T, int d, hipStream_t s) {
    hy::moe_combine_kernel<<<dim3(T, (d + 2047) / 2048), 256, 0, s>>>(h, nullptr, nullptr, nullptr, nullptr, out, d, 0, 0, 0);
}

void launch_hy_moe_grouped(const uint16_t* h, const int32_t* idx, const float* wt, const uint16_t* w_up,
                           const uint16_t* w_down, uint16_t* out, int32_t* meta, uint16_t* z, uint16_t* yrows, int T,
                           int d, int F, int E, int top, int act, hipStream_t s) {
    if (T == 0) return;
    if (top == 0) return moe_no_choice(h, out, T, d, s);
    const int tm = hy_moe_tile(T * top, E, d, F, F);
#define HY_MOE(TM, ACT) moe_grouped<TM, ACT>(h, idx, wt, w_up, w_down, out, meta, z, yrows, T, d, F, E, top, 0.f, 0.f, 0.f, s)
    if (act == 0) { if (tm == 32) HY_MOE(32, 0); else if (tm == 64) HY_MOE(64, 0); else if (tm == 128) HY_MOE(128, 0); else HY_MOE(256, 0); }
    else { if (tm == 32) HY_MOE(32, 1); else if (tm == 64) HY_MOE(64, 1); else if (tm == 128) HY_MOE(128, 1); else HY_MOE(256, 1); }
#undef HY_MOE
}

// Gated experts.  w_gu: bf16 [E, 2F, d] in the tile order of moe_glu_row_order; needs d % 128 == 0 and F % 128 == 0 (the down
// GEMM's k-steps and the up GEMM's 64-output tiles).
void launch_hy_moe_glu_grouped(const uint16_t* h, const int32_t* idx, const float* wt, const uint16_t* w_gu,
                               const uint16_t* w_down, uint16_t* out, int32_t* meta, uint16_t* z, uint16_t* yrows, int T,
                               int d, int F, int E, int top, float limit, float slope, float shift, hipStream_t s) {
    if (T == 0) return;
    if (top == 0) return moe_no_choice(h, out, T, d, s);
    const int tm = hy_moe_tile(T * top, E, d, F, 2 * F);
#define HY_MOE(TM) moe_grouped<TM, hy::kActGlu>(h, idx, wt, w_gu, w_down, out, meta, z, yrows, T, d, F, E, top, limit, slope, shift, s)
    if (tm == 32) HY_MOE(32);
    else if (tm == 64) HY_MOE(64);
    else if (tm == 128) HY_MOE(128);
    else HY_MOE(256);
#undef HY_MOE
}

}  // namespace chronos
