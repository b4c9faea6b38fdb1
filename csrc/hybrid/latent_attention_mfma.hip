// latent_attention_mfma.hip — the bfloat16 latent attention on the matrix cores (see latent_attention.hip for the
// math: one cached row per token, key = the whole row, value = its first `rank` columns, shared by all heads).
//
// One workgroup takes up to 128 (token, head) rows of one sequence — 16 per wave, rows are (token * H + head), so any
// head count tiles the same way — and walks the sequence's keys 64 at a time:
//   * the key tile goes from memory straight into LDS (no staging registers), row-major [KT][DK], NB tiles deep: the
//     next ones are on their way while one is computed, one barrier per tile.  Both MFMA operands want 8
//     k-values per lane — dims for the scores, KEYS for the weighted sum: the scores read rows as they lie, the sum
//     reads the same image through gfx950's transposing LDS reads (4 keys of 16 columns each).
//   * scores  S^T = K Q^T : 16x16x32 MFMAs with the key rows as A operand and the wave's 16 query rows (held in
//     registers for the whole kernel) as B operand, so a lane ends up with 4 keys x 1 query row per 16-key tile;
//   * softmax in float per query row (lane & 15): causal mask by the row's own position, running maximum and sum,
//     reductions over the 4 lane groups by two shuffles;
//   * sum  O^T = V^T P^T : the lane's 8 weights of two neighbouring 16-key tiles ARE a B operand (the k index is a
//     fixed permutation of the 32 keys, the same one the value columns are read with), so the weights never
//     leave registers.  Accumulators: rank / 16 tiles x 4 registers.  Optionally each weight enters as two
//     bfloat16 terms (rounded value + remainder), which keeps the float softmax weights nearly exact.
// After the last key a sink per head may join the denominator.
// With a window a row sees only its last `window` positions: the walk starts at the tile of the first row's first
// visible key and every row masks by its own position.
// Sizes: DK % 8 == 0 (the scores' steps past it are zero), rank % 16 == 0, DK <= 576, rank <= 512.
// Everything else takes latent_attention.hip.
#include "hybrid_common.h"

namespace chronos {
namespace hy {

constexpr int MKT = 64;  // keys per tile (decode of wide rows: 32)
constexpr int kRowsAhead = 1024;   // keys whose cache rows are looked up at a time
constexpr float kLog2e = 1.4426950408889634f;

// NS: k-steps of the scores (DK / 32) at most; NCT: 16-column tiles of the output (rank / 16) at most.  All of them are
// computed whatever the sizes (a run-time test in front of every product would serialise the loop); the surplus is zero
// times a real number or never stored.
// NW: waves per workgroup, 4 or 8 (16 query rows each): with 8 a staged key tile serves 128 rows and every SIMD holds two
// waves, so one wave's softmax and staging run beside the other's MFMAs.
// TT: weights as two bfloat16 terms.
// KT, NB: keys per tile and tiles in LDS; CS: waves that share the output columns.  A decode launch (up to 32 rows per
// sequence) has one workgroup per CU and is a chain of latencies: with an operand read behind every product, a row look-up
// behind every 1 KiB piece and one tile on its way, a tile of 64 keys of 576 columns took 8 us.  There (NB > 2) the operands
// of a tile are read together, the row numbers too, two (rows over 320 columns: three, of 32 keys) tiles are on their way,
// and in rows over 320 columns 8 waves take 16 keys and half of the output columns each (the scores twice; half of the
// accumulators, so two waves fit a SIMD).  With its combine, 64 sequences of 1230 - 2870 keys, mean 2048: 576 columns, 32
// heads 67.7 -> 59.5 us, 16 heads 60.6 -> 46.9, 320 columns, 16 heads 37.7 -> 32.7, 32 heads 41.4 -> 36.4; one sequence of
// 700, 576 columns, 16 heads 26.1 -> 21.3.  All of equal length 51.8 (2.9 TB/s; the longest sequence's splits are the rest).
// Four waves with three tiles ahead, operands read one by one: 68.  Rows up to 192 columns: several workgroups per CU, as before.
// KS: waves that share 16 query rows.  With few rows (decode) a tile's keys are dealt to 2 or 4 waves, each with a softmax
// of its own over its keys (16 keys per wave: 16x16x16 products in the sum), and merged through LDS at the end.
template <int NS, int NCT, int NW, int KS, int CS, int KT, int NB, bool TT>
__global__ void __launch_bounds__(64 * NW) latent_attention_mfma_kernel(
        const uint16_t* __restrict__ qa, const uint16_t* __restrict__ cache, const int32_t* __restrict__ block_table,
        int max_blocks, const int32_t* __restrict__ q_start, const int32_t* __restrict__ pos,
        const float* __restrict__ gate, uint16_t* __restrict__ out, int H, int DK, int rank, int BS, float scale,
        int window, int nsplit, float* __restrict__ part_o, float* __restrict__ part_ml, int bs_shift,
        const float* __restrict__ sink) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    const int b = blockIdx.x;
    const int t0 = q_start[b], t1 = q_start[b + 1];
    const int rows_total = (t1 - t0) * H;
    constexpr int RPB = 16 * NW / (KS * CS);  // query rows per workgroup
    constexpr int NCW = NCT / CS;             // column tiles per wave
    constexpr bool AHEAD = NB > 2;            // decode: operands read in front of the products, deeper staging
    const int rb0 = blockIdx.y * RPB;
    if (rb0 >= rows_total) return;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, g = lane >> 4, qi = lane & 15;
    const int nct = rank / 16;
    constexpr int CPR = NS * 4 + 1, krs = CPR * 16;   // key row in LDS: 16-byte chunks, bytes
    constexpr int PT = (KT * CPR + 63) / 64, PW = (PT + NW - 1) / NW, TB = PT * 1024;   // 1 KiB pieces per tile and per wave; a tile's bytes
    __shared__ int krow[kRowsAhead];  // cache row (page * page size + slot) of the keys of the next tiles
    // this lane's query row (for the B operand and for the softmax): row r of the sequence, token t0 + r / H
    const int kpart = wv % KS;   // which part of a tile's keys this wave takes
    const int c0 = CS > 1 ? wv / KS % CS * NCW : 0, wr = wv / (KS * CS) * 16;   // its first column tile, its first row
    const int r = rb0 + wr + qi;
    const bool rok = r < rows_total;
    const int rc = rok ? r : rows_total - 1;
    const int64_t grow = (int64_t)t0 * H + rc;              // row of qa / out / gate
    const int prow = rok ? pos[t0 + rc / H] : -1;
    const int last_row = min(rows_total, rb0 + RPB) - 1;
    const int pmax = pos[t0 + last_row / H];                // positions grow along the sequence
    const int k_lo = window > 0 ? max(0, pos[t0 + rb0 / H] - window + 1) / KT * KT : 0;
    const int row_lo = window > 0 ? prow - window + 1 : 0;  // the first key this lane's row sees
    bf16x8 qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {   // columns past the row's end are zero here (and real numbers in the key image)
        const u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
        qf[s] = 32 * s + 8 * g < DK ? *reinterpret_cast<const bf16x8*>(qa + grow * DK + 32 * s + 8 * g)
                                    : __builtin_bit_cast(bf16x8, z);
    }
    f32x4 O[NCW];
#pragma unroll
    for (int c = 0; c < NCW; ++c) O[c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrow = -INFINITY, lrow = 0.f;
    const float scale2 = scale * kLog2e;   // scores, maxima and sums live in the base-2 domain
    const int32_t* bt = block_table + (int64_t)b * max_blocks;
    const int chunks = DK / 8;
    const uint32_t lds0 = lds_offset(smem);
    // key tiles are dealt round-robin to the nsplit workgroups of this row block (blockIdx.z): the context length is
    // only known on the device, and a split that gets no tile contributes an empty partial
    const int kfirst = k_lo + blockIdx.z * KT, kstep = KT * nsplit;
    const int n = __builtin_amdgcn_readfirstlane(kfirst <= pmax ? (pmax - kfirst) / kstep + 1 : 0);   // tiles of this workgroup
    constexpr int RA = kRowsAhead / KT;
    auto look_up = [&](int t0) {   // cache rows of tiles t0 .. t0 + RA - 1
        for (int i = threadIdx.x; i < min(RA, n - t0) * KT; i += 64 * NW) {
            const int key = min(kfirst + (t0 + i / KT) * kstep + i % KT, pmax);  // past the end: a real row, masked below
            krow[i] = bs_shift >= 0 ? ((bt[key >> bs_shift] << bs_shift) + (key & (BS - 1))) : (bt[key / BS] * BS + key % BS);
        }
    };
    const int wu = __builtin_amdgcn_readfirstlane(wv);
    int prow_of[AHEAD ? PW : 1], pcol[AHEAD ? PW : 1];   // row of the tile and column of this lane's chunk of each piece
    if constexpr (AHEAD) {
#pragma unroll
        for (int j = 0; j < PW; ++j) {
            const int i = min(wu + j * NW, PT - 1) * 64 + lane, at = i / CPR;
            prow_of[j] = min(at, KT - 1);
            pcol[j] = min(i - at * CPR, chunks - 1) * 8;
        }
    }
    auto stage = [&](int t) {
        if constexpr (AHEAD) {   // counted waits: every wave as many pieces (the last ones of some twice)
            int kr[PW];
#pragma unroll
            for (int j = 0; j < PW; ++j) kr[j] = krow[t % RA * KT + prow_of[j]];
#pragma unroll
            for (int j = 0; j < PW; ++j)
                dma_1k(cache + ((int64_t)kr[j] * DK + pcol[j]), lds0 + t % NB * TB + min(wu + j * NW, PT - 1) * 1024);
        } else {
#pragma unroll
            for (int j = wv; j < PT; j += NW)
                dma_rows<CPR, KT>(cache, krow + t % RA * KT, DK, chunks, j, lds0 + t % NB * TB, lane);
        }
    };
    look_up(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t + 1 < NB; ++t)
        if (t < n) stage(t);
    const bool wave_on = rb0 + wr < rows_total;   // (a wave without rows only helps to stage)
    for (int t = 0; t < n; ++t) {
        const int k0 = kfirst + t * kstep;
        // this wave's pieces of the tile have landed; behind the barrier: everyone's, and the tile before it has been read by all
        dma_wait_for<PW, NB - 2>(n - 1 - t);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t + NB - 1 < n) {
            if ((t + NB - 1) % RA == 0) {   // (every kRowsAhead keys)
                look_up(t + NB - 1);
                __syncthreads();
            }
            stage(t + NB - 1);
        }
        const unsigned char* kimg = smem + t % NB * TB;
        if (wave_on) {
        // ---- scores: KT / 16 key tiles of 16; lane gets keys 16 kt + 4 g + i of query row qi
        constexpr int NKT = KT / 16 / KS;
        const int key0 = kpart * (KT / KS);
        f32x4 S[NKT];
        const unsigned char* vt = kimg + (key0 + 4 * g + (qi >> 2)) * krs + (qi & 3) * 8 + c0 * 32;
        bf16x4 vr[AHEAD ? NKT : 1][AHEAD ? NCW : 1];
        if constexpr (AHEAD) {
            // The compiler would read each operand into the registers of the one before it, behind its product: all of the
            // scores' are read first, then, behind their products and under the softmax, all of the sum's.
            bf16x8 kf[NKT][NS];
            f32x4 odd[NKT];
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) {
#pragma unroll
                for (int s = 0; s < NS; ++s)
                    kf[kt][s] = *reinterpret_cast<const bf16x8*>(kimg + (key0 + 16 * kt + qi) * krs + g * 16 + s * 64);
                S[kt] = odd[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int s = 0; s < NS; ++s)
#pragma unroll
                for (int kt = 0; kt < NKT; ++kt)
                    (s & 1 ? odd[kt] : S[kt]) = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[kt][s], qf[s], s & 1 ? odd[kt] : S[kt], 0, 0, 0);
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt) S[kt] += odd[kt];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
                for (int c = 0; c < NCW; ++c) vr[kt][c] = lds_read_tr4(vt + 16 * kt * krs + c * 32);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int kt = 0; kt < NKT && !AHEAD; ++kt) {
            S[kt] = f32x4{0.f, 0.f, 0.f, 0.f};
            const unsigned char* arow = kimg + (key0 + 16 * kt + qi) * krs + g * 16;
#pragma unroll
            for (int s = 0; s < NS; ++s)
                S[kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(arow + s * 64), qf[s],
                                                                S[kt], 0, 0, 0);
        }
        // ---- softmax over the tile for query row qi (this lane and the 3 other lane groups hold its keys)
        float mx = -INFINITY;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = k0 + key0 + 16 * kt + 4 * g + i;
                const float sv = key <= prow && key >= row_lo ? S[kt][i] * scale2 : -INFINITY;
                S[kt][i] = sv;
                mx = fmaxf(mx, sv);
            }
        mx = rows_max(mx);
        const float mn = fmaxf(mrow, mx);
        const float corr = (mn == -INFINITY) ? 1.f : __builtin_amdgcn_exp2f(mrow - mn);
        const float mref = (mn == -INFINITY) ? 0.f : mn;   // (all masked: every exponent is -inf, every weight 0)
        float sum = 0.f;
#pragma unroll
        for (int kt = 0; kt < NKT; ++kt)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float p = __builtin_amdgcn_exp2f(S[kt][i] - mref);
                S[kt][i] = p;
                sum += p;
            }
        sum = rows_sum(sum);
        lrow = lrow * corr + sum;
        mrow = mn;
        // ---- weighted sum of the value columns: k index of step u = [tile 2u keys 4g..4g+3 | tile 2u+1 keys 4g..4g+3]
        constexpr int NU = NKT / 2;
        if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0) {   // (rarely, once the maxima have settled)
#pragma unroll
            for (int c = 0; c < NCW; ++c) O[c] *= corr;
        }
        if constexpr (NKT == 1) {
            bf16x4 pf, pl;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                pf[e] = (__bf16)S[0][e];
                if constexpr (TT) pl[e] = (__bf16)(S[0][e] - (float)pf[e]);
            }
#pragma unroll
            for (int c = 0; c < NCW; ++c) {
                const bf16x4 vf = AHEAD ? vr[0][AHEAD ? c : 0] : lds_read_tr4(vt + c * 32);
                O[c] = mfma_16x16x16(vf, pf, O[c]);
                if constexpr (TT) O[c] = mfma_16x16x16(vf, pl, O[c]);
            }
        }
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            bf16x8 pf, pl;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float w = S[2 * u + (e >> 2)][e & 3];
                pf[e] = (__bf16)w;
                if constexpr (TT) pl[e] = (__bf16)(w - (float)pf[e]);
            }
#pragma unroll
            for (int c = 0; c < NCW; ++c) {
                const bf16x4 lo = AHEAD ? vr[AHEAD ? 2 * u : 0][AHEAD ? c : 0] : lds_read_tr4(vt + 32 * u * krs + c * 32);
                const bf16x4 hi = AHEAD ? vr[AHEAD ? 2 * u + 1 : 0][AHEAD ? c : 0] : lds_read_tr4(vt + (32 * u + 16) * krs + c * 32);
                const bf16x8 vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                O[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pf, O[c], 0, 0, 0);
                if constexpr (TT) O[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vf, pl, O[c], 0, 0, 0);
            }
        }
        }
    }
    if constexpr (KS > 1) {   // the waves that share these rows merge their partial results; the first one goes on
        constexpr int MS = NCW * 16 + 4;    // floats per row (padded)
        float* mb = reinterpret_cast<float*>(smem);
        static_assert(NW * 16 * MS * 4 <= NB * TB, "the partial rows fit the key tiles' LDS");
        __shared__ float ml[NW][16][2];
        __syncthreads();                    // everyone is done with the key tiles
#pragma unroll
        for (int c = 0; c < NCW; ++c) *reinterpret_cast<f32x4*>(mb + (wv * 16 + qi) * MS + 16 * c + 4 * g) = O[c];
        if (g == 0) {
            ml[wv][qi][0] = mrow;
            ml[wv][qi][1] = lrow;
        }
        __syncthreads();
        if (kpart != 0) return;
        float mn = mrow, e[KS];
#pragma unroll
        for (int k = 1; k < KS; ++k) mn = fmaxf(mn, ml[wv + k][qi][0]);
        const float mref = mn == -INFINITY ? 0.f : mn;
        e[0] = exp2f(mrow - mref);
        lrow *= e[0];
#pragma unroll
        for (int k = 1; k < KS; ++k) {
            e[k] = exp2f(ml[wv + k][qi][0] - mref);
            lrow += e[k] * ml[wv + k][qi][1];
        }
        mrow = mn;
#pragma unroll
        for (int c = 0; c < NCW; ++c) {
            O[c] *= e[0];
#pragma unroll
            for (int k = 1; k < KS; ++k)
                O[c] += e[k] * *reinterpret_cast<const f32x4*>(mb + ((wv + k) * 16 + qi) * MS + 16 * c + 4 * g);
        }
    }
    if (!rok) return;
    if (nsplit > 1) {  // unnormalised partial: the combine kernel merges the splits
        const int64_t pr = grow * nsplit + blockIdx.z;
        if (g == 0 && c0 == 0) {
            part_ml[pr * 2] = mrow;
            part_ml[pr * 2 + 1] = lrow;
        }
#pragma unroll
        for (int c = 0; c < NCW; ++c)
            if (c0 + c < nct) *reinterpret_cast<f32x4*>(part_o + pr * rank + 16 * (c0 + c) + 4 * g) = O[c];
        return;
    }
    float f = 1.f / lrow;
    if (sink != nullptr) {   // exp(sink) joins the denominator, without a value
        const float sk = sink[rc % H] * kLog2e, mn = fmaxf(mrow, sk), c = exp2f(mrow - mn);
        f = c / (lrow * c + exp2f(sk - mn));
    }
    if (gate != nullptr) f *= sigmoidf_(gate[grow]);
    // lane holds O^T[col = 16 c + 4 g + i][query row qi]
#pragma unroll
    for (int c = 0; c < NCW; ++c)
        if (c0 + c < nct) {
            const u16x4 o = u16x4{f2bf(O[c][0] * f), f2bf(O[c][1] * f), f2bf(O[c][2] * f), f2bf(O[c][3] * f)};
            *reinterpret_cast<u16x4*>(out + grow * rank + 16 * (c0 + c) + 4 * g) = o;
        }
}

// one wave per (token, head) row and 256 columns: out = sum_z 2^(m_z - m) O_z / (sum_z 2^(m_z - m) l_z + 2^(sink log2 e - m)) * sigmoid(gate)
// (the partial maxima are in the base-2 domain: score * scale * log2 e).  Lane z holds
// split z's maximum and sum; a lane then sums 4 neighbouring columns over the splits, all on their way before
// the maxima are looked at: a few rows are one memory latency, not one per four splits behind another: 6 rows of 8 heads in 13 splits 6.7 -> 3.6 us.
constexpr int kLatentSplits = 16;   // at most (hy_latent_nsplit)
__global__ void __launch_bounds__(256) latent_combine_kernel(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                             const float* __restrict__ gate, uint16_t* __restrict__ out,
                                                             int64_t rows, int rank, int nsplit,
                                                             const float* __restrict__ sink, int H) {
    const int lane = threadIdx.x & 63;
    const int nc = (rank + 255) / 256;
    const int64_t it = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6), r = it / nc;
    if (r >= rows) return;
    const int c = (int)(it - r * nc) * 256 + lane * 4;    // (rank is a multiple of 16; lanes past it read its last columns)
    const float* const po = part_o + r * nsplit * rank + min(c, rank - 4);
    f32x4 v[kLatentSplits];
#pragma unroll
    for (int z = 0; z < kLatentSplits; ++z)
        if (z < nsplit) v[z] = *reinterpret_cast<const f32x4*>(po + (int64_t)z * rank);
    const float mz = lane < nsplit ? part_ml[(r * nsplit + lane) * 2] : -INFINITY;
    const float lz = lane < nsplit ? part_ml[(r * nsplit + lane) * 2 + 1] : 0.f;
    const float sk = sink != nullptr ? sink[r % H] * kLog2e : -INFINITY;
    const float m = fmaxf(wave_max(mz), sk);
    float e = mz == -INFINITY ? 0.f : exp2f(mz - m);   // (a split without a visible key adds nothing)
    const float l = wave_sum(e * lz) + (sink != nullptr ? exp2f(sk - m) : 0.f);
    e *= (gate != nullptr ? sigmoidf_(gate[r]) : 1.f) / l;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int z = 0; z < kLatentSplits; ++z)
        if (z < nsplit) acc += __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(e), z)) * v[z];
    if (c < rank) *reinterpret_cast<u16x4*>(out + r * rank + c) = u16x4{f2bf(acc[0]), f2bf(acc[1]), f2bf(acc[2]), f2bf(acc[3])};
}

}  // namespace hy

template <int NS, int NCT, int NW, int KS, int CS, int KT, int NB, bool TT>
static void la_mfma_launch(const uint16_t* qa, const uint16_t* cache, const int32_t* bt, int max_blocks,
                           const int32_t* q_start, const int32_t* pos, const float* gate, uint16_t* out, int B, int H,
                           int DK, int rank, int BS, int max_q, float scale, int window, int nsplit, float* part_o,
                           float* part_ml, const float* sink, hipStream_t s) {
    auto kern = hy::latent_attention_mfma_kernel<NS, NCT, NW, KS, CS, KT, NB, TT>;
    constexpr int bytes = NB * ((KT * (NS * 4 + 1) + 63) / 64) * 1024;
    static_assert(bytes <= 152 * 1024, "LDS");
    static int set_bytes = 0;
    if (bytes > set_bytes) {
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        set_bytes = bytes;
    }
    constexpr int rpb = 16 * NW / (KS * CS);
    const dim3 grid(B, (max_q * H + rpb - 1) / rpb, nsplit);
    const int bs_shift = (BS & (BS - 1)) == 0 ? __builtin_ctz(BS) : -1;
    kern<<<grid, 64 * NW, bytes, s>>>(qa, cache, bt, max_blocks, q_start, pos, gate, out, H, DK, rank, BS, scale, window,
                                  nsplit, part_o, part_ml, bs_shift, sink);
}

bool hy_latent_mfma_ok(int DK, int rank) { return !(DK % 8 || rank % 16 || DK > 576 || rank > 512 || rank > DK); }

// Splits of the key range (flash-decoding) for a launch of `wgs` workgroups over contexts of at most max_ctx keys:
// enough workgroups to cover the chip, at least one key tile per split (2 behind a window, whose few tiles are all of the
// walk), at most 16.  A tile of a few rows is a chain of latencies, dearer than its partials: at least 4 tiles, 2 tiles and one, us with the combining,
// 1 sequence of 700 keys, 8 heads of 288 columns 15.1, 12.1, 11.1, 32 heads of 576 30.8, 21.0, 17.8; 6 of about 200 12.2, 12.2, 11.0, 23.5, 20.5,
// 17.7; 16 of about 700 15.3, 12.5, 11.2.  Not two splits: 1 of 120 keys 8.2, 9.4.  32 splits: 6 of about 2000, 32 heads 24.1 -> 26.2.
// Three only where the rank is large and workgroups few: 200 keys, us, whole and in three: 16 heads of rank 128, 1 and 64 sequences 9.1, 9.8 and 9.4, 11.1; 8 of rank 256
// 11.7, 11.6 and 12.3, 12.9; 32 of rank 512 21.3, 18.6 and 22.1, 24.8 (16 sequences 21.6, 20.0; 32 level).
int hy_latent_nsplit(int wgs, int max_ctx, bool windowed, int rank) {
    if (wgs >= 128) return 1;
    int want = (256 + wgs - 1) / wgs, cap = max_ctx / ((windowed ? 2 : 1) * hy::MKT);
    if (!windowed && cap < (rank > 256 && wgs <= 32 ? 3 : 4)) cap = 1;
    if (want > hy::kLatentSplits) want = hy::kLatentSplits;
    if (want > cap) want = cap;
    return want < 1 ? 1 : want;
}

// false: these sizes are not served here (the caller takes the general kernel).  nsplit > 1: part_o float
// [T * H * nsplit, rank] and part_ml float [T * H * nsplit, 2] scratch.
bool launch_hy_latent_attention_mfma(const uint16_t* qa, const uint16_t* cache, const int32_t* bt, int max_blocks,
                                     const int32_t* q_start, const int32_t* pos, const float* gate, uint16_t* out, int B,
                                     int H, int DK, int rank, int BS, int max_q, float scale, int window, bool two_term,
                                     int nsplit, float* part_o, float* part_ml, int64_t total_rows, const float* sink,
                                     hipStream_t s) {
    if (!hy_latent_mfma_ok(DK, rank)) return false;
    if (B == 0 || max_q == 0) return true;
#define HY_LAM(NS, NCT, NW, KS, CS, KT, NB, TT) la_mfma_launch<NS, NCT, NW, KS, CS, KT, NB, TT>(qa, cache, bt, max_blocks, q_start, pos, gate, out, B, H, DK, rank, BS, max_q, scale, window, nsplit, part_o, part_ml, sink, s)
    // 8 waves per workgroup when a sequence brings more than 64 rows; up to 32 or 16 rows 2 or 4 waves share them (each
    // instance's figures stand at the kernel)
    const int rows = max_q * H;
#define HY_LAM_R(NS, NCT, TT)                             \
    do {                                                  \
        if (rows > 64) HY_LAM(NS, NCT, 8, 1, 1, 64, 2, TT);      \
        else if (rows > 32) HY_LAM(NS, NCT, 4, 1, 1, 64, 2, TT); \
        else if (NS > 10 || rows > 16) HY_LAM(NS, NCT, (NS > 10 ? 8 : 4), 2, (NS > 10 ? 2 : 1), (NS > 10 ? 32 : 64), (NS > 10 ? 4 : NS > 6 ? 3 : 2), TT); \
        else HY_LAM(NS, NCT, (NS > 10 ? 8 : 4), (NS > 10 ? 2 : 4), (NS > 10 ? 2 : 1), (NS > 10 ? 32 : 64), (NS > 10 ? 4 : NS > 6 ? 3 : 2), TT); \
    } while (0)
#define HY_LAM_T(NS, NCT)                                                                       \
    do {                                                                                        \
        if (two_term) HY_LAM_R(NS, NCT, true); else HY_LAM_R(NS, NCT, false);                   \
    } while (0)
    if (DK <= 128 && rank <= 64) HY_LAM_T(4, 4);
    else if (DK <= 192 && rank <= 128) HY_LAM_T(6, 8);
    else if (DK <= 320 && rank <= 256) HY_LAM_T(10, 16);
    else HY_LAM_T(18, 32);
#undef HY_LAM_T
#undef HY_LAM_R
#undef HY_LAM
    if (nsplit > 1)
        hy::latent_combine_kernel<<<(unsigned)((total_rows * ((rank + 255) / 256) + 3) / 4), 256, 0, s>>>(part_o, part_ml, gate, out, total_rows, rank, nsplit, sink, H);
    return true;
}

}  // namespace chronos
