// chunk_scan.hip — the linear-state recurrences of linear_scan.hip and mlstm.hip with one decay per head and token, on the
// matrix cores: prompt portions are taken 64 tokens at a time.  With L_t = sum of the log decays of a chunk's tokens up to
// t, S the state before the chunk, w_s the factor on what token s writes and r_t the factor on what token t reads,
//
//     o_t = r_t ( e^L_t S^T q_t + sum_(s <= t) e^(L_t - L_s) w_s (k_s . q_t) v_s )
//     S  <- e^L_C S + sum_s k_s (e^(L_C - L_s) w_s v_s)^T
//
// which are the sums of the token-by-token form in another order.  With the delta rule a token writes u_s = beta_s (v_s - what
// the state before it reads at k_s) in place of v_s; with A[t, s] = beta_t e^(L_t - L_s) w_t w_s (k_t . k_s) below the
// diagonal (w: the scale of k), (I + A) u = beta (v - e^L w S^T k), solved 16 rows at a time with the diagonal tiles' inverses.
//
// Precision: q, k and v are bfloat16, everything else stays float32.  A float32 operand of a matrix product (the state, the
// weights of a chunk's tokens, the scaled values) enters as three bfloat16 terms whose sum is exactly that number, so a
// product costs three matrix instructions and loses nothing (two float32 operands: six of the nine products of terms, the
// rest is below 2^-26), and all products accumulate in float32.  L is summed in float64: differences of sums over strong
// decays keep their digits.  Terms by truncation cost 3% less time, but leave the errors one-sided and larger (the state
// after the state-space form: 4.8e-8 of its norm off the float64 recurrence; nearest terms 3.9e-8; token by token 4.2e-8).
// The delta rule's solve carries what its sums round off along: the state is 5.7e-8 off (token by token 5.8e-8; without,
// 6.1e-8, and 9.3e-8 with the products added to the sum one by one).
//
// Where something is infinite or NaN, or overflows on the way, a weight of 0 above the diagonal times a later token's value would reach
// back to earlier tokens, and a number without three finite terms would turn to NaN: a wave that has met such a thing in its read-outs
// or its state takes the sequence's tokens again at the end, one by one, from the state before them.
//
// A workgroup is NW waves and serves 16 NW value columns of one (sequence, head); a wave keeps all D rows of its 16 columns
// of S in accumulators, which are in the operand layout of the read-out's product as they stand.  A chunk's q, k, v rows
// come by DMA into one of two LDS buffers while the chunk before is computed; 16-byte pieces are permuted within a row by a
// function of the row, so that neither the row-wise reads nor the transposing ones meet in a bank.  The waves share the
// 64 x 64 weights (ten 16 x 16 tiles on and below the diagonal) through LDS; the delta rule's tiles lie beside.
//
// What bounds it: the chain of a sequence's chunks, one wave per SIMD: vector instructions (the cutting into terms, the
// exponentials) and 114 matrix instructions (delta: 162) per chunk and wave at D = 128, and two barriers, 5 us a chunk (delta: 10, 4.8 with
// its tiles made ahead).
// Measured, 4 sequences of 2048 tokens, token by token -> this: retention, 8 heads of 128 x 128: 797 -> 177 us, in four
// segments 73; 32 heads: 857 -> 182; state-space form, 128 heads of 128 x 64: 1058 -> 442; mlstm, 4 heads of 128 x 256: 1987
// -> 220, in four segments 95, 4 heads of 256 x 512: 3050 -> 299, in two 213; delta rule, 32 heads of 128 x 128: 959 -> 352,
// with the tiles ahead 270.
// One and two waves per workgroup: 436 and 302 us where four took 233 (of 171, before addresses, weights and stores lost
// their branches).
#include "chronos_lds.h"
#include "chunk_common.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace chronos {
namespace hy {

constexpr int kCH = 64;   // tokens per chunk
constexpr int kCW = 4;    // waves per workgroup (NW above)

// e^x with x's digits beyond float32 kept
__device__ __forceinline__ float exp_d(double x) {
    const float h = (float)x, e = expf(h);
    return e + e * (float)(x - h);
}

// acc, or NaN where one of x is infinite or NaN
__device__ __forceinline__ float not_finite(const f32x4& x, float acc) {
#pragma unroll
    for (int r = 0; r < 4; ++r) acc = __builtin_fmaf(x[r], 0.f, acc);
    return acc;
}

// Running sum over the wave's lanes (lane l: the sum of lanes 0 .. l): within rows of 16 lanes, then from row to row.
__device__ __forceinline__ double lanes_running_sum(double x) {
    auto from = [](double v, auto ctrl, auto rows) {
        const uint64_t u = __builtin_bit_cast(uint64_t, v);
        const uint32_t lo = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)u, decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
        const uint32_t hi = __builtin_amdgcn_update_dpp(0, (int)(uint32_t)(u >> 32), decltype(ctrl)::value, decltype(rows)::value, 0xf, true);
        return __builtin_bit_cast(double, (uint64_t)hi << 32 | lo);
    };
    using std::integral_constant;
    constexpr integral_constant<int, 0xf> all{};
    x += from(x, integral_constant<int, 0x111>{}, all);                              // one lane to the right
    x += from(x, integral_constant<int, 0x112>{}, all);
    x += from(x, integral_constant<int, 0x114>{}, all);
    x += from(x, integral_constant<int, 0x118>{}, all);
    x += from(x, integral_constant<int, 0x142>{}, integral_constant<int, 0xa>{});    // lane 15 of rows 0, 2 to rows 1, 3
    x += from(x, integral_constant<int, 0x143>{}, integral_constant<int, 0xc>{});    // lane 31 to rows 2 and 3
    return x;
}

// What the forms read per token: plain: decay (one per token and head, or dts = 0: per head), qscale, kscale, vscale
// (any of the three may be absent); delta: the same without vscale, and beta; mlstm: the log decays, log write factors and
// e^-m of mlstm_gates_kernel.
struct ChunkScan {
    const uint16_t* proj;
    int ldp, q_off, k_off, v_off;
    const float *qscale, *kscale, *vscale, *decay, *beta;
    int dts;
    float q_mul;
    const float *la, *lb, *em;
    const int32_t *q_start, *pos0, *slots;
    const float* n0;   // [B, H, D]: the normaliser before the step (workgroups of one (sequence, head) start at any time)
    float *S, *n, *o;
    int B, HK, H, Dv, T;
    // more than one segment per sequence: states before it [B, H, D, Dv], then of each segment but the last; mlstm: normalisers and all:
    // products of decays of each segment but the last, [segs - 1, B, H, ..]
    int segs;
    float *seg_s, *seg_n, *seg_d;
    unsigned char* tiles;   // delta: [slots, H, kDeltaTiles] of delta_tiles_kernel, or nullptr
};

// What the delta rule's chunks need of their q, k and decays alone, per chunk and head, written by delta_tiles_kernel (bytes): tiles as three terms, 512
// bytes a term: the weights [10], the solve's below the diagonal [6], the inverses of its diagonal ones less the identity [4] | floats: beta,
// beta k-scale e^L, c, e^L, r [64] each, e^L_C
constexpr int kDtTile = 1536, kDtA = 10 * kDtTile, kDtT = 16 * kDtTile, kDtSc = 20 * kDtTile, kDtEnd = kDtSc + 5 * kCH * 4, kDeltaTiles = 32 * 1024;
static_assert(kDtEnd + 4 <= kDeltaTiles, "tiles of a chunk");
// Chunk c of sequence b, tokens from s0 on, is chunk s0 / 64 + b + c of the launch: no two alike, T / 64 + B + 1 of them at most.
__host__ __device__ constexpr int64_t delta_slots(int T, int B) { return (int64_t)T / kCH + B + 1; }
__device__ __forceinline__ Terms4 load_terms(const unsigned char* tile, int lane) {
    const bf16x4* const at = reinterpret_cast<const bf16x4*>(tile) + lane;
    return {at[0], at[64], at[128]};
}

// LDS (bytes): two buffers of q | k | v | weight tiles [10][64 lanes] x 16 (delta: and the solve's tiles [10], the inverses of
// the diagonal ones [4]) | every wave's own copy of the scalars (L in float64, w, c; delta: beta, beta k-scale, and that times
// e^L) | mlstm: the weight tiles' sums over s [10][16] and the waves' parts of n . q [NW][64].  PRE: two buffers of q | k | v | delta_tiles_kernel's.
template <int D, int MODE, bool PRE> struct ChunkLds {
    static constexpr int Q = kCH * D * 2, V = kCH * kCW * 32, BUF = 2 * Q + V + (PRE ? kDeltaTiles : 0);
    static constexpr int PT = 2 * BUF, AT = PT + (PRE ? 0 : 10 * 1024), TT = AT + (MODE == kScanDelta && !PRE ? 10 * 1024 : 0);
    static constexpr int OWN = TT + (MODE == kScanDelta && !PRE ? 4 * 1024 : 0), OWN_SIZE = PRE ? 0 : kCH * (MODE == kScanDelta ? 28 : 16);
    static constexpr int SUM = OWN + kCW * OWN_SIZE, SIZE = SUM + (MODE == kScanMlstm ? 640 + kCW * 256 : 0);
};

// A chunk's scalars, lane t token t of nt: its sum of log decays, the factors on what it writes (w) and reads (rd), the sign gC of the product of the
// chunk's decays, and their sum LC
template <bool MLSTM>
__device__ __forceinline__ double chunk_logs(bool valid, float sd, float sw, int lane, float& w, float& rd, float& gC, double& LC) {
    double L = 0.0;
    w = 0.f;
    gC = 1.f;
    if (valid) {
        if constexpr (MLSTM) {
            L = sd;
            w = expf(sw);
        } else {
            const float lg = logf(fabsf(sd));
            L = lg < -110.f ? -110.f : lg;   // e^-110 is 0 in float32, as a decay of 0 is
            w = sw;
        }
    }
    if constexpr (!MLSTM) {   // the sign of a product of decays up to t goes with what t writes and reads
        const uint64_t neg = __ballot(valid && sd < 0.f);
        if (__popcll(neg & (~0ull >> (63 - lane))) & 1) {
            w = -w;
            rd = -rd;
        }
        if (__popcll(neg) & 1) gC = -1.f;
    }
    L = lanes_running_sum(L);
    LC = __builtin_bit_cast(double, (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(__builtin_bit_cast(uint64_t, L) >> 32), 63) << 32 |
                                        (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)__builtin_bit_cast(uint64_t, L), 63));
    return L;
}

// Rows 16 i + ln of a chunk's q or k, columns 32 kk + 8 g ..: either operand of a product over columns
template <int D> __device__ __forceinline__ bf16x8 chunk_row8(const unsigned char* base, int i, int kk, int ln, int g) {
    return *reinterpret_cast<const bf16x8*>(base + (16 * i + ln) * (D * 2) + (((kk * 4 + g) ^ spread<D / 8>(ln)) * 16));
}
// Weights: tile (i, j) holds rows s = 16 j.. (4 g + r) and columns t = 16 i.. (ln): k_s . tbase_t times e^(L_t - L_s) w_s, for s <= t
template <int D>
__device__ __forceinline__ f32x4 chunk_weights(const unsigned char* kb, const unsigned char* tbase, int i, int j, const double* Ls, const float* ws, int ln, int g) {
    constexpr int KK = D / 32;
    bf16x8 x[KK], y[KK];
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) { x[kk] = chunk_row8<D>(kb, j, kk, ln, g); y[kk] = chunk_row8<D>(tbase, i, kk, ln, g); }
    f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) acc[kk & 1] = mfma_16x16x32(x[kk], y[kk], acc[kk & 1]);
    f32x4 v = acc[0];
    if (KK > 1) v += acc[1];
    const int t = 16 * i + ln;
    const double Lt = Ls[t];
    const f32x4 wsv = *reinterpret_cast<const f32x4*>(ws + 16 * j + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int s = 16 * j + 4 * g + r;
        v[r] = s <= t ? v[r] * (wsv[r] * exp_d(Lt - Ls[s])) : 0.f;
    }
    return v;
}
// Delta: tile (i, j) of -A, A[t, s] = beta_t k-scale_t k-scale_s e^(L_t - L_s) (k_t . k_s) for s < t (bk: beta k-scale)
template <int D>
__device__ __forceinline__ f32x4 chunk_minus_a(const unsigned char* kb, int i, int j, const double* Ls, const float* ws, const float* bk, int ln, int g) {
    const int t = 16 * i + ln;
    f32x4 v = chunk_weights<D>(kb, kb, i, j, Ls, ws, ln, g);
    const float f = -bk[t];
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = 16 * j + 4 * g + r < t ? v[r] * f : 0.f;
    return v;
}
// (I + A)^-1 - I of a diagonal tile whose -A is at `a`, by forward substitution, lane n column n, to `out` in operand layout: lane (t, g) holds
// columns 4 g ..  A wave by itself.
__device__ __forceinline__ void chunk_inverse(const f32x4* a, float* out, int ln, int g) {
    __builtin_amdgcn_wave_barrier();   // the wave's own writes
    float x[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        float acc[4] = {r == ln ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < (r + 3) / 4; ++q) {
            const f32x4 row = a[q * 16 + r];   // -A[r][4 q ..]
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * q + e < r) acc[e] += row[e] * x[4 * q + e];
        }
        x[r] = (acc[0] + acc[1]) + (acc[2] + acc[3]);
    }
    if (g == 0) {
#pragma unroll
        for (int r = 0; r < 16; ++r) out[((ln >> 2) * 16 + r) * 4 + (ln & 3)] = r == ln ? 0.f : x[r];
    }
}

// The delta rule's tiles and scalars of every chunk and head, all chunks side by side: what the walk over a sequence's chunks had done between its steps, half
// of a chunk's time there, and once for every 64 value columns.  Same arithmetic, same bits.  Both launches, us, heads of 128 x 128, before -> this: 8
// heads, one sequence of 4000 tokens 670 -> 306 (14 of them this launch), 113 29 -> 23, 21 of about 100 52 -> 40; 32 heads, one of 1351 240 -> 124, 4 of 2048 383 -> 292
// (74: 32 KB written per chunk and head, three workgroups per CU; the walk then reads 3.9 TB/s).  A workgroup per chunk and head; in small
// launches bound by one chunk's latencies.
template <int D>
__global__ void __launch_bounds__(256) delta_tiles_kernel(const ChunkScan a) {
    constexpr int CPR = D / 8, NW = 4, Q = kCH * D * 2;
    extern __shared__ __attribute__((aligned(1024))) unsigned char cs_smem[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane & 15, g = lane >> 4;
    const int hd = blockIdx.x % a.H, slot = blockIdx.x / a.H, hk = hd / (a.H / a.HK);
    int upto = 0;   // sequences whose first chunk is this one or an earlier one
    for (int j = 0; j < a.B; j += 64) {
        const int q = j + lane;
        upto += __popcll(__ballot(q < a.B && (a.q_start[min(q, a.B - 1)] >> 6) + q <= slot));
    }
    if (upto == 0) return;
    const int b = upto - 1, s0 = a.q_start[b], t1 = a.q_start[b + 1], tb = s0 + (slot - (s0 >> 6) - b) * kCH;
    if (tb >= t1) return;
    const int nt = min(kCH, t1 - tb), last = nt - 1, nrow = (nt + 15) / 16;
    unsigned char* const qb = cs_smem;
    unsigned char* const kb = cs_smem + Q;
    f32x4* const diag = reinterpret_cast<f32x4*>(cs_smem + 2 * Q) + wv * 64;
    float* const inv = reinterpret_cast<float*>(cs_smem + 2 * Q + 4096) + wv * 256;
    double* const Ls = reinterpret_cast<double*>(cs_smem + 2 * Q + 8192 + wv * 1024);
    float *const ws = reinterpret_cast<float*>(Ls + kCH), *const bk = ws + kCH;
    const uint32_t lds0 = lds_offset(cs_smem);
    const uint16_t* const q = a.proj + a.q_off + (int64_t)hk * D + (int64_t)tb * a.ldp;
    const uint16_t* const k = a.proj + a.k_off + (int64_t)hk * D + (int64_t)tb * a.ldp;
#pragma unroll
    for (int u = 0; u < (CPR + NW - 1) / NW; ++u) {
        const int j = wv + NW * u, i = j * 64 + lane, row = i / CPR, c = (i % CPR) ^ spread<CPR>(row);
        if (CPR % NW == 0 || j < CPR) {
            const int64_t at = (int64_t)min(row, last) * a.ldp + c * 8;
            dma_1k(q + at, __builtin_amdgcn_readfirstlane(lds0 + j * 1024));
            dma_1k(k + at, __builtin_amdgcn_readfirstlane(lds0 + Q + j * 1024));
        }
    }
    const int64_t t = min(tb + lane, t1 - 1);
    const bool valid = lane < nt;
    const float sd = a.dts != 0 ? a.decay[t * a.dts + hd] : a.decay[hd];
    float rd = a.qscale != nullptr ? a.qscale[t * a.HK + hk] : a.q_mul, w, gC;
    const float sb = a.beta[t * a.H + hd];
    double LC;
    const double L = chunk_logs<false>(valid, sd, a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f, lane, w, rd, gC, LC);
    const float eL = exp_d(L), bt = valid ? sb : 0.f;
    Ls[lane] = L;
    ws[lane] = w;
    bk[lane] = bt * w;
    unsigned char* const out = a.tiles + ((int64_t)slot * a.H + hd) * kDeltaTiles;
    if (wv == 0) {
        float* const sc = reinterpret_cast<float*>(out + kDtSc);
        sc[lane] = bt;
        sc[kCH + lane] = bt * w * eL;
        sc[2 * kCH + lane] = gC * exp_d(LC - L) * w;
        sc[3 * kCH + lane] = eL;
        sc[4 * kCH + lane] = rd;
        if (lane == 0) sc[5 * kCH] = gC * exp_d(LC);
    }
    auto put = [&](int at, const Terms4& v) {
        bf16x4* const to = reinterpret_cast<bf16x4*>(out + at) + lane;
        to[0] = v.h;
        to[64] = v.m;
        to[128] = v.l;
    };
    dma_wait();
    __syncthreads();
    for (int p = wv; p < 10; p += NW) {
        const int i = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, j = p - i * (i + 1) / 2;
        if (i < nrow) put(p * kDtTile, split3(chunk_weights<D>(kb, qb, i, j, Ls, ws, ln, g)));
    }
    for (int p = NW - 1 - wv; p < 6; p += NW) {   // (the last waves had a tile less)
        const int i = p < 1 ? 1 : p < 3 ? 2 : 3, j = p - i * (i - 1) / 2;
        if (i < nrow) put(kDtA + p * kDtTile, split3(chunk_minus_a<D>(kb, i, j, Ls, ws, bk, ln, g)));
    }
    if (wv < nrow) {
        diag[lane] = chunk_minus_a<D>(kb, wv, wv, Ls, ws, bk, ln, g);
        chunk_inverse(diag, inv, ln, g);
        __builtin_amdgcn_wave_barrier();
        put(kDtT + wv * kDtTile, split3(reinterpret_cast<const f32x4*>(inv)[lane]));
    }
}

// STATE: the first pass over segments, which only carries the state on (each from 0, the first from the sequence's state)
// PRE (delta): the tiles and scalars of the chunks come from delta_tiles_kernel
template <int D, int MODE, bool STATE, bool PRE = false>
__global__ void __launch_bounds__(64 * kCW, 1) __attribute__((amdgpu_waves_per_eu(1, 1))) chunk_scan_kernel(const ChunkScan a) {
    using M = ChunkLds<D, MODE, PRE>;
    static_assert(!PRE || (MODE == kScanDelta && !STATE), "tiles ahead: the delta rule");
    constexpr bool DELTA = MODE == kScanDelta, MLSTM = MODE == kScanMlstm;
    constexpr int NW = kCW, CPR = D / 8, VC = 2 * NW, KK = D / 32;   // 16-byte pieces per row of q and k, of v; 32-row steps of the state
    extern __shared__ __attribute__((aligned(1024))) unsigned char cs_smem[];
    f32x4* const pt = reinterpret_cast<f32x4*>(cs_smem + M::PT);
    f32x4* const at = reinterpret_cast<f32x4*>(cs_smem + M::AT);
    f32x4* const tt = reinterpret_cast<f32x4*>(cs_smem + M::TT);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), ln = lane & 15, g = lane >> 4;
    unsigned char* const own = cs_smem + M::OWN + wv * M::OWN_SIZE;
    double* const Ls = reinterpret_cast<double*>(own);
    float* const ws = reinterpret_cast<float*>(own + kCH * 8);
    float* const cs = ws + kCH;
    float *const bs = cs + kCH, *const bk = bs + kCH, *const be = bk + kCH;            // delta
    float* const psum = reinterpret_cast<float*>(cs_smem + M::SUM);                    // mlstm
    float* const nq = psum + 160;
    // groups of workgroups that share q and k rows go to one XCD (workgroup i runs on XCD i % 8), the next segment's behind them: less
    // than 8 groups leave XCDs free
    const int nslab = (a.Dv + 16 * NW - 1) / (16 * NW), id = blockIdx.x >> 3, seg = blockIdx.y;
    const int group = (id / nslab) * 8 + ((blockIdx.x - seg * a.B * a.H) & 7), slab = id % nslab;
    if (group >= a.B * a.H) return;
    const int b = group / a.H, hd = group % a.H, hk = hd / (a.H / a.HK);
    const int s0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= s0) return;
    const int chunks = (t1 - s0 + kCH - 1) / kCH;
    const int t0 = s0 + chunks * seg / a.segs * kCH, te = min(t1, s0 + chunks * (seg + 1) / a.segs * kCH);   // this segment's tokens
    const int64_t cells = (int64_t)a.B * a.H;
    const int c0 = slab * 16 * NW, col = c0 + wv * 16 + ln;
    const bool live = col < a.Dv;
    const int64_t srow = (int64_t)a.slots[b] * a.H + hd;
    float* const Sp = a.S + srow * D * a.Dv + col;
    const bool fresh = a.pos0[b] == 0;
    // S[2 kk + h], element r of lane group g: row 32 kk + 8 g + 4 h + r (what the read-out's product takes from that lane)
    f32x4 S[2 * KK];
    auto row_of = [&](int i, int r) { return (i >> 1) * 32 + 8 * g + 4 * (i & 1) + r; };
    // element r of S[i] of a state at `at` (this lane's column of its first row)
    auto take = [&](const float* at, int i, int r) { return live ? at[(int64_t)row_of(i, r) * a.Dv] : 0.f; };
    // the normaliser n likewise, the 32-row steps dealt to the waves (every column of the accumulator the same)
    constexpr int NO = MLSTM ? (KK + NW - 1) / NW : 1;
    f32x4 nst[2 * NO];
    auto n_row = [&](int i, int r) {
        const int kk = wv + NW * (i >> 1);
        return kk < KK ? kk * 32 + 8 * g + 4 * (i & 1) + r : -1;
    };
    float* const seg0 = a.segs > 1 ? a.seg_s + (int64_t)group * D * a.Dv + col : nullptr;   // the state before the step, kept by the first pass
    const bool first = seg == 0, from0 = fresh || (STATE && !first);
    {
        const float* const at = STATE || a.segs == 1 ? Sp : first ? seg0 : seg0 + cells * D * a.Dv;
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[i][r] = from0 && (STATE || first) ? 0.f : take(at, i, r);
        if (STATE && first && !fresh && live) {
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) seg0[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
        }
        if constexpr (MLSTM) {
            const float* const nat = STATE || first ? a.n0 + (int64_t)group * D : a.seg_n + (int64_t)group * D;
#pragma unroll
            for (int i = 0; i < 2 * NO; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) nst[i][r] = (STATE && !first) || n_row(i, r) < 0 ? 0.f : nat[n_row(i, r)];
        }
    }
    if constexpr (!STATE && !DELTA) {
        for (int j = 1; j < seg; ++j) {   // over the segments between: S <- (product of decays) S + what they write
            const float d = a.seg_d[cells * j + group];
            const float* const at = seg0 + cells * (j + 1) * D * a.Dv;
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[i][r] = d * S[i][r] + take(at, i, r);
            if constexpr (MLSTM) {
#pragma unroll
                for (int i = 0; i < 2 * NO; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (n_row(i, r) >= 0) nst[i][r] = d * nst[i][r] + a.seg_n[(cells * j + group) * D + n_row(i, r)];
            }
        }
    }
    double Lseg = 0.0;   // STATE: the sum of the segment's log decays, and the sign of their product
    float gseg = 1.f;
    float odd = 0.f;     // NaN once something was not finite
    const uint16_t* const qp = a.proj + a.q_off + (int64_t)hk * D;
    const uint16_t* const kp = a.proj + a.k_off + (int64_t)hk * D;
    const uint16_t* const vp = a.proj + a.v_off + (int64_t)hd * a.Dv + c0;
    const int vn = min(VC, (a.Dv - c0) / 8);
    const uint32_t lds0 = lds_offset(cs_smem);
    // A chunk's rows into buffer `buf`: pieces wv, wv + NW, .. of each operand, 64 / CPR rows each.  Rows past the last token
    // repeat it (their weights are 0), columns past Dv the last ones (not stored).
    auto fetch = [&](int tb, int buf) {
        const int last = t1 - 1 - tb;
        const uint32_t dst = lds0 + buf * M::BUF;
        const uint16_t *const q = qp + (int64_t)tb * a.ldp, *const k = kp + (int64_t)tb * a.ldp, *const v = vp + (int64_t)tb * a.ldp;
#pragma unroll
        for (int u = 0; u < (CPR + NW - 1) / NW; ++u) {
            const int j = wv + NW * u, i = j * 64 + lane, row = i / CPR, c = (i % CPR) ^ spread<CPR>(row);
            if (CPR % NW == 0 || j < CPR) {
                const int64_t at = (int64_t)min(row, last) * a.ldp + c * 8;
                if (!STATE) dma_1k(q + at, __builtin_amdgcn_readfirstlane(dst + j * 1024));
                dma_1k(k + at, __builtin_amdgcn_readfirstlane(dst + M::Q + j * 1024));
            }
        }
#pragma unroll
        for (int u = 0; u < VC / NW; ++u) {
            const int j = wv + NW * u, i = j * 64 + lane, row = i / VC, c = (i % VC) ^ spread<VC>(row);
            dma_1k(v + (int64_t)min(row, last) * a.ldp + min(c, vn - 1) * 8, __builtin_amdgcn_readfirstlane(dst + 2 * M::Q + j * 1024));
        }
        if constexpr (PRE) {
            const unsigned char* const from = a.tiles + ((int64_t)((s0 >> 6) + b + (tb - s0) / kCH) * a.H + hd) * kDeltaTiles + lane * 16;
#pragma unroll
            for (int u = 0; u < kDeltaTiles / 1024 / NW; ++u)
                dma_1k(from + (wv + NW * u) * 1024, __builtin_amdgcn_readfirstlane(dst + 2 * M::Q + M::V + (wv + NW * u) * 1024));
        }
    };
    // the scalars of token tb + lane, as loaded; past the range: nothing decays, nothing is written
    float sd = 1.f, sw = 0.f, sr = 0.f, sb = 0.f;
    const float fixed = !MLSTM && a.dts == 0 ? a.decay[hd] : 1.f;
    auto scalars = [&](int tb) {
        const int64_t t = min(tb + lane, t1 - 1);
        if constexpr (MLSTM) {
            sd = a.la[t * a.H + hd];
            sw = a.lb[t * a.H + hd];
            sr = a.em[t * a.H + hd];
        } else {
            sd = a.dts != 0 ? a.decay[t * a.dts + hd] : fixed;
            sw = a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f;
            if (!DELTA && a.vscale != nullptr) sw *= a.vscale[t * a.H + hd];
            sr = a.qscale != nullptr ? a.qscale[t * a.HK + hk] : a.q_mul;
            if constexpr (DELTA) sb = a.beta[t * a.H + hd];
        }
    };
    // stores of the read-out: past the chunk's last token and past Dv the descriptor's range drops them
    const uint32_t orow = (uint32_t)a.H * a.Dv * 4, ocol = live ? (uint32_t)col * 4 : 0x80000000u;
    if (t0 < te) {
        fetch(t0, 0);
        if constexpr (!PRE) scalars(t0);
    }
    for (int tb = t0, buf = 0; tb < te; tb += kCH, buf ^= 1) {
        const int nt = min(kCH, te - tb);
        // (PRE: the chunk before, a whole one, issued 16 stores after this one's pieces; they need not be done)
        if (PRE && tb != t0) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else dma_wait();
        // ---- the chunk's scalars (before the next chunk's DMA is issued: what waits for them would wait for that, too)
        const bool valid = lane < nt;
        double LC = 0.0;
        float w, rd = sr, gC = 1.f, eL = 0.f;
        if constexpr (!PRE) {
        const double L = chunk_logs<MLSTM>(valid, sd, sw, lane, w, rd, gC, LC);
        if constexpr (STATE) {
            Lseg += LC;
            gseg *= gC;
        }
        eL = exp_d(L);
        Ls[lane] = L;
        ws[lane] = w;
        cs[lane] = gC * exp_d(LC - L) * w;
        if constexpr (DELTA) {
            const float bt = valid ? sb : 0.f;
            bs[lane] = bt;
            bk[lane] = bt * w;
            be[lane] = bt * w * eL;
        }
        }
        __syncthreads();   // this chunk's rows are in LDS; nobody reads the other buffer or the last chunk's weights any more
        if (tb + kCH < te) {
            fetch(tb + kCH, buf ^ 1);
            if constexpr (!PRE) scalars(tb + kCH);
        }
        const unsigned char* const qb = cs_smem + buf * M::BUF;
        const unsigned char* const kb = qb + M::Q;
        const unsigned char* const vb = kb + M::Q;
        const unsigned char* const pre = vb + M::V;   // PRE
        const float* const psc = reinterpret_cast<const float*>(pre + kDtSc);
        auto row8 = [&](const unsigned char* base, int i, int kk) { return chunk_row8<D>(base, i, kk, ln, g); };
        // k rows 32 p + 4 g + (0..3), 32 p + 16 + 4 g + (0..3), column 32 kk + 8 (ln / 4) + 4 h + ln % 4: the update's left operand
        const int r4 = 4 * g + (ln >> 2), sp4 = spread<CPR>(r4);
        auto kcol8 = [&](int p, int kk, int h) {
            const unsigned char* at = kb + (32 * p + r4) * (D * 2) + ((kk * 4 + (ln & 3)) ^ sp4) * 16 + h * 8;
            return join8(lds_read_tr4(at), lds_read_tr4(at + 16 * (D * 2)));
        };
        const int nrow = (nt + 15) / 16;   // 16-token rows of tiles that hold tokens
        for (int p = STATE || PRE ? 10 : wv; p < 10; p += NW) {
            const int i = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, j = p - i * (i + 1) / 2;
            if (i >= nrow) continue;
            const f32x4 v = chunk_weights<D>(kb, qb, i, j, Ls, ws, ln, g);
            pt[p * 64 + lane] = v;
            if constexpr (MLSTM) {
                float sum = (v[0] + v[1]) + (v[2] + v[3]);
                sum = rows_sum(sum);
                if (g == 0) psum[p * 16 + ln] = sum;
            }
        }
        if constexpr (DELTA && !PRE) {   // wave w the tiles of column w of -A, and the diagonal one's inverse
            for (int i = wv; i < nrow; ++i) {
                const int p = i * (i + 1) / 2 + wv;
                at[p * 64 + lane] = chunk_minus_a<D>(kb, i, wv, Ls, ws, bk, ln, g);
                if (i == wv) chunk_inverse(at + p * 64, reinterpret_cast<float*>(tt + wv * 64), ln, g);
            }
        }
        if constexpr (MLSTM && !STATE) {   // n . q of the state before the chunk, this wave's rows
            f32x4 acc[4] = {};
#pragma unroll
            for (int u = 0; u < NO; ++u) {
                const int kk = wv + NW * u;
                if (kk < KK) {
                    const float x[8] = {nst[2 * u][0], nst[2 * u][1], nst[2 * u][2], nst[2 * u][3],
                                        nst[2 * u + 1][0], nst[2 * u + 1][1], nst[2 * u + 1][2], nst[2 * u + 1][3]};
                    const Terms n = split3(x);
                    bf16x8 q[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) q[i] = row8(qb, i, kk);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = mfma_16x16x32(q[i], n.l, acc[i]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = mfma_16x16x32(q[i], n.m, acc[i]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) acc[i] = mfma_16x16x32(q[i], n.h, acc[i]);
                }
            }
            if (ln == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(nq + wv * kCH + 16 * i + 4 * g) = acc[i];
            }
        }
        if constexpr (!STATE && !PRE) __syncthreads();   // the weights are there
        float fr = rd;
        if constexpr (MLSTM && !STATE) {
            const int i = lane >> 4, p0 = i * (i + 1) / 2;
            float intra = 0.f, inter = 0.f;
            for (int j = 0; j <= i; ++j) intra += psum[(p0 + j) * 16 + ln];
#pragma unroll
            for (int u = 0; u < NW; ++u) inter += nq[u * kCH + lane];
            odd = __builtin_fmaf(inter, 0.f, odd);
            fr = a.q_mul / (fmaxf(fabsf((intra + eL * inter) * a.q_mul), rd) + 1e-6f);
        }
        const float eC = PRE ? psc[5 * kCH] : gC * exp_d(LC);
        // ---- read-out and the state after the chunk, NI rows of tiles
        auto rest = [&](auto ni) {
            constexpr int NI = decltype(ni)::value;
            bf16x8 v[NI / 2];   // v rows 32 p + 4 g + (0..3), 32 p + 16 + 4 g + (0..3) of this lane's column
#pragma unroll
            for (int p = 0; p < NI / 2; ++p) {
                const unsigned char* at = vb + (32 * p + r4) * (VC * 16) + ((wv * 2 + ((ln & 3) >> 1)) ^ spread<VC>(r4)) * 16 + (ln & 1) * 8;
                v[p] = join8(lds_read_tr4(at), lds_read_tr4(at + 16 * (VC * 16)));
            }
            f32x4 U[NI];   // delta: what the chunk's tokens write, before the scales
            if constexpr (!STATE) {
            // the state before the chunk times q (delta: and k), a 32-row step of it at a time
            f32x4 oq[NI], ok[NI];
#pragma unroll
            for (int i = 0; i < NI; ++i) oq[i] = ok[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                bf16x8 q[NI], k[NI];
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    q[i] = row8(qb, i, kk);
                    if constexpr (DELTA) k[i] = row8(kb, i, kk);
                }
                const float x[8] = {S[2 * kk][0], S[2 * kk][1], S[2 * kk][2], S[2 * kk][3],
                                    S[2 * kk + 1][0], S[2 * kk + 1][1], S[2 * kk + 1][2], S[2 * kk + 1][3]};
                const Terms st = split3(x);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    const bf16x8 term = c == 0 ? st.l : c == 1 ? st.m : st.h;
#pragma unroll
                    for (int i = 0; i < NI; ++i) {
                        oq[i] = mfma_16x16x32(q[i], term, oq[i]);
                        if constexpr (DELTA) ok[i] = mfma_16x16x32(k[i], term, ok[i]);
                    }
                }
            }
            float el[NI][4], fo[NI][4];
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    el[i][r] = PRE ? psc[3 * kCH + 16 * i + 4 * g + r] : __shfl(eL, 16 * i + 4 * g + r, 64);
                    fo[i][r] = PRE ? psc[4 * kCH + 16 * i + 4 * g + r] : __shfl(fr, 16 * i + 4 * g + r, 64);
                    oq[i][r] *= el[i][r];
                }
            if constexpr (DELTA) {
                const float *const bsp = PRE ? psc : bs, *const bep = PRE ? psc + kCH : be;
                auto tile_a = [&](int i, int j) {
                    if constexpr (PRE) return load_terms(pre + kDtA + (i * (i - 1) / 2 + j) * kDtTile, lane);
                    else return split3(at[(i * (i + 1) / 2 + j) * 64 + lane]);
                };
                auto tile_t = [&](int i) {
                    if constexpr (PRE) return load_terms(pre + kDtT + i * kDtTile, lane);
                    else return split3(tt[i * 64 + lane]);
                };
                auto tile_p = [&](int i, int j) {
                    if constexpr (PRE) return load_terms(pre + (i * (i + 1) / 2 + j) * kDtTile, lane);
                    else return split3(pt[(i * (i + 1) / 2 + j) * 64 + lane]);
                };
                // (I + A) U = beta (v - e^L k-scale S^T k), 16 rows at a time
                Terms4 ut[NI];
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    const f32x4 b0 = *reinterpret_cast<const f32x4*>(bsp + 16 * i + 4 * g), b1 = *reinterpret_cast<const f32x4*>(bep + 16 * i + 4 * g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float p = b1[r] * ok[i][r];
                        U[i][r] = b0[r] * (float)v[i / 2][4 * (i & 1) + r] - p;
                        ok[i][r] = -__builtin_fmaf(b1[r], ok[i][r], -p);   // what rounding p and the sum below took, for the last sum
                    }
                }
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    if (i > 0 && i >= nrow) {   // (rows without tokens: nothing)
                        ut[i] = split3(U[i]);
                        continue;
                    }
                    // the small products first, and all of them before they meet the sum: one rounding at its size
                    if (i > 0) {
                        Terms4 w[NI];
                        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int j = 0; j < i; ++j) acc = mul_low(w[j] = tile_a(i, j), ut[j], acc);
#pragma unroll
                        for (int j = 0; j < i; ++j) acc = mul_high(w[j], ut[j], acc);
                        const f32x4 sum = U[i] + acc, part = sum - U[i];
                        ok[i] += (U[i] - (sum - part)) + (acc - part);
                        U[i] = sum;
                    }
                    const Terms4 w = tile_t(i), u = split3(U[i]);
                    U[i] += mul_high(w, u, mul_low(w, u, ok[i]));
                    ut[i] = split3(U[i]);
                }
#pragma unroll
                for (int i = 0; i < NI; ++i) {
                    if (i > 0 && i >= nrow) continue;
                    Terms4 w[NI];
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int j = 0; j <= i; ++j) acc = mul_low(w[j] = tile_p(i, j), ut[j], acc);
#pragma unroll
                    for (int j = 0; j <= i; ++j) acc = mul_high(w[j], ut[j], acc);
                    oq[i] += acc;
                }
            } else {
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int p = 0; p <= i / 2; ++p) {
                        const f32x4 x0 = pt[(i * (i + 1) / 2 + 2 * p) * 64 + lane];
                        f32x4 x1 = {0.f, 0.f, 0.f, 0.f};
                        if (2 * p + 1 <= i) x1 = pt[(i * (i + 1) / 2 + 2 * p + 1) * 64 + lane];
                        const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                        const Terms w3 = split3(x);
                        oq[i] = mfma_16x16x32(w3.h, v[p], mfma_16x16x32(w3.m, v[p], mfma_16x16x32(w3.l, v[p], oq[i])));
                    }
            }
#pragma unroll
            for (int i = 0; i < NI; ++i) {   // (rows without tokens hold what was in LDS)
                const float met = not_finite(oq[i], odd);
                odd = i == 0 || i < nrow ? met : odd;
            }
            const auto ord = __builtin_amdgcn_make_buffer_rsrc(a.o + ((int64_t)tb * a.H + hd) * a.Dv, (short)0, (int)(nt * orow), 0x00020000);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(oq[i][r] * fo[i][r]), ord, ocol + (16 * i + 4 * g + r) * orow, 0, 0);
            }
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) S[i] *= eC;
            if constexpr (MLSTM) {
#pragma unroll
                for (int i = 0; i < 2 * NO; ++i) nst[i] *= eC;
            }
#pragma unroll
            for (int p = 0; p < NI / 2; ++p) {
                const float* const csp = PRE ? psc + 2 * kCH : cs;
                const f32x4 f0 = *reinterpret_cast<const f32x4*>(csp + 32 * p + 4 * g);
                const f32x4 f1 = *reinterpret_cast<const f32x4*>(csp + 32 * p + 16 + 4 * g);
                const float f[8] = {f0[0], f0[1], f0[2], f0[3], f1[0], f1[1], f1[2], f1[3]};
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = f[e] * (DELTA ? U[2 * p + (e >> 2)][e & 3] : (float)v[p][e]);
                const Terms u = split3(x);
                Terms un;
                if constexpr (MLSTM) un = split3(f);
#pragma unroll
                for (int k2 = 0; k2 < KK; k2 += 2) {   // four tiles of the state at a time
                    constexpr int NT = KK > 1 ? 4 : 2;
                    bf16x8 kc[NT];
#pragma unroll
                    for (int y = 0; y < NT; ++y) kc[y] = kcol8(p, k2 + (y >> 1), y & 1);
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        const bf16x8 term = c == 0 ? u.l : c == 1 ? u.m : u.h;
#pragma unroll
                        for (int y = 0; y < NT; ++y) S[2 * k2 + y] = mfma_16x16x32(kc[y], term, S[2 * k2 + y]);
                    }
                    if constexpr (MLSTM) {
#pragma unroll
                        for (int y = 0; y < NT; ++y) {
                            const int kk = k2 + (y >> 1);
                            if (kk % NW == wv) {
                                f32x4& nn = nst[2 * (kk / NW) + (y & 1)];
                                nn = mfma_16x16x32(kc[y], un.h, mfma_16x16x32(kc[y], un.m, mfma_16x16x32(kc[y], un.l, nn)));
                            }
                        }
                    }
                }
            }
        };
        if (nt > 32) rest(std::integral_constant<int, 4>{});
        else rest(std::integral_constant<int, 2>{});
    }
    bool again = false;
    float nl[(D + 63) / 64] = {};   // mlstm: rows lane, lane + 64 .. of the normaliser
    if constexpr (!STATE) {         // (a segment's state that is not finite shows in the next one's)
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i) odd = not_finite(S[i], odd);
        again = __builtin_amdgcn_ballot_w64(odd != odd) != 0;   // (wave-uniform)
    }
    if (again) {   // from the sequence's first token
        dma_wait();   // what the chunks stored is there before the same places are written
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[i][r] = fresh ? 0.f : take(a.segs == 1 ? Sp : seg0, i, r);
        if constexpr (MLSTM) {
#pragma unroll
            for (int j = 0; j < (D + 63) / 64; ++j) nl[j] = a.n0[(int64_t)group * D + min(lane + 64 * j, D - 1)];
        }
        auto over_rows = [](float x) {   // lanes of the same column hold a quarter of the rows each
            return rows_sum(x);
        };
        for (int64_t t = s0; t < te; ++t) {
            float d, w, rr = a.q_mul;
            if constexpr (MLSTM) {
                d = expf(a.la[t * a.H + hd]);
                w = expf(a.lb[t * a.H + hd]);
            } else {
                d = a.dts != 0 ? a.decay[t * a.dts + hd] : fixed;
                w = a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f;
                if (!DELTA && a.vscale != nullptr) w *= a.vscale[t * a.H + hd];
                if (a.qscale != nullptr) rr = a.qscale[t * a.HK + hk];
            }
            const uint16_t *const q = qp + t * a.ldp, *const k = kp + t * a.ldp;
            if constexpr (MLSTM) {
                float x = 0.f;
#pragma unroll
                for (int j = 0; j < (D + 63) / 64; ++j)
                    if (lane + 64 * j < D) {
                        nl[j] = d * nl[j] + bf2f(k[lane + 64 * j]) * w;
                        x += nl[j] * bf2f(q[lane + 64 * j]);
                    }
                rr = a.q_mul / (fmaxf(fabsf(wave_sum(x) * a.q_mul), a.em[t * a.H + hd]) + 1e-6f);
            }
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) S[i] *= d;
            float u = live ? bf2f(vp[t * a.ldp + wv * 16 + ln]) : 0.f;
            if constexpr (DELTA) {
                float x = 0.f;
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    float kf[8];
                    ld8(k + 32 * kk + 8 * g, kf);
#pragma unroll
                    for (int e = 0; e < 8; ++e) x += S[2 * kk + (e >> 2)][e & 3] * kf[e];
                }
                u = (u - over_rows(x) * w) * a.beta[t * a.H + hd];
            }
            u *= w;
            float y = 0.f;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                float kf[8], qf[8];
                ld8(k + 32 * kk + 8 * g, kf);
                ld8(q + 32 * kk + 8 * g, qf);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    f32x4& s = S[2 * kk + (e >> 2)];
                    s[e & 3] += kf[e] * u;
                    y += s[e & 3] * qf[e];
                }
            }
            y = over_rows(y) * rr;
            if (t >= t0 && g == 0 && live) a.o[(t * a.H + hd) * a.Dv + col] = y;
        }
    }
    if (!STATE && seg != a.segs - 1) return;
    float* const dst = STATE ? seg0 + cells * (seg + 1) * D * a.Dv : Sp;
    if (live) {
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) dst[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
    }
    if (slab != 0) return;
    if constexpr (MLSTM) {
        float* const nd = STATE ? a.seg_n + (cells * seg + group) * D : a.n + srow * D;
        if (again) {
#pragma unroll
            for (int j = 0; j < (D + 63) / 64; ++j) {
                const int row = lane + 64 * j;
                if (row < D && (row / 32) % NW == wv) nd[row] = nl[j];
            }
        } else if (ln == 0) {
#pragma unroll
            for (int i = 0; i < 2 * NO; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (n_row(i, r) >= 0) nd[n_row(i, r)] = nst[i][r];
        }
    }
    if (STATE && threadIdx.x == 0) a.seg_d[cells * seg + group] = gseg * exp_d(Lseg);
}

// The scalar recurrences of mlstm.hip for a whole prompt portion: m_t = max(f_t + m_(t-1), i_t) is a prefix of the pairs
// (f, i) under (f1, i1)(f2, i2) = (f1 + f2, max(i1 + f2, i2)), taken 256 tokens at a time in float64.  One workgroup per
// (sequence, head) leaves log a, log b and e^-m per token, m in its slot and n as it was before the step in n0.
__global__ void __launch_bounds__(256) mlstm_gates_kernel(const float* __restrict__ gate_pre, const int32_t* __restrict__ q_start,
                                                          const int32_t* __restrict__ pos0, const int32_t* __restrict__ slots,
                                                          const float* __restrict__ n_state, float* __restrict__ m_state,
                                                          float* __restrict__ n0, float* __restrict__ la, float* __restrict__ lb,
                                                          float* __restrict__ em, int H, int D, float cap) {
    __shared__ double wF[4], wM[4];
    __shared__ float ms[257];
    const int b = blockIdx.x, hd = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int t0 = q_start[b], t1 = q_start[b + 1];
    if (t1 <= t0) return;
    const int64_t row = (int64_t)slots[b] * H + hd;
    const bool fresh = pos0[b] == 0;
    for (int d = tid; d < D; d += 256) n0[((int64_t)b * H + hd) * D + d] = fresh ? 0.f : n_state[row * D + d];
    float m = fresh ? 0.f : m_state[row];
    for (int tb = t0; tb < t1; tb += 256) {
        const int nt = min(256, t1 - tb);
        const int64_t t = tb + min(tid, nt - 1);
        const float ig = cap * tanhf(gate_pre[t * 2 * H + hd] / cap);
        const float fg = logsigmoidf_(cap * tanhf(gate_pre[t * 2 * H + H + hd] / cap));
        double F = fg, M = ig;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double pF = __shfl_up(F, o, 64), pM = __shfl_up(M, o, 64);
            if (lane >= o) {
                M = fmax(pM + F, M);
                F += pF;
            }
        }
        if (lane == 63) {
            wF[wv] = F;
            wM[wv] = M;
        }
        __syncthreads();
        double in = m;   // the running maximum in front of this wave
        for (int u = 0; u < wv; ++u) in = fmax(in + wF[u], wM[u]);
        const float mt = (float)fmax(in + F, M);
        ms[tid + 1] = mt;
        if (tid == 0) ms[0] = m;
        __syncthreads();
        if (tid < nt) {
            const double prev = ms[tid];
            la[t * H + hd] = (float)(fg + prev - mt);
            lb[t * H + hd] = (float)((double)ig - mt);
            em[t * H + hd] = expf(-mt);
        }
        m = ms[nt];
        __syncthreads();
    }
    if (tid == 0) m_state[row] = m;
}

}  // namespace hy

int hy_chunk_segments(int B, int H, int D, int Dv, int longest, int least);

// Whether a launch takes less time in chunks than token by token.  A chunk costs the same whether it is full or not: a range of one token
// costs a workgroup 6 to 10 us per slab, token by token little more than its state's bytes, so that a short prompt beside many decode
// rows is faster there: retention, 8 heads of 128 x 128, us in chunks / token by token: 16 tokens beside 256 decode rows 118 / 50, 117 beside
// 256 115 / 95, 117 beside 64 35 / 64, 2048 beside 256 176 / 957; delta rule, 32 heads: 40 beside 64 142 / 65, 117 beside 256 550 / 296, 2048
// beside 256 622 / 1214.  Alone, 32 sequences of n tokens: 15.5 / 10.7 at n = 4, 15.4 / 17.1 at 16, 33 / 71 at 117.  The times are
// modelled: the chain of the longest range (in segments side by side, which walk it 1.6 times) or the chunks of all over 256 CUs, the chain
// of tokens or all tokens, and the states' megabytes; fitted per form on 2639 launches of 14 shapes (rms 0.13 .. 0.15 of a time;
// profiles/recurrence_forms.json).  Chunked where that is 0.8 of the other at most: 2 of the 2639 are then slower than token by token by more
// than 3% (by 6), always chunked 445 (by up to 140); 2% on average off the better of the two.
bool hy_chunk_scan_pays(int mode, int T, int B, int H, int D, int Dv, int longest) {
    struct Cost {
        double c0, chain, work, t0, step, steps, mb;
    };
    constexpr Cost costs[3] = {{4.7, 5.7, 6.5, 2.8, 0.465, 0.277, 0.175}, {10.3, 7.1, 7.7, 9.1, 1.0, 0.54, 0.295}, {6.5, 11.4, 9.8, 4.3, 0.475, 0.52, 0.18}};
    const Cost& c = costs[mode];
    const int segs = mode == hy::kScanDelta ? 1 : hy_chunk_segments(B, H, D, Dv, longest, 256), most = (longest + 63) / 64;
    const double slabs = (double)H * ((Dv + 63) / 64), size = std::sqrt(D / 128.0);
    const double chunks = most + std::max(B - 1.0, (T - longest) / 64.0 + (B - 1) / 2.0);
    const double chunked = c.c0 + std::max(c.chain * most / segs * (segs > 1 ? 1.6 : 1.0), c.work * slabs * chunks / 256) * size;
    const double token = c.t0 + std::max(c.step * longest * size, c.steps * T * slabs * D / 128 / 256) + c.mb * B * H * D * Dv * 8e-6;
    return chunked <= 0.8 * token;
}

// When the chunked form serves a launch: bfloat16 rows of q, k and v on 16-byte boundaries, a state of 32, 64, 128 or 256
// rows, a sequence with at least 16 new tokens, with the delta rule 32 (longest: the most that any sequence brings), and a launch that
// gains (above).  The delta rule's tiles leave no room for D = 256.
bool hy_chunk_scan_ok(const void* proj, int ldp, int q_off, int k_off, int v_off, int T, int B, int H, int D, int Dv, int longest, int mode) {
    const bool delta = mode == hy::kScanDelta;
    return longest >= (delta ? 32 : 16) && (D == 32 || D == 64 || D == 128 || (D == 256 && !delta)) && Dv % 8 == 0 && ((uintptr_t)proj & 15) == 0 &&
           ((ldp | q_off | k_off | v_off) & 7) == 0 && ldp < 1 << 23 &&   // (64 rows of o, no wider than proj's, within 2^31 bytes)
           hy_chunk_scan_pays(mode, T, B, H, D, Dv, longest);
}

template <int D, int MODE, bool STATE, bool PRE = false>
static void chunk_scan_pass(const hy::ChunkScan& a, int segs, hipStream_t s) {
    constexpr int lds = hy::ChunkLds<D, MODE, PRE>::SIZE;
    static_assert(lds <= 160 * 1024, "LDS of one workgroup");
    constexpr auto kern = hy::chunk_scan_kernel<D, MODE, STATE, PRE>;
    lds_limit<kern>(lds);
    const int nslab = (a.Dv + 16 * hy::kCW - 1) / (16 * hy::kCW);
    kern<<<dim3((a.B * a.H + 7) / 8 * 8 * nslab, segs), 64 * hy::kCW, lds, s>>>(a);
}
template <int D, int MODE>
static void chunk_scan_run(const hy::ChunkScan& a, hipStream_t s) {
    if constexpr (MODE != hy::kScanDelta) {
        if (a.segs > 1) chunk_scan_pass<D, MODE, true>(a, a.segs - 1, s);
    } else if (a.tiles != nullptr) {
        constexpr int lds = 4 * hy::kCH * D + 8192 + 4 * 1024;
        constexpr auto kern = hy::delta_tiles_kernel<D>;
        lds_limit<kern>(lds);
        kern<<<(unsigned)(hy::delta_slots(a.T, a.B) * a.H), 256, lds, s>>>(a);
        return chunk_scan_pass<D, MODE, false, true>(a, a.segs, s);
    }
    chunk_scan_pass<D, MODE, false>(a, a.segs, s);
}

// Bytes of scratch for the delta rule's tiles, or 0: made between the steps, as where no sequence has two chunks, and of launches whose tiles would take more
// than `most` (512 MB: a prompt portion of 32768 tokens and 16 heads takes 270).
int64_t hy_delta_tiles_bytes(const void* proj, int ldp, int q_off, int k_off, int v_off, int T, int B, int H, int D, int Dv, int longest, int64_t most) {
    const int64_t n = hy::delta_slots(T, B) * H * hy::kDeltaTiles;
    return longest > hy::kCH && n <= most && hy_chunk_scan_ok(proj, ldp, q_off, k_off, v_off, T, B, H, D, Dv, longest, hy::kScanDelta) ? n : 0;
}

// Segments that a sequence's chunks are dealt to, here and in gla_scan.hip: launches that leave half of the CUs or more without a
// workgroup carry the states over segments first (half a chunk's work) and take all of them side by side then: of at least `least`
// tokens in the longest sequence, counted up to a chunk (449 tokens: two of 224 for 256), of less or none in the others.  Not with the
// delta rule, whose step from state to state is a matrix.  256 tokens here (four chunks), 128 in gla_scan.hip (eight,
// slower ones).  Measured, one pass -> segments (profiles/prompt_form_rules.json, 82 launches, one of them slower, by 1 %): retention, 8 heads of
// 128 x 128, 4 sequences of 512 tokens (two segments) 48 -> 39 us, one of 512 (two) 47 -> 36, 4096 (16) 346 -> 57; mlstm, 4 heads of
// 256 x 512, one of 512 (two) 81 -> 67, 4096 (eight) 579 -> 157, of 32768 4701 -> 1009; state-space form, 128 heads of 128 x 64, one of
// 512 (two) 50 -> 43.  At most four segments: 118 and 232 us for the two of 4096.  One decay per row, heads of 128 x 256: 16 heads, 2
// sequences of 256 tokens (two segments) 52 both, one of 2048 (four) 371 -> 174; 4 heads, 4 of 256 (two) 51 -> 50, of 512 (four) 96 -> 55,
// one of 512 (four) 96 -> 51, of 2048 (16) 369 -> 79.
int hy_chunk_segments(int B, int H, int D, int Dv, int longest, int least) {
    if (D != 32 && D != 64 && D != 128 && D != 256) return 1;
    const int64_t wgs = (int64_t)B * H * ((Dv + 63) / 64);
    const int64_t segs = std::min<int64_t>({wgs > 0 ? 256 / wgs : 1, (longest + 63) / least, 16});
    return segs > 1 ? (int)segs : 1;
}
// floats of scratch: the states before the step and of all segments but the last; normalisers and products of decays of those
int64_t hy_chunk_segment_floats(int B, int H, int D, int Dv, int segs) {
    return segs > 1 ? (int64_t)B * H * ((int64_t)segs * D * Dv + (segs - 1) * (int64_t)(D + 1)) : 0;
}
static void chunk_scan_scratch(hy::ChunkScan& a, int D, int segs, float* seg) {
    a.segs = segs;
    const int64_t cells = (int64_t)a.B * a.H;
    a.seg_s = seg;
    a.seg_n = seg + cells * segs * D * a.Dv;
    a.seg_d = a.seg_n + cells * (segs - 1) * D;
}

template <int MODE>
static void chunk_scan_d(int D, const hy::ChunkScan& a, hipStream_t s) {
    if (D == 32) chunk_scan_run<32, MODE>(a, s);
    else if (D == 64) chunk_scan_run<64, MODE>(a, s);
    else if (D == 128) chunk_scan_run<128, MODE>(a, s);
    else if constexpr (MODE != hy::kScanDelta) chunk_scan_run<256, MODE>(a, s);   // (delta: its tiles do not fit the LDS beside)
}

// One decay per head and token (dts = H) or per head (dts = 0), with beta the delta correction (D <= 128); see
// launch_hy_linear_scan.  seg: hy_chunk_segment_floats, with beta hy_delta_tiles_bytes or nullptr.
void launch_hy_chunk_scan(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, const float* qscale, const float* kscale,
                          float q_mul, const float* decay, int dts, const float* beta, const int32_t* q_start,
                          const int32_t* pos0, const int32_t* slots, float* S, float* o, int T, int B, int HK, int H, int D, int Dv, const float* vscale,
                          int segs, float* seg, hipStream_t s) {
    hy::ChunkScan a{proj, ldp, q_off, k_off, v_off, qscale, kscale, vscale, decay, beta, dts, q_mul, nullptr, nullptr, nullptr,
                    q_start, pos0, slots, nullptr, S, nullptr, o, B, HK, H, Dv, T, 1, nullptr, nullptr, nullptr, beta != nullptr ? reinterpret_cast<unsigned char*>(seg) : nullptr};
    if (beta == nullptr && segs > 1) chunk_scan_scratch(a, D, segs, seg);
    if (beta != nullptr) chunk_scan_d<hy::kScanDelta>(D, a, s);
    else chunk_scan_d<hy::kScanPlain>(D, a, s);
}

// segs: hy_chunk_segments (1: none).  scratch: 3 T H + B H D + hy_chunk_segment_floats floats
void launch_hy_chunk_mlstm(const uint16_t* proj, int ldp, const float* gate_pre, const int32_t* q_start, const int32_t* pos0,
                           const int32_t* slots, float* S, float* n, float* m, float* scratch, float* o, int T, int B, int H,
                           int D, int Dv, float cap, int segs, hipStream_t s) {
    const int64_t th = (int64_t)T * H;
    float *la = scratch, *lb = la + th, *em = lb + th, *n0 = em + th;
    hy::mlstm_gates_kernel<<<dim3(B, H), 256, 0, s>>>(gate_pre, q_start, pos0, slots, n, m, n0, la, lb, em, H, D, cap);
    hy::ChunkScan a{proj, ldp, 0, H * D, 2 * H * D, nullptr, nullptr, nullptr, nullptr, nullptr, H, 1.f / sqrtf((float)D), la, lb, em,
                    q_start, pos0, slots, n0, S, n, o, B, H, H, Dv, T, 1, nullptr, nullptr, nullptr, nullptr};
    if (segs > 1) chunk_scan_scratch(a, D, segs, n0 + (int64_t)B * H * D);
    chunk_scan_d<hy::kScanMlstm>(D, a, s);
}

}  // namespace chronos
