// gla_scan.hip — the recurrence of linear_scan.hip with one decay per state row and no delta correction (gated linear
// attention), bfloat16 rows, 16 tokens at a time on the matrix cores.  With d_t the decays of token t, F_t = d_1 .. d_t (products over the
// chunk's tokens, row by row), S the state before the chunk, w_s and r_t the factors on what token s writes and token t reads,
//
//     o_t = r_t ( (F_t q_t)^T S + sum_(s <= t) P[t, s] v_s ),   P[t, s] = (F_t q_t) . (w_s k_s / F_s)
//     S  <- F_16 (S + sum_s (w_s k_s / F_s) v_s^T)
//
// A chunk in which some |F_t| leaves [2^-40, 2^40] (a decay of 0, say) is taken token by token instead, by the same waves; so is one with
// infinities, NaN or numbers beyond 2^25 among k, w and v, or whose read-out is not finite: a weight of 0 above the diagonal times a
// later token's infinite value would reach back, and an infinity has no terms.
// Precision: as chunk_scan.hip, all but q, k, v is float32; a float32 operand of a matrix product enters as three bfloat16 terms
// whose sum it is, two of them as the six leading of the nine products of terms.
//
// A workgroup is 4 waves and serves 64 value columns of one (sequence, head); a wave keeps all D rows of its 16 columns of S in
// accumulators.  A chunk's rows come by DMA into one of two LDS buffers while the chunk before is computed.  Half of the threads form
// F q, half w k / F (two rows of 8 tokens each), shared through LDS as terms, and each wave reads out and updates its columns.
//
// What bounds it: the chain of a sequence's chunks, one wave per SIMD: about 600 vector and 66 matrix instructions a chunk and wave at
// D = 128, two barriers and the LDS reads between them, 2.8 us.  Measured, 4 sequences of 2048 tokens, 16 heads of 128 x 256: token by
// token 988 us, this 375; one of 4000, 8 heads: 1684 and 694, in eight segments 172.  P on the vector ALUs from running products: 648 us, and the same
// with F in float32: state 9.6e-8 of its norm off the float64 recurrence (token by token 8.7e-8, this 7.8e-8); with the stores of a
// chunk waited for by the next: 482 us, with that 448, and the terms rounded in pairs 403 (382 as measured for the 375).
#include "chronos_lds.h"
#include "chunk_common.h"

#include <type_traits>

namespace chronos {
namespace hy {

struct GlaScan {
    const uint16_t* proj;
    int ldp, q_off, k_off, v_off;
    const float *qscale, *kscale, *vscale, *decay;   // decay [T, H, D]; the others as in linear_scan.hip, may be nullptr
    float q_mul;
    const int32_t *q_start, *pos0, *slots;
    float *S, *o;
    int B, HK, H, Dv, T;
    // segments of a sequence side by side (1: none), as in chunk_scan.hip: the state before the step and, of each segment but the last,
    // what it writes, [segs, B, H, D, Dv]; products of its decays [segs - 1, B, H, D]
    int segs;
    float *seg_s, *seg_d;
    unsigned char* tiles;   // [gla_slots, H, GlaTile::SIZE] of gla_tiles_kernel, or nullptr
};

constexpr int kGC = 16;   // tokens per chunk
constexpr uint16_t kBig = 0x4c00;   // 2^25 as bfloat16: sums of products of three such and 2^40 stay finite

typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
// the larger magnitudes of two and of a pair of bfloat16, as bits
__device__ __forceinline__ u16x2 max_bits(u16x2 m, uint32_t pair) { return __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, pair & 0x7fff7fffu)); }

// Waits for the wave's DMA pieces when `STORES` of its stores (all that it issued after them) may still be under way: memory
// instructions of a wave complete in the order of issue, and a store takes as long as a chunk's arithmetic.
// Values loaded beside the pieces are received before the stores, too (received()), else the compiler waits for everything.
template <int STORES> __device__ __forceinline__ void dma_wait_before_stores() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(STORES) : "memory"); }
__device__ __forceinline__ void received(float& a) { asm volatile("" : "+v"(a)); }

// What a chunk needs of its q, k and decays alone, per chunk and head, written by gla_tiles_kernel (bytes): F q, w k / F, three terms each, as they lie
// in LDS | P over the rows of each of the walk's RW waves of a column, three terms, 512 bytes a term | F_16 | the factors w and r | F_16 in float64 | whether the chunk goes token by token
template <int D> struct GlaTile {
    static constexpr int RW = D >= 128 ? D / 64 : 1, Q = kGC * D * 2, P = 6 * Q, F = P + RW * 3 * 512, W = F + D * 4, X = W + 2 * kGC * 4, BAD = X + D * 8, SIZE = (BAD + 4 + 1023) / 1024 * 1024;
};
// Chunk c of sequence b, tokens from s0 on, is chunk s0 / 16 + b + c of the launch: no two alike, T / 16 + B + 1 of them at most.
__host__ __device__ constexpr int64_t gla_slots(int T, int B) { return (int64_t)T / kGC + B + 1; }

// Rows 2 rp, 2 rp + 1 of 8 of a chunk's tokens (half: the last 8): d their decays, d0 those of the first 8 tokens, q two rows of q or k each, w (k only) the
// factors on what is written.  F q or w k / F to put(token, x, y), F_16 to `last` (of q's threads with half).  Returns whether the chunk goes token by token.
// F in float64, so that F_t / F_s carries the rounding of its two ends and not of the steps between.
template <typename Put, typename Last>
__device__ __forceinline__ bool gla_rows(bool keys, int half, const float2 (&d)[8], const float2 (&d0)[8], const uint32_t (&q)[8], const float (&w)[8], Put&& put, Last&& last) {
    double X = 1.0, Y = 1.0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        X *= d0[e].x;
        Y *= d0[e].y;
    }
    if (!half) X = Y = 1.0;
    float x[8], y[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        X *= d[e].x;
        Y *= d[e].y;
        x[e] = (float)X;
        y[e] = (float)Y;
    }
    bool bad = false;
    if (keys) {
        float lo = 1.f, hi = 1.f;
        u16x2 big = {0, 0};   // (largest magnitudes as bits: a NaN is above all)
#pragma unroll
        for (int e = 0; e < 8; ++e) big = max_bits(big, q[e]);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            lo = fminf(lo, fminf(fabsf(x[e]), fabsf(y[e])));
            hi = fmaxf(hi, fmaxf(fabsf(x[e]), fabsf(y[e])));
        }
        // (fminf and fmaxf drop a NaN, X and Y keep it)
        bad = !(lo >= 0x1p-40f) || !(hi <= 0x1p40f) || X != X || Y != Y || big[0] >= kBig || big[1] >= kBig;
        auto inverse = [](float v) {   // to half a last place in the range that counts
            const float r = __builtin_amdgcn_rcpf(v);
            return __builtin_fmaf(__builtin_fmaf(-v, r, 1.f), r, r);
        };
#pragma unroll
        for (int e = 0; e < 8; ++e)
            put(8 * half + e, w[e] * __uint_as_float(q[e] << 16) * inverse(x[e]), w[e] * __uint_as_float(q[e] & 0xffff0000u) * inverse(y[e]));
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) put(8 * half + e, __uint_as_float(q[e] << 16) * x[e], __uint_as_float(q[e] & 0xffff0000u) * y[e]);
        if (half) last(X, Y);
    }
    return bad;
}
// Rows 2 rp, 2 rp + 1 of token t of F q or w k / F into the three terms at `base`
template <int D> __device__ __forceinline__ void gla_put(unsigned char* base, int t, int rp, float x, float y) {
    unsigned char* at = base + t * (D * 2) + (((rp >> 2) ^ spread<D / 8>(t)) * 16) + (rp & 3) * 4;
#pragma unroll
    for (int k = 0; k < 3; ++k) *reinterpret_cast<uint32_t*>(at + k * (kGC * D * 2)) = round_pair(x, y);
}
// P of the terms at `base`, rows s = 4 g + r and columns t = ln, 0 above the diagonal
struct GlaP {
    f32x4 small, big;
};
__device__ __forceinline__ void gla_weights(GlaP& p, const bf16x8 (&q)[3], const bf16x8 (&k)[3]) {
    p.small = mfma_16x16x32(k[2], q[0], p.small);
    p.small = mfma_16x16x32(k[1], q[1], p.small);
    p.small = mfma_16x16x32(k[0], q[2], p.small);
    p.small = mfma_16x16x32(k[1], q[0], p.small);
    p.small = mfma_16x16x32(k[0], q[1], p.small);
    p.big = mfma_16x16x32(k[0], q[0], p.big);
}
__device__ __forceinline__ Terms4 gla_weight_terms(const GlaP& p, int ln, int g) {
    f32x4 P = p.small + p.big;
#pragma unroll
    for (int r = 0; r < 4; ++r) P[r] = 4 * g + r <= ln ? P[r] : 0.f;
    return split3(P);
}

// A workgroup per chunk and head: the chunk's tile, all chunks side by side (see GlaTile)
template <int D>
__global__ void __launch_bounds__(256) gla_tiles_kernel(const GlaScan a) {
    using G = GlaTile<D>;
    __shared__ __attribute__((aligned(16))) unsigned char im[6 * G::Q];
    __shared__ float ws[kGC];
    __shared__ int bad;
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 15, g = lane >> 4;
    const int hd = blockIdx.x % a.H, slot = blockIdx.x / a.H, hk = hd / (a.H / a.HK);
    int upto = 0;   // sequences whose first chunk is this one or an earlier one
    for (int j = 0; j < a.B; j += 64) {
        const int q = j + lane;
        upto += __popcll(__ballot(q < a.B && a.q_start[min(q, a.B - 1)] / kGC + q <= slot));
    }
    if (upto == 0) return;
    const int b = upto - 1, s0 = a.q_start[b], t1 = a.q_start[b + 1], tb = s0 + (slot - s0 / kGC - b) * kGC;
    if (tb >= t1) return;
    const int nt = min(kGC, t1 - tb);
    unsigned char* const out = a.tiles + ((int64_t)slot * a.H + hd) * G::SIZE;
    const bool keys = tid >= 128;   // (wave-uniform)
    const uint16_t* const src = a.proj + (keys ? a.k_off : a.q_off) + (int64_t)hk * D;
    const float* const dp = a.decay + (int64_t)hd * D;
    const int64_t ldd = (int64_t)a.H * D;
    constexpr int NI = (D + 127) / 128;
    float2 d[NI][8], d0[NI][8];
    uint32_t q[NI][8];
#pragma unroll
    for (int it = 0; it < NI; ++it) {
        const int i = (tid & 127) + 128 * it, rp = i % (D / 2), half = i / (D / 2) & 1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {   // tokens past the range decay nothing, rows past it repeat the last
            const float2 one = {1.f, 1.f};
            const int t = 8 * half + e;
            d0[it][e] = e < nt ? *reinterpret_cast<const float2*>(dp + (tb + e) * ldd + 2 * rp) : one;
            d[it][e] = t < nt ? *reinterpret_cast<const float2*>(dp + (tb + t) * ldd + 2 * rp) : one;
            q[it][e] = *reinterpret_cast<const uint32_t*>(src + (int64_t)min(tb + t, t1 - 1) * a.ldp + 2 * rp);
        }
    }
    if (tid == 0) bad = 0;
    __syncthreads();
    if (tid < kGC) {
        const int64_t t = min(tb + tid, t1 - 1);
        float sw = a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f;
        if (a.vscale != nullptr) sw *= a.vscale[t * a.H + hd];
        const float w = tid < nt ? sw : 0.f;
        ws[tid] = w;
        if (!(fabsf(sw) < 0x1p25f)) bad = 1;
        float* const fac = reinterpret_cast<float*>(out + G::W);
        fac[tid] = w;
        fac[kGC + tid] = a.qscale != nullptr ? a.qscale[t * a.HK + hk] : a.q_mul;
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < NI; ++it) {
        const int i = (tid & 127) + 128 * it, rp = i % (D / 2), half = i / (D / 2);
        if (D % 128 == 0 || i < D) {
            float w[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) w[e] = keys ? ws[8 * half + e] : 1.f;
            if (gla_rows(keys, half, d[it], d0[it], q[it], w, [&](int t, float x, float y) { gla_put<D>(im + (keys ? 3 * G::Q : 0), t, rp, x, y); },
                         [&](double X, double Y) {
                             *reinterpret_cast<float2*>(out + G::F + rp * 8) = float2{(float)X, (float)Y};
                             *reinterpret_cast<double2*>(out + G::X + rp * 16) = double2{X, Y};
                         }))
                bad = 1;
        }
    }
    __syncthreads();
    if (wv < G::RW) {
        const int sp = spread<D / 8>(ln);
        GlaP p{{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int j = 0; j < D / 32 / G::RW; ++j) {
            const int kk = wv * (D / 32 / G::RW) + j;
            const unsigned char* at = im + ln * (D * 2) + ((kk * 4 + g) ^ sp) * 16;
            auto term = [&](int k) { return *reinterpret_cast<const bf16x8*>(at + k * G::Q); };
            const bf16x8 qt[3] = {term(0), term(1), term(2)}, kt[3] = {term(3), term(4), term(5)};
            gla_weights(p, qt, kt);
        }
        const Terms4 pt = gla_weight_terms(p, ln, g);
        bf16x4* const to = reinterpret_cast<bf16x4*>(out + G::P + wv * 1536) + lane;
        to[0] = pt.h;
        to[64] = pt.m;
        to[128] = pt.l;
        if (tid == 0) *reinterpret_cast<int*>(out + G::BAD) = bad;
    }
    for (int i = tid; i < 6 * G::Q / 16; i += 256) reinterpret_cast<u16x8*>(out)[i] = reinterpret_cast<const u16x8*>(im)[i];
}

// LDS (bytes): two buffers of q | k | decays (float) | v (64 columns), rows as they lie | F q and w k / F, three terms each | F_16 |
// the factors w and r of two chunks | whether a chunk goes token by token, for three chunks, and whether the segment starts at the sequence's
template <int D> struct GlaLds {
    static constexpr int Q = kGC * D * 2, DEC = 2 * Q, V = DEC + kGC * D * 4, BUF = V + kGC * 128;
    static constexpr int TQ = 2 * BUF, TK = TQ + 3 * Q, F = TK + 3 * Q, SC = F + D * 4, BAD = SC + 4 * kGC * 4, SIZE = BAD + 16;
};

// STATE: the first pass over segments, which only carries the state on (each from 0, the first from the sequence's state)
template <int D, bool STATE>
__global__ void __launch_bounds__(256, 1) gla_scan_kernel(const GlaScan a) {
    using M = GlaLds<D>;
    constexpr int CPR = D / 8, KK = D / 32;   // 16-byte pieces per row of q and k; 32-row steps
    extern __shared__ __attribute__((aligned(1024))) unsigned char gs_smem[];
    float* const fs = reinterpret_cast<float*>(gs_smem + M::F);
    float* const sc = reinterpret_cast<float*>(gs_smem + M::SC);
    int* const bad = reinterpret_cast<int*>(gs_smem + M::BAD);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), ln = lane & 15, g = lane >> 4;
    // groups of workgroups that share q, k and decay rows go to one XCD (workgroup i runs on XCD i % 8), the next segment's behind them
    const int nslab = (a.Dv + 63) / 64, id = blockIdx.x >> 3, seg = blockIdx.y, slab = id % nslab;
    const int group = (id / nslab) * 8 + ((blockIdx.x - seg * a.B * a.H) & 7);
    if (group >= a.B * a.H) return;
    const int b = group / a.H, hd = group % a.H, hk = hd / (a.H / a.HK);
    const int s0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= s0) return;
    const int chunks = (t1 - s0 + kGC - 1) / kGC;
    const int own = s0 + chunks * seg / a.segs * kGC, te = min(t1, s0 + chunks * (seg + 1) / a.segs * kGC);   // this segment's tokens
    const int64_t cells = (int64_t)a.B * a.H;
    const int c0 = slab * 64, col = c0 + wv * 16 + ln;
    const bool live = col < a.Dv;
    float* const Sp = a.S + ((int64_t)a.slots[b] * a.H + hd) * D * a.Dv + col;
    const bool fresh = a.pos0[b] == 0;
    // S[2 kk + h], element r of lane group g: row 32 kk + 8 g + 4 h + r (what the read-out's product takes from that lane)
    f32x4 S[2 * KK];
    auto row_of = [&](int i, int r) { return (i >> 1) * 32 + 8 * g + 4 * (i & 1) + r; };
    float* const seg0 = a.segs > 1 ? a.seg_s + (int64_t)group * D * a.Dv + col : nullptr;   // the state before the step, kept by the first pass
    {
        const bool first = seg == 0, zero = !live || (STATE ? !first || fresh : first && fresh);
        const float* const at = STATE || a.segs == 1 ? Sp : first ? seg0 : seg0 + cells * D * a.Dv;
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[i][r] = zero ? 0.f : at[(int64_t)row_of(i, r) * a.Dv];
        if (STATE && first && !zero) {
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) seg0[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
        }
    }
    if constexpr (!STATE) {
        for (int j = 1; j < seg; ++j) {   // over the segments between: S <- (products of decays) S + what they write
            const float *const at = seg0 + cells * (j + 1) * D * a.Dv, *const d = a.seg_d + (cells * j + group) * D;
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[i][r] = d[row_of(i, r)] * S[i][r] + (live ? at[(int64_t)row_of(i, r) * a.Dv] : 0.f);
        }
    }
    int t0 = own;
    if (tid < 4) bad[tid] = 0;
    if constexpr (!STATE)
        if (seg != 0) {   // products of decays cannot carry on a state that is not finite: then from the sequence's first token
            f32x4 odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) odd += S[i] * 0.f;
            __syncthreads();
            if (!(odd[0] + odd[1] + odd[2] + odd[3] == 0.f)) bad[3] = 1;
            __syncthreads();
            if (bad[3] != 0) {
                t0 = s0;
#pragma unroll
                for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[i][r] = live && !fresh ? seg0[(int64_t)row_of(i, r) * a.Dv] : 0.f;
            }
        }
    double dx[(D + 127) / 128], dy[(D + 127) / 128];   // STATE: the products of the segment's decays so far (rows as F q below)
#pragma unroll
    for (int it = 0; it < (D + 127) / 128; ++it) dx[it] = dy[it] = 1.0;
    const uint16_t* const qp = a.proj + a.q_off + (int64_t)hk * D;
    const uint16_t* const kp = a.proj + a.k_off + (int64_t)hk * D;
    const uint16_t* const vp = a.proj + a.v_off + (int64_t)hd * a.Dv + c0;
    const float* const dp = a.decay + (int64_t)hd * D;
    const int64_t ldd = (int64_t)a.H * D;
    const int vn = min(8, (a.Dv - c0) / 8);
    const uint32_t lds0 = lds_offset(gs_smem);
    // A chunk's rows into a buffer, pieces of 1 KiB dealt to the waves: q D / 32, k D / 32, decays D / 16, v 2.  Rows past the last
    // token repeat it, columns past Dv the last ones (not stored).
    constexpr int NP = (D / 8 + 2 + 3) / 4;
    const char* from[NP];
    int64_t step[NP];
    int prow[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        const int p = wv + 4 * u;   // wave-uniform
        if (p < D / 16) {
            const int i = (p % (D / 32)) * 64 + lane;
            prow[u] = i / CPR;
            from[u] = reinterpret_cast<const char*>((p < D / 32 ? qp : kp) + i % CPR * 8);
            step[u] = (int64_t)a.ldp * 2;
        } else if (p < D / 8) {
            const int i = (p - D / 16) * 64 + lane;
            prow[u] = i / (2 * CPR);
            from[u] = reinterpret_cast<const char*>(dp + i % (2 * CPR) * 4);
            step[u] = ldd * 4;
        } else {
            const int i = ((p - D / 8) & 1) * 64 + lane;
            prow[u] = i / 8;
            from[u] = reinterpret_cast<const char*>(vp + min(i % 8, vn - 1) * 8);
            step[u] = (int64_t)a.ldp * 2;
        }
    }
    auto fetch = [&](int tb, int buf) {
#pragma unroll
        for (int u = 0; u < NP; ++u)
            if (wv + 4 * u < D / 8 + 2)
                dma_1k(from[u] + min(tb + prow[u], t1 - 1) * step[u], __builtin_amdgcn_readfirstlane(lds0 + buf * M::BUF + (wv + 4 * u) * 1024));
    };
    float sw = 0.f, sr = 0.f;   // the factors of token tb + tid % 16, as loaded
    auto scalars = [&](int tb) {
        const int64_t t = min(tb + ln, t1 - 1);
        sw = a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f;
        if (a.vscale != nullptr) sw *= a.vscale[t * a.H + hd];
        sr = a.qscale != nullptr ? a.qscale[t * a.HK + hk] : a.q_mul;
    };
    const uint32_t orow = (uint32_t)a.H * a.Dv * 4, ocol = live ? (uint32_t)col * 4 : 0x80000000u;
    if (t0 < te) {
        fetch(t0, 0);
        scalars(t0);
    }
    received(sw);
    received(sr);
    for (int tb = t0, buf = 0, turn = 0; tb < te; tb += kGC, buf ^= 1, turn = turn == 2 ? 0 : turn + 1) {
        const int nt = min(kGC, te - tb);
        unsigned char* const raw = gs_smem + buf * M::BUF;
        const uint16_t* const qs = reinterpret_cast<const uint16_t*>(raw);
        const uint16_t* const ks = reinterpret_cast<const uint16_t*>(raw + M::Q);
        float* const ds = reinterpret_cast<float*>(raw + M::DEC);
        float* const ws = sc + buf * 2 * kGC;
        // (each earlier chunk issued 4 stores or 16 after this chunk's pieces)
        if (STATE || tb == t0) dma_wait();
        else dma_wait_before_stores<4>();
        if (tid < kGC) {
            ws[tid] = tid < nt ? sw : 0.f;
            ws[kGC + tid] = sr;
            if (!(fabsf(sw) < 0x1p25f)) bad[turn] = 1;
        }
        __syncthreads();   // the rows are there; nobody reads the other buffer or the last chunk's products any more
        if (nt < kGC) {    // tokens past the range decay nothing
            for (int i = nt * D + tid; i < kGC * D; i += 256) ds[i] = 1.f;
            __syncthreads();
        }
        if (tb + kGC < te) {
            fetch(tb + kGC, buf ^ 1);
            scalars(tb + kGC);
        }
        Terms st[KK];   // of the state before the chunk
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const float x[8] = {S[2 * kk][0], S[2 * kk][1], S[2 * kk][2], S[2 * kk][3],
                                S[2 * kk + 1][0], S[2 * kk + 1][1], S[2 * kk + 1][2], S[2 * kk + 1][3]};
            st[kk] = split3(x);
        }
        // ---- F q (threads 0 .. 127) and w k / F (the others): two rows, 8 tokens
        const bool keys = tid >= 128;   // (wave-uniform)
        const uint16_t* const src = keys ? ks : qs;
#pragma unroll
        for (int it = 0; it < (D + 127) / 128; ++it) {
            const int i = (tid & 127) + 128 * it, rp = i % (D / 2), half = i / (D / 2);
            if (D % 128 == 0 || i < D) {
                // everything read first (the compiler keeps reads behind the writes below)
                float2 d[8], d0[8];
                uint32_t q[8];
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    d0[e] = *reinterpret_cast<const float2*>(ds + e * D + 2 * rp);
                    d[e] = *reinterpret_cast<const float2*>(ds + (8 * half + e) * D + 2 * rp);
                    q[e] = *reinterpret_cast<const uint32_t*>(src + (8 * half + e) * D + 2 * rp);
                    w[e] = keys ? ws[8 * half + e] : 1.f;
                }
                if (gla_rows(keys, half, d, d0, q, w, [&](int t, float x, float y) { gla_put<D>(gs_smem + (keys ? M::TK : M::TQ), t, rp, x, y); },
                             [&](double X, double Y) {
                                 fs[2 * rp] = (float)X;
                                 fs[2 * rp + 1] = (float)Y;
                                 if constexpr (STATE) {
                                     dx[it] *= X;
                                     dy[it] *= Y;
                                 }
                             }))
                    bad[turn] = 1;
            }
        }
        if (tid == 0) bad[turn == 2 ? 0 : turn + 1] = 0;   // (the next chunk's; last read two barriers ago)
        __syncthreads();   // all of it is there
        received(sw);
        received(sr);
        const f32x4 fr = *reinterpret_cast<const f32x4*>(ws + kGC + 4 * g);
        const auto ord = __builtin_amdgcn_make_buffer_rsrc(a.o + ((int64_t)tb * a.H + hd) * a.Dv, (short)0, tb < own ? 0 : (int)(nt * orow), 0x00020000);
        const bf16x4 v4 = lds_read_tr4(raw + M::V + (4 * g + (ln >> 2)) * 128 + wv * 32 + (ln & 3) * 8);   // tokens 4 g ..
        const bf16x8 vv = join8(v4, v4);
        const bf16x4 none = {};
        const uint2 vw = __builtin_bit_cast(uint2, v4);
        const u16x2 vbig = max_bits(max_bits(u16x2{0, 0}, vw.x), vw.y);
        bool apart = __builtin_amdgcn_ballot_w64(bad[turn] != 0 || (!STATE && (vbig[0] >= kBig || vbig[1] >= kBig))) != 0;   // (wave-uniform)
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        if (!STATE && !apart) {
            // ---- read-out: o = (F q)^T S, and P with rows s = 4 g + r and columns t = ln (as its product with v takes it)
            const int sp = spread<CPR>(ln);
            f32x4 small = {0.f, 0.f, 0.f, 0.f}, big = small;
            GlaP p{small, small};
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const unsigned char* at = gs_smem + M::TQ + ln * (D * 2) + ((kk * 4 + g) ^ sp) * 16;
                auto term = [&](int k) { return *reinterpret_cast<const bf16x8*>(at + k * M::Q); };
                const bf16x8 q[3] = {term(0), term(1), term(2)}, k[3] = {term(3), term(4), term(5)};
                gla_weights(p, q, k);
                small = mfma_16x16x32(q[2], st[kk].h, small);
                small = mfma_16x16x32(q[1], st[kk].m, small);
                small = mfma_16x16x32(q[0], st[kk].l, small);
                small = mfma_16x16x32(q[1], st[kk].h, small);
                small = mfma_16x16x32(q[0], st[kk].m, small);
                big = mfma_16x16x32(q[0], st[kk].h, big);
            }
            const Terms4 pt = gla_weight_terms(p, ln, g);
            small = mfma_16x16x32(join8(pt.l, none), vv, small);
            big = mfma_16x16x32(join8(pt.h, pt.m), vv, big);
            o = small + big;
            apart = __builtin_amdgcn_ballot_w64(!(__builtin_fmaf(o[0], 0.f, o[1] * 0.f) + __builtin_fmaf(o[2], 0.f, o[3] * 0.f) == 0.f)) != 0;
        }
        if (apart) {   // token by token
            const uint16_t* const vs = reinterpret_cast<const uint16_t*>(raw + M::V) + wv * 16 + ln;
            for (int t = 0; t < nt; ++t) {
                const float u = bf2f(vs[t * 64]) * ws[t];
                float acc[2] = {0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = t * D + (i >> 1) * 32 + 8 * g + 4 * (i & 1) + r;
                        S[i][r] = ds[row] * S[i][r] + bf2f(ks[row]) * u;
                        acc[r & 1] += bf2f(qs[row]) * S[i][r];
                    }
                float x = acc[0] + acc[1];
                x = rows_sum(x);
                if (!STATE && g == 0) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x * ws[kGC + t]), ord, ocol + t * orow, 0, 0);
            }
            continue;
        }
        if constexpr (!STATE) {
#pragma unroll
            for (int r = 0; r < 4; ++r)   // (past the last token and past Dv the descriptor's range drops the store)
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[r] * fr[r]), ord, ocol + (4 * g + r) * orow, 0, 0);
        }
        // ---- the state after the chunk
        const int r4 = 4 * g + (ln >> 2), sp4 = spread<CPR>(r4);
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i) {
            const int kk = i >> 1, h = i & 1;
            const unsigned char* at = gs_smem + M::TK + r4 * (D * 2) + ((kk * 4 + (ln & 3)) ^ sp4) * 16 + h * 8;
            const bf16x4 kh = lds_read_tr4(at), km = lds_read_tr4(at + M::Q), kl = lds_read_tr4(at + 2 * M::Q);
            S[i] = mfma_16x16x32(join8(kl, none), vv, S[i]);
            S[i] = mfma_16x16x32(join8(kh, km), vv, S[i]);
            S[i] *= *reinterpret_cast<const f32x4*>(fs + kk * 32 + 8 * g + 4 * h);
        }
    }
    if (!STATE && seg != a.segs - 1) return;
    if (live) {
        float* const out = STATE ? seg0 + cells * (seg + 1) * D * a.Dv : Sp;
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
    }
    if constexpr (STATE) {
#pragma unroll
        for (int it = 0; it < (D + 127) / 128; ++it) {
            const int i = (tid & 127) + 128 * it, rp = i % (D / 2);
            if (tid < 128 && (D % 128 == 0 || i < D) && i / (D / 2) == 1) {   // (every slab the same)
                float* const d = a.seg_d + (cells * seg + group) * D + 2 * rp;
                d[0] = (float)dx[it];
                d[1] = (float)dy[it];
            }
        }
    }
}

// LDS (bytes): two buffers of gla_tiles_kernel's tile | v; the waves' parts of the read-outs of two chunks; whether the segment starts at the sequence's
template <int D> struct GlaWalkLds {
    static constexpr int NW = 4 * GlaTile<D>::RW, V = GlaTile<D>::SIZE, BUF = V + kGC * 128, O = 2 * BUF, BAD = O + (NW > 4 ? 2 * NW * 1024 : 0), SIZE = BAD + 16;
};

// The walk over tiles made ahead: as gla_scan_kernel, but RW waves share 16 columns of S, each with its D / RW rows, its part of P and of the read-out; the
// parts meet in LDS behind the next chunk's barrier.  The terms were made between the steps, once for every 64 value columns, half of a chunk's
// time.  Both launches, us, heads of 128 x 256, before -> this: 16 heads, 4 sequences of 2048 tokens 376 -> 300 (72 of them the tiles: 28 KB written per chunk and head),
// 8 of 1000 271 -> 229, 2 of 256 50 -> 35; 8 heads, one of 4000 (eight segments) 172 -> 102; 4 heads, one of 2048 76 -> 55, 21 of 117 38.6 -> 33.4; 8 of
// 256 x 256, 4 of 500 148 -> 86.  With one wave per 16 columns 300 and 58.7 us where this took 288 and 55; with three or four buffers and one workgroup per CU 350
// and 48, 21 of 117 43: what bounds it is the work of the waves that a CU holds, 212 vector and 22 matrix instructions of each per chunk and 1200 cycles
// of its LDS, two workgroups per CU (hence 128 registers).
template <int D, bool STATE>
__global__ void __launch_bounds__(256 * GlaTile<D>::RW) __attribute__((amdgpu_waves_per_eu(D >= 128 ? 4 : 2))) gla_walk_kernel(const GlaScan a) {
    using G = GlaTile<D>;
    using M = GlaWalkLds<D>;
    constexpr int NW = M::NW, RW = G::RW, CPR = D / 8, KK = D / 32 / RW;
    extern __shared__ __attribute__((aligned(1024))) unsigned char gs_smem[];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6), cw = wv & 3, part = wv >> 2, ln = lane & 15, g = lane >> 4;
    // groups of workgroups that share tiles go to one XCD (workgroup i runs on XCD i % 8), the next segment's behind them
    const int nslab = (a.Dv + 63) / 64, id = blockIdx.x >> 3, seg = blockIdx.y, slab = id % nslab;
    const int group = (id / nslab) * 8 + ((blockIdx.x - seg * a.B * a.H) & 7);
    if (group >= a.B * a.H) return;
    const int b = group / a.H, hd = group % a.H, hk = hd / (a.H / a.HK);
    const int s0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= s0) return;
    const int chunks = (t1 - s0 + kGC - 1) / kGC;
    const int own = s0 + chunks * seg / a.segs * kGC, te = min(t1, s0 + chunks * (seg + 1) / a.segs * kGC);   // this segment's tokens
    const int64_t cells = (int64_t)a.B * a.H;
    const int c0 = slab * 64, col = c0 + cw * 16 + ln;
    const bool live = col < a.Dv;
    // S[2 kk + h], element r of lane group g: the part's row 32 kk + 8 g + 4 h + r
    f32x4 S[2 * KK];
    auto row_of = [&](int i, int r) { return part * (D / RW) + (i >> 1) * 32 + 8 * g + 4 * (i & 1) + r; };
    float* const Sp = a.S + ((int64_t)a.slots[b] * a.H + hd) * D * a.Dv + col;
    const bool fresh = a.pos0[b] == 0;
    float* const seg0 = a.segs > 1 ? a.seg_s + (int64_t)group * D * a.Dv + col : nullptr;   // the state before the step, kept by the first pass
    {
        const bool first = seg == 0, zero = !live || (STATE ? !first || fresh : first && fresh);
        const float* const at = STATE || a.segs == 1 ? Sp : first ? seg0 : seg0 + cells * D * a.Dv;
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) S[i][r] = zero ? 0.f : at[(int64_t)row_of(i, r) * a.Dv];
        if (STATE && first && !zero) {
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) seg0[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
        }
    }
    int t0 = own;
    if constexpr (!STATE) {
        for (int j = 1; j < seg; ++j) {   // over the segments between: S <- (products of decays) S + what they write
            const float *const at = seg0 + cells * (j + 1) * D * a.Dv, *const d = a.seg_d + (cells * j + group) * D;
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) S[i][r] = d[row_of(i, r)] * S[i][r] + (live ? at[(int64_t)row_of(i, r) * a.Dv] : 0.f);
        }
        if (seg != 0) {   // products of decays cannot carry on a state that is not finite: then from the sequence's first token
            int* const bad = reinterpret_cast<int*>(gs_smem + M::BAD);
            f32x4 odd = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) odd += S[i] * 0.f;
            if (tid == 0) *bad = 0;
            __syncthreads();
            if (!(odd[0] + odd[1] + odd[2] + odd[3] == 0.f)) *bad = 1;
            __syncthreads();
            if (*bad != 0) {
                t0 = s0;
#pragma unroll
                for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) S[i][r] = live && !fresh ? seg0[(int64_t)row_of(i, r) * a.Dv] : 0.f;
            }
        }
    }
    // STATE: the products of the segment's decays so far, thread i's of row i (D <= threads)
    double dx = 1.0;
    const uint16_t* const qp = a.proj + a.q_off + (int64_t)hk * D;
    const uint16_t* const kp = a.proj + a.k_off + (int64_t)hk * D;
    const uint16_t* const vp = a.proj + a.v_off + (int64_t)hd * a.Dv + c0;
    const float* const dp = a.decay + (int64_t)hd * D;
    const int64_t ldd = (int64_t)a.H * D;
    const int vn = min(8, (a.Dv - c0) / 8);
    const uint32_t lds0 = lds_offset(gs_smem);
    // A chunk's tile and rows of v into a buffer, pieces of 1 KiB dealt to the waves.  v: rows past the last token repeat it, columns past
    // Dv the last ones (not stored).
    constexpr int NR = G::SIZE / 1024, NP = (NR + 2 + NW - 1) / NW;
    const unsigned char* const tiles = a.tiles + ((int64_t)(s0 / kGC + b) * a.H + hd) * G::SIZE + lane * 16;
    auto fetch = [&](int tb, int buf) {
        const unsigned char* const tile = tiles + (int64_t)((tb - s0) / kGC) * a.H * G::SIZE;
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int p = wv + NW * u;   // wave-uniform
            const uint32_t to = __builtin_amdgcn_readfirstlane(lds0 + buf * M::BUF + p * 1024);
            if (p < NR) dma_1k(tile + p * 1024, to);
            else if (p < NR + 2) {
                const int i = (p - NR) * 64 + lane;
                dma_1k(vp + (int64_t)min(tb + i / 8, t1 - 1) * a.ldp + min(i % 8, vn - 1) * 8, to);
            }
        }
    };
    const uint32_t orow = (uint32_t)a.H * a.Dv * 4, ocol = live ? (uint32_t)col * 4 : 0x80000000u;
    // A chunk's outputs of token 4 g + r for the r of this wave's part (past the last token and past Dv the descriptor's range drops the store)
    f32x4 last = {0.f, 0.f, 0.f, 0.f}, fr = last;   // RW 1: the chunk's read-out; the factors r
    constexpr int STORES = 4 / RW;
    auto store = [&](int tb, int buf) {
        const int nt = min(kGC, te - tb);
        const auto ord = __builtin_amdgcn_make_buffer_rsrc(a.o + ((int64_t)tb * a.H + hd) * a.Dv, (short)0, tb < own ? 0 : (int)(nt * orow), 0x00020000);
        const float* const at = reinterpret_cast<const float*>(gs_smem + M::O + (buf * NW + cw) * 1024) + lane * 4 + part * STORES;
#pragma unroll
        for (int r = 0; r < STORES; ++r) {
            float x = RW == 1 ? last[r] : at[r];
#pragma unroll
            for (int k = 1; k < RW; ++k) x += at[k * 4 * 256 + r];
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x * fr[r]), ord, ocol + (4 * g + part * STORES + r) * orow, 0, 0);
        }
    };
    if (t0 < te) fetch(t0, 0);
    for (int tb = t0, buf = 0; tb < te; tb += kGC, buf ^= 1) {
        const int nt = min(kGC, te - tb);
        unsigned char* const raw = gs_smem + buf * M::BUF;
        const float* const ws = reinterpret_cast<const float*>(raw + G::W);
        // (from the third chunk on, the one before issued its predecessor's stores after this chunk's pieces)
        if (STATE || tb < t0 + 2 * kGC) dma_wait();
        else dma_wait_before_stores<STORES>();
        __syncthreads();   // the tile is there; nobody reads the other buffer any more; the parts of the last chunk's read-out are there
        if (tb + kGC < te) fetch(tb + kGC, buf ^ 1);
        asm volatile("" ::: "memory");   // (the count above takes the stores behind the pieces)
        if (!STATE && tb != t0) store(tb - kGC, buf ^ 1);
        if constexpr (!STATE) {
#pragma unroll
            for (int r = 0; r < STORES; ++r) fr[r] = ws[kGC + 4 * g + part * STORES + r];
        } else if (tid < D) {
            dx *= *reinterpret_cast<const double*>(raw + G::X + tid * 8);
        }
        const bf16x4 v4 = lds_read_tr4(raw + M::V + (4 * g + (ln >> 2)) * 128 + cw * 32 + (ln & 3) * 8);   // tokens 4 g ..
        const bf16x4 none = {};
        const bf16x8 vv = join8(v4, v4);
        const uint2 vw = __builtin_bit_cast(uint2, v4);
        const u16x2 vbig = max_bits(max_bits(u16x2{0, 0}, vw.x), vw.y);
        const int bad = __builtin_amdgcn_readfirstlane(*reinterpret_cast<const int*>(raw + G::BAD));
        bool apart = bad != 0 || (!STATE && __builtin_amdgcn_ballot_w64(vbig[0] >= kBig || vbig[1] >= kBig) != 0);   // (wave-uniform)
        f32x4* const mine = reinterpret_cast<f32x4*>(gs_smem + M::O + (buf * NW + wv) * 1024) + lane;
        f32x4 N[2 * KK];   // the state after the chunk
        if (!apart) {
            const int r4 = 4 * g + (ln >> 2), sp4 = spread<CPR>(r4), sp = spread<CPR>(ln);
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) {
                const int kk = part * KK + (i >> 1), h = i & 1;
                const unsigned char* at = raw + 3 * G::Q + r4 * (D * 2) + ((kk * 4 + (ln & 3)) ^ sp4) * 16 + h * 8;
                const bf16x4 kh = lds_read_tr4(at), km = lds_read_tr4(at + G::Q), kl = lds_read_tr4(at + 2 * G::Q);
                N[i] = mfma_16x16x32(join8(kl, none), vv, S[i]);
                N[i] = mfma_16x16x32(join8(kh, km), vv, N[i]);
                N[i] *= *reinterpret_cast<const f32x4*>(reinterpret_cast<const float*>(raw + G::F) + kk * 32 + 8 * g + 4 * h);
            }
            if constexpr (!STATE) {
                // ---- this part's read-out: (F q)^T S + P v
                f32x4 small = {0.f, 0.f, 0.f, 0.f}, big = small, less = small;
#pragma unroll
                for (int j = 0; j < KK; ++j) {
                    const unsigned char* at = raw + ln * (D * 2) + (((part * KK + j) * 4 + g) ^ sp) * 16;
                    auto term = [&](int k) { return *reinterpret_cast<const bf16x8*>(at + k * G::Q); };
                    const bf16x8 q[3] = {term(0), term(1), term(2)};
                    const float x[8] = {S[2 * j][0], S[2 * j][1], S[2 * j][2], S[2 * j][3], S[2 * j + 1][0], S[2 * j + 1][1], S[2 * j + 1][2], S[2 * j + 1][3]};
                    const Terms st = split3(x);
                    less = mfma_16x16x32(q[2], st.h, less);
                    small = mfma_16x16x32(q[1], st.h, small);
                    big = mfma_16x16x32(q[0], st.h, big);
                    less = mfma_16x16x32(q[1], st.m, less);
                    small = mfma_16x16x32(q[0], st.m, small);
                    less = mfma_16x16x32(q[0], st.l, less);
                }
                const bf16x4* const pt = reinterpret_cast<const bf16x4*>(raw + G::P + part * 1536) + lane;
                less = mfma_16x16x32(join8(pt[128], none), vv, less);
                big = mfma_16x16x32(join8(pt[0], pt[64]), vv, big);
                last = (less + small) + big;
                apart = __builtin_amdgcn_ballot_w64(!(__builtin_fmaf(last[0], 0.f, last[1] * 0.f) + __builtin_fmaf(last[2], 0.f, last[3] * 0.f) == 0.f)) != 0;
                if (RW > 1) *mine = last;
            }
        }
        if (!apart) {
#pragma unroll
            for (int i = 0; i < 2 * KK; ++i) S[i] = N[i];
            continue;
        }
        // ---- token by token
        auto tokens = [&](const uint16_t* q, const uint16_t* k, int64_t ld, const float* d, int64_t ld4) {
            const uint16_t* const vs = reinterpret_cast<const uint16_t*>(raw + M::V) + cw * 16 + ln;
            for (int t = 0; t < nt; ++t) {
                const float u = bf2f(vs[t * 64]) * ws[t];
                float acc[2] = {0.f, 0.f};
#pragma unroll
                for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int row = row_of(i, r);
                        S[i][r] = d[t * ld4 + row] * S[i][r] + bf2f(k[t * ld + row]) * u;
                        acc[r & 1] += bf2f(q[t * ld + row]) * S[i][r];
                    }
                float x = acc[0] + acc[1];
                x = rows_sum(x);
#pragma unroll
                for (int r = 0; r < 4; ++r) last[r] = t == 4 * g + r ? x : last[r];
            }
        };
        if (bad != 0) {   // all waves: the chunk's rows come where the terms are
            uint16_t* const qs = reinterpret_cast<uint16_t*>(raw);
#pragma unroll
            for (int u = 0; u < (D / 8 + NW - 1) / NW; ++u) {
                const int pc = wv + NW * u, i = (pc % (D / 32)) * 64 + lane, j = (pc - D / 16) * 64 + lane;
                if (pc < D / 8)
                    dma_1k(pc < D / 16 ? reinterpret_cast<const void*>((pc < D / 32 ? qp : kp) + min(tb + i / CPR, t1 - 1) * (int64_t)a.ldp + i % CPR * 8)
                                       : reinterpret_cast<const void*>(dp + min(tb + j / (2 * CPR), t1 - 1) * ldd + j % (2 * CPR) * 4),
                           __builtin_amdgcn_readfirstlane(lds0 + buf * M::BUF + pc * 1024));
            }
            dma_wait();
            __syncthreads();
            tokens(qs, qs + kGC * D, D, reinterpret_cast<const float*>(qs + 2 * kGC * D), D);
        } else {
            tokens(qp + (int64_t)tb * a.ldp, kp + (int64_t)tb * a.ldp, a.ldp, dp + tb * ldd, ldd);
        }
        if (!STATE && RW > 1) *mine = last;
    }
    if (!STATE && t0 < te) {
        __syncthreads();
        store(t0 + (te - 1 - t0) / kGC * kGC, (te - 1 - t0) / kGC & 1);
    }
    if (!STATE && seg != a.segs - 1) return;
    if (live) {
        float* const out = STATE ? seg0 + cells * (seg + 1) * D * a.Dv : Sp;
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(int64_t)row_of(i, r) * a.Dv] = S[i][r];
    }
    if (STATE && tid < D) a.seg_d[(cells * seg + group) * D + tid] = (float)dx;   // (every slab the same)
}

}  // namespace hy

// Whether a launch takes less time in chunks than token by token: ranges of 8 tokens on average, or one of 24.  A chunk costs the same
// whether it is full or not: 21 sequences of n tokens, 4 heads of 128 x 256, token by token / here, us: 9.2 / 9.8 at n = 2, 10.9 / 9.8 at 4, 14.0 / 9.8
// at 8, 21 / 9.9 at 16, 109 / 39 at 117; one of n beside 64 ranges of one token: 19.7 / 25.8 at 4, 25.2 / 26.0 at 16, beside 256 63.8 / 74.3 at 16,
// 68.6 / 73.6 at 24.  Of 905 launches of 4 shapes (profiles/recurrence_forms.json) 2 lose by more than 3% (the worst by 8); from 4 tokens for the longest
// on 66 did (by up to 45).
bool hy_gla_scan_pays(int T, int B, int longest) { return longest >= 24 || (longest >= 4 && T >= 8 * (int64_t)B); }

// When this form serves a launch: bfloat16 rows of q, k, v and rows of decays on 16-byte boundaries, a state of 32, 64, 128 or 256
// rows, and a launch that gains (longest: the most new tokens that any sequence brings).
bool hy_gla_scan_ok(const void* proj, const void* decay, int ldp, int q_off, int k_off, int v_off, int T, int B, int D, int Dv, int longest) {
    return hy_gla_scan_pays(T, B, longest) && (D == 32 || D == 64 || D == 128 || D == 256) && Dv % 8 == 0 && hy::aligned16(proj, decay) &&
           ((ldp | q_off | k_off | v_off) & 7) == 0 && ldp < 1 << 23;
}

template <int D, bool STATE>
static void gla_scan_pass(const hy::GlaScan& a, int segs, hipStream_t s) {
    const unsigned groups = (a.B * a.H + 7) / 8 * 8;
    const dim3 grid(groups * ((a.Dv + 63) / 64), segs);
    auto go = [&](auto kern, int threads, int lds) { kern<<<grid, threads, lds, s>>>(a); };
    if (a.tiles != nullptr) {
        using M = hy::GlaWalkLds<D>;
        static_assert(M::SIZE <= 160 * 1024 && D <= 64 * M::NW, "LDS of one workgroup, a row per thread");
        lds_limit<hy::gla_walk_kernel<D, STATE>>(M::SIZE);
        return go(hy::gla_walk_kernel<D, STATE>, 64 * M::NW, M::SIZE);
    }
    constexpr int lds = hy::GlaLds<D>::SIZE;
    static_assert(lds <= 160 * 1024, "LDS of one workgroup");
    lds_limit<hy::gla_scan_kernel<D, STATE>>(lds);
    go(hy::gla_scan_kernel<D, STATE>, 256, lds);
}
template <int D>
static void gla_scan_run(const hy::GlaScan& a, hipStream_t s) {
    if (a.tiles != nullptr) hy::gla_tiles_kernel<D><<<(unsigned)(hy::gla_slots(a.T, a.B) * a.H), 256, 0, s>>>(a);
    if (a.segs > 1) gla_scan_pass<D, true>(a, a.segs - 1, s);
    gla_scan_pass<D, false>(a, a.segs, s);
}

// Bytes of scratch for the chunks' tiles, or 0: made between the steps, as where no sequence has more than five chunks (the launch more costs 2.5 us: 21
// sequences of 64 tokens, 4 heads of 128 x 256, 21.8 us so, 23.5 with tiles ahead, of 117 38.6 and 33.4), and of launches whose tiles would take more than
// `most` (512 MB: a prompt portion of 16384 tokens and 16 heads of 128 takes 470).
int64_t hy_gla_tiles_bytes(const void* proj, const void* decay, int ldp, int q_off, int k_off, int v_off, int T, int B, int H, int D, int Dv, int longest, int64_t most) {
    const int size = D == 32 ? hy::GlaTile<32>::SIZE : D == 64 ? hy::GlaTile<64>::SIZE : D == 128 ? hy::GlaTile<128>::SIZE : hy::GlaTile<256>::SIZE;
    const int64_t n = hy::gla_slots(T, B) * H * size;
    return longest > 5 * hy::kGC && n <= most && hy_gla_scan_ok(proj, decay, ldp, q_off, k_off, v_off, T, B, D, Dv, longest) ? n : 0;
}

void launch_hy_gla_scan(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, const float* qscale, const float* kscale,
                        float q_mul, const float* decay, const int32_t* q_start, const int32_t* pos0, const int32_t* slots,
                        float* S, float* o, int T, int B, int HK, int H, int D, int Dv, const float* vscale, int segs, float* seg, void* tiles, hipStream_t s) {
    const hy::GlaScan a{proj, ldp, q_off, k_off, v_off, qscale, kscale, vscale, decay, q_mul, q_start, pos0, slots, S, o, B, HK, H, Dv, T,
                        segs, seg, segs > 1 ? seg + (int64_t)segs * B * H * D * Dv : nullptr, static_cast<unsigned char*>(tiles)};
    if (D == 32) gla_scan_run<32>(a, s);
    else if (D == 64) gla_scan_run<64>(a, s);
    else if (D == 128) gla_scan_run<128>(a, s);
    else gla_scan_run<256>(a, s);
}

}  // namespace chronos
