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
    int B, HK, H, Dv;
    // segments of a sequence side by side (1: none), as in chunk_scan.hip: the state before the step and, of each segment but the last,
    // what it writes, [segs, B, H, D, Dv]; products of its decays [segs - 1, B, H, D]
    int segs;
    float *seg_s, *seg_d;
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
        auto put = [&](int base, int t, int rp, float x, float y) {   // the terms of rows 2 rp, 2 rp + 1 of token t
            unsigned char* at = gs_smem + base + t * (D * 2) + (((rp >> 2) ^ spread<CPR>(t)) * 16) + (rp & 3) * 4;
#pragma unroll
            for (int k = 0; k < 3; ++k) *reinterpret_cast<uint32_t*>(at + k * M::Q) = round_pair(x, y);
        };
        const bool keys = tid >= 128;   // (wave-uniform)
        const uint16_t* const src = keys ? ks : qs;
#pragma unroll
        for (int it = 0; it < (D + 127) / 128; ++it) {
            const int i = (tid & 127) + 128 * it, rp = i % (D / 2), half = i / (D / 2);
            if (D % 128 == 0 || i < D) {
                // everything read first (the compiler keeps reads behind the writes below); F in float64, so that F_t / F_s carries
                // the rounding of its two ends and not of the steps between
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
                    if (!(lo >= 0x1p-40f) || !(hi <= 0x1p40f) || X != X || Y != Y || big[0] >= kBig || big[1] >= kBig) bad[turn] = 1;
                    auto inverse = [](float v) {   // to half a last place in the range that counts
                        const float r = __builtin_amdgcn_rcpf(v);
                        return __builtin_fmaf(__builtin_fmaf(-v, r, 1.f), r, r);
                    };
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        put(M::TK, 8 * half + e, rp, w[e] * __uint_as_float(q[e] << 16) * inverse(x[e]),
                            w[e] * __uint_as_float(q[e] & 0xffff0000u) * inverse(y[e]));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        put(M::TQ, 8 * half + e, rp, __uint_as_float(q[e] << 16) * x[e], __uint_as_float(q[e] & 0xffff0000u) * y[e]);
                }
                if (!keys && half) {
                    fs[2 * rp] = x[7];
                    fs[2 * rp + 1] = y[7];
                    if constexpr (STATE) {
                        dx[it] *= X;
                        dy[it] *= Y;
                    }
                }
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
            f32x4 small = {0.f, 0.f, 0.f, 0.f}, big = small, psmall = small, pbig = small;
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) {
                const unsigned char* at = gs_smem + M::TQ + ln * (D * 2) + ((kk * 4 + g) ^ sp) * 16;
                auto term = [&](int base) { return *reinterpret_cast<const bf16x8*>(at + base); };
                const bf16x8 qh = term(0), qm = term(M::Q), ql = term(2 * M::Q), kh = term(3 * M::Q), km = term(4 * M::Q), kl = term(5 * M::Q);
                psmall = mfma_16x16x32(kl, qh, psmall);
                psmall = mfma_16x16x32(km, qm, psmall);
                psmall = mfma_16x16x32(kh, ql, psmall);
                psmall = mfma_16x16x32(km, qh, psmall);
                psmall = mfma_16x16x32(kh, qm, psmall);
                pbig = mfma_16x16x32(kh, qh, pbig);
                small = mfma_16x16x32(ql, st[kk].h, small);
                small = mfma_16x16x32(qm, st[kk].m, small);
                small = mfma_16x16x32(qh, st[kk].l, small);
                small = mfma_16x16x32(qm, st[kk].h, small);
                small = mfma_16x16x32(qh, st[kk].m, small);
                big = mfma_16x16x32(qh, st[kk].h, big);
            }
            f32x4 P = psmall + pbig;
#pragma unroll
            for (int r = 0; r < 4; ++r) P[r] = 4 * g + r <= ln ? P[r] : 0.f;
            const Terms4 pt = split3(P);
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
                x += __shfl_xor(x, 16, 64);
                x += __shfl_xor(x, 32, 64);
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
    constexpr int lds = hy::GlaLds<D>::SIZE;
    static_assert(lds <= 160 * 1024, "LDS of one workgroup");
    const auto kern = hy::gla_scan_kernel<D, STATE>;
    static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)set;
    const int groups = (a.B * a.H + 7) / 8 * 8;
    kern<<<dim3(groups * ((a.Dv + 63) / 64), segs), 256, lds, s>>>(a);
}
template <int D>
static void gla_scan_run(const hy::GlaScan& a, hipStream_t s) {
    if (a.segs > 1) gla_scan_pass<D, true>(a, a.segs - 1, s);
    gla_scan_pass<D, false>(a, a.segs, s);
}

void launch_hy_gla_scan(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, const float* qscale, const float* kscale,
                        float q_mul, const float* decay, const int32_t* q_start, const int32_t* pos0, const int32_t* slots,
                        float* S, float* o, int B, int HK, int H, int D, int Dv, const float* vscale, int segs, float* seg, hipStream_t s) {
    const hy::GlaScan a{proj, ldp, q_off, k_off, v_off, qscale, kscale, vscale, decay, q_mul, q_start, pos0, slots, S, o, B, HK, H, Dv,
                        segs, seg, segs > 1 ? seg + (int64_t)segs * B * H * D * Dv : nullptr};
    if (D == 32) gla_scan_run<32>(a, s);
    else if (D == 64) gla_scan_run<64>(a, s);
    else if (D == 128) gla_scan_run<128>(a, s);
    else gla_scan_run<256>(a, s);
}

}  // namespace chronos
