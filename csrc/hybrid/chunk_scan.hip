// chunk_scan.hip — the linear-state recurrences of linear_scan.hip and mlstm.hip with one decay per head and token, on the
// matrix cores: prompt portions are taken 64 tokens at a time.  With L_t = sum of the log decays of a chunk's tokens up to
// t, S the state before the chunk, w_s the factor on what token s writes and r_t the factor on what token t reads,
//
//     o_t = r_t ( e^L_t S^T q_t + sum_(s <= t) e^(L_t - L_s) w_s (k_s . q_t) v_s )
//     S  <- e^L_C S + sum_s k_s (e^(L_C - L_s) w_s v_s)^T
//
// which are the sums of the token-by-token form in another order.  Precision: q, k and v are bfloat16, everything else
// stays float32.  A float32 operand of a matrix product (the state, the weights of a chunk's tokens, the scaled values)
// enters as three bfloat16 terms cut off its 24-bit mantissa — exactly that number, so a product costs three matrix
// instructions and loses nothing — and all products accumulate in float32.  L is summed in float64: differences of sums
// over strong decays keep their digits.
//
// A workgroup is NW waves and serves 16 NW value columns of one (sequence, head); a wave keeps all D rows of its 16 columns
// of S in accumulators, which are in the operand layout of the read-out's product as they stand.  A chunk's q, k, v rows
// come by DMA into one of two LDS buffers while the chunk before is computed; 16-byte pieces are permuted within a row by a
// function of the row, so that neither the row-wise reads nor the transposing ones meet in a bank.  The waves share the
// 64 x 64 weights (ten 16 x 16 tiles on and below the diagonal) through LDS.
//
// What bounds it: the chain of a sequence's chunks, one wave per SIMD: about 1300 vector instructions (the cutting into
// terms, the exponentials) and 114 matrix instructions per chunk and wave at D = 128, and two barriers, 7 us a chunk.
// Measured, 4 sequences of 2048 tokens, token by token -> this: retention, 8 heads of 128 x 128: 797 -> 233 us; 32 heads:
// 857 -> 243; state-space form, 128 heads of 128 x 64: 1101 -> 527; mlstm, 4 heads of 128 x 256: 1987 -> 301, 4 heads of
// 256 x 512: 3058 -> 462, 8 heads: 3228 -> 472.  One and two waves per workgroup: 436 and 302 us where four take 233.
#include "hybrid_common.h"

namespace chronos {
namespace hy {

constexpr int kCH = 64;   // tokens per chunk
constexpr int kCW = 4;    // waves per workgroup (NW above)

__device__ __forceinline__ f32x4 mfma_16x16x32(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// x = h + m + l exactly: the upper, middle and lower 8 bits of the mantissa
struct Terms {
    bf16x8 h, m, l;
};
__device__ __forceinline__ Terms split3(const float (&x)[8]) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 t[3];
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = x[i];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = __float_as_uint(a[2 * i]), v = __float_as_uint(a[2 * i + 1]);
            t[k][i] = __builtin_amdgcn_perm(v, u, 0x07060302);   // (upper half of v) << 16 | upper half of u
            if (k < 2) {
                a[2 * i] -= __uint_as_float(u & 0xffff0000u);
                a[2 * i + 1] -= __uint_as_float(v & 0xffff0000u);
            }
        }
    }
    return {__builtin_bit_cast(bf16x8, t[0]), __builtin_bit_cast(bf16x8, t[1]), __builtin_bit_cast(bf16x8, t[2])};
}
__device__ __forceinline__ bf16x8 join8(bf16x4 a, bf16x4 b) { return __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7); }

// e^x with x's digits beyond float32 kept
__device__ __forceinline__ float exp_d(double x) {
    const float h = (float)x, e = expf(h);
    return e + e * (float)(x - h);
}

// Where piece c (16 bytes) of row r of a tile with CPR pieces per row lies: c ^ spread<CPR>(r).  16 rows at the same c, and
// 4 rows at 4 neighbouring c, fall on different banks.
template <int CPR> __device__ __forceinline__ int spread(int r) {
    if constexpr (CPR >= 16) return ((r & 3) << 2) | ((r >> 2) & 3);
    else if constexpr (CPR == 8) return ((r & 2) << 1) | ((r >> 2) & 3);
    else if constexpr (CPR == 4) return (r >> 2) & 3;
    else return 0;
}

// 64 rows of CPR pieces from src (rows ld elements apart, last: the last row there is, n: real pieces per row) into LDS:
// piece j of CPR, one per 64 lanes.
template <int CPR> __device__ __forceinline__ void dma_tile(const uint16_t* src, int64_t ld, int last, int n, int j, uint32_t lds,
                                                            int lane) {
    const int i = j * 64 + lane, row = i / CPR, c = (i % CPR) ^ spread<CPR>(row);
    dma_1k(src + min(row, last) * ld + min(c, n - 1) * 8, __builtin_amdgcn_readfirstlane(lds + j * 1024));
}

enum { kScanPlain = 0, kScanMlstm = 1 };

// What the two forms read per token: plain: decay (one per token and head, or dts = 0: per head), qscale, kscale, vscale
// (any of the three may be absent); mlstm: the log decays, log write factors and e^-m of mlstm_gates_kernel.
struct ChunkScan {
    const uint16_t* proj;
    int ldp, q_off, k_off, v_off;
    const float *qscale, *kscale, *vscale, *decay;
    int dts;
    float q_mul;
    const float *la, *lb, *em;
    const int32_t *q_start, *pos0, *slots;
    const float* n0;   // [B, H, D]: the normaliser before the step (workgroups of one (sequence, head) start at any time)
    float *S, *n, *o;
    int B, HK, H, Dv;
};

template <int D> constexpr int chunk_scan_lds() {
    constexpr int NW = kCW;
    return 2 * kCH * (2 * D + 16 * NW) * 2 + 10 * 1024 + NW * (kCH * 16) + 10 * 16 * 4 + NW * kCH * 4;
}

template <int D, int MODE>
__global__ void __launch_bounds__(64 * kCW, 1) chunk_scan_kernel(const ChunkScan a) {
    constexpr int NW = kCW, CPR = D / 8, VC = 2 * NW, KK = D / 32;   // 16-byte pieces per row of q and k, of v; 32-row steps of the state
    constexpr int QB = kCH * D * 2, VB = kCH * VC * 16, BUF = 2 * QB + VB;
    extern __shared__ __attribute__((aligned(1024))) unsigned char cs_smem[];
    f32x4* const pt = reinterpret_cast<f32x4*>(cs_smem + 2 * BUF);                 // weight tiles, [10][64 lanes]
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ln = lane & 15, g = lane >> 4;
    unsigned char* const own = cs_smem + 2 * BUF + 10 * 1024 + wv * (kCH * 16);     // the wave's own copy of the scalars
    double* const Ls = reinterpret_cast<double*>(own);
    float* const ws = reinterpret_cast<float*>(own + kCH * 8);
    float* const cs = ws + kCH;
    float* const psum = reinterpret_cast<float*>(cs_smem + 2 * BUF + 10 * 1024 + NW * (kCH * 16));   // [10][16]
    float* const nq = psum + 160;                                                                    // [NW][64]
    // groups of workgroups that share q and k rows go to one XCD (workgroup i runs on XCD i % 8)
    const int nslab = (a.Dv + 16 * NW - 1) / (16 * NW), id = blockIdx.x >> 3;
    const int group = (id / nslab) * 8 + (blockIdx.x & 7), slab = id % nslab;
    if (group >= a.B * a.H) return;
    const int b = group / a.H, hd = group % a.H, hk = hd / (a.H / a.HK);
    const int t0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= t0) return;
    const int c0 = slab * 16 * NW, col = c0 + wv * 16 + ln;
    const bool live = col < a.Dv;
    const int64_t srow = (int64_t)a.slots[b] * a.H + hd;
    float* const Sp = a.S + srow * D * a.Dv + col;
    const bool fresh = a.pos0[b] == 0;
    // S[2 kk + h], element r of lane group g: row 32 kk + 8 g + 4 h + r (what the read-out's product takes from that lane)
    f32x4 S[2 * KK];
#pragma unroll
    for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) S[i][r] = !fresh && live ? Sp[(int64_t)((i >> 1) * 32 + 8 * g + 4 * (i & 1) + r) * a.Dv] : 0.f;
    // mlstm: the normaliser n likewise, the 32-row steps dealt to the waves (every column of the accumulator the same)
    constexpr int NO = MODE == kScanMlstm ? (KK + NW - 1) / NW : 1;
    f32x4 nst[2 * NO];
    if constexpr (MODE == kScanMlstm) {
#pragma unroll
        for (int i = 0; i < 2 * NO; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int kk = wv + NW * (i >> 1);
                nst[i][r] = kk < KK ? a.n0[(int64_t)group * D + kk * 32 + 8 * g + 4 * (i & 1) + r] : 0.f;
            }
    }
    const uint16_t* const qp = a.proj + a.q_off + (int64_t)hk * D;
    const uint16_t* const kp = a.proj + a.k_off + (int64_t)hk * D;
    const uint16_t* const vp = a.proj + a.v_off + (int64_t)hd * a.Dv + c0;
    const int vn = min(VC, (a.Dv - c0) / 8);
    const uint32_t lds0 = lds_offset(cs_smem);
    auto fetch = [&](int tb, int buf) {
        const int64_t at = (int64_t)tb * a.ldp;
        const int last = t1 - 1 - tb;
        const uint32_t dst = lds0 + buf * BUF;
        for (int j = wv; j < 2 * CPR + VC; j += NW) {
            if (j < CPR) dma_tile<CPR>(qp + at, a.ldp, last, CPR, j, dst, lane);
            else if (j < 2 * CPR) dma_tile<CPR>(kp + at, a.ldp, last, CPR, j - CPR, dst + QB, lane);
            else dma_tile<VC>(vp + at, a.ldp, last, vn, j - 2 * CPR, dst + 2 * QB, lane);
        }
    };
    // the scalars of token tb + lane, as loaded; past the range: nothing decays, nothing is written
    float sd = 1.f, sw = 0.f, sr = 0.f;
    const float fixed = MODE == kScanPlain && a.dts == 0 ? a.decay[hd] : 1.f;
    auto scalars = [&](int tb) {
        const int64_t t = min(tb + lane, t1 - 1);
        if constexpr (MODE == kScanMlstm) {
            sd = a.la[t * a.H + hd];
            sw = a.lb[t * a.H + hd];
            sr = a.em[t * a.H + hd];
        } else {
            sd = a.dts != 0 ? a.decay[t * a.dts + hd] : fixed;
            sw = a.kscale != nullptr ? a.kscale[t * a.HK + hk] : 1.f;
            if (a.vscale != nullptr) sw *= a.vscale[t * a.H + hd];
            sr = a.qscale != nullptr ? a.qscale[t * a.HK + hk] : a.q_mul;
        }
    };
    fetch(t0, 0);
    scalars(t0);
    for (int tb = t0, buf = 0; tb < t1; tb += kCH, buf ^= 1) {
        const int nt = min(kCH, t1 - tb);
        dma_wait();
        // ---- the chunk's scalars (before the next chunk's DMA is issued: what waits for them would wait for that, too)
        const bool valid = lane < nt;
        double L = 0.0;
        float w = 0.f;
        const float rd = sr;
        if (valid) {
            if constexpr (MODE == kScanMlstm) {
                L = sd;
                w = expf(sw);
            } else {
                const float lg = logf(sd);
                L = lg < -110.f ? -110.f : lg;   // e^-110 is 0 in float32, as a decay of 0 is
                w = sw;
            }
        }
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const double up = __shfl_up(L, o, 64);
            if (lane >= o) L += up;
        }
        const double LC = __shfl(L, 63, 64);
        Ls[lane] = L;
        ws[lane] = w;
        cs[lane] = exp_d(LC - L) * w;
        __builtin_amdgcn_wave_barrier();
        __syncthreads();   // this chunk's rows are in LDS; nobody reads the other buffer or the last chunk's weights any more
        if (tb + kCH < t1) {
            fetch(tb + kCH, buf ^ 1);
            scalars(tb + kCH);
        }
        const unsigned char* const qb = cs_smem + buf * BUF;
        const unsigned char* const kb = qb + QB;
        const unsigned char* const vb = kb + QB;
        // rows 16 i + ln of q or k, columns 32 kk + 8 g ..: either operand of a product over columns
        auto row8 = [&](const unsigned char* base, int i, int kk) {
            const int r = 16 * i + ln;
            return *reinterpret_cast<const bf16x8*>(base + r * (D * 2) + (((kk * 4 + g) ^ spread<CPR>(r)) * 16));
        };
        // k rows 32 p + 4 g + (0..3), 32 p + 16 + 4 g + (0..3), column 32 kk + 8 (ln / 4) + 4 h + ln % 4: the update's left operand
        auto kcol8 = [&](int p, int kk, int h) {
            const int r = 32 * p + 4 * g + (ln >> 2), c = ((kk * 4 + (ln & 3)) ^ spread<CPR>(r)) * 16 + h * 8;
            return join8(lds_read_tr4(kb + r * (D * 2) + c), lds_read_tr4(kb + (r + 16) * (D * 2) + c));   // (spread: period 16)
        };
        // ---- weights: tile p = (i, j) holds rows s = 16 j.. (4 g + r) and columns t = 16 i.. (ln)
        for (int p = wv; p < 10; p += NW) {
            const int i = p < 1 ? 0 : p < 3 ? 1 : p < 6 ? 2 : 3, j = p - i * (i + 1) / 2;
            if (16 * i >= nt) continue;
            f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
            for (int kk = 0; kk < KK; ++kk) acc[kk & 1] = mfma_16x16x32(row8(kb, j, kk), row8(qb, i, kk), acc[kk & 1]);
            const int t = 16 * i + ln;
            const double Lt = Ls[t];
            f32x4 v;
            float sum = 0.f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int s = 16 * j + 4 * g + r;
                v[r] = s <= t ? (acc[0][r] + acc[1][r]) * (ws[s] * exp_d(Lt - Ls[s])) : 0.f;
                sum += v[r];
            }
            pt[p * 64 + lane] = v;
            if constexpr (MODE == kScanMlstm) {
                sum += __shfl_xor(sum, 16, 64);
                sum += __shfl_xor(sum, 32, 64);
                if (g == 0) psum[p * 16 + ln] = sum;
            }
        }
        if constexpr (MODE == kScanMlstm) {   // n . q of the state before the chunk, this wave's rows
            f32x4 acc[4] = {};
#pragma unroll
            for (int u = 0; u < NO; ++u) {
                const int kk = wv + NW * u;
                if (kk < KK) {
                    const float x[8] = {nst[2 * u][0], nst[2 * u][1], nst[2 * u][2], nst[2 * u][3],
                                        nst[2 * u + 1][0], nst[2 * u + 1][1], nst[2 * u + 1][2], nst[2 * u + 1][3]};
                    const Terms n = split3(x);
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const bf16x8 q = row8(qb, i, kk);
                        acc[i] = mfma_16x16x32(q, n.h, mfma_16x16x32(q, n.m, mfma_16x16x32(q, n.l, acc[i])));
                    }
                }
            }
            if (ln == 0) {
#pragma unroll
                for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(nq + wv * kCH + 16 * i + 4 * g) = acc[i];
            }
        }
        __syncthreads();   // the weights are there
        const float eL = exp_d(L);
        float fr = rd;
        if constexpr (MODE == kScanMlstm) {
            const int i = lane >> 4, p0 = i * (i + 1) / 2;
            float intra = 0.f, inter = 0.f;
            for (int j = 0; j <= i; ++j) intra += psum[(p0 + j) * 16 + ln];
#pragma unroll
            for (int u = 0; u < NW; ++u) inter += nq[u * kCH + lane];
            fr = a.q_mul / (fmaxf(fabsf((intra + eL * inter) * a.q_mul), rd) + 1e-6f);
        }
        // ---- read-out: state before the chunk, then the chunk's own tokens
        Terms st[KK];
#pragma unroll
        for (int kk = 0; kk < KK; ++kk) {
            const float x[8] = {S[2 * kk][0], S[2 * kk][1], S[2 * kk][2], S[2 * kk][3],
                                S[2 * kk + 1][0], S[2 * kk + 1][1], S[2 * kk + 1][2], S[2 * kk + 1][3]};
            st[kk] = split3(x);
        }
        bf16x8 v[2];   // v rows 32 p + 4 g + (0..3), 32 p + 16 + 4 g + (0..3) of this lane's column
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            const int r = 32 * p + 4 * g + (ln >> 2), c = ((wv * 2 + ((ln & 3) >> 1)) ^ spread<VC>(r)) * 16 + (ln & 1) * 8;
            v[p] = join8(lds_read_tr4(vb + r * (VC * 16) + c), lds_read_tr4(vb + (r + 16) * (VC * 16) + c));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (16 * i < nt) {
                f32x4 ah = {0.f, 0.f, 0.f, 0.f}, am = ah, al = ah;
#pragma unroll
                for (int kk = 0; kk < KK; ++kk) {
                    const bf16x8 q = row8(qb, i, kk);
                    ah = mfma_16x16x32(q, st[kk].h, ah);
                    am = mfma_16x16x32(q, st[kk].m, am);
                    al = mfma_16x16x32(q, st[kk].l, al);
                }
                f32x4 acc;
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[r] = (ah[r] + (am[r] + al[r])) * __shfl(eL, 16 * i + 4 * g + r, 64);
#pragma unroll
                for (int p = 0; p <= i / 2; ++p) {
                    const f32x4 x0 = pt[(i * (i + 1) / 2 + 2 * p) * 64 + lane];
                    f32x4 x1 = {0.f, 0.f, 0.f, 0.f};
                    if (2 * p + 1 <= i) x1 = pt[(i * (i + 1) / 2 + 2 * p + 1) * 64 + lane];
                    const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                    const Terms w3 = split3(x);
                    acc = mfma_16x16x32(w3.h, v[p], mfma_16x16x32(w3.m, v[p], mfma_16x16x32(w3.l, v[p], acc)));
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = 16 * i + 4 * g + r;
                    const float f = __shfl(fr, t, 64);
                    if (t < nt && live) a.o[((int64_t)(tb + t) * a.H + hd) * a.Dv + col] = acc[r] * f;
                }
            }
        }
        // ---- the state after the chunk
        const float eC = exp_d(LC);
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i) S[i] *= eC;
        if constexpr (MODE == kScanMlstm) {
#pragma unroll
            for (int i = 0; i < 2 * NO; ++i) nst[i] *= eC;
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (32 * p >= nt) break;
            const f32x4 f0 = *reinterpret_cast<const f32x4*>(cs + 32 * p + 4 * g);
            const f32x4 f1 = *reinterpret_cast<const f32x4*>(cs + 32 * p + 16 + 4 * g);
            const float f[8] = {f0[0], f0[1], f0[2], f0[3], f1[0], f1[1], f1[2], f1[3]};
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = f[e] * (float)v[p][e];
            const Terms u = split3(x);
            Terms un;
            if constexpr (MODE == kScanMlstm) un = split3(f);
#pragma unroll
            for (int kk = 0; kk < KK; ++kk)
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const bf16x8 kc = kcol8(p, kk, h);
                    f32x4& s = S[2 * kk + h];
                    s = mfma_16x16x32(kc, u.h, mfma_16x16x32(kc, u.m, mfma_16x16x32(kc, u.l, s)));
                    if constexpr (MODE == kScanMlstm) {
                        if (kk % NW == wv) {
                            f32x4& nn = nst[2 * (kk / NW) + h];
                            nn = mfma_16x16x32(kc, un.h, mfma_16x16x32(kc, un.m, mfma_16x16x32(kc, un.l, nn)));
                        }
                    }
                }
        }
    }
    if (live) {
#pragma unroll
        for (int i = 0; i < 2 * KK; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) Sp[(int64_t)((i >> 1) * 32 + 8 * g + 4 * (i & 1) + r) * a.Dv] = S[i][r];
    }
    if constexpr (MODE == kScanMlstm) {
        if (slab == 0 && ln == 0) {
#pragma unroll
            for (int i = 0; i < 2 * NO; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int kk = wv + NW * (i >> 1);
                    if (kk < KK) a.n[srow * D + kk * 32 + 8 * g + 4 * (i & 1) + r] = nst[i][r];
                }
        }
    }
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

// When the chunked form serves a launch: bfloat16 rows of q, k and v on 16-byte boundaries, a state of 32, 64, 128 or 256
// rows, and a sequence with at least 16 new tokens (longest: the most that any sequence brings).  A chunk costs the same
// whether it is full or not, the token-by-token kernels cost per token: 32 sequences of n tokens take (token by token /
// chunked, us) 9.9 / 16.5 at n = 4, 11.7 / 16.4 at 8, 15.9 / 16.1 at 16, 71.5 / 39.3 at 117 (8 heads of 128 x 128, fixed
// decays), and 50 / 68, 61 / 67, 85 / 67, 444 / 144 (mlstm, 4 heads of 256 x 512).
bool hy_chunk_scan_ok(const void* proj, int ldp, int q_off, int k_off, int v_off, int D, int Dv, int longest) {
    return longest >= 16 && (D == 32 || D == 64 || D == 128 || D == 256) && Dv % 8 == 0 && ((uintptr_t)proj & 15) == 0 &&
           ((ldp | q_off | k_off | v_off) & 7) == 0;
}

template <int D, int MODE>
static void chunk_scan_run(const hy::ChunkScan& a, hipStream_t s) {
    constexpr int lds = hy::chunk_scan_lds<D>();
    static_assert(lds <= 160 * 1024, "LDS of one workgroup");
    const auto kern = hy::chunk_scan_kernel<D, MODE>;
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    const int nslab = (a.Dv + 16 * hy::kCW - 1) / (16 * hy::kCW);
    kern<<<(a.B * a.H + 7) / 8 * 8 * nslab, 64 * hy::kCW, lds, s>>>(a);
}

template <int MODE>
static void chunk_scan_d(int D, const hy::ChunkScan& a, hipStream_t s) {
    if (D == 32) chunk_scan_run<32, MODE>(a, s);
    else if (D == 64) chunk_scan_run<64, MODE>(a, s);
    else if (D == 128) chunk_scan_run<128, MODE>(a, s);
    else chunk_scan_run<256, MODE>(a, s);
}

// One decay per head and token (dts = H) or per head (dts = 0), no delta correction; see launch_hy_linear_scan.
void launch_hy_chunk_scan(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, const float* qscale, const float* kscale,
                          float q_mul, const float* decay, int dts, const int32_t* q_start, const int32_t* pos0,
                          const int32_t* slots, float* S, float* o, int B, int HK, int H, int D, int Dv, const float* vscale,
                          hipStream_t s) {
    hy::ChunkScan a{proj, ldp, q_off, k_off, v_off, qscale, kscale, vscale, decay, dts, q_mul, nullptr, nullptr, nullptr,
                    q_start, pos0, slots, nullptr, S, nullptr, o, B, HK, H, Dv};
    chunk_scan_d<hy::kScanPlain>(D, a, s);
}

// scratch: 3 T H + B H D floats
void launch_hy_chunk_mlstm(const uint16_t* proj, int ldp, const float* gate_pre, const int32_t* q_start, const int32_t* pos0,
                           const int32_t* slots, float* S, float* n, float* m, float* scratch, float* o, int T, int B, int H,
                           int D, int Dv, float cap, hipStream_t s) {
    const int64_t th = (int64_t)T * H;
    float *la = scratch, *lb = la + th, *em = lb + th, *n0 = em + th;
    hy::mlstm_gates_kernel<<<dim3(B, H), 256, 0, s>>>(gate_pre, q_start, pos0, slots, n, m, n0, la, lb, em, H, D, cap);
    hy::ChunkScan a{proj, ldp, 0, H * D, 2 * H * D, nullptr, nullptr, nullptr, nullptr, H, 1.f / sqrtf((float)D), la, lb, em,
                    q_start, pos0, slots, n0, S, n, o, B, H, H, Dv};
    chunk_scan_d<hy::kScanMlstm>(D, a, s);
}

}  // namespace chronos
