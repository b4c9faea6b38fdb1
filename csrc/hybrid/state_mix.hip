// state_mix.hip — the recurrent mixers of decode rows between their two projections in one launch: preparation, state step (state_step.hip), and
// the read-out's norm and gate.  bfloat16 rows, one token per sequence; a longer range is walked token by token, so the launch's hint need not
// be true.
//
//   delta    q, k, v pass the short convolution (4 taps, SiLU) over the sequence's history, which is moved on; q and k are scaled to unit
//            length; decay exp(-exp(A) softplus(a)), write strength sigmoid(b); the delta rule
//   rows     decay of every state row sigmoid(b + low W)^p
//   gates    matrix memory: input and forget gates, running maximum, normaliser n and denominator (mlstm.hip)
//   then     y = o / rms(o) * w * gate,  gate = silu(g) or sigmoid(g)
//
// A workgroup holds whole heads (of the delta rule the HPW value heads of one key head: they share its history, which one of them alone could
// not rewrite while the others read it), the layout of state_step.hip with all columns of a head in one workgroup.  What was
// 3 or 4 launches, each a few us of latency between a product and the next, is one; the state's bytes bound many rows as before.
// us, launches -> one: delta rule, 8 heads of 128 by 128, 1 and 64 sequences 13.0 -> 7.7, 23.1 -> 14.1, 32 heads 18.5 -> 7.9, 63.3 -> 60.6; rows, 4 heads of
// 128 by 256 8.6 -> 6.8, 18.4 -> 12.8, 16 heads 9.2 -> 6.9, 57.1 -> 56.6; gates, 4 heads of 128 by 256 10.7 -> 6.9, 18.6 -> 12.1.
#include "hybrid_common.h"

#include <type_traits>

namespace chronos {
namespace hy {

enum { kMixDelta = 0, kMixRows = 1, kMixGates = 2 };

struct StateMix {
    const uint16_t* proj;
    int ldp, q_off, k_off, v_off, g_off;
    const int32_t *q_start, *pos0, *slots;
    float* S;
    uint16_t* y;
    const float* w;
    float eps, q_mul;
    int HK, H, Dv, silu;
    const float *taps, *ab, *a_log;   // delta: taps [C, 4] of the columns q_off .. , pre-activations [T, 2H], [H]
    uint16_t* hist;                   // [slots, 3, C]
    int C;
    const float *low, *w2, *b2;       // rows: [T, R], [R, H D], [H D]
    int R;
    float p;
    const float* gate_pre;            // gates: [T, 2H]
    float *n, *m, cap;                // [slots, H, D], [slots, H]
};

constexpr int mix_threads(int D) { return D >= 128 ? 2 * D : 256; }

// ONCE: the states are read and written as data used once (nt).  (A template: of two branches the compiler makes one again and drops the mark.)
template <int D, int CL, int HPW, int FORM, bool ONCE>
__global__ void __launch_bounds__(HPW * mix_threads(D)) state_mix_kernel(const StateMix a) {
    constexpr int NT = mix_threads(D), NW = NT / 64, RI = 64 / CL, NI = D / (NW * RI);
    constexpr bool ROWS = FORM == kMixRows, DELTA = FORM == kMixDelta, GATES = FORM == kMixGates;
    static_assert(NW * RI * NI == D && (HPW == 1 || DELTA) && 2 * D <= HPW * NT && D % 64 == 0, "every wave its rows");
    __shared__ float qs[D], ks[D], ds[ROWS ? D : 1], red[2 * D / 64];
    __shared__ __attribute__((aligned(16))) f32x4 part[HPW][NW][CL];
    const int b = blockIdx.x, hk = blockIdx.y, sub = threadIdx.x / NT, tid = threadIdx.x % NT, hd = hk * HPW + sub;
    const int t0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= t0) return;
    const int lane = tid & 63, wv = tid >> 6, cl = lane % CL, rl = lane / CL, col = cl * 4;
    const bool live = col < a.Dv, fresh = a.pos0[b] == 0, past = a.pos0[b] > 0;
    const int row0 = wv * (NI * RI) + rl, slot = a.slots[b];
    float* const Sp = a.S + (((int64_t)slot * a.H + hd) * D + row0) * a.Dv + col;
    f32x4 S[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const f32x4* const p = reinterpret_cast<const f32x4*>(Sp + (int64_t)(RI * i) * a.Dv);
        S[i] = !live || fresh ? f32x4{0.f, 0.f, 0.f, 0.f} : ONCE ? __builtin_nontemporal_load(p) : *p;
    }
    f32x4 wn = {0.f, 0.f, 0.f, 0.f};
    if (live) wn = *reinterpret_cast<const f32x4*>(a.w + (int64_t)hd * a.Dv + col);
    // this thread's row of q or k (delta: q rows, then k rows), and what it keeps between tokens
    const int r = threadIdx.x;
    const int qc = DELTA ? (r < D ? a.q_off + hk * D + r : a.k_off + hk * D + r - D) : 0;
    uint16_t* const hrow = DELTA ? a.hist + (int64_t)slot * 3 * a.C - a.q_off : nullptr;   // (by column of proj)
    uint16_t qin[4];
    u16x4 vin[4];
    float nr = 0.f, mr = 0.f;
    float* const np = GATES ? a.n + ((int64_t)slot * a.H + hd) * D + r : nullptr;
    if constexpr (GATES) {
        if (!fresh && r < D) nr = *np;
        if (!fresh) mr = a.m[(int64_t)slot * a.H + hd];
    }
    auto total = [&](f32x4 x) {   // the sum over all rows of this lane's columns, in every lane
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = across_sum<CL>(x[e]);
        if (rl == 0) part[sub][wv][cl] = x;
        __syncthreads();
        x = part[sub][0][cl];
#pragma unroll
        for (int i = 1; i < NW; ++i) x += part[sub][i][cl];
        return x;
    };
    auto step = [&](int t) {
        const uint16_t* const p = a.proj + (int64_t)t * a.ldp;
        float g = 1.f, w = 1.f, rd = a.q_mul, bt = 1.f;
        f32x4 u = {0.f, 0.f, 0.f, 0.f}, gv = u;
        if (live) {
            const u16x4 gq = *reinterpret_cast<const u16x4*>(p + a.g_off + (int64_t)hd * a.Dv + col);
            gv = f32x4{bf2f(gq[0]), bf2f(gq[1]), bf2f(gq[2]), bf2f(gq[3])};
        }
        if constexpr (DELTA) {
            // inputs 3 tokens back to this one: this range's, or the history's
            const int vc = a.v_off + hd * a.Dv + col;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int s = t - 3 + i;
                const bool here = s >= t0;
                const uint16_t* const src = here ? a.proj + (int64_t)s * a.ldp : hrow + (int64_t)(3 + s - t0) * a.C;
                qin[i] = r < 2 * D && (here || past) ? src[qc] : (uint16_t)0;
                vin[i] = live && (here || past) ? *reinterpret_cast<const u16x4*>(src + vc) : u16x4{0, 0, 0, 0};
            }
            if (r < 2 * D) {
                const f32x4 tp = *reinterpret_cast<const f32x4*>(a.taps + (int64_t)(qc - a.q_off) * 4);
                float z = 0.f;
#pragma unroll
                for (int i = 0; i < 4; ++i) z += tp[i] * bf2f(qin[i]);
                z *= sigmoid_act<uint16_t>(z);
                (r < D ? qs : ks)[r < D ? r : r - D] = z;
                const float ss = wave_sum(z * z);
                if ((r & 63) == 0) red[r >> 6] = ss;
            }
            if (live) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const f32x4 tp = *reinterpret_cast<const f32x4*>(a.taps + (int64_t)(vc - a.q_off + e) * 4);
                    float z = 0.f;
#pragma unroll
                    for (int i = 0; i < 4; ++i) z += tp[i] * bf2f(vin[i][e]);
                    u[e] = z * sigmoid_act<uint16_t>(z);
                }
            }
            const float av = a.ab[(int64_t)t * 2 * a.H + hd], bv = a.ab[(int64_t)t * 2 * a.H + a.H + hd];
            g = expf(-expf(a.a_log[hd]) * (av > 20.f ? av : log1pf(expf(av))));
            bt = sigmoidf_(bv);
            __syncthreads();
            float sq = 0.f, sk = 0.f;
#pragma unroll
            for (int i = 0; i < D / 64; ++i) {
                sq += red[i];
                sk += red[D / 64 + i];
            }
            rd = a.q_mul / sqrtf(sq + 1e-6f);
            w = 1.f / sqrtf(sk + 1e-6f);
        } else {
            if (live) {
                const u16x4 v = *reinterpret_cast<const u16x4*>(p + a.v_off + (int64_t)hd * a.Dv + col);
                u = f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
            }
            float qv = 0.f, kv = 0.f;
            if (r < D) {
                qs[r] = qv = bf2f(p[a.q_off + hk * D + r]);
                ks[r] = kv = bf2f(p[a.k_off + hk * D + r]);
                if constexpr (ROWS) {
                    const int c = hd * D + r;
                    float z = a.b2[c];
#pragma unroll 4
                    for (int j = 0; j < a.R; ++j) z += a.low[(int64_t)t * a.R + j] * a.w2[(int64_t)j * a.H * D + c];
                    ds[r] = expf(logsigmoidf_(z) * a.p);
                }
            }
            if constexpr (GATES) {
                const float zi = a.gate_pre[(int64_t)t * 2 * a.H + hd], zf = a.gate_pre[(int64_t)t * 2 * a.H + a.H + hd];
                const float ig = a.cap * tanhf(zi / a.cap), fg = logsigmoidf_(a.cap * tanhf(zf / a.cap));
                const float mn = fmaxf(fg + mr, ig);
                g = expf(fg + mr - mn);
                w = expf(ig - mn);
                mr = mn;
                nr = g * nr + w * kv;
                if (r < D) {
                    const float ss = wave_sum(nr * (qv * a.q_mul));
                    if ((r & 63) == 0) red[r >> 6] = ss;
                }
            }
            __syncthreads();
            if constexpr (GATES) {
                float dot = 0.f;
#pragma unroll
                for (int i = 0; i < D / 64; ++i) dot += red[i];
                rd = a.q_mul / (fmaxf(fabsf(dot), expf(-mr)) + 1e-6f);
            }
        }
#pragma unroll
        for (int i = 0; i < NI; ++i) S[i] *= ROWS ? ds[row0 + RI * i] : g;
        if constexpr (DELTA) {
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < NI; ++i) x += S[i] * ks[row0 + RI * i];
            u = (u - total(x) * w) * bt;
            __syncthreads();   // part is read
        }
        u *= w;
        f32x4 x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            S[i] += u * ks[row0 + RI * i];
            x[i & 1] += S[i] * qs[row0 + RI * i];
        }
        if (live && t + 1 == t1)
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                f32x4* const p = reinterpret_cast<f32x4*>(Sp + (int64_t)(RI * i) * a.Dv);
                if constexpr (ONCE) __builtin_nontemporal_store(S[i], p);
                else *p = S[i];
            }
        const f32x4 o = total(x[0] + x[1]) * rd;
        // the head's norm and gate: a row's columns lie over CL lanes (dead ones hold 0)
        float ss = o[0] * o[0] + o[1] * o[1] + o[2] * o[2] + o[3] * o[3];
        ss = group_sum(ss, CL);
        const float inv = 1.f / sqrtf(ss / (float)a.Dv + a.eps);
        if (wv == 0 && rl == 0 && live) {
            u16x4 out;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float sg = sigmoid_act<uint16_t>(gv[e]);
                out[e] = f2bf(o[e] * inv * wn[e] * (a.silu ? gv[e] * sg : sg));
            }
            *reinterpret_cast<u16x4*>(a.y + ((int64_t)t * a.H + hd) * a.Dv + col) = out;
        }
    };
    step(t0);
    for (int t = t0 + 1; t < t1; ++t) {   // ranges longer than the launch was told
        __syncthreads();                  // the last token's LDS is read
        step(t);
    }
    // (all waves have used the history that they read: their sums in the last exchange depend on it)
    if constexpr (DELTA) {
        if (r < 2 * D)
#pragma unroll
            for (int i = 0; i < 3; ++i) hrow[(int64_t)i * a.C + qc] = qin[i + 1];
        if (wv == 0 && rl == 0 && live)
#pragma unroll
            for (int i = 0; i < 3; ++i) *reinterpret_cast<u16x4*>(hrow + (int64_t)i * a.C + a.v_off + hd * a.Dv + col) = vin[i + 1];
    }
    if constexpr (GATES) {
        if (r < D) *np = nr;
        if (r == 0) a.m[(int64_t)slot * a.H + hd] = mr;
    }
}

}  // namespace hy

// Heads of 64, 128 or 256 rows by up to 256 columns in fours; of the delta rule one or two value heads per key head.  Offsets and rows in fours
// (8-byte loads), the state, taps and weights on 16 bytes.
bool hy_state_mix_ok(int D, int Dv, int heads_per_key) {
    return (D == 64 || D == 128 || D == 256) && Dv % 4 == 0 && Dv >= 4 && Dv <= 256 && (heads_per_key == 1 || (heads_per_key == 2 && D <= 128));
}

template <int D, int HPW, int FORM, bool ONCE>
static void state_mix_cols(const hy::StateMix& a, int B, hipStream_t s) {
    const dim3 grid(B, a.HK);
    constexpr int nt = HPW * hy::mix_threads(D);
    if (a.Dv <= 64) hy::state_mix_kernel<D, 16, HPW, FORM, ONCE><<<grid, nt, 0, s>>>(a);
    else if (a.Dv <= 128) hy::state_mix_kernel<D, 32, HPW, FORM, ONCE><<<grid, nt, 0, s>>>(a);
    else hy::state_mix_kernel<D, 64, HPW, FORM, ONCE><<<grid, nt, 0, s>>>(a);
}
template <int HPW, int FORM>
static void state_mix(const hy::StateMix& a, int B, int D, hipStream_t s) {
    if (B == 0) return;
    // states beyond an L2; smaller ones are found there again at the next step: a decode step of four layers, us, 64 rows of 16 heads (134 MB in two
    // layers) 758 -> 714, 11 rows (6 MB) 175 -> 171; but 6 rows (3 MB) 169 -> 171, one row 154.6 -> 157.5
    const bool once = (int64_t)B * a.H * D * a.Dv * 4 >= 4 << 20;
    auto cols = [&](auto DC) {
        once ? state_mix_cols<decltype(DC)::value, HPW, FORM, true>(a, B, s) : state_mix_cols<decltype(DC)::value, HPW, FORM, false>(a, B, s);
    };
    if (D == 64) cols(std::integral_constant<int, 64>{});
    else if (D == 128) cols(std::integral_constant<int, 128>{});
    else if constexpr (HPW == 1) cols(std::integral_constant<int, 256>{});
}

void launch_hy_delta_step(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, int g_off, const float* taps, const float* ab, const float* a_log,
                          const int32_t* q_start, const int32_t* pos0, const int32_t* slots, uint16_t* hist, int C, float* S, const float* w, uint16_t* y,
                          int B, int HK, int H, int D, int Dv, float q_mul, float eps, hipStream_t s) {
    hy::StateMix a{};
    a.proj = proj, a.ldp = ldp, a.q_off = q_off, a.k_off = k_off, a.v_off = v_off, a.g_off = g_off;
    a.q_start = q_start, a.pos0 = pos0, a.slots = slots, a.S = S, a.y = y, a.w = w, a.eps = eps, a.q_mul = q_mul;
    a.HK = HK, a.H = H, a.Dv = Dv, a.silu = 1;
    a.taps = taps, a.ab = ab, a.a_log = a_log, a.hist = hist, a.C = C;
    if (H == HK) state_mix<1, hy::kMixDelta>(a, B, D, s);
    else state_mix<2, hy::kMixDelta>(a, B, D, s);
}

void launch_hy_rows_step(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, int g_off, const float* low, const float* w2, const float* b2,
                         int R, float p, const int32_t* q_start, const int32_t* pos0, const int32_t* slots, float* S, const float* w, uint16_t* y, int B,
                         int H, int D, int Dv, float q_mul, float eps, hipStream_t s) {
    hy::StateMix a{};
    a.proj = proj, a.ldp = ldp, a.q_off = q_off, a.k_off = k_off, a.v_off = v_off, a.g_off = g_off;
    a.q_start = q_start, a.pos0 = pos0, a.slots = slots, a.S = S, a.y = y, a.w = w, a.eps = eps, a.q_mul = q_mul;
    a.HK = H, a.H = H, a.Dv = Dv, a.silu = 1;
    a.low = low, a.w2 = w2, a.b2 = b2, a.R = R, a.p = p;
    state_mix<1, hy::kMixRows>(a, B, D, s);
}

void launch_hy_mlstm_step(const uint16_t* proj, int ldp, int g_off, const float* gate_pre, const int32_t* q_start, const int32_t* pos0,
                          const int32_t* slots, float* S, float* n, float* m, const float* w, uint16_t* y, int B, int H, int D, int Dv, float cap,
                          float eps, hipStream_t s) {
    hy::StateMix a{};
    a.proj = proj, a.ldp = ldp, a.q_off = 0, a.k_off = H * D, a.v_off = 2 * H * D, a.g_off = g_off;
    a.q_start = q_start, a.pos0 = pos0, a.slots = slots, a.S = S, a.y = y, a.w = w, a.eps = eps, a.q_mul = 1.f / sqrtf((float)D);
    a.HK = H, a.H = H, a.Dv = Dv, a.silu = 0;
    a.gate_pre = gate_pre, a.n = n, a.m = m, a.cap = cap;
    state_mix<1, hy::kMixGates>(a, B, D, s);
}

}  // namespace chronos
