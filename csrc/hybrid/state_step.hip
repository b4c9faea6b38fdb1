// state_step.hip — the recurrences of linear_scan.hip and mlstm.hip for one token per sequence (decode): the state is read once,
// stepped and written once, bfloat16 rows.  A longer range is walked token by token, so the launch's hint need not be true.
//
//     plain:   S <- d S + k (w v),  o = r q^T S          d: one decay per head (fixed or per token) or per state row
//     delta:   u = beta (v - w k^T (d S)),  S <- d S + k (w u),  o = r q^T S
//     mlstm:   S <- a S + k (b v),  o = q^T S / den      (a, b, den of the gate kernel)
//
// What bounds it is the state's traffic, so a lane takes 16 bytes of a row: CL lanes a row's 4 CL columns, 64 / CL rows per
// instruction.  A workgroup of 4 waves (8 for 256 rows) holds all rows of its columns in registers, every load in flight at once.
//  q and k are handed to the lanes through LDS, sums over rows go over the lanes of a column, then over the waves.
// Measured, 64 sequences, 8 heads of 256 x 512 float32 (537 MB read and written): a lane per column took 157 us, this 92; one sequence: 16.9 and
// 10.5 us with the gate kernel; delta rule, 16 sequences, 32 heads of 128 x 128: 13.7 and 10.8.
// The state is read and written as data used once (nt).  Eight layers' states in turn, us, plain, reads alone marked, writes alone, both: 64 sequences
// 116, 112, 120, 107 (5.0 TB/s); 16 28.9, 24.2, 29.9, 22.9; 4 9.8, 9.4, 9.8, 7.9; one 5.7, 5.8, 5.6, 5.4; heads of 32 x 64 and 64 x 64 level.  (One
// state stepped over and over, which no decoder does, finds half of itself in the memory-side cache unmarked: 84, marked 106.)  More is gained by
// what stays cached beside it: in a decode step of 64 rows, two of four layers so, the kernel takes 106 us for 100 and the latent attention behind it
// 52 for 71; the step 878 for 913 (reads alone 901, writes alone 907), 32 rows 650 for 683, 16 rows and fewer level.
#include "hybrid_common.h"

namespace chronos {
namespace hy {

struct StateStep {
    const uint16_t* proj;
    int ldp, q_off, k_off, v_off;
    const float *qscale, *kscale, *vscale, *decay, *beta;   // as in linear_scan.hip; mlstm: vscale = b, decay = a
    const float* den;                                       // mlstm [T, H]
    float q_mul;
    int dts;                                                // decays per token (0: the same for every token)
    const int32_t *q_start, *pos0, *slots;
    float *S, *o;
    int HK, H, Dv;
};

// The waves share the D rows; NI: instructions (16 bytes each) per lane
template <int D, int CL, bool ROWS, bool DELTA>
__global__ void __launch_bounds__(D >= 128 ? 2 * D : 256) state_step_kernel(const StateStep a) {
    constexpr int NT = D >= 128 ? 2 * D : 256, NW = NT / 64;         // threads, waves
    constexpr int RI = 64 / CL, NI = D / (NW * RI);   // rows per instruction, instructions per lane
    static_assert(NW * RI * NI == D, "every wave its rows");
    __shared__ float qs[D], ks[D], ds[ROWS ? D : 1];
    __shared__ __attribute__((aligned(16))) f32x4 part[NW][CL];
    const int b = blockIdx.x, hd = blockIdx.y, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int t0 = a.q_start[b], t1 = a.q_start[b + 1];
    if (t1 <= t0) return;
    const int cl = lane % CL, rl = lane / CL, col = (blockIdx.z * CL + cl) * 4, hk = hd / (a.H / a.HK);
    const bool live = col < a.Dv, fresh = a.pos0[b] == 0;
    const int row0 = wv * (NI * RI) + rl;                            // this lane's rows: row0 + RI i
    float* const Sp = a.S + (((int64_t)a.slots[b] * a.H + hd) * D + row0) * a.Dv + col;
    f32x4 S[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
        S[i] = live && !fresh ? __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(Sp + (int64_t)(RI * i) * a.Dv)) : f32x4{0.f, 0.f, 0.f, 0.f};
    auto total = [&](f32x4 x) {   // the sum over all rows of this lane's columns, in every lane
#pragma unroll
        for (int e = 0; e < 4; ++e) x[e] = across_sum<CL>(x[e]);
        if (rl == 0) part[wv][cl] = x;
        __syncthreads();
        x = part[0][cl];
#pragma unroll
        for (int i = 1; i < NW; ++i) x += part[i][cl];
        return x;
    };
    auto step = [&](int t) {
        const uint16_t* const p = a.proj + (int64_t)t * a.ldp;
        for (int r = threadIdx.x; r < D; r += NT) {
            qs[r] = bf2f(p[a.q_off + hk * D + r]);
            ks[r] = bf2f(p[a.k_off + hk * D + r]);
            if constexpr (ROWS) ds[r] = a.decay[((int64_t)t * a.H + hd) * D + r];
        }
        const float g = ROWS ? 1.f : a.decay[(int64_t)t * a.dts + hd];
        float w = a.kscale != nullptr ? a.kscale[(int64_t)t * a.HK + hk] : 1.f;
        if (a.vscale != nullptr) w *= a.vscale[(int64_t)t * a.H + hd];
        float r = a.qscale != nullptr ? a.qscale[(int64_t)t * a.HK + hk] : a.q_mul;
        if (a.den != nullptr) r /= a.den[(int64_t)t * a.H + hd];
        const float bt = DELTA ? a.beta[(int64_t)t * a.H + hd] : 1.f;
        f32x4 u = {0.f, 0.f, 0.f, 0.f};
        if (live) {
            const u16x4 v = *reinterpret_cast<const u16x4*>(p + a.v_off + (int64_t)hd * a.Dv + col);
            u = f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
        }
        __syncthreads();
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
            for (int i = 0; i < NI; ++i) __builtin_nontemporal_store(S[i], reinterpret_cast<f32x4*>(Sp + (int64_t)(RI * i) * a.Dv));
        const f32x4 y = total(x[0] + x[1]) * r;
        if (wv == 0 && rl == 0 && live) *reinterpret_cast<f32x4*>(a.o + ((int64_t)t * a.H + hd) * a.Dv + col) = y;
    };
    step(t0);   // (apart from the loop: in front of one the compiler waits for the whole state)
    for (int t = t0 + 1; t < t1; ++t) step(t);   // ranges longer than the launch was told
}

}  // namespace hy

// bfloat16 rows, one token per sequence (longest: the most that any sequence brings, as far as the caller knows), a state of 32, 64,
// 128 or 256 rows of a multiple of 4 columns, v on 8-byte and the state and o on 16-byte boundaries
bool hy_state_step_ok(const void* proj, const void* S, const void* o, int ldp, int v_off, int D, int Dv, int longest) {
    return longest == 1 && (D == 32 || D == 64 || D == 128 || D == 256) && Dv % 4 == 0 && (reinterpret_cast<uintptr_t>(proj) & 7) == 0 &&
           ((ldp | v_off) & 3) == 0 && hy::aligned16(S, o);
}

template <int D, int CL>
static void state_step_run(const hy::StateStep& a, bool rows, int B, hipStream_t s) {
    const dim3 grid(B, a.H, (a.Dv + 4 * CL - 1) / (4 * CL));
    constexpr int nt = D >= 128 ? 2 * D : 256;
    if (a.beta != nullptr) {
        if (rows) hy::state_step_kernel<D, CL, true, true><<<grid, nt, 0, s>>>(a);
        else hy::state_step_kernel<D, CL, false, true><<<grid, nt, 0, s>>>(a);
    } else {
        if (rows) hy::state_step_kernel<D, CL, true, false><<<grid, nt, 0, s>>>(a);
        else hy::state_step_kernel<D, CL, false, false><<<grid, nt, 0, s>>>(a);
    }
}

// rows: decay [T, H, D]; else per head (dts = H) or fixed (dts = 0).  den != nullptr: mlstm (vscale = b, decay = a).
void launch_hy_state_step(const uint16_t* proj, int ldp, int q_off, int k_off, int v_off, const float* qscale, const float* kscale,
                          float q_mul, const float* decay, bool rows, int dts, const float* beta, const float* den,
                          const int32_t* q_start, const int32_t* pos0, const int32_t* slots, float* S, float* o, int B, int HK, int H,
                          int D, int Dv, const float* vscale, hipStream_t s) {
    const hy::StateStep a{proj, ldp, q_off, k_off, v_off, qscale, kscale, vscale, decay, beta, den, q_mul, dts, q_start, pos0, slots, S, o, HK, H, Dv};
    // 256 columns per workgroup where that gives every CU one, else 64
    const bool many = (int64_t)B * H * ((Dv + 255) / 256) >= 256;
#define HY_STEP(DD)                                                  \
    do {                                                             \
        if (many && Dv > 128) state_step_run<DD, 64>(a, rows, B, s); \
        else if (many && Dv > 64) state_step_run<DD, 32>(a, rows, B, s); \
        else state_step_run<DD, 16>(a, rows, B, s);                  \
    } while (0)
    if (D == 32) HY_STEP(32);
    else if (D == 64) HY_STEP(64);
    else if (D == 128) HY_STEP(128);
    else HY_STEP(256);
#undef HY_STEP
}

}  // namespace chronos
