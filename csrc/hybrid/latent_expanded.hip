// latent_expanded.hip — latent attention of whole prompts with the keys and values written out, bfloat16 on the matrix cores.
//
// A prompt step whose sequences all start at position 0 has every key's latent among its own tokens.  Then one product
// c W_kv^T [T, H (D + Dv)] gives each head its keys and values, at exactly the cost of carrying the queries into the latent
// space and the output back, and attention runs over D + R and Dv columns per head and not over rank + R and rank
// (128 + 64 and 128 against 576 and 512: 320 multiplications per score against 1088).  The cached rows are the same.
//
// A workgroup takes 32 NW query rows of one (sequence, head), 32 per wave, and walks the keys 64 at a time:
//   * a tile's keys ([k | shared rotated part], from two arrays) and values go from memory straight into LDS, two tiles deep;
//     rows end in a 16-byte pad, so that 16 rows at one column fall on different banks;
//   * scores S^T = K Q^T and sum O^T = V^T P^T as in latent_attention_mfma.hip: a lane holds 4 keys of one query row, its
//     weights are the sum's right operand as they stand, the values are read by transposing LDS reads.  Each key and value
//     operand serves the wave's two sets of 16 rows: with one set per wave the LDS reads take twice the matrix cores' time;
//   * masks only where a tile reaches past a row's own position (or a window's edge); waves skip tiles they do not see.
// blockIdx.x is the (sequence, head): where their number is a multiple of 8 the workgroups of one run on one XCD and share its L2, else they
// are dealt over the XCDs; the longest walks start first.
//
// What bounds it: per tile and wave 80 matrix instructions of 16 cycles (D + R = 192, Dv = 128) beside about 1000 cycles of
// softmax on the vector ALUs, two waves per SIMD.  Measured, 4 sequences of 2048 tokens, 16 heads of 128 + 64 and 128, rank 512: through
// the latents 557 us and 121 for the two products around it; this 136 (640 TFLOP/s) and 47 for the product in front.
//
// Precision: through the latents the query in latent space and the weighted latents are rounded to bfloat16, here the keys and the values;
// weights and result in both.  Error of a layer's output against float64, of its norm, prompts of 117 to 2048 tokens, through the latents / here:
// scores of deviation 1 0.00271 .. 0.00292 / 0.00266 .. 0.00283, a third of it 0.00256 .. 0.00277 / 0.00255 .. 0.00276, three times 0.00318 .. 0.00354
// / 0.00323 .. 0.00368 (rounded values no longer average out over the keys).  Logits of whole prompt steps, 15 of 1872 to 8192 tokens:
// 0.00962 and 0.00951 on average, the smaller one here in 9.
#include "hybrid_common.h"

namespace chronos {
namespace hy {

struct LatentExpanded {
    const uint16_t* q;        // [T, H, D + R] (row stride ldq): rotated part last
    int64_t ldq;
    const uint16_t* kv;       // [T, H, D + Dv]
    const uint16_t* kr;       // [T, R] (row stride ldr): the shared rotated keys
    int64_t ldr;
    const int32_t* q_start;
    const float* gate;        // [T, H] or nullptr
    const uint16_t* gcols;    // [T, H Dv] (row stride ldg) or nullptr
    int64_t ldg;
    const float* sink;        // [H] or nullptr
    uint16_t* out;            // [T, H, Dv] (row stride ldo)
    int64_t ldo;
    int H, D, R, Dv, window;
    float scale;
};

// NS: k-steps of the scores, (D + R) / 32 at most; NCT: 16-column tiles of the values, Dv / 16 at most
template <int NS, int NCT, int NW>
__global__ void __launch_bounds__(64 * NW) latent_expanded_kernel(const LatentExpanded a) {
    constexpr int KT = 64, RPB = 32 * NW, CK = NS * 4 + 1, CV = NCT * 2 + 1, NP = (CK + CV + NW - 1) / NW;
    constexpr float kLog2e = 1.4426950408889634f;
    extern __shared__ __attribute__((aligned(1024))) unsigned char le_smem[];   // 2 x (64 CK + 64 CV) 16-byte chunks
    const int h = blockIdx.x % a.H, b = blockIdx.x / a.H;
    const int t0 = a.q_start[b], n = a.q_start[b + 1] - t0;
    const int rb0 = (gridDim.y - 1 - blockIdx.y) * RPB;
    if (rb0 >= n) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, qi = lane & 15;
    const int DK = a.D + a.R, dkv = a.D + a.Dv;
    const int64_t ldkv = (int64_t)a.H * dkv;
    const int row0 = rb0 + 32 * wv, rlast = min(row0 + 31, n - 1), kend = min(rb0 + RPB, n) - 1;   // this wave's rows; the block's last key
    bf16x8 qf[2][NS];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint16_t* qr = a.q + (int64_t)(t0 + min(row0 + 16 * j + qi, n - 1)) * a.ldq + (int64_t)h * DK;
#pragma unroll
        for (int s = 0; s < NS; ++s) {   // columns past the row's end are zero here (and real numbers in the key image)
            const u16x8 z = {0, 0, 0, 0, 0, 0, 0, 0};
            qf[j][s] = 32 * s + 8 * g < DK ? *reinterpret_cast<const bf16x8*>(qr + 32 * s + 8 * g) : __builtin_bit_cast(bf16x8, z);
        }
    }
    // this lane's part of a tile's pieces wv, wv + NW, .. (64 chunks each: the keys' CK pieces, then the values' CV)
    const uint16_t* src[NP];
    int64_t step[NP];
    int krow[NP];
#pragma unroll
    for (int u = 0; u < NP; ++u) {
        const int p = wv + NW * u;
        const bool key = p < CK;
        const int i = (key ? p : p - CK) * 64 + lane, row = key ? i / CK : i / CV, c = key ? i - row * CK : i - row * CV;
        krow[u] = row;
        if (key) {
            const int cc = min(c, DK / 8 - 1);
            const bool rot = cc >= a.D / 8;
            src[u] = rot ? a.kr + (int64_t)t0 * a.ldr + (cc - a.D / 8) * 8 : a.kv + t0 * ldkv + (int64_t)h * dkv + cc * 8;
            step[u] = rot ? a.ldr : ldkv;
        } else {
            src[u] = a.kv + t0 * ldkv + (int64_t)h * dkv + a.D + min(c, a.Dv / 8 - 1) * 8;
            step[u] = ldkv;
        }
    }
    const uint32_t lds0 = lds_offset(le_smem);
    auto stage = [&](int k0, int buf) {   // (keys past the block's last one repeat it, masked below)
#pragma unroll
        for (int u = 0; u < NP; ++u)
            if (wv + NW * u < CK + CV)
                dma_1k(src[u] + min(k0 + krow[u], kend) * step[u],
                       __builtin_amdgcn_readfirstlane(lds0 + (buf * (CK + CV) + wv + NW * u) * 1024));
    };
    f32x4 O[2][NCT];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int c = 0; c < NCT; ++c) O[j][c] = f32x4{0.f, 0.f, 0.f, 0.f};
    float mrow[2] = {-INFINITY, -INFINITY}, lrow[2] = {0.f, 0.f};
    const float scale2 = a.scale * kLog2e;   // maxima and sums live in the base-2 domain
    const int kfirst = a.window > 0 ? max(0, rb0 - a.window + 1) / KT * KT : 0;
    stage(kfirst, 0);
    int buf = 0;
    for (int k0 = kfirst; k0 <= kend; k0 += KT, buf ^= 1) {
        dma_wait();
        __syncthreads();   // the tile is there; everyone has read the other buffer's
        if (k0 + KT <= kend) stage(k0 + KT, buf ^ 1);
        if (k0 > rlast || row0 >= n || (a.window > 0 && k0 + KT - 1 < row0 - a.window + 1)) continue;   // (wave-uniform)
        const unsigned char* kimg = le_smem + buf * (CK + CV) * 1024;
        const unsigned char* vimg = kimg + CK * 1024;
        f32x4 S[2][4];
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) {
            S[0][kt] = S[1][kt] = f32x4{0.f, 0.f, 0.f, 0.f};
            const unsigned char* arow = kimg + (16 * kt + qi) * (CK * 16) + g * 16;
#pragma unroll
            for (int s = 0; s < NS; ++s) {
                const bf16x8 k = *reinterpret_cast<const bf16x8*>(arow + s * 64);
                S[0][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[0][s], S[0][kt], 0, 0, 0);
                S[1][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k, qf[1][s], S[1][kt], 0, 0, 0);
            }
        }
        if (k0 + KT - 1 > row0 || (a.window > 0 && k0 < rlast - a.window + 1)) {
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = row0 + 16 * j + qi, lo = a.window > 0 ? row - a.window + 1 : 0;
#pragma unroll
                for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const int key = k0 + 16 * kt + 4 * g + i;
                        S[j][kt][i] = key <= row && key >= lo ? S[j][kt][i] : -INFINITY;
                    }
            }
        }
        bf16x8 pf[2][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {   // the scale is positive (host-checked): the largest score is the largest product
            float mx = -INFINITY;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt) mx = fmaxf(fmaxf(mx, fmaxf(S[j][kt][0], S[j][kt][1])), fmaxf(S[j][kt][2], S[j][kt][3]));
            mx = rows_max(mx);
            const float mn = fmaxf(mrow[j], mx * scale2);
            const float corr = mn == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(mrow[j] - mn);
            const float mref = mn == -INFINITY ? 0.f : mn;   // (all masked: every weight is 0)
            float sum = 0.f;
#pragma unroll
            for (int kt = 0; kt < 4; ++kt)
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(S[j][kt][i], scale2, -mref));
                    sum += p;
                    pf[j][kt >> 1][4 * (kt & 1) + i] = (__bf16)p;
                }
            sum = rows_sum(sum);
            lrow[j] = lrow[j] * corr + sum;
            mrow[j] = mn;
            if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0) {   // (rarely, once the maxima have settled)
#pragma unroll
                for (int c = 0; c < NCT; ++c) O[j][c] *= corr;
            }
        }
        const unsigned char* vt = vimg + (4 * g + (qi >> 2)) * (CV * 16) + (qi & 3) * 8;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int c = 0; c < NCT; ++c) {
                const bf16x4 lo = lds_read_tr4(vt + 32 * u * (CV * 16) + c * 32);
                const bf16x4 hi = lds_read_tr4(vt + (32 * u + 16) * (CV * 16) + c * 32);
                const bf16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
                O[0][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf[0][u], O[0][c], 0, 0, 0);
                O[1][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v, pf[1][u], O[1][c], 0, 0, 0);
            }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = row0 + 16 * j + qi;
        if (row >= n) continue;
        const int64_t t = t0 + row;
        float f = 1.f / lrow[j];
        if (a.sink != nullptr) {   // exp(sink) joins the denominator, without a value
            const float sk = a.sink[h] * kLog2e, mn = fmaxf(mrow[j], sk), c = exp2f(mrow[j] - mn);
            f = c / (lrow[j] * c + exp2f(sk - mn));
        }
        if (a.gate != nullptr) f *= sigmoidf_(a.gate[t * a.H + h]);
        // lane holds O^T[col = 16 c + 4 g + i][query row]
#pragma unroll
        for (int c = 0; c < NCT; ++c)
            if (16 * c < a.Dv) {
                f32x4 o = O[j][c] * f;
                if (a.gcols != nullptr)
#pragma unroll
                    for (int i = 0; i < 4; ++i) o[i] *= sigmoidf_(ld<uint16_t>(a.gcols + t * a.ldg + (int64_t)h * a.Dv + 16 * c + 4 * g + i));
                *reinterpret_cast<u16x4*>(a.out + t * a.ldo + (int64_t)h * a.Dv + 16 * c + 4 * g) = u16x4{f2bf(o[0]), f2bf(o[1]), f2bf(o[2]), f2bf(o[3])};
            }
    }
}

}  // namespace hy

template <int NS, int NCT, int NW>
static void latent_expanded_run(const hy::LatentExpanded& a, int B, int max_q, hipStream_t s) {
    auto kern = hy::latent_expanded_kernel<NS, NCT, NW>;
    constexpr int bytes = 2 * (NS * 4 + 1 + NCT * 2 + 1) * 1024;
    static const hipError_t set = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    (void)set;
    kern<<<dim3(B * a.H, (max_q + 32 * NW - 1) / (32 * NW)), 64 * NW, bytes, s>>>(a);
}

// D, R, Dv in elements; rows of q, kv and kr on 16-byte boundaries, of out on 8-byte ones (host-checked)
bool hy_latent_expanded_ok(int D, int R, int Dv) { return D % 8 == 0 && R % 8 == 0 && D > 0 && R >= 0 && D + R <= 192 && Dv % 16 == 0 && Dv > 0 && Dv <= 128; }

void launch_hy_latent_expanded(const uint16_t* q, int64_t ldq, const uint16_t* kv, const uint16_t* kr, int64_t ldr,
                               const int32_t* q_start, const float* gate, const uint16_t* gcols, int64_t ldg, const float* sink,
                               uint16_t* out, int64_t ldo, int B, int H, int D, int R, int Dv, float scale, int window, int max_q,
                               hipStream_t s) {
    if (B == 0 || max_q == 0) return;
    const hy::LatentExpanded a{q, ldq, kv, kr, ldr, q_start, gate, gcols, ldg, sink, out, ldo, H, D, R, Dv, window, scale};
    // 256 rows per workgroup where that still gives every CU two (their walks differ in length), else 128
    const bool wide = (int64_t)B * H * ((max_q + 255) / 256) >= 512;
    if (D + R <= 96 && Dv <= 64) {
        if (wide) latent_expanded_run<3, 4, 8>(a, B, max_q, s);
        else latent_expanded_run<3, 4, 4>(a, B, max_q, s);
    } else {
        if (wide) latent_expanded_run<6, 8, 8>(a, B, max_q, s);
        else latent_expanded_run<6, 8, 4>(a, B, max_q, s);
    }
}

}  // namespace chronos
