// moe.hip — mixture-of-experts feed-forward of the hybrid decoders.
//
//   route   per token: float router logits (N = experts + identity outputs; the few-row projection of
//           hybrid_elementwise.hip), then one wave per token: softmax over all N, the `top` largest
//           of score + correction chosen (the correction steers the choice only), weights = the chosen outputs' plain
//           scores, not renormalised.  Ties go to the lower index.
//   route_group  sigmoid scores; the outputs form equal groups of neighbours, a group scores its top two
//           scores added up, only the best `keep` groups stay eligible, the `top` largest eligible scores are chosen and
//           weighted by score / (sum of the chosen + 1e-20) * scale.
//   ffn     per token: sum over its chosen experts of weight * W_down act(W_up h); an index >= E is an identity
//           expert (weight * h).  Token-parallel form: one workgroup per token streams the chosen experts' weights
//           (the decode regime: few tokens, every expert matrix read about once; float accumulation throughout).
//
// No step of either kernel depends on the host knowing the routing: both capture into a graph.
#include "hybrid_common.h"
#include "rowdot_tile.h"

#include <type_traits>

namespace chronos {
namespace hy {

__device__ __forceinline__ void unpack8(const uint4& r, float (&v)[8]) {
    const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        v[2 * i] = __uint_as_float(w[i] << 16);
        v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}


// The choice of one token by one wave: zr its N <= 256 logits (4 per lane; LDS or memory) -> idx[top], wt[top].  Softmax over all N, the largest of
// score + correction chosen, plain scores as weights.
__device__ __forceinline__ void select_softmax(const float* zr, const float* __restrict__ corr, int32_t* __restrict__ idx, float* __restrict__ wt,
                                               int N, int top) {
    const int lane = threadIdx.x & 63;
    float s[4], c[4];
    float mx = -INFINITY;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        s[j] = e < N ? zr[e] : -INFINITY;
        mx = fmaxf(mx, s[j]);
    }
    mx = wave_max(mx);
    float sum = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        s[j] = (lane + 64 * j < N) ? expf(s[j] - mx) : 0.f;
        sum += s[j];
    }
    sum = wave_sum(sum);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        s[j] = s[j] / sum;
        c[j] = e < N ? s[j] + corr[e] : -INFINITY;
    }
    for (int k = 0; k < top; ++k) {
        // the wave's best (value, lowest index): a lane's own candidates first, then across lanes
        float bv = -INFINITY, bs = 0.f;
        int be = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            if (c[j] > bv || (c[j] == bv && e < be && c[j] != -INFINITY)) {
                bv = c[j]; be = e; bs = s[j];
            }
        }
        lanes_best(bv, be, bs);
        if (lane == 0) {
            idx[k] = be;
            wt[k] = bs;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j == be) c[j] = -INFINITY;
    }
}

// LDS: h row (d floats) | z (F floats) | out (d floats).
template <typename T>
__global__ void __launch_bounds__(256) moe_ffn_token_kernel(const T* __restrict__ h, const int32_t* __restrict__ idx,
                                                            const float* __restrict__ wt, const T* __restrict__ w_up,
                                                            const T* __restrict__ w_down, T* __restrict__ out, int d,
                                                            int F, int E, int top, int act) {
    extern __shared__ float sm[];
    float* hs = sm;
    float* zs = hs + d;
    float* os = zs + F;
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < d; i += 256) {
        hs[i] = ld<T>(h + t * d + i);
        os[i] = 0.f;
    }
    __syncthreads();
    for (int k = 0; k < top; ++k) {
        const int e = idx[t * top + k];
        const float g = wt[t * top + k];
        if (e >= E) {  // identity expert (uniform over the workgroup)
            for (int i = threadIdx.x; i < d; i += 256) os[i] += g * hs[i];
            __syncthreads();
            continue;
        }
        const T* wu = w_up + (int64_t)e * F * d;
        for (int f = wv; f < F; f += 4) {
            const T* wr = wu + (int64_t)f * d;
            float acc = 0.f;
            for (int i = lane; i < d; i += 64) acc += ld<T>(wr + i) * hs[i];
            acc = wave_sum(acc);
            if (lane == 0) zs[f] = act_apply(rnd<T>(acc), act);
        }
        __syncthreads();
        const T* wd = w_down + (int64_t)e * d * F;
        for (int r = wv; r < d; r += 4) {
            const T* wr = wd + (int64_t)r * F;
            float acc = 0.f;
            for (int i = lane; i < F; i += 64) acc += ld<T>(wr + i) * zs[i];
            acc = wave_sum(acc);
            if (lane == 0) os[r] += g * acc;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < d; i += 256) st<T>(out + t * d + i, os[i]);
}

// ... the `top` largest logits (ties: the lower index), weighted by the softmax over the chosen only.  top <= 64 (lane k keeps the k-th choice).
__device__ __forceinline__ void select_topk(const float* zr, int32_t* __restrict__ idx, float* __restrict__ wt, int N, int top) {
    const int lane = threadIdx.x & 63;
    float c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        c[j] = e < N ? zr[e] : -INFINITY;
    }
    float first = 0.f, sum = 0.f, mine = 0.f;  // lane k keeps the k-th chosen logit's exponential
    for (int k = 0; k < top; ++k) {
        float bv = -INFINITY;
        int be = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            if (e < N && (c[j] > bv || (c[j] == bv && e < be))) {
                bv = c[j]; be = e;
            }
        }
        float none = 0.f;
        lanes_best(bv, be, none);
        if (k == 0) first = bv;  // the largest logit: the softmax's reference point
        const float ex = expf(bv - first);
        sum += ex;
        if (k == lane) {
            mine = ex;
            idx[k] = be;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j == be) c[j] = -INFINITY;
    }
    if (lane < top) wt[lane] = mine / sum;
}

// ... sigmoid scores, the choice limited to the best groups (ng groups of N / ng neighbouring outputs, a group's score = its top two scores added up,
// the `keep` best stay; ties: the lower index), then the `top` largest eligible scores (ties: the lower index), weights = score / (their sum +
// 1e-20) * scale.  ng <= 64 (lane g ranks group g), top <= 64.  sc, okg: LDS of the wave's own, N scores and ng flags.
__device__ __forceinline__ void select_group(const float* zr, int32_t* __restrict__ idx, float* __restrict__ wt, int N, int top, int ng, int keep,
                                             float scale, float* sc, int* okg) {
    const int lane = threadIdx.x & 63;
    const int per = N / ng;
    float s[4], c[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        s[j] = e < N ? sigmoidf_(zr[e]) : 0.f;
        if (e < N) sc[e] = s[j];
    }
    // (wave-private LDS rows: a wave's own writes are visible to its later reads)
    if (keep < ng) {
        float gsc = -INFINITY;
        if (lane < ng) {
            float a = -INFINITY, b = -INFINITY;   // the group's two largest
            for (int i = 0; i < per; ++i) {
                const float v = sc[lane * per + i];
                if (v > a) { b = a; a = v; }
                else if (v > b) b = v;
            }
            gsc = per > 1 ? a + b : a;
        }
        int rank = 0;   // groups that come before this one
        for (int g = 0; g < ng; ++g) {
            const float o = __shfl(gsc, g, 64);
            rank += (o > gsc || (o == gsc && g < lane)) ? 1 : 0;
        }
        if (lane < ng) okg[lane] = rank < keep ? 1 : 0;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int e = lane + 64 * j;
        c[j] = (e < N && (keep >= ng || okg[e / per])) ? s[j] : -INFINITY;
    }
    float sum = 0.f, mine = 0.f;
    for (int k = 0; k < top; ++k) {
        float bv = -INFINITY;
        int be = 0x7fffffff;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = lane + 64 * j;
            if (e < N && (c[j] > bv || (c[j] == bv && e < be && c[j] != -INFINITY))) {
                bv = c[j]; be = e;
            }
        }
        float none = 0.f;
        lanes_best(bv, be, none);
        sum += bv;
        if (k == lane) {
            mine = bv;
            idx[k] = be;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (lane + 64 * j == be) c[j] = -INFINITY;
    }
    if (lane < top) wt[lane] = mine / (sum + 1e-20f) * scale;
}

struct Choice {   // which of the three, and its parameters
    const float* corr;   // softmax form
    int N, top, ng, keep;
    float scale;
};
enum { kSoftmax = 0, kTopk = 1, kGroups = 2 };
template <int FORM>
__device__ __forceinline__ void select_any(const float* zr, int32_t* idx, float* wt, const Choice& c, float* sc, int* okg) {
    if constexpr (FORM == kSoftmax) select_softmax(zr, c.corr, idx, wt, c.N, c.top);
    else if constexpr (FORM == kTopk) select_topk(zr, idx, wt, c.N, c.top);
    else select_group(zr, idx, wt, c.N, c.top, c.ng, c.keep, c.scale, sc, okg);
}

// One wave per token of logits z [T, N].
template <int FORM>
__global__ void __launch_bounds__(256) moe_select_kernel(const float* __restrict__ z, int32_t* __restrict__ idx, float* __restrict__ wt, int rows, Choice c) {
    __shared__ float sc[FORM == kGroups ? 4 : 1][256];
    __shared__ int okg[FORM == kGroups ? 4 : 1][64];
    const int wv = FORM == kGroups ? threadIdx.x >> 6 : 0;
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= rows) return;   // (a whole wave leaves; the waves of a block share no barrier)
    select_any<FORM>(z + t * c.N, idx + t * c.top, wt + t * c.top, c, sc[wv], okg[wv]);
}

// Projection and choice of one token by one workgroup: 16 waves share the N rows of w (N <= 64), the first wave chooses.  For up to 256 tokens, which
// as a projection and a choice were two launches and two chains of latencies.  What bounds it is latency: a wave has up to 16 loads of 16
// bytes a lane on their way.  us, two launches -> this: 1 token of 1024 by 10 rows 6.0 -> 5.2, 64 of 2048 by 18 11.4 -> 7.5, of 4096 by 34 12.6 -> 9.8, 256 of
// 4096 by 64 13.9 -> 12.2; 300 tokens, more than there are CUs, 8.0 -> 9.5, 11.5 -> 13.5 and 14.9 -> 21.8.  Up to 2^18 weights, which every token's workgroup reads: 7168 by 34 (238 K) 12.8 -> 12.1 at 64
// tokens, by 48 (336 K) 13.0 -> 13.6, by 64 (448 K) 12.8 -> 14.9; one token 14.8 -> 14.3, 200 18.6 -> 15.7.
constexpr int kRouteN = 64, kRouteWaves = 16;
template <int FORM>
__global__ void __launch_bounds__(64 * kRouteWaves) moe_route_token_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ w,
                                                                           const float* __restrict__ bias, int32_t* __restrict__ idx,
                                                                           float* __restrict__ wt, int d, Choice c) {
    __shared__ float z[kRouteN], sc[FORM == kGroups ? kRouteN : 1];
    __shared__ int okg[FORM == kGroups ? kRouteN : 1];
    constexpr int R = kRouteN / kRouteWaves;   // rows of a wave: wave, wave + 16, ..
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n = (c.N - wave + kRouteWaves - 1) / kRouteWaves;
    const uint16_t *hr = h + t * d, *wr = w + (int64_t)wave * d;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.f;
    auto part = [&](auto MC, auto UC, int k) {   // M rows by U runs of 512 columns
        constexpr int M = decltype(MC)::value, U = decltype(UC)::value;
        uint4 hq[U], q[M][U];
#pragma unroll
        for (int u = 0; u < U; ++u) hq[u] = *reinterpret_cast<const uint4*>(hr + k + 512 * u);
#pragma unroll
        for (int r = 0; r < M; ++r)
#pragma unroll
            for (int u = 0; u < U; ++u) q[r][u] = *reinterpret_cast<const uint4*>(wr + (int64_t)r * kRouteWaves * d + k + 512 * u);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float hv[8], wv[8];
            unpack8(hq[u], hv);
#pragma unroll
            for (int r = 0; r < M; ++r) {
                unpack8(q[r][u], wv);
#pragma unroll
                for (int e = 0; e < 8; ++e) acc[r] += hv[e] * wv[e];
            }
        }
    };
    auto rows = [&](auto MC) {
        constexpr int M = decltype(MC)::value, U = M == 1 ? 8 : M <= 3 ? 4 : 2;
        int k = 0;
        for (; k + 512 * U <= d; k += 512 * U) part(MC, std::integral_constant<int, U>{}, k + lane * 8);
        if constexpr (U > 4)
            for (; k + 2048 <= d; k += 2048) part(MC, std::integral_constant<int, 4>{}, k + lane * 8);
        if constexpr (U > 2)
            for (; k + 1024 <= d; k += 1024) part(MC, std::integral_constant<int, 2>{}, k + lane * 8);
        for (k += lane * 8; k < d; k += 512) part(MC, std::integral_constant<int, 1>{}, k);
    };
    if (n == 1) rows(std::integral_constant<int, 1>{});
    else if (n == 2) rows(std::integral_constant<int, 2>{});
    else if (n == 3) rows(std::integral_constant<int, 3>{});
    else if (n == 4) rows(std::integral_constant<int, 4>{});
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float v = wave_sum(acc[r]);
        if (lane == 0 && r < n) z[wave + kRouteWaves * r] = v + (bias != nullptr ? bias[wave + kRouteWaves * r] : 0.f);
    }
    __syncthreads();
    if (wave == 0) select_any<FORM>(z, idx + t * c.top, wt + t * c.top, c, sc, okg);
}

// Projection and choice of many tokens: a workgroup takes 16 tokens by all N <= 16 NT rows of w, its 8 waves then choose for two of them each; the
// logits stay in LDS and are those of the projection by itself, bit for bit.  us, two launches -> this, softmax and top-k: 600 tokens of 1024 by 8 rows 8.0, 7.0 -> 7.4,
// 5.8; 2446 of 2048 by 18 13.0, 11.5 -> 12.6, 10.2; 8192 of 2048 by 16 21.1, 17.1 -> 17.8, 14.2; of 4096 by 32 34.8, 31.0 -> 30.3, 27.6.  Beyond 32 rows the choices, two
// after each other in a wave, take longer than the launch: 8192 of 4096 by 34 31.4, 27.8 -> 34.4, 31.5, by 64 43.8, 38.2 -> 48.3, 44.8; 1000 by 64 28.8, 27.3 -> 30.2, 27.2.
template <int FORM, int NT>
__global__ void __launch_bounds__(512) moe_route_tile_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ w, const float* __restrict__ bias,
                                                             int32_t* __restrict__ idx, float* __restrict__ wt, int rows, int d, Choice c) {
    __shared__ f32x4 red[8][NT][64];
    __shared__ float z[16][16 * NT], sc[FORM == kGroups ? 8 : 1][16 * NT];
    __shared__ int okg[FORM == kGroups ? 8 : 1][64];
    const int64_t t0 = (int64_t)blockIdx.x * 16;
    const int wv = threadIdx.x >> 6;
    rowdot_tile<1, NT, 8>(h, w, bias, t0, 0, rows, d, c.N, red, [&](int64_t t, int r, float v) { z[t - t0][r] = v; });
    __syncthreads();
    for (int i = wv; i < 16 && t0 + i < rows; i += 8)
        select_any<FORM>(z[i], idx + (t0 + i) * c.top, wt + (t0 + i) * c.top, c, sc[FORM == kGroups ? wv : 0], okg[FORM == kGroups ? wv : 0]);
}

// Gated experts: per token sum_k weight_k * W_down,e ( g sigmoid(slope g) (u + shift) ), g = min(W_gate,e h, limit),
// u = clamp(W_up,e h, +-limit).  w_gu [E, 2F, d]: gate rows then up rows, or (tiled) in the grouped path's tile order.
// LDS: h (d) | gate, up (2F) | out (d).
template <typename T>
__global__ void __launch_bounds__(256) moe_glu_token_kernel(const T* __restrict__ h, const int32_t* __restrict__ idx,
                                                            const float* __restrict__ wt, const T* __restrict__ w_gu,
                                                            const T* __restrict__ w_down, T* __restrict__ out, int d,
                                                            int F, int E, int top, float limit, float slope,
                                                            float shift, int tiled) {
    extern __shared__ float sm[];
    float* hs = sm;
    float* zs = hs + d;
    float* os = zs + 2 * F;
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < d; i += 256) {
        hs[i] = ld<T>(h + t * d + i);
        os[i] = 0.f;
    }
    __syncthreads();
    for (int k = 0; k < top; ++k) {
        const int e = idx[t * top + k];
        const float g = wt[t * top + k];
        if (e < 0 || e >= E) continue;  // (uniform over the workgroup)
        const T* wu = w_gu + (int64_t)e * 2 * F * d;
        for (int f = wv; f < 2 * F; f += 4) {
            int row = f;
            if (tiled) {  // the grouped path's row order: per 128-row tile and 64-row half, 32 gate rows then their up rows
                const int c = f < F ? f : f - F;
                row = (c >> 6) * 128 + ((c >> 5) & 1) * 64 + (c & 31) + (f < F ? 0 : 32);
            }
            const T* wr = wu + (int64_t)row * d;
            float acc = 0.f;
            for (int i = lane; i < d; i += 64) acc += ld<T>(wr + i) * hs[i];
            acc = wave_sum(acc);
            if (lane == 0) zs[f] = rnd<T>(acc);
        }
        __syncthreads();
        for (int f = threadIdx.x; f < F; f += 256) {
            const float a = fminf(zs[f], limit), u = fminf(fmaxf(zs[F + f], -limit), limit);
            zs[f] = rnd<T>(a * sigmoidf_(slope * a) * (u + shift));
        }
        __syncthreads();
        const T* wd = w_down + (int64_t)e * d * F;
        for (int r = wv; r < d; r += 4) {
            const T* wr = wd + (int64_t)r * F;
            float acc = 0.f;
            for (int i = lane; i < F; i += 64) acc += ld<T>(wr + i) * zs[i];
            acc = wave_sum(acc);
            if (lane == 0) os[r] += g * rnd<T>(acc);
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < d; i += 256) st<T>(out + t * d + i, os[i]);
}

}  // namespace hy

void launch_hy_rowdot(const void*, const void*, const float*, float*, int, int, int, bool, hipStream_t);

bool hy_moe_route_one(int T, int N, int d) {
    const int64_t nd = (int64_t)N * d;
    return T <= 256 && N <= hy::kRouteN && d % 8 == 0 && (nd <= 1 << 18 || (nd <= 1 << 19 && (T == 1 || T > 160)));
}
// z: float [T, N] scratch for the router logits (the few-row float32-output projection, then the selection); not touched where one launch does both
template <int FORM>
static void moe_route(const void* h, const void* w, const float* bias, float* z, int32_t* idx, float* wt, int T, int d, const hy::Choice& c, bool f32,
                      hipStream_t s) {
    if (T == 0) return;
    if (!f32 && hy_moe_route_one(T, c.N, d) && hy::aligned16(h, w)) {
        hy::moe_route_token_kernel<FORM><<<T, 64 * hy::kRouteWaves, 0, s>>>((const uint16_t*)h, (const uint16_t*)w, bias, idx, wt, d, c);
        return;
    }
    if (!f32 && T > 512 && c.N > 0 && c.N <= 32 && d % 64 == 0 && hy::aligned16(h, w)) {
        const uint16_t *hb = (const uint16_t*)h, *wb = (const uint16_t*)w;
        const unsigned wgs = (T + 15) / 16;
        if (c.N <= 16) hy::moe_route_tile_kernel<FORM, 1><<<wgs, 512, 0, s>>>(hb, wb, bias, idx, wt, T, d, c);
        else hy::moe_route_tile_kernel<FORM, 2><<<wgs, 512, 0, s>>>(hb, wb, bias, idx, wt, T, d, c);
        return;
    }
    launch_hy_rowdot(h, w, bias, z, T, d, c.N, f32, s);
    hy::moe_select_kernel<FORM><<<(T + 3) / 4, 256, 0, s>>>(z, idx, wt, T, c);
}

void launch_hy_moe_route(const void* h, const void* w, const float* corr, float* z, int32_t* idx, float* wt, int T, int d,
                         int N, int top, bool f32, hipStream_t s) {
    moe_route<hy::kSoftmax>(h, w, nullptr, z, idx, wt, T, d, {corr, N, top, 0, 0, 0.f}, f32, s);
}

void launch_hy_moe_ffn_token(const void* h, const int32_t* idx, const float* wt, const void* w_up, const void* w_down,
                             void* out, int T, int d, int F, int E, int top, int act, bool f32, hipStream_t s) {
    if (T == 0) return;
    const int bytes = (2 * d + F) * 4;
    if (f32) {
        auto kern = hy::moe_ffn_token_kernel<float>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        kern<<<T, 256, bytes, s>>>((const float*)h, idx, wt, (const float*)w_up, (const float*)w_down, (float*)out, d, F, E, top, act);
    } else {
        auto kern = hy::moe_ffn_token_kernel<uint16_t>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        kern<<<T, 256, bytes, s>>>((const uint16_t*)h, idx, wt, (const uint16_t*)w_up, (const uint16_t*)w_down, (uint16_t*)out, d, F, E, top, act);
    }
}

// z: float [T, N] scratch for the router logits (bias added by the projection), N <= 256
void launch_hy_moe_route_topk(const void* h, const void* w, const float* bias, float* z, int32_t* idx, float* wt, int T,
                              int d, int N, int top, bool f32, hipStream_t s) {
    moe_route<hy::kTopk>(h, w, bias, z, idx, wt, T, d, {nullptr, N, top, 0, 0, 0.f}, f32, s);
}

// z: float [T, N] scratch for the router logits, N <= 256, groups <= 64, top <= 64
void launch_hy_moe_route_group(const void* h, const void* w, float* z, int32_t* idx, float* wt, int T, int d, int N,
                               int top, int ng, int keep, float scale, bool f32, hipStream_t s) {
    moe_route<hy::kGroups>(h, w, nullptr, z, idx, wt, T, d, {nullptr, N, top, ng, keep, scale}, f32, s);
}

void launch_hy_moe_glu_token(const void* h, const int32_t* idx, const float* wt, const void* w_gu, const void* w_down,
                             void* out, int T, int d, int F, int E, int top, float limit, float slope, float shift,
                             bool tiled, bool f32, hipStream_t s) {
    if (T == 0) return;
    const int bytes = (2 * d + 2 * F) * 4;
    if (f32) {
        auto kern = hy::moe_glu_token_kernel<float>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        kern<<<T, 256, bytes, s>>>((const float*)h, idx, wt, (const float*)w_gu, (const float*)w_down, (float*)out, d, F, E, top, limit, slope, shift, tiled);
    } else {
        auto kern = hy::moe_glu_token_kernel<uint16_t>;
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        kern<<<T, 256, bytes, s>>>((const uint16_t*)h, idx, wt, (const uint16_t*)w_gu, (const uint16_t*)w_down, (uint16_t*)out, d, F, E, top, limit, slope, shift, tiled);
    }
}

}  // namespace chronos
