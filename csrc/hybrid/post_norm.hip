// post_norm.hip — the float32 residual stream of post-norm hybrid decoders and their gated feed-forward activation.
//
//   rms_norm          h = T(x / sqrt(mean(x^2) + eps) * w)                       (the model's final norm)
//   scale_add_rms     x <- (alpha x + y) / sqrt(mean((alpha x + y)^2) + eps) * w;  h = T(x)
//                     The norm sits AFTER the residual sum, so the stream itself is what the next sublayer reads:
//                     one kernel reads the sublayer output y (activation type) and the stream, does all arithmetic in
//                     float, rewrites the stream in place and emits its copy in the activation type.
//   glu               y = g sigmoid(slope g) (u + shift),  g = min(gate, limit),  u = clamp(up, -limit, limit), from
//                     a [T, 2F] projection whose first F columns are the gate and last F the up part.
//   decay_pow         z <- sigmoid(z)^p through exp(p log sigmoid(z)), float, in place (per-channel decays).
//
// Rows whose width is a multiple of 4 move 16 bytes (float) / 8 bytes (bfloat16) per lane and keep up to 16 values per
// thread in registers between the statistics pass and the write pass (d <= 4096 is read once).
#include "hybrid_common.h"

namespace chronos {
namespace hy {

template <typename T> __device__ __forceinline__ f32x4 ld4(const T* p);
template <> __device__ __forceinline__ f32x4 ld4<float>(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
template <> __device__ __forceinline__ f32x4 ld4<uint16_t>(const uint16_t* p) {
    const u16x4 v = *reinterpret_cast<const u16x4*>(p);
    return f32x4{bf2f(v[0]), bf2f(v[1]), bf2f(v[2]), bf2f(v[3])};
}
template <typename T> __device__ __forceinline__ void st4(T* p, const f32x4& v);
template <> __device__ __forceinline__ void st4<float>(float* p, const f32x4& v) { *reinterpret_cast<f32x4*>(p) = v; }
template <> __device__ __forceinline__ void st4<uint16_t>(uint16_t* p, const f32x4& v) {
    *reinterpret_cast<u16x4*>(p) = u16x4{f2bf(v[0]), f2bf(v[1]), f2bf(v[2]), f2bf(v[3])};
}

// S float32 slices of a product, summed in order and rounded where the product would be
struct Slices {
    const float* p;
    int S;
    int64_t stride;
};
// x <- norm(alpha * x + y) * w, h <- x in bfloat16, as below with y in slices, d % 4 == 0: a launch less than a sum before it (a
// decode step of one row at width 1024 189 -> 185 us, of 8 rows 207 -> 204).  NT threads take a row, 4 columns each NJ times, and everything that
// they read is on its way before the first sum: a few rows are a chain of latencies (256 threads that took one piece after the other: 26 rows of
// 4096 in 4 slices 5.8 us, now 3.3; 64 rows of 8192 in 8 10.2, now 5.8; one row of 1024 in 4 3.2, now 2.5).
template <int NT, int NJ>
__global__ void __launch_bounds__(NT) rms_norm_slices_kernel(Slices y, float* __restrict__ x, const float* __restrict__ w,
                                                             uint16_t* __restrict__ h, int d, float alpha, float eps) {
    __shared__ float red[NT / 64];
    const int64_t at = blockIdx.x * (int64_t)d;
    f32x4 c[NJ], wv[NJ];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int i = min((int)(threadIdx.x + NT * j) * 4, d - 4);   // (past the row: its last columns again, not counted)
        const float* const p = y.p + at + i;
        f32x4 v = *reinterpret_cast<const f32x4*>(p);
        c[j] = *reinterpret_cast<const f32x4*>(x + at + i);
        wv[j] = *reinterpret_cast<const f32x4*>(w + i);
#pragma unroll 4
        for (int k = 1; k < y.S; ++k) v += *reinterpret_cast<const f32x4*>(p + k * y.stride);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = bf2f(f2bf(v[e]));
        v = c[j] * alpha + v;
        c[j] = v;
        if ((int)(threadIdx.x + NT * j) * 4 < d) ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    float sum = 0.f;
#pragma unroll
    for (int k = 0; k < NT / 64; ++k) sum += red[k];
    const float rstd = 1.f / sqrtf(sum / (float)d + eps);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int i = (threadIdx.x + NT * j) * 4;
        if (i < d) {
            const f32x4 v = c[j] * rstd * wv[j];
            *reinterpret_cast<f32x4*>(x + at + i) = v;
            st4<uint16_t>(h + at + i, v);
        }
    }
}

// JOIN: v = alpha * x + y (y in TY), x <- norm(v) * w, h <- TH(x).   plain: v = x (float), h <- TH(norm(v) * w); with `rows` (VEC only) v = x's
// row rows[r] of `total`, NaN where there is none.
template <typename TY, typename TH, bool JOIN, bool VEC>
__global__ void __launch_bounds__(256) rms_norm_kernel(const TY* __restrict__ y, float* __restrict__ x,
                                                       const float* __restrict__ w, TH* __restrict__ h, int d,
                                                       float alpha, float eps, const int64_t* __restrict__ rows, int total) {
    __shared__ float red[16];
    const int64_t row = blockIdx.x, src = !JOIN && VEC && rows != nullptr ? rows[row] : row;
    const bool there = JOIN || !VEC || (src >= 0 && src < total);
    float* xr = x + (there ? src : 0) * d;
    const TY* yr = JOIN ? y + row * d : nullptr;
    TH* hr = h != nullptr ? h + row * d : nullptr;
    float ss = 0.f;
    if constexpr (VEC) {
        f32x4 c[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = (threadIdx.x + 256 * j) * 4;
            c[j] = f32x4{0.f, 0.f, 0.f, 0.f};
            if (i < d) {
                f32x4 v = *reinterpret_cast<const f32x4*>(xr + i);
                if constexpr (JOIN) v = v * alpha + ld4<TY>(yr + i);
                if (!there) v *= NAN;
                c[j] = v;
                ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
            }
        }
        for (int i = (threadIdx.x + 1024) * 4; i < d; i += 1024) {
            f32x4 v = *reinterpret_cast<const f32x4*>(xr + i);
            if constexpr (JOIN) v = v * alpha + ld4<TY>(yr + i);
            ss += v[0] * v[0] + v[1] * v[1] + v[2] * v[2] + v[3] * v[3];
        }
        const float rstd = 1.f / sqrtf(block_sum(ss, red) / (float)d + eps);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int i = (threadIdx.x + 256 * j) * 4;
            if (i < d) {
                const f32x4 v = c[j] * rstd * *reinterpret_cast<const f32x4*>(w + i);
                if constexpr (JOIN) *reinterpret_cast<f32x4*>(xr + i) = v;
                if (hr != nullptr) st4<TH>(hr + i, v);
            }
        }
        for (int i = (threadIdx.x + 1024) * 4; i < d; i += 1024) {
            f32x4 v = *reinterpret_cast<const f32x4*>(xr + i);
            if constexpr (JOIN) v = v * alpha + ld4<TY>(yr + i);
            v = v * rstd * *reinterpret_cast<const f32x4*>(w + i);   // (of no row there is: rstd is NaN)
            if constexpr (JOIN) *reinterpret_cast<f32x4*>(xr + i) = v;
            if (hr != nullptr) st4<TH>(hr + i, v);
        }
    } else {
        for (int i = threadIdx.x; i < d; i += 256) {
            float v = xr[i];
            if constexpr (JOIN) v = v * alpha + ld<TY>(yr + i);
            ss += v * v;
        }
        const float rstd = 1.f / sqrtf(block_sum(ss, red) / (float)d + eps);
        for (int i = threadIdx.x; i < d; i += 256) {
            float v = xr[i];
            if constexpr (JOIN) v = v * alpha + ld<TY>(yr + i);
            v = v * rstd * w[i];
            if constexpr (JOIN) xr[i] = v;
            if (hr != nullptr) st<TH>(hr + i, v);
        }
    }
}

// grid (rows, column blocks); rows of gu (gate columns, then up columns) and of y may be parts of wider ones
template <typename T, bool VEC>
__global__ void __launch_bounds__(256) glu_kernel(const T* __restrict__ gu, int64_t ldg, T* __restrict__ y, int64_t ldy, int F,
                                                  float limit, float slope, float shift) {
    constexpr int E = VEC ? 4 : 1;
    const int64_t r = blockIdx.x;
    const int c = (int)(blockIdx.y * blockDim.x + threadIdx.x) * E;
    if (c >= F) return;
    const T* g = gu + r * ldg + c;
    if constexpr (VEC) {
        const f32x4 gv = ld4<T>(g), uv = ld4<T>(g + F);
        f32x4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float a = fminf(gv[k], limit), u = fminf(fmaxf(uv[k], -limit), limit);
            o[k] = a * sigmoid_act<T>(slope * a) * (u + shift);
        }
        st4<T>(y + r * ldy + c, o);
    } else {
        const float a = fminf(ld<T>(g), limit), u = fminf(fmaxf(ld<T>(g + F), -limit), limit);
        st<T>(y + r * ldy + c, a * sigmoid_act<T>(slope * a) * (u + shift));
    }
}

// 16 bytes per lane: 8192 x 2 x 11008, 540 MB: 127 us at 8 bytes per lane, 120 so; 2457 x 2 x 2816: 10.6 and 9.1
__global__ void __launch_bounds__(256) glu_vec_kernel(const uint16_t* __restrict__ gu, int64_t ldg, uint16_t* __restrict__ y, int64_t ldy,
                                                      int F, float limit, float slope, float shift) {
    const int64_t r = blockIdx.x;
    const int c = (int)(blockIdx.y * blockDim.x + threadIdx.x) * 8;
    if (c >= F) return;
    float g[8], u[8];
    ld8(gu + r * ldg + c, g);
    ld8(gu + r * ldg + F + c, u);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float a = fminf(g[k], limit), b = fminf(fmaxf(u[k], -limit), limit);
        g[k] = a * sigmoid_act<uint16_t>(slope * a) * (b + shift);
    }
    st8(y + r * ldy + c, g);
}

// p <= 1/16: log sigmoid(z) = min(z, 0) - log(1 + e^-|z|) with the second part through the hardware's exp2 and log2, whose absolute error of
// 1e-7 times p is a small part of a last place of the result; the outer exponential is the library's.  Largest error and root mean square in
// units of the result's last place at p = 1/16, this and the library throughout: z in -100 .. -20 0.83, 0.300 both; -20 .. -6 1.14, 0.344 and
// 1.08, 0.343; -0.1 .. 0.1 0.67, 0.292 and 0.64, 0.291 (at p = 1/8 0.90, 0.315 and 0.89, 0.308, hence the line).  Through exp2 to the end the
// rounding of z p log2 e shows: 4.2, 1.33 at z < -40.  16 bytes per lane.  8192 x 2048 values: 67 us with the library, which bounds it, 20 so.
__device__ __forceinline__ f32x4 decay_pow4(f32x4 v, float p) {
    constexpr float kLog2e = 1.4426950408889634f, kLn2 = 0.6931471805599453f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const float t = __builtin_amdgcn_exp2f(-fabsf(v[e]) * kLog2e);
        v[e] = expf(p * __builtin_fmaf(-kLn2, __builtin_amdgcn_logf(1.f + t), fminf(v[e], 0.f)));
    }
    return v;
}
__global__ void __launch_bounds__(256) decay_pow_vec_kernel(f32x4* __restrict__ z, int64_t n4, float p) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    z[i] = decay_pow4(z[i], p);
}

__global__ void __launch_bounds__(256) decay_pow_kernel(float* __restrict__ z, int64_t n, float p) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) z[i] = expf(logsigmoidf_(z[i]) * p);
}

// Decays of a gated linear recurrence from their low-rank logits, in one pass: out[t, c] = sigmoid(b[c] + sum_r a[t, r] w[r, c])^p, float
// throughout, the sum in the order of r.  A thread takes 4 channels of TT tokens, so that w is read once for them; the tokens' a is
// the same in all lanes.  Bound by writing out (8192 x 4096
// of rank 16: 28 us, 4.8 TB/s, 38 where launches follow each other); a library product, the copy of its bias and decay_pow took 120 there, 15 for 2446 x 512 (8 so), 16 for a single
// token (6).
template <int TT, bool POW4>
__global__ void __launch_bounds__(256) low_rank_decay_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                             const float* __restrict__ b, float* __restrict__ out, int T, int R, int C,
                                                             float p, bool tokens_x) {
    const int c = ((tokens_x ? blockIdx.y : blockIdx.x) * 256 + threadIdx.x) * 4;
    if (c >= C) return;
    const int t0 = (tokens_x ? blockIdx.x : blockIdx.y) * TT;
    f32x4 z[TT];
#pragma unroll
    for (int u = 0; u < TT; ++u) z[u] = *reinterpret_cast<const f32x4*>(b + c);
    for (int r = 0; r < R; ++r) {
        const f32x4 wr = *reinterpret_cast<const f32x4*>(w + (int64_t)r * C + c);
#pragma unroll
        for (int u = 0; u < TT; ++u) {
            const float av = a[(int64_t)min(t0 + u, T - 1) * R + r];
#pragma unroll
            for (int e = 0; e < 4; ++e) z[u][e] = __builtin_fmaf(av, wr[e], z[u][e]);
        }
    }
#pragma unroll
    for (int u = 0; u < TT; ++u) {
        if (t0 + u >= T) break;
        f32x4 v = z[u];
        if constexpr (POW4) v = decay_pow4(v, p);
        else
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = expf(logsigmoidf_(v[e]) * p);
        *reinterpret_cast<f32x4*>(out + (int64_t)(t0 + u) * C + c) = v;
    }
}

}  // namespace hy

// C % 4 == 0, w, b and out on 16 bytes
void launch_hy_low_rank_decay(const float* a, const float* w, const float* b, float* out, int T, int R, int C, float p, hipStream_t s) {
    if (T == 0 || C == 0) return;
    const int gx = (C / 4 + 255) / 256;
    const bool pow4 = p > 0.f && p <= 0.0625f;   // (as in launch_hy_decay_pow)
    // the workgroups of the same tokens side by side (8192 x 4096: 38 us, 40 the other way round) as long as the second axis holds the
    // tokens: the device states 65536 blocks for it
#define HY_LRD(TT) do { \
        const int gt = (T + TT - 1) / TT; \
        const bool tx = gt > 65535; \
        const dim3 grid(tx ? gt : gx, tx ? gx : gt); \
        if (pow4) hy::low_rank_decay_kernel<TT, true><<<grid, 256, 0, s>>>(a, w, b, out, T, R, C, p, tx); \
        else hy::low_rank_decay_kernel<TT, false><<<grid, 256, 0, s>>>(a, w, b, out, T, R, C, p, tx); \
    } while (0)
    if ((int64_t)gx * T >= 4096) HY_LRD(4);   // (four tokens a thread once that leaves four workgroups per CU)
    else HY_LRD(1);
#undef HY_LRD
}

// y == nullptr: plain norm of x (h in float when out_f32, else bfloat16).  Otherwise the joined form; y is in the
// activation type (float when out_f32), h may be nullptr (float activations read the stream itself).
void launch_hy_rms_norm(const void* y, float* x, const float* w, void* h, bool out_f32, int rows, int d, float alpha,
                        float eps, hipStream_t s) {
    if (rows == 0) return;
    const bool vec = d % 4 == 0;
#define HY_RN(TY, TH, JOIN)                                                                                           \
    do {                                                                                                              \
        if (vec) hy::rms_norm_kernel<TY, TH, JOIN, true><<<rows, 256, 0, s>>>((const TY*)y, x, w, (TH*)h, d, alpha, eps, nullptr, rows); \
        else hy::rms_norm_kernel<TY, TH, JOIN, false><<<rows, 256, 0, s>>>((const TY*)y, x, w, (TH*)h, d, alpha, eps, nullptr, rows);    \
    } while (0)
    if (y != nullptr) {
        if (out_f32) HY_RN(float, float, true);
        else HY_RN(uint16_t, uint16_t, true);
    } else {
        if (out_f32) HY_RN(float, float, false);
        else HY_RN(float, uint16_t, false);
    }
#undef HY_RN
}

// the plain norm of rows[0 .. n) of x's `total` rows, d % 4 == 0
void launch_hy_rms_norm_rows(const float* x, const int64_t* rows, int total, const float* w, void* h, bool out_f32, int n, int d, float eps,
                             hipStream_t s) {
    if (n == 0) return;
    float* const xs = const_cast<float*>(x);
    if (out_f32) hy::rms_norm_kernel<float, float, false, true><<<n, 256, 0, s>>>(nullptr, xs, w, (float*)h, d, 1.f, eps, rows, total);
    else hy::rms_norm_kernel<float, uint16_t, false, true><<<n, 256, 0, s>>>(nullptr, xs, w, (uint16_t*)h, d, 1.f, eps, rows, total);
}

void launch_hy_rms_norm_slices(const float* ys, int S, float* x, const float* w, uint16_t* h, int rows, int d, float alpha, float eps,
                               hipStream_t s) {
    if (rows == 0) return;
    const hy::Slices y{ys, S, (int64_t)rows * d};   // (d <= 8192)
    if (d <= 1024) hy::rms_norm_slices_kernel<256, 1><<<rows, 256, 0, s>>>(y, x, w, h, d, alpha, eps);
    else if (d <= 2048) hy::rms_norm_slices_kernel<512, 1><<<rows, 512, 0, s>>>(y, x, w, h, d, alpha, eps);
    else if (d <= 4096) hy::rms_norm_slices_kernel<1024, 1><<<rows, 1024, 0, s>>>(y, x, w, h, d, alpha, eps);
    else hy::rms_norm_slices_kernel<1024, 2><<<rows, 1024, 0, s>>>(y, x, w, h, d, alpha, eps);
}

// ldg, ldy: row strides of gu and y
void launch_hy_glu(const void* gu, int64_t ldg, void* y, int64_t ldy, int64_t rows, int F, float limit, float slope,
                   float shift, bool f32, hipStream_t s) {
    if (rows == 0 || F == 0) return;
    auto al = [&](const void* p) { return reinterpret_cast<uintptr_t>(p) % (f32 ? 16 : 8) == 0; };
    const bool vec = F % 4 == 0 && ldg % 4 == 0 && ldy % 4 == 0 && al(gu) && al(y);
    if (!f32 && F % 8 == 0 && (ldg | ldy) % 8 == 0 && hy::aligned16(gu, y)) {
        const int per = F / 8, nt = per < 256 ? (per + 63) / 64 * 64 : 256;
        hy::glu_vec_kernel<<<dim3((unsigned)rows, (per + nt - 1) / nt), nt, 0, s>>>((const uint16_t*)gu, ldg, (uint16_t*)y, ldy, F, limit, slope, shift);
        return;
    }
    const int per = vec ? F / 4 : F, nt = per < 256 ? (per + 63) / 64 * 64 : 256;
    const dim3 grid((unsigned)rows, (per + nt - 1) / nt);
#define HY_GLU(T, VEC) hy::glu_kernel<T, VEC><<<grid, nt, 0, s>>>((const T*)gu, ldg, (T*)y, ldy, F, limit, slope, shift)
    if (f32) { if (vec) HY_GLU(float, true); else HY_GLU(float, false); }
    else { if (vec) HY_GLU(uint16_t, true); else HY_GLU(uint16_t, false); }
#undef HY_GLU
}

void launch_hy_decay_pow(float* z, int64_t n, float p, hipStream_t s) {
    if (n == 0) return;
    if (p > 0.f && p <= 0.0625f && n % 4 == 0 && hy::aligned16(z)) {
        hy::decay_pow_vec_kernel<<<(unsigned)((n / 4 + 255) / 256), 256, 0, s>>>(reinterpret_cast<f32x4*>(z), n / 4, p);
        return;
    }
    hy::decay_pow_kernel<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(z, n, p);
}

}  // namespace chronos
