// hybrid_elementwise.hip — the float32 residual stream of the hybrid decoders: embedding rows, layer norm (weight, no
// bias) with the residual add fused, the few-row float32-output projections, activations.
//
// The sublayers' outputs are normalised and ADDED to the stream (x <- x + norm(y)), so the norm kernel reads the
// sublayer output in the activation type, does all its arithmetic in float, updates the float stream in place and
// emits the stream's copy in the activation type for the next sublayer's GEMMs (one pass, nothing re-read from HBM).
#include "hybrid_common.h"
#include "rowdot_tile.h"

namespace chronos {
namespace hy {

// h (or nullptr): the rows in bfloat16 as well.  pos0 (or nullptr) [B]: pos at every sequence's first token, which a prompt step's recurrences
// ask for; sequences without tokens read the next one's, or the last.  Here it costs nothing (three launches of torch's, 4.7 us each and 10 us of the host's
// time, which is what bounds prompts of a few hundred tokens).
template <typename T>
__global__ void __launch_bounds__(256) embed_kernel(const int32_t* __restrict__ ids, const T* __restrict__ table,
                                                    float* __restrict__ x, uint16_t* __restrict__ h, int d, float scale,
                                                    const int32_t* __restrict__ pos, const int32_t* __restrict__ q_start,
                                                    int32_t* __restrict__ pos0, int B) {
    const int64_t t = blockIdx.x;
    if (pos0 != nullptr && t == 0)
        for (int b = threadIdx.x; b < B; b += 256) pos0[b] = pos[min(max(q_start[b], 0), (int)gridDim.x - 1)];
    const T* src = table + (int64_t)ids[t] * d;
    if constexpr (sizeof(T) == 2) {
        if (d % 8 == 0 && ((reinterpret_cast<uintptr_t>(table) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(h)) & 15) == 0) {   // 8 columns a thread
            for (int i = threadIdx.x * 8; i < d; i += 2048) {
                float v[8];
                ld8(src + i, v);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] *= scale;
                st8f(x + t * d + i, v);
                if (h != nullptr) st8(h + t * d + i, v);
            }
            return;
        }
    }
    for (int i = threadIdx.x; i < d; i += blockDim.x) {
        const float v = ld<T>(src + i) * scale;
        x[t * d + i] = v;
        if (h != nullptr) h[t * d + i] = f2bf(v);
    }
}

// y [rows, d] (activation type, or float for the plain norm of the stream itself) -> float statistics in two passes
// (mean, then the mean of squared deviations), then
//   ADD:   x[row] += (y - mean) * rstd * w;   h[row] = T(x[row])   (h == nullptr: not written)
//   plain: h[row] = T((y - mean) * rstd * w)
template <typename TY, typename TH, bool ADD>
__global__ void __launch_bounds__(256) layer_norm_kernel(const TY* __restrict__ y, float* __restrict__ x,
                                                         const float* __restrict__ w, TH* __restrict__ h, int d,
                                                         float eps) {
    __shared__ float red[16];
    const int64_t row = blockIdx.x;
    const TY* yr = y + row * d;
    float s = 0.f;
    for (int i = threadIdx.x; i < d; i += 256) s += ld<TY>(yr + i);
    const float mean = block_sum(s, red) / (float)d;
    float q = 0.f;
    for (int i = threadIdx.x; i < d; i += 256) {
        const float c = ld<TY>(yr + i) - mean;
        q += c * c;
    }
    const float rstd = 1.f / sqrtf(block_sum(q, red) / (float)d + eps);
    for (int i = threadIdx.x; i < d; i += 256) {
        float v = (ld<TY>(yr + i) - mean) * rstd * w[i];
        if constexpr (ADD) {
            v += x[row * d + i];
            x[row * d + i] = v;
        }
        if (h != nullptr) st<TH>(h + row * d + i, v);
    }
}

// The plain norm of float rows of a multiple of 4 columns up to 4096, read once (the same three passes' arithmetic; 64 rows of 4096: 13.6 us in
// three strided passes, 5.0 so).
template <typename TH>
__global__ void __launch_bounds__(256) layer_norm_plain_kernel(const float* __restrict__ y, const float* __restrict__ w, TH* __restrict__ h,
                                                               int d, float eps, const int64_t* __restrict__ rows, int total) {
    __shared__ float red[16];
    const int64_t row = blockIdx.x, src = rows != nullptr ? rows[row] : row;
    const bool there = src >= 0 && src < total;
    f32x4 v[4];
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = (threadIdx.x + 256 * j) * 4;
        v[j] = i < d ? there ? *reinterpret_cast<const f32x4*>(y + src * d + i) : f32x4{NAN, NAN, NAN, NAN} : f32x4{0.f, 0.f, 0.f, 0.f};
        s += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
    }
    const float mean = block_sum(s, red) / (float)d;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
        if ((threadIdx.x + 256 * j) * 4 < d)
#pragma unroll
            for (int e = 0; e < 4; ++e) q += (v[j][e] - mean) * (v[j][e] - mean);
    const float rstd = 1.f / sqrtf(block_sum(q, red) / (float)d + eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int i = (threadIdx.x + 256 * j) * 4;
        if (i < d) {
            const f32x4 o = (v[j] - mean) * rstd * *reinterpret_cast<const f32x4*>(w + i);
            if constexpr (sizeof(TH) == 4) *reinterpret_cast<f32x4*>(h + row * d + i) = o;
            else *reinterpret_cast<u16x4*>(h + row * d + i) = u16x4{f2bf(o[0]), f2bf(o[1]), f2bf(o[2]), f2bf(o[3])};
        }
    }
}

// The added norm for bfloat16 rows of a multiple of 8 columns up to 8192, read once: a row's values (and the stream's) wait
// in registers between the statistics and the write, 8 columns per lane and step.  W waves share a row (1: four rows per
// workgroup, no barrier; 4: one row).  Bound by the bytes of y, x in and out and h: 8192 x 2048 takes 35 us (5.8 TB/s) where
// three strided passes took 68; 64 rows of 4096 take 5 us, not 14.
template <int W, int NV>
__global__ void __launch_bounds__(256) layer_norm_vec_kernel(const uint16_t* __restrict__ y, float* __restrict__ x, const float* __restrict__ w,
                                                             uint16_t* __restrict__ h, int rows, int d, float eps) {
    __shared__ float red[2][4];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t row = W == 1 ? (int64_t)blockIdx.x * 4 + wv : blockIdx.x;
    if (row >= rows) return;   // (W == 4: never)
    const int c0 = (W == 1 ? lane : threadIdx.x) * 8;
    constexpr int STEP = 64 * W * 8;
    float v[NV][8], xs[NV][8];
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + j * STEP;
        if (c < d) {
            ld8(y + row * d + c, v[j]);
            ld8f(x + row * d + c, xs[j]);
#pragma unroll
            for (int e = 0; e < 8; ++e) s += v[j][e];
        }
    }
    auto total = [&](float a, int k) {
        a = wave_sum(a);
        if constexpr (W == 4) {
            if (lane == 0) red[k][wv] = a;
            __syncthreads();
            a = (red[k][0] + red[k][1]) + (red[k][2] + red[k][3]);
        }
        return a;
    };
    const float mean = total(s, 0) / (float)d;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if (c0 + j * STEP < d)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float c = v[j][e] - mean;
                q += c * c;
            }
    const float rstd = 1.f / sqrtf(total(q, 1) / (float)d + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = c0 + j * STEP;
        if (c < d) {
            float wf[8];
            ld8f(w + c, wf);
#pragma unroll
            for (int e = 0; e < 8; ++e) xs[j][e] += (v[j][e] - mean) * rstd * wf[e];
            st8f(x + row * d + c, xs[j]);
            if (h != nullptr) st8(h + row * d + c, xs[j]);
        }
    }
}

// The same with y as S float32 slices [rows, d] of a product of few rows, summed in order and rounded here, d % 4 == 0 (a launch of 3 - 5 us less).  NT threads
// take a row, 4 columns each NJ times, everything that they read on its way before the first sum, as in post_norm.hip's.  64 rows of 4096 in 8
// slices 5.0 us with 256 threads, 4.3 so; of 8192 7.6 and 6.3.
template <int NT, int NJ>
__global__ void __launch_bounds__(NT) layer_norm_slices_kernel(const float* __restrict__ ys, int S, int64_t stride, float* __restrict__ x,
                                                               const float* __restrict__ w, uint16_t* __restrict__ h, int d, float eps) {
    __shared__ float red[2][NT / 64];
    const int64_t at = blockIdx.x * (int64_t)d;
    f32x4 v[NJ], xs[NJ], wv[NJ];
    bool in[NJ];
    auto total = [&](float a, int k) {
        a = wave_sum(a);
        if ((threadIdx.x & 63) == 0) red[k][threadIdx.x >> 6] = a;
        __syncthreads();
        a = 0.f;
#pragma unroll
        for (int i = 0; i < NT / 64; ++i) a += red[k][i];
        return a;
    };
    float s = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        in[j] = (int)(threadIdx.x + NT * j) * 4 < d;
        const int i = min((int)(threadIdx.x + NT * j) * 4, d - 4);   // (past the row: its last columns again, not counted)
        const float* const p = ys + at + i;
        v[j] = *reinterpret_cast<const f32x4*>(p);
        xs[j] = *reinterpret_cast<const f32x4*>(x + at + i);
        wv[j] = *reinterpret_cast<const f32x4*>(w + i);
#pragma unroll 4
        for (int k = 1; k < S; ++k) v[j] += *reinterpret_cast<const f32x4*>(p + k * stride);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[j][e] = bf2f(f2bf(v[j][e]));
        if (in[j]) s += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
    }
    const float mean = total(s, 0) / (float)d;
    float q = 0.f;
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (in[j])
#pragma unroll
            for (int e = 0; e < 4; ++e) q += (v[j][e] - mean) * (v[j][e] - mean);
    const float rstd = 1.f / sqrtf(total(q, 1) / (float)d + eps);
#pragma unroll
    for (int j = 0; j < NJ; ++j)
        if (in[j]) {
            const int64_t i = at + (threadIdx.x + NT * j) * 4;
            const f32x4 o = xs[j] + (v[j] - mean) * rstd * wv[j];
            *reinterpret_cast<f32x4*>(x + i) = o;
            *reinterpret_cast<u16x4*>(h + i) = u16x4{f2bf(o[0]), f2bf(o[1]), f2bf(o[2]), f2bf(o[3])};
        }
}

// out[t, n] = sum_k h[t, k] * w[n, k] (+ bias[n]) in float.  A workgroup takes TB tokens (their rows sit in LDS) and
// 4 output rows, one per wave: a weight row is read ONCE for all TB tokens, 16 bytes per lane when the row length
// allows (VEC), and the grid's second axis spreads the output rows over workgroups so a handful of decode rows still
// fills many CUs.
template <typename T> struct Vec16 { static constexpr int E = 16 / (int)sizeof(T); };
template <typename T> __device__ __forceinline__ void unpack16(const uint4& v, float* f);
template <> __device__ __forceinline__ void unpack16<uint16_t>(const uint4& v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __uint_as_float(w[i] << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}
template <> __device__ __forceinline__ void unpack16<float>(const uint4& v, float* f) {
    f[0] = __uint_as_float(v.x); f[1] = __uint_as_float(v.y); f[2] = __uint_as_float(v.z); f[3] = __uint_as_float(v.w);
}

template <typename T, int TB, bool VEC>
__global__ void __launch_bounds__(256) rowdot_kernel(const T* __restrict__ h, const T* __restrict__ w,
                                                     const float* __restrict__ bias, float* __restrict__ out, int rows,
                                                     int d, int n) {
    extern __shared__ __attribute__((aligned(16))) unsigned char rd_smem[];
    T* hs = reinterpret_cast<T*>(rd_smem);
    constexpr int E = Vec16<T>::E;
    const int64_t t0 = (int64_t)blockIdx.x * TB;
    const int nt = (int)min((int64_t)TB, rows - t0);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if constexpr (VEC) {
        const uint4* src = reinterpret_cast<const uint4*>(h + t0 * d);
        for (int i = threadIdx.x; i < nt * d / E; i += 256) reinterpret_cast<uint4*>(hs)[i] = src[i];
    } else {
        for (int i = threadIdx.x; i < nt * d; i += 256) hs[i] = h[t0 * d + i];
    }
    __syncthreads();
    const int r = blockIdx.y * 4 + wv;
    if (r >= n) return;
    const T* wr = w + (int64_t)r * d;
    float acc[TB];
#pragma unroll
    for (int u = 0; u < TB; ++u) acc[u] = 0.f;
    if constexpr (VEC) {
        for (int k = lane * E; k < d; k += 64 * E) {
            float wf[E];
            unpack16<T>(*reinterpret_cast<const uint4*>(wr + k), wf);
#pragma unroll
            for (int u = 0; u < TB; ++u)
                if (u < nt) {
                    float hf[E];
                    unpack16<T>(*reinterpret_cast<const uint4*>(hs + u * d + k), hf);
#pragma unroll
                    for (int i = 0; i < E; ++i) acc[u] += hf[i] * wf[i];
                }
        }
    } else {
        for (int k = lane; k < d; k += 64) {
            const float wk = ld<T>(wr + k);
#pragma unroll
            for (int u = 0; u < TB; ++u)
                if (u < nt) acc[u] += ld<T>(hs + u * d + k) * wk;
        }
    }
#pragma unroll
    for (int u = 0; u < TB; ++u) {
        const float v = wave_sum(acc[u]);
        if (lane == 0 && u < nt) out[(t0 + u) * n + r] = v + (bias != nullptr ? bias[r] : 0.f);
    }
}

// The same on the matrix cores, for bfloat16 rows of whole 64-element steps (products of bfloat16 pairs are exact in
// float32, and so are their sums' roundings: the precision of the kernel above).  A workgroup takes 16 TT tokens and 16 NT
// output rows and splits d over its NWV waves, 64 elements at a time, straight from memory into operands; the waves' sums
// meet in LDS.  Bound by reading h once (26 us for 8192 x 4096 by 64 rows, 2.6 TB/s; the kernel above reads every token's row
// from LDS once per output row: 268 us).  Errors against float64 are the same: chains of four matrix products.
template <int TT, int NT, int NWV>
__global__ void __launch_bounds__(64 * NWV) rowdot_mfma_kernel(const uint16_t* __restrict__ h, const uint16_t* __restrict__ w,
                                                               const float* __restrict__ bias, float* __restrict__ out, int rows,
                                                               int d, int n) {
    __shared__ f32x4 red[NWV][TT * NT][64];
    rowdot_tile<TT, NT, NWV>(h, w, bias, (int64_t)blockIdx.x * 16 * TT, blockIdx.y * 16 * NT, rows, d, n, red,
                             [&](int64_t t, int r, float v) { out[t * n + r] = v; });
}

template <typename T>
__global__ void __launch_bounds__(256) act_kernel(T* __restrict__ x, int64_t n, int kind) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) st<T>(x + i, act_apply(ld<T>(x + i), kind));
}

// 8 activations per thread, 16-byte loads and stores: 8192 x 8192 squared ReLUs in 44 us (6.1 TB/s) where one activation per
// thread took 127
__global__ void __launch_bounds__(256) act_vec_kernel(uint16_t* __restrict__ x, int64_t n8, int kind) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    float v[8];
    ld8(x + i * 8, v);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = act_apply(v[e], kind);
    st8(x + i * 8, v);
}

}  // namespace hy

void launch_hy_embed(const int32_t* ids, const void* table, float* x, uint16_t* h, int T, int d, float scale, bool f32, const int32_t* pos,
                     const int32_t* q_start, int32_t* pos0, int B, hipStream_t s) {
    if (T == 0) return;
    if (f32) hy::embed_kernel<float><<<T, 256, 0, s>>>(ids, (const float*)table, x, h, d, scale, pos, q_start, pos0, B);
    else hy::embed_kernel<uint16_t><<<T, 256, 0, s>>>(ids, (const uint16_t*)table, x, h, d, scale, pos, q_start, pos0, B);
}
// Row r of a norm over chosen rows: row rows[r] of the `total` there are (none of them: NaN, as memory past the stream is not its)
bool hy_rows_norm_ok(int d) { return d % 4 == 0 && d <= 4096; }
void launch_hy_layer_norm_rows(const float* x, const int64_t* rows, int total, const float* w, void* h, bool out_f32, int n, int d, float eps,
                               hipStream_t s) {
    if (n == 0) return;
    if (out_f32) hy::layer_norm_plain_kernel<float><<<n, 256, 0, s>>>(x, w, (float*)h, d, eps, rows, total);
    else hy::layer_norm_plain_kernel<uint16_t><<<n, 256, 0, s>>>(x, w, (uint16_t*)h, d, eps, rows, total);
}
// y_f32: the input is float (the plain norm of the stream); out_f32: h is float.  x == nullptr: plain norm.
void launch_hy_layer_norm(const void* y, bool y_f32, float* x, const float* w, void* h, bool out_f32, int rows, int d,
                          float eps, hipStream_t s) {
    if (rows == 0) return;
    if (x != nullptr && !y_f32 && d % 8 == 0 && d <= 8192 && hy::aligned16(y, x, w, h)) {
        const uint16_t* yb = (const uint16_t*)y;
        uint16_t* hb = (uint16_t*)h;
        if (d <= 1024) hy::layer_norm_vec_kernel<1, 2><<<(rows + 3) / 4, 256, 0, s>>>(yb, x, w, hb, rows, d, eps);
        else if (d <= 2048) hy::layer_norm_vec_kernel<4, 1><<<rows, 256, 0, s>>>(yb, x, w, hb, rows, d, eps);
        else if (d <= 4096) hy::layer_norm_vec_kernel<4, 2><<<rows, 256, 0, s>>>(yb, x, w, hb, rows, d, eps);
        else hy::layer_norm_vec_kernel<4, 4><<<rows, 256, 0, s>>>(yb, x, w, hb, rows, d, eps);
    } else if (x != nullptr) {
        if (y_f32) hy::layer_norm_kernel<float, float, true><<<rows, 256, 0, s>>>((const float*)y, x, w, (float*)h, d, eps);
        else hy::layer_norm_kernel<uint16_t, uint16_t, true><<<rows, 256, 0, s>>>((const uint16_t*)y, x, w, (uint16_t*)h, d, eps);
    } else if (y_f32 && d % 4 == 0 && d <= 4096 && hy::aligned16(y, w, h)) {
        if (out_f32) hy::layer_norm_plain_kernel<float><<<rows, 256, 0, s>>>((const float*)y, w, (float*)h, d, eps, nullptr, rows);
        else hy::layer_norm_plain_kernel<uint16_t><<<rows, 256, 0, s>>>((const float*)y, w, (uint16_t*)h, d, eps, nullptr, rows);
    } else {
        if (out_f32) hy::layer_norm_kernel<float, float, false><<<rows, 256, 0, s>>>((const float*)y, nullptr, w, (float*)h, d, eps);
        else hy::layer_norm_kernel<float, uint16_t, false><<<rows, 256, 0, s>>>((const float*)y, nullptr, w, (uint16_t*)h, d, eps);
    }
}
// d % 8 == 0, d <= 8192, everything on 16 bytes
void launch_hy_layer_norm_slices(const float* ys, int S, float* x, const float* w, uint16_t* h, int rows, int d, float eps, hipStream_t s) {
    if (rows == 0) return;
    const int64_t n = (int64_t)rows * d;
    if (d <= 1024) hy::layer_norm_slices_kernel<256, 1><<<rows, 256, 0, s>>>(ys, S, n, x, w, h, d, eps);
    else if (d <= 2048) hy::layer_norm_slices_kernel<512, 1><<<rows, 512, 0, s>>>(ys, S, n, x, w, h, d, eps);
    else if (d <= 4096) hy::layer_norm_slices_kernel<1024, 1><<<rows, 1024, 0, s>>>(ys, S, n, x, w, h, d, eps);
    else hy::layer_norm_slices_kernel<1024, 2><<<rows, 1024, 0, s>>>(ys, S, n, x, w, h, d, eps);
}
template <typename T>
static void rowdot_t(const T* h, const T* w, const float* bias, float* out, int rows, int d, int n, hipStream_t s) {
    // tokens per workgroup: as many (up to 8) as keep the staged rows within 48 KB
    const int fit = (48 * 1024) / (d * (int)sizeof(T));
    const bool vec = d % hy::Vec16<T>::E == 0;
    const int ny = (n + 3) / 4;
#define HY_RD(TB)                                                                                                  \
    do {                                                                                                           \
        const dim3 grid((rows + TB - 1) / TB, ny);                                                                 \
        if (vec) hy::rowdot_kernel<T, TB, true><<<grid, 256, TB * d * sizeof(T), s>>>(h, w, bias, out, rows, d, n); \
        else hy::rowdot_kernel<T, TB, false><<<grid, 256, TB * d * sizeof(T), s>>>(h, w, bias, out, rows, d, n);    \
    } while (0)
    if (fit >= 8 && rows >= 8) HY_RD(8);
    else if (fit >= 4 && rows >= 4) HY_RD(4);
    else if (fit >= 2 && rows >= 2) HY_RD(2);
    else {
        auto kern = hy::rowdot_kernel<T, 1, false>;
        const int bytes = d * (int)sizeof(T);
        if (bytes > 48 * 1024)
            (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
        kern<<<dim3(rows, ny), 256, bytes, s>>>(h, w, bias, out, rows, d, n);
    }
#undef HY_RD
}

// Few tokens: 16 output rows per workgroup and d over 16 waves, so that a decode row's chain is short and its workgroups are
// many; more: up to 64 output rows, and two tiles of tokens where that leaves a workgroup per CU, to read w less often.
template <int TT, int NT, int NWV>
static void rowdot_mfma(const uint16_t* h, const uint16_t* w, const float* bias, float* out, int rows, int d, int n, hipStream_t s) {
    const dim3 grid((rows + 16 * TT - 1) / (16 * TT), (n + 16 * NT - 1) / (16 * NT));
    hy::rowdot_mfma_kernel<TT, NT, NWV><<<grid, 64 * NWV, 0, s>>>(h, w, bias, out, rows, d, n);
}

void launch_hy_rowdot(const void* h, const void* w, const float* bias, float* out, int T, int d, int n, bool f32,
                      hipStream_t s) {
    if (T == 0 || n == 0) return;
    // (us, vector ALUs / matrix cores: 16 tokens of 1024 by 8 rows 5.1 / 3.5, of 2048 by 200 rows 7.5 / 5.7, of 4096 by 64 rows
    // 6.8 / 9.0; 200 tokens of 4096 by 64 rows 8.2 / 9.2; 1 token of it 9.8 / 6.1, 1024 tokens 28 / 20, 8192 tokens 268 / 26:
    // a workgroup's 16 tokens share one CU's loads, which a few tokens of long rows would rather spread)
    const bool spread = d > 2048 && T >= 2 && T <= 256;
    if (!f32 && d % 64 == 0 && !spread && (((uintptr_t)h | (uintptr_t)w) & 15) == 0) {
        const uint16_t *hb = (const uint16_t*)h, *wb = (const uint16_t*)w;
        if (T <= 512) rowdot_mfma<1, 1, 16>(hb, wb, bias, out, T, d, n, s);
        else if (n <= 16) rowdot_mfma<1, 1, 8>(hb, wb, bias, out, T, d, n, s);
        else if (n <= 32) rowdot_mfma<1, 2, 8>(hb, wb, bias, out, T, d, n, s);
        else if (T < 4096) rowdot_mfma<1, 4, 8>(hb, wb, bias, out, T, d, n, s);
        else rowdot_mfma<2, 4, 8>(hb, wb, bias, out, T, d, n, s);
        return;
    }
    if (f32) rowdot_t<float>((const float*)h, (const float*)w, bias, out, T, d, n, s);
    else rowdot_t<uint16_t>((const uint16_t*)h, (const uint16_t*)w, bias, out, T, d, n, s);
}
void launch_hy_act(void* x, int64_t n, int kind, bool f32, hipStream_t s) {
    if (n == 0) return;
    if (!f32 && n % 8 == 0 && hy::aligned16(x)) {
        hy::act_vec_kernel<<<(unsigned)((n / 8 + 255) / 256), 256, 0, s>>>((uint16_t*)x, n / 8, kind);
        return;
    }
    const int64_t blocks = (n + 255) / 256;
    if (f32) hy::act_kernel<float><<<(unsigned)blocks, 256, 0, s>>>((float*)x, n, kind);
    else hy::act_kernel<uint16_t><<<(unsigned)blocks, 256, 0, s>>>((uint16_t*)x, n, kind);
}

}  // namespace chronos
