// chronos_act.h — activations of the hybrid decoders' feed-forwards, for their own kernels and the epilogues of the projections.
#pragma once
#include <hip/hip_runtime.h>

namespace chronos {
namespace hy {

__device__ __forceinline__ float sigmoidf_(float z) { return 1.f / (1.f + expf(-z)); }

// sigmoidf_ for values that end up in activation type T.  For bfloat16 through the hardware's exponential and reciprocal, each with its
// remainder: e^-z = 2^h (1 + l), h the rounded product and l = -z - h ln 2, and one Newton step of the reciprocal that takes 2^h l along.
// Its error is that of the library's exponential and a division (units of float32's last place, largest and root mean square: z in -20 .. -6
// 2.5, 0.472, theirs 2.6, 0.476; -2 .. -0.1 2.1, 0.518 and 2.2, 0.520; 2 .. 20 1.5, 0.572 both), in half of the instructions; without the
// remainders it grows with |z|, to 64 units at -87.  The scale 2^-24 keeps what v_rcp_f32 would flush (z < -87.3).
template <typename T> __device__ __forceinline__ float sigmoid_act(float z) {
    if constexpr (sizeof(T) == 4) return sigmoidf_(z);
    else {
        constexpr float kLog2e = 1.44269504088896340736f, kLn2 = 0.693147182464599609375f, kLn2Low = -1.904654299957767e-9f;
        const float h = z * -kLog2e, e = __builtin_amdgcn_exp2f(h);
        const float l = __builtin_fmaf(h, -kLn2Low, __builtin_fmaf(h, -kLn2, -z));
        const float d = __builtin_fmaf(e, 0x1p-24f, 0x1p-24f), r = __builtin_amdgcn_rcpf(d);
        const float q = __builtin_fmaf(e * -0x1p-24f * l, r, __builtin_fmaf(-d, r, 1.f));
        return (fabsf(h) < 128.f ? __builtin_fmaf(q, r, r) : r) * 0x1p-24f;   // (beyond: 0, 1, or z's NaN)
    }
}

constexpr int kActRelu2 = 0, kActGelu = 1;
__device__ __forceinline__ float act_apply(float z, int kind) {
    if (kind == kActRelu2) {
        const float r = fmaxf(z, 0.f);
        return r * r;
    }
    return 0.5f * z * (1.f + erff(z * 0.70710678118654752440f));
}

}  // namespace hy
}  // namespace chronos
