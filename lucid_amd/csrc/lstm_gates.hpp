// The gate functions of the LSTM kernels, one definition for all of them: which kernel takes a layer does not show in its bits.
#pragma once
#include "common.hpp"

namespace lq {

// They are on the chain of a step of the recurrence, so both are straight-line code (the library's expf and tanhf branch, and both
// sides run in a wavefront).  Against float64, 4 M points of each range, largest error in units of the last place and relative root
// mean square, in brackets 1 / (1 + expf(-x)) and tanhf:
//   sigmoid  -10 .. 10    2.02 (2.18)  3.1e-8 (3.8e-8)       tanh  -0.7 .. 0.7  1.25 (1.37)  2.8e-8 (2.9e-8)
//            -60 .. -10   1.64 (2.61)  2.9e-8 (3.7e-8)             -10 .. 10    1.19 (1.37)  1.88e-8 (1.93e-8)
//            -110 .. -60  0.89 (1.78 to -87; beyond -88.7 the library's is 0)
// Without the reduction to a whole and a fraction the exponential alone takes sigmoid to 2.77.

constexpr float kLog2e = 1.44269502f, kLog2eLow = 1.92596299e-8f, kLn2 = 0.693147182f;

// 1 / (1 + e) for 0 <= e <= 1: 1 - r is exact, so the correction sees no rounding of 1 + e
__device__ __forceinline__ float reciprocal_above_one(float e) {
    const float r = __builtin_amdgcn_rcpf(1.0f + e);
    return __builtin_fmaf(r, __builtin_fmaf(-r, e, 1.0f - r), r);
}
__device__ __forceinline__ float sigmoid(float x) {  // (a NaN fails the comparisons and stays one)
    const float a = __builtin_fabsf(x), to = a > 110.0f ? 110.0f : a;
    const float t = to * -kLog2e, whole = __builtin_rintf(t);
    const float low = __builtin_fmaf(to, -kLog2eLow, __builtin_fmaf(to, -kLog2e, -t));  // what t lost
    const float e = __builtin_ldexpf(__builtin_amdgcn_exp2f((t - whole) + low), int(whole));  // exp(-|x|), subnormals too
    const float s = reciprocal_above_one(e);
    return x < 0.0f ? e * s : s;
}
__device__ __forceinline__ float tanh_gate(float x) {
    const float a = __builtin_fabsf(x), u = x * x;
    // below 0.6 a + a^3 P(a^2): P fitted for the least relative error, 2.8e-9
    float q = __builtin_fmaf(u, -0x1.8257d2p-8f, 0x1.54b882p-6f);
    q = __builtin_fmaf(q, u, -0x1.b898dap-5f);
    q = __builtin_fmaf(q, u, 0x1.1109aep-3f);
    q = __builtin_fmaf(q, u, -0x1.55553ep-2f);
    const float small = __builtin_fmaf(a * u, q, a);
    // 1 - 2 e / (1 + e) with e = exp(-2 a); what t lost goes onto e itself
    const float a2 = a > 20.0f ? 40.0f : 2.0f * a, t = a2 * -kLog2e;
    const float low = __builtin_fmaf(a2, -kLog2eLow, __builtin_fmaf(a2, -kLog2e, -t)), e2 = __builtin_amdgcn_exp2f(t);
    const float e = __builtin_fmaf(e2, low * kLn2, e2);
    const float large = __builtin_fmaf(-2.0f * e, reciprocal_above_one(e), 1.0f);
    return __builtin_copysignf(a < 0.6f ? small : large, x);
}

}  // namespace lq
