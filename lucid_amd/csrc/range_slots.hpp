// Running min / max of a tensor kept by the kernel that produces it, so that a
// dynamic quantizer downstream needs no pass of its own over the tensor.
//
// A range buffer is kRangeWords 32-bit words: word 0 = number of partial slots
// in use, then kRangeSlots minima and kRangeSlots maxima.  Every block of the
// producing kernel writes its own slot (no atomics, nothing to initialise);
// the consumer reduces the slots.  fminf / fmaxf drop NaNs, so a block that saw
// a NaN stores NaN in both of its slots and the reduction propagates it (the
// reference's reductions propagate NaN, lucid/_C/backend/cpu/Reduce.cpp:87-125).
// min and max are exact and order-independent, so the result is bit-identical
// to a separate min / max pass.
#pragma once
#include "wave_reduce.hpp"

namespace lq {

constexpr int kRangeSlots = 16384;
constexpr int kRangeWords = 4 + 2 * kRangeSlots;

// Folds one (lo, hi, nan) per lane of a block (up to 1024 threads) into the
// block's slot.  All threads of the block must call it; gridDim.x * gridDim.y
// must not exceed kRangeSlots.
__device__ __forceinline__ void range_block_store(float* range, float lo, float hi, int nan) {
    block_minmax(lo, hi, nan);
    if (threadIdx.x == 0) {
        if (nan) lo = hi = __builtin_nanf("");
        const unsigned slot = blockIdx.y * gridDim.x + blockIdx.x;
        range[4 + slot] = lo;
        range[4 + kRangeSlots + slot] = hi;
        if (slot == 0) reinterpret_cast<unsigned*>(range)[0] = gridDim.x * gridDim.y;
    }
}

// The range a lane keeps of what it writes: IEEE 754-2019 minimum / maximum, which a NaN passes through (one
// v_minimum3_f32 / v_maximum3_f32 per two values; fminf / fmaxf beside a NaN flag take five instructions per value).
struct RangeKeep {
    float lo = __builtin_inff(), hi = -__builtin_inff();
    __device__ __forceinline__ void add(float y) {
        lo = __builtin_elementwise_minimum(lo, y);
        hi = __builtin_elementwise_maximum(hi, y);
    }
    __device__ __forceinline__ void store(float* range) const { range_block_store(range, lo, hi, lo != lo); }
};

// The range itself, for every thread of a block (up to 1024; all must call it): the reduction of the slots.  The first
// AHEAD slots of each thread are requested together with their number, which would otherwise be a memory round trip
// before them (they are words of the buffer in any case; what lies past the number is not looked at).
template <int AHEAD>
__device__ __forceinline__ void range_block_load(const float* __restrict__ range, float& mn, float& mx) {
    static_assert(AHEAD * 1024 <= kRangeSlots, "within the buffer for blocks of up to 1024 threads");
    float a[AHEAD], b[AHEAD];
#pragma unroll
    for (int u = 0; u < AHEAD; ++u) {
        const unsigned i = threadIdx.x + u * blockDim.x;
        a[u] = range[4 + i], b[u] = range[4 + kRangeSlots + i];
    }
    const unsigned n = reinterpret_cast<const unsigned*>(range)[0];
    float lo = __builtin_inff(), hi = -__builtin_inff();
    auto add = [&](float x, float y) {
        lo = __builtin_elementwise_minimum(lo, x);
        hi = __builtin_elementwise_maximum(hi, y);
    };
#pragma unroll
    for (int u = 0; u < AHEAD; ++u)
        if (threadIdx.x + u * blockDim.x < n) add(a[u], b[u]);
    for (unsigned i = threadIdx.x + AHEAD * blockDim.x; i < n; i += blockDim.x) add(range[4 + i], range[4 + kRangeSlots + i]);
    int nan = (lo != lo) | (hi != hi);
    block_minmax(lo, hi, nan);
    mn = nan ? __builtin_nanf("") : lo, mx = nan ? __builtin_nanf("") : hi;
}

// vDSP_vmax / vDSP_vmin single precision propagate NaN (Vdsp.cpp:140-151).
__device__ __forceinline__ float vmaxf(float a, float b) {
    if (a != a || b != b) return __builtin_nanf("");
    return a > b ? a : b;
}
__device__ __forceinline__ float vminf(float a, float b) {
    if (a != a || b != b) return __builtin_nanf("");
    return a < b ? a : b;
}

// lucid/quantization/_qparams.py:198-215, float32 throughout.
__device__ __forceinline__ void qparams_of(float mn, float mx, int symmetric, int qmin, int qmax,
                                           int is_signed, float eps, float half_range, float* scale,
                                           float* zp) {
    float lo = vminf(mn, 0.0f);
    float hi = vmaxf(mx, 0.0f);
    if (symmetric) {
        float max_abs = vmaxf(fabsf(lo), fabsf(hi));
        *scale = vmaxf(max_abs / half_range, eps);
        *zp = is_signed ? 0.0f : float((qmax + qmin + 1) >> 1);
    } else {
        float s = vmaxf((hi - lo) / float(qmax - qmin), eps);
        float z = float(qmin) - __builtin_rintf(lo / s);
        float qlo = float(qmin), qhi = float(qmax);
        z = (z < qlo) ? qlo : ((z > qhi) ? qhi : z);
        *scale = s;
        *zp = z;
    }
}

}  // namespace lq
