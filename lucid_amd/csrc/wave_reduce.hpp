// Min / max over a wavefront through the vector unit's own lane moves (DPP): six steps of a few cycles
// each, where a butterfly of __shfl_xor sends every step through the LDS unit (about 100 cycles).
#pragma once
#include "common.hpp"

namespace lq {

namespace wave_reduce_detail {
// the value of another lane of the row / of an earlier row; lanes without a source keep their own
template <int CTRL, int ROWS>
__device__ __forceinline__ float dpp(float v) {
    const int b = int(__float_as_uint(v));
    return __uint_as_float(unsigned(__builtin_amdgcn_update_dpp(b, b, CTRL, ROWS, 0xf, false)));
}
template <bool MAX>
__device__ __forceinline__ float pick(float a, float b) { return MAX ? fmaxf(a, b) : fminf(a, b); }
// over each row of 16 lanes: lane 15 of the row holds the result
template <bool MAX>
__device__ __forceinline__ float row(float v) {
    v = pick<MAX>(v, dpp<0x111, 0xf>(v));  // row_shr 1, 2, 4, 8
    v = pick<MAX>(v, dpp<0x112, 0xf>(v));
    v = pick<MAX>(v, dpp<0x114, 0xf>(v));
    return pick<MAX>(v, dpp<0x118, 0xf>(v));
}
template <bool MAX>
__device__ __forceinline__ float wave(float v) {
    v = row<MAX>(v);
    v = pick<MAX>(v, dpp<0x142, 0xa>(v));  // row_bcast 15 into rows 1 and 3
    v = pick<MAX>(v, dpp<0x143, 0xc>(v));  // row_bcast 31 into rows 2 and 3: lane 63 holds the result
    return __uint_as_float(unsigned(__builtin_amdgcn_readlane(int(__float_as_uint(v)), 63)));
}
}  // namespace wave_reduce_detail

// NaNs are dropped (fminf / fmaxf); every lane gets the result.  All 64 lanes must be active.
__device__ __forceinline__ float wave_min(float v) { return wave_reduce_detail::wave<false>(v); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce_detail::wave<true>(v); }
__device__ __forceinline__ bool wave_any(int v) { return __builtin_amdgcn_ballot_w64(v != 0) != 0; }

// (lo, hi, nan) over a block of up to 1024 threads, every thread gets it.  One barrier; the LDS words are free
// again after the next one.
__device__ __forceinline__ void block_minmax(float& lo, float& hi, int& nan) {
    __shared__ float s_lo[16], s_hi[16];
    __shared__ int s_nan[16];
    lo = wave_min(lo), hi = wave_max(hi), nan = wave_any(nan);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = (blockDim.x + 63) >> 6;
    if (lane == 0) s_lo[wave] = lo, s_hi[wave] = hi, s_nan[wave] = nan;
    lds_barrier();
    const int w = (lane & 15) < waves ? lane & 15 : 0;
    lo = wave_reduce_detail::row<false>(s_lo[w]), hi = wave_reduce_detail::row<true>(s_hi[w]);
    lo = __uint_as_float(unsigned(__builtin_amdgcn_readlane(int(__float_as_uint(lo)), 15)));
    hi = __uint_as_float(unsigned(__builtin_amdgcn_readlane(int(__float_as_uint(hi)), 15)));
    nan = wave_any(s_nan[w]);
}

}  // namespace lq
