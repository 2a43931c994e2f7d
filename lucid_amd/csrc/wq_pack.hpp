// How packed codes meet the bfloat16 matrix instruction: shared by the small-batch and the
// large-batch weight-only products.
#pragma once
#include "common.hpp"

namespace lq {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));

template <int BITS>
struct WqGeom {
    static constexpr int CODES = 128 / BITS;  // codes per 16-byte load: 32 or 16
    static constexpr int WK = 4 * CODES;      // k per window: 128 or 64
    static constexpr int NI = WK / 32;        // instructions (k steps of 32) per window: 4 or 2
};

// How the registers are exchanged for a group size: 0 = not at all, 1 = between lane halves,
// 2 = transposed; the window then holds 1, 2 or 4 group segments.
__host__ __device__ inline int wq_swap_mode(int bits, int gs) {
    const int window = 512 / bits;
    return gs >= window ? 0 : (gs * 2 == window ? 1 : 2);
}

// After the exchange, register rho of quarter q holds what quarter q_src loaded as register j_src.
__host__ __device__ inline void wq_source(int sw, int rho, int q, int& q_src, int& j_src) {
    q_src = q, j_src = rho;
    if (sw == 1 && (rho < 2) != (q < 2)) {
        q_src = rho < 2 ? q - 2 : q + 2;
        j_src = rho < 2 ? rho + 2 : rho - 2;
    } else if (sw == 2) {
        q_src = rho, j_src = q;
    }
}

// upper lane half of a <-> lower lane half of b
__device__ __forceinline__ void wq_swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0], b = r[1];
}
// odd 16-lane rows of a <-> even 16-lane rows of b
__device__ __forceinline__ void wq_swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0], b = r[1];
}
template <int SW>
__device__ __forceinline__ void wq_exchange(uint32_t (&wd)[4]) {
    if (SW >= 1) wq_swap32(wd[0], wd[2]), wq_swap32(wd[1], wd[3]);
    if (SW == 2) wq_swap16(wd[0], wd[1]), wq_swap16(wd[2], wd[3]);
}

// The codes of instruction i of a window as an operand.  A byte as a float has zeros below bit 16: its
// upper half is the bfloat16.  A 4-bit code enters as OFF + c, for which a bit pattern needs no
// conversion: 0x4180 | c << 3 = 16 + c, or 0x4300 | c = 128 + c; slots 2d and 2d + 1 pair nibble d with
// nibble d + 4.  What the offset adds to the sums is taken out again with the bias, and the larger it is
// the more of the sums' precision goes with it: against float64, relative, 1e-6 with 16 and 5e-6 with 128.
template <int BITS, int OFF>
__device__ __forceinline__ uint4 wq_codes(const uint32_t (&wd)[4], int i) {
    static_assert(BITS == 8 ? OFF == 0 : (OFF == 16 || OFF == 128), "");
    constexpr int SH = OFF == 16 ? 3 : 0;  // where the nibble goes in its half word
    uint4 f;
    if (BITS == 4) {
        const uint32_t c = wd[i];
        uint32_t mask = 0x000f000fu << SH, one = OFF == 16 ? 0x41804180u : 0x43004300u;
        asm("" : "+s"(mask));  // in registers: an AND-OR takes one literal at most
        asm("" : "+v"(one));
        f.x = ((c << SH) & mask) | one;
        f.y = ((c >> (4 - SH)) & mask) | one;
        f.z = ((c >> (8 - SH)) & mask) | one;
        f.w = ((c >> (12 - SH)) & mask) | one;
    } else {
        const uint32_t a = wd[(2 * i) & 3], b = wd[(2 * i + 1) & 3];
        const uint32_t a0 = __float_as_uint(float(a & 0xffu)), a1 = __float_as_uint(float((a >> 8) & 0xffu));
        const uint32_t a2 = __float_as_uint(float((a >> 16) & 0xffu)), a3 = __float_as_uint(float(a >> 24));
        const uint32_t b0 = __float_as_uint(float(b & 0xffu)), b1 = __float_as_uint(float((b >> 8) & 0xffu));
        const uint32_t b2 = __float_as_uint(float((b >> 16) & 0xffu)), b3 = __float_as_uint(float(b >> 24));
        f.x = __builtin_amdgcn_perm(a1, a0, 0x07060302u);
        f.y = __builtin_amdgcn_perm(a3, a2, 0x07060302u);
        f.z = __builtin_amdgcn_perm(b1, b0, 0x07060302u);
        f.w = __builtin_amdgcn_perm(b3, b2, 0x07060302u);
    }
    return f;
}

// (e0, e1) = h + m + l part by part, each part a pair of bfloat16 (e0's in the low half): the
// packed conversion rounds to nearest, the remainders are exact (8 + 8 + 8 significant bits with
// signed remainders).  A NaN stays a NaN in every part; an infinity turns into a NaN in the
// lower parts, so a non-finite x gives a non-finite y.
typedef __bf16 wq_bf2 __attribute__((ext_vector_type(2)));
typedef float wq_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t wq_pk(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(wq_f2{a, b}, wq_bf2));
}
__device__ __forceinline__ void wq_split3x2(float e0, float e1, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = wq_pk(e0, e1);
    e0 -= __uint_as_float(h << 16), e1 -= __uint_as_float(h & 0xffff0000u);
    m = wq_pk(e0, e1);
    e0 -= __uint_as_float(m << 16), e1 -= __uint_as_float(m & 0xffff0000u);
    l = wq_pk(e0, e1);
}

}  // namespace

// Large-batch product (wq_gemm.hip), and whether it is the faster of the two for a problem.
bool wq_gemm_beats_small_batch(int M, int N, int K, int gs, int bits);
int launch_wq_gemm(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N,
                   int K, int gs, int bits, float* out, hipStream_t st);
}  // namespace lq
