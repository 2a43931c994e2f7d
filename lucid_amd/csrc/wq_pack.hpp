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

// The codes of instruction i of a window as an operand; slots 2d and 2d + 1 pair code d with code d + 4 (4-bit) or
// are codes 2d and 2d + 1.  A code c enters as (c + centre) / unit, and the centre is taken out again with the bias: with
// centre = -2^(bits-1) the sums stay as small as the products are.  4 bits: with the top bit flipped a nibble is
// the signed code, and v_cvt_off_f32_i4 gives a sixteenth of that as a float whose upper half is the bfloat16.  8 bits: the
// signed byte as a float, likewise.
// PATTERN (4 bits): c as the bit pattern 0x4300 | c = 128 + c, which needs no conversion (8 instructions in place of 14): the
// calls that have always had it, 2 .. 64 rows of whole windows, keep their bits.  Its sums grow with the mean of x and are
// cancelled by the bias afterwards: against float64, K = 4096, groups of 128, relative, x normal / after a ReLU: 8e-6 / 4e-5,
// 8 bits uncentred 4e-7 / 1.4e-6; centred 1.5e-7 / 3e-7, and 1e-6 when the weight is decoded first.
template <int BITS>
constexpr int kWqCentre = -(1 << (BITS - 1));
template <int BITS>
constexpr float kWqUnit = BITS == 4 ? 16.0f : 1.0f;  // (not of PATTERN)

template <int BITS, bool PATTERN = false>
__device__ __forceinline__ uint4 wq_codes(const uint32_t (&wd)[4], int i) {
    static_assert(!PATTERN || BITS == 4, "");
    auto upper = [](float lo, float hi) { return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u); };
    uint4 f;
    if constexpr (PATTERN) {
        const uint32_t c = wd[i];
        uint32_t mask = 0x000f000fu, one = 0x43004300u;
        asm("" : "+s"(mask));  // in registers: an AND-OR takes one literal at most
        asm("" : "+v"(one));
        f.x = (c & mask) | one;
        f.y = ((c >> 4) & mask) | one;
        f.z = ((c >> 8) & mask) | one;
        f.w = ((c >> 12) & mask) | one;
    } else if constexpr (BITS == 4) {
        const uint32_t even = wd[i] ^ 0x88888888u, odd = even >> 4;
        auto at = [](uint32_t w, int byte) { return __builtin_amdgcn_cvt_off_f32_i4(int((w >> (8 * byte)) & 0xffu)); };
        f.x = upper(at(even, 0), at(even, 2));
        f.y = upper(at(odd, 0), at(odd, 2));
        f.z = upper(at(even, 1), at(even, 3));
        f.w = upper(at(odd, 1), at(odd, 3));
    } else {
        const uint32_t a = wd[(2 * i) & 3] ^ 0x80808080u, b = wd[(2 * i + 1) & 3] ^ 0x80808080u;
        auto at = [](uint32_t w, int byte) { return float(int8_t((w >> (8 * byte)) & 0xffu)); };
        f.x = upper(at(a, 0), at(a, 1));
        f.y = upper(at(a, 2), at(a, 3));
        f.z = upper(at(b, 0), at(b, 1));
        f.w = upper(at(b, 2), at(b, 3));
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
