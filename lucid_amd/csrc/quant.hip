// quantize / dequantize / fake_quantize / min-max / calculate_qparams for
// gfx950.  All of them are HBM-bound: the kernels issue 128-bit loads that a
// wavefront covers contiguously, keep several loads in flight per lane, and
// do the arithmetic in the order Lucid's CPU path does it
// (lucid/quantization/_functional.py:180, 281, 311-313): IEEE division,
// round-half-even, add zero point, clamp, cast.  No reciprocal, no FMA.
#include <mutex>
#include <type_traits>
#include "common.hpp"
#include "qgemm.hpp"
#include "range_slots.hpp"

using namespace lq;

namespace {

constexpr int kThreads = 256;

// Streaming access: float values are touched once, so their loads and stores carry the
// non-temporal hint and do not displace what is still needed in L2 / Infinity Cache.
// (Measured on MI355X: 5 B/element quantize 239 us -> 207 us on 268 M elements.)
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ float4 nt_load(const float4* p) {
    f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4*>(p));
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void nt_store(float4* p, float4 v) {
    f32x4 t = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(t, reinterpret_cast<f32x4*>(p));
}

// ---------------------------------------------------------------- element math
// clip keeps NaN (CpuBackend.h:6880-6891); the float->int cast maps NaN to 0.
__device__ __forceinline__ float q_core(float x, float s, float z, float lo, float hi) {
    float t = x / s;
    float r = __builtin_rintf(t);
    float u = r + z;
    u = (u < lo) ? lo : ((u > hi) ? hi : u);
    return u;
}

__device__ __forceinline__ int to_code(float c) { return (c != c) ? 0 : int(c); }

// rint(x / s) without dividing, bit-identical to the division.
// t0 = x * r with r = fl(1/s) is within 3 * 2^-24 * |x/s| of the correctly
// rounded quotient.  If t0 is further than that (with margin) from the nearest
// half-integer, both round to the same integer.  Otherwise - ties, near-ties,
// huge, infinite or NaN quotients - the lane redoes the IEEE division.
__device__ __forceinline__ bool rint_quotient_safe(float t0, float n) {
    const float frac = __builtin_fabsf(t0 - n);  // <= 0.5
    // false for NaN / inf t0 as well
    return (0.5f - frac) > 4.0e-7f * __builtin_fabsf(t0) && __builtin_fabsf(t0) < 4.0e6f;
}

__device__ __forceinline__ float clamp_code(float r, float z, float lo, float hi) {
    float u = r + z;
    return (u < lo) ? lo : ((u > hi) ? hi : u);
}

// four quotients at once; `r` is fl(1/s)
__device__ __forceinline__ float4 rint_div4(float4 v, float4 s, float4 r) {
    float4 t = {v.x * r.x, v.y * r.y, v.z * r.z, v.w * r.w};
    float4 n = {__builtin_rintf(t.x), __builtin_rintf(t.y), __builtin_rintf(t.z), __builtin_rintf(t.w)};
    // branch-free conjunction: the four tests are evaluated unconditionally
    const bool ok = (int(rint_quotient_safe(t.x, n.x)) & int(rint_quotient_safe(t.y, n.y)) &
                     int(rint_quotient_safe(t.z, n.z)) & int(rint_quotient_safe(t.w, n.w))) != 0;
    if (__builtin_expect(!ok, 0)) {
        n.x = __builtin_rintf(v.x / s.x);
        n.y = __builtin_rintf(v.y / s.y);
        n.z = __builtin_rintf(v.z / s.z);
        n.w = __builtin_rintf(v.w / s.w);
    }
    return n;
}

__device__ __forceinline__ float4 splat(float v) { return float4{v, v, v, v}; }

struct alignas(4) Code8x4 {
    int8_t v[4];
};
struct alignas(8) Code16x4 {
    int16_t v[4];
};

__device__ __forceinline__ Code8x4 nt_load(const Code8x4* p) {
    unsigned w = __builtin_nontemporal_load(reinterpret_cast<const unsigned*>(p));
    Code8x4 c;
    __builtin_memcpy(&c, &w, 4);
    return c;
}
__device__ __forceinline__ Code16x4 nt_load(const Code16x4* p) {
    u32x2 w = __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(p));
    Code16x4 c;
    __builtin_memcpy(&c, &w, 8);
    return c;
}

template <typename CodeT>
struct CodeVec;
template <>
struct CodeVec<int8_t> {
    using type = Code8x4;
};
template <>
struct CodeVec<int16_t> {
    using type = Code16x4;
};

// ---------------------------------------------------------------- segment ops
// Each op works on groups of four consecutive elements ("quads") that share
// one (scale, zero_point).
template <typename CodeT>
struct QuantizeOp {
    using In = float4;
    using Vec = typename CodeVec<CodeT>::type;
    const float4* __restrict__ x;
    Vec* __restrict__ q;
    float lo, hi;
    int off;
    __device__ __forceinline__ In load(size_t i) const { return nt_load(&x[i]); }
    static constexpr int kMaxU = 2;  // loads in flight per lane; measured best for 4 B in / 1 B out
    static constexpr bool kDivides = true;
    __device__ __forceinline__ Vec pack(In v, float4 s, float4 z, float4 r) const {
        const float4 n = rint_div4(v, s, r);
        Vec o;
        o.v[0] = CodeT(to_code(clamp_code(n.x, z.x, lo, hi)) + off);
        o.v[1] = CodeT(to_code(clamp_code(n.y, z.y, lo, hi)) + off);
        o.v[2] = CodeT(to_code(clamp_code(n.z, z.z, lo, hi)) + off);
        o.v[3] = CodeT(to_code(clamp_code(n.w, z.w, lo, hi)) + off);
        return o;
    }
    __device__ __forceinline__ Vec pack(In v, float s, float z, float r) const {
        return pack(v, splat(s), splat(z), splat(r));
    }
    // Codes are stored with no hint, unlike what this file streams otherwise: a GEMM or a dequantize reads
    // them next.  (2048 x 8192 onto 4096 with per-token scales 96.6 -> 90.5 us; range + quantize + dequantize of
    // 64 Mi elements 157 -> 152, of 16 Mi 52.7 -> 50.6, of 256 Mi, whose codes no cache holds, 597 -> 590.  2048 x 4096 onto 11008 with
    // per-token scales, an output of 45 MB: 81.5 -> 82.1 over 16 random placements of its buffers, 87.7 -> 93.5 in one that was found; a quantization
    // whose codes nobody reads: 16 Mi elements 16.3 -> 15.6, rows of 8192 x 16384 122 -> 131.)
    __device__ __forceinline__ void store(size_t i, In v, float4 s, float4 z, float4 r) const { q[i] = pack(v, s, z, r); }
    // scalar tail / generic path
    __device__ __forceinline__ void scalar(size_t e, float s, float z) const {
        const float* xs = reinterpret_cast<const float*>(x);
        CodeT* qs = reinterpret_cast<CodeT*>(q);
        qs[e] = CodeT(to_code(q_core(xs[e], s, z, lo, hi)) + off);
    }
};

template <typename CodeT>
struct DequantizeOp {
    using Vec = typename CodeVec<CodeT>::type;
    using In = Vec;
    static constexpr int kMaxU = 8;
    static constexpr bool kDivides = false;
    const Vec* __restrict__ q;
    float4* __restrict__ out;
    int off;
    __device__ __forceinline__ In load(size_t i) const { return nt_load(&q[i]); }
    __device__ __forceinline__ void store(size_t i, In v, float4 s, float4 z, float4) const {
        float4 o;
        o.x = (float(int(v.v[0]) - off) - z.x) * s.x;
        o.y = (float(int(v.v[1]) - off) - z.y) * s.y;
        o.z = (float(int(v.v[2]) - off) - z.z) * s.z;
        o.w = (float(int(v.v[3]) - off) - z.w) * s.w;
        nt_store(&out[i], o);
    }
    __device__ __forceinline__ void scalar(size_t e, float s, float z) const {
        const CodeT* qs = reinterpret_cast<const CodeT*>(q);
        float* os = reinterpret_cast<float*>(out);
        os[e] = (float(int(qs[e]) - off) - z) * s;
    }
};

struct FakeQuantizeOp {
    using In = float4;
    static constexpr int kMaxU = 4;
    static constexpr bool kDivides = true;
    const float4* __restrict__ x;
    float4* __restrict__ out;
    float lo, hi;
    __device__ __forceinline__ In load(size_t i) const { return nt_load(&x[i]); }
    __device__ __forceinline__ void store(size_t i, In v, float4 s, float4 z, float4 r) const {
        const float4 n = rint_div4(v, s, r);
        float4 o;
        o.x = (clamp_code(n.x, z.x, lo, hi) - z.x) * s.x;
        o.y = (clamp_code(n.y, z.y, lo, hi) - z.y) * s.y;
        o.z = (clamp_code(n.z, z.z, lo, hi) - z.z) * s.z;
        o.w = (clamp_code(n.w, z.w, lo, hi) - z.w) * s.w;
        nt_store(&out[i], o);
    }
    __device__ __forceinline__ void scalar(size_t e, float s, float z) const {
        const float* xs = reinterpret_cast<const float*>(x);
        float* os = reinterpret_cast<float*>(out);
        os[e] = (q_core(xs[e], s, z, lo, hi) - z) * s;
    }
};

struct QParams {
    const float* scale;  // device, length C, or nullptr -> use the by-value pair
    const float* zp;
    float s_host, z_host;
};

// One block = one chunk of U*256 quads inside one [outer][C] segment, so the
// (scale, zero_point) pair is uniform across the block.  All U loads are
// issued before the first store.
// `tail` elements (a single segment only) behind its last quad are left to the first block.
template <typename Op, int U>
__global__ __launch_bounds__(kThreads) void seg_kernel(Op op, size_t inner4, unsigned tail,
                                                       unsigned chunks_per_seg, size_t C,
                                                       QParams qp) {
    const size_t seg = blockIdx.x / chunks_per_seg;
    const unsigned chunk = blockIdx.x - unsigned(seg * chunks_per_seg);
    float s, z;
    if (qp.scale) {
        const size_t c = seg % C;
        s = qp.scale[c];
        z = qp.zp[c];
    } else {
        s = qp.s_host;
        z = qp.z_host;
    }
    const float r = 1.0f / s;  // once per lane; the per-element quotients use it under a guard
    if (blockIdx.x == 0 && threadIdx.x < tail) op.scalar(inner4 * 4 + threadIdx.x, s, z);
    const size_t base = seg * inner4;
    const size_t i0 = size_t(chunk) * (U * kThreads) + threadIdx.x;
    typename Op::In v[U];
    if (size_t(chunk + 1) * (U * kThreads) <= inner4) {  // whole chunk in range: no predicates
#pragma unroll
        for (int j = 0; j < U; ++j) v[j] = op.load(base + i0 + size_t(j) * kThreads);
#pragma unroll
        for (int j = 0; j < U; ++j) op.store(base + i0 + size_t(j) * kThreads, v[j], splat(s), splat(z), splat(r));
        return;
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
        size_t i = i0 + size_t(j) * kThreads;
        if (i < inner4) v[j] = op.load(base + i);
    }
#pragma unroll
    for (int j = 0; j < U; ++j) {
        size_t i = i0 + size_t(j) * kThreads;
        if (i < inner4) op.store(base + i, v[j], splat(s), splat(z), splat(r));
    }
}

// Segments that no block can have to itself (short, or not whole quads; the channel-last layouts among them): quads
// of consecutive elements whatever segment they are of.  CHANNELS: most channels a quad can be of - 2 where a segment is
// at least 4 elements, 4 below.
// SHARED: a thread's quads are `stride` apart, a whole number of rounds of the channels, so that they are all of the same
// channels at the same places: those, their qparams and reciprocals are found once per U quads.  Groups of `stride`
// threads take U * stride quads.  Otherwise they are found per quad.
// (Quantize / dequantize / fake-quantize, us, per quad and shared by four: 5000 x 3000 x 7 along the last axis 166 / 181 / 191 and
// 93 / 105 / 142, 8192 x 8192 along the last 127 / 135 / 149 and 52 / 72 / 84, where memory takes 52 / 56 / 84 with a channel per row;
// 4096 x 512 x 8 along the last 25.7 / 29.4 / 32.9 and 15.0 / 16.3 / 22.5, along the middle 18.1 / - / 25.0 and 15.9 / - / 22.6.
// Two quads per thread: 115 / 125 / 148 for the first; eight: 89 / 108 / 156.)
template <typename Op, int U, int CHANNELS, bool SHARED>
__global__ __launch_bounds__(kThreads) void flat_kernel(Op op, unsigned n, FastDiv stride, FastDiv inner, FastDiv C,
                                                        QParams qp) {
    const unsigned n4 = n / 4, t = blockIdx.x * unsigned(kThreads) + threadIdx.x;
    const unsigned step = SHARED ? stride.d : unsigned(kThreads);
    const unsigned i0 = SHARED ? t + stride(t) * (U - 1) * stride.d : blockIdx.x * unsigned(U * kThreads) + threadIdx.x;
    typename Op::In v[U];
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const unsigned i = i0 + j * step;
        v[j] = op.load(i < n4 ? i : n4 - 1);
    }
    float s[4], z[4], r[4];
    auto find = [&](unsigned i) {
        unsigned seg = inner(i * 4), at = i * 4 - seg * inner.d, c = seg - C(seg) * C.d;
        if constexpr (CHANNELS == 2) {
            const unsigned next = c + 1 == C.d ? 0 : c + 1, left = inner.d - at;
            const float s0 = qp.scale[c], z0 = qp.zp[c], s1 = qp.scale[next], z1 = qp.zp[next];
            const float r0 = 1.0f / s0, r1 = 1.0f / s1;
#pragma unroll
            for (unsigned e = 0; e < 4; ++e) s[e] = e < left ? s0 : s1, z[e] = e < left ? z0 : z1, r[e] = e < left ? r0 : r1;
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                s[e] = qp.scale[c], z[e] = qp.zp[c];
                const bool wrap = ++at == inner.d;
                at = wrap ? 0 : at;
                c = wrap ? (c + 1 == C.d ? 0 : c + 1) : c;
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) r[e] = 1.0f / s[e];
        }
    };
    if (SHARED && i0 < n4) find(i0);
#pragma unroll
    for (int j = 0; j < U; ++j) {
        const unsigned i = i0 + j * step;
        if (i >= n4) break;
        if (!SHARED) find(i);
        op.store(i, v[j], float4{s[0], s[1], s[2], s[3]}, float4{z[0], z[1], z[2], z[3]}, float4{r[0], r[1], r[2], r[3]});
    }
    if (blockIdx.x == 0 && threadIdx.x < n % 4) {
        const unsigned e = n4 * 4 + threadIdx.x, seg = inner(e), c = seg - C(seg) * C.d;
        op.scalar(e, qp.scale[c], qp.zp[c]);
    }
}

// Any shape, any alignment: one element per thread, channel looked up per element.  For tensors
// whose first element is not aligned, and 2^31 elements and more of short segments.
template <typename Op>
__global__ __launch_bounds__(kThreads) void generic_kernel(Op op, size_t n, size_t C, size_t inner,
                                                           QParams qp) {
    size_t e = size_t(blockIdx.x) * kThreads + threadIdx.x;
    const size_t stride = size_t(gridDim.x) * kThreads;
    for (; e < n; e += stride) {
        float s, z;
        if (qp.scale) {
            const size_t c = (e / inner) % C;
            s = qp.scale[c];
            z = qp.zp[c];
        } else {
            s = qp.s_host;
            z = qp.z_host;
        }
        op.scalar(e, s, z);
    }
}

template <typename Op>
int launch_elementwise(Op op, size_t outer, size_t C, size_t inner, QParams qp, bool vec_ok,
                       hipStream_t st, const char* name) {
    const size_t n = outer * C * inner;
    if (n == 0) return LQ_OK;
    size_t segs = outer * C;
    if (C == 1) segs = 1, inner = n;  // one (scale, zero_point): one run, whatever its shape
    const size_t tail = C == 1 ? n % 4 : 0;
    if (vec_ok && inner >= 256 && inner % 4 == tail) {
        const size_t inner4 = inner / 4;
        int U = inner4 >= 8 * kThreads ? 8 : (inner4 >= 4 * kThreads ? 4 : (inner4 >= 2 * kThreads ? 2 : 1));
        if (U > Op::kMaxU) U = Op::kMaxU;
        const size_t per_block = size_t(U) * kThreads;
        const size_t chunks = (inner4 + per_block - 1) / per_block;
        const size_t blocks = chunks * segs;
        LQ_REQUIRE(blocks <= 0x7fffffffull && chunks <= 0xffffffffull, LQ_ERR_SHAPE,
                   "%s: tensor too large for one launch (%zu blocks)", name, blocks);
        dim3 grid{unsigned(blocks)}, block{kThreads};
        switch (U) {
        case 8: hipLaunchKernelGGL((seg_kernel<Op, 8>), grid, block, 0, st, op, inner4, unsigned(tail), unsigned(chunks), C, qp); break;
        case 4: hipLaunchKernelGGL((seg_kernel<Op, 4>), grid, block, 0, st, op, inner4, unsigned(tail), unsigned(chunks), C, qp); break;
        case 2: hipLaunchKernelGGL((seg_kernel<Op, 2>), grid, block, 0, st, op, inner4, unsigned(tail), unsigned(chunks), C, qp); break;
        default: hipLaunchKernelGGL((seg_kernel<Op, 1>), grid, block, 0, st, op, inner4, unsigned(tail), unsigned(chunks), C, qp); break;
        }
    } else if (vec_ok && n >= 4 && n < (size_t(1) << 31) && qp.scale) {
        // `round`: quads after which the channels come round again.  A stride of whole rounds that is not much more than
        // a block keeps a thread's quads near each other; where that would be fewer than 16 groups of threads, one group.
        const size_t quads = n / 4, cols = C * inner, round = cols % 4 == 0 ? cols / 4 : (cols % 2 == 0 ? cols / 2 : cols);
        const FastDiv by_inner{unsigned(inner)}, by_c{unsigned(C)};
        auto launch = [&](auto kernel, size_t threads, size_t stride) {
            hipLaunchKernelGGL(kernel, dim3(unsigned((threads + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, op,
                               unsigned(n), FastDiv{unsigned(stride)}, by_inner, by_c, qp);
        };
        // Found per quad: channels that come round less than twice, and what has two channels to find and nothing to divide by
        // (dequantize of 5000 x 3000 x 7 along the middle axis: 92.6 us, shared 96.1).  So does a quantization of so few that a CU has
        // less than three blocks either way: it takes two quads per thread by itself, four would halve the blocks (us, per quad /
        // shared, replayed from a graph: 300 x 39 x 28 3.1 / 3.5, 1777 x 20 x 2 3.0 / 3.3, 796 x 63 x 10 3.1 / 3.4; 143 x 3027 x 2 and 1215 x
        // 49 x 15 3.6 and 3.5 either way, 132 x 5645 x 2 4.5 / 4.2).
        if (quads >= 2 * round && (inner < 4 || Op::kDivides) && (Op::kMaxU >= 4 || quads >= 768 * kThreads)) {
            constexpr int U = 4;
            size_t stride = (kThreads + round - 1) / round * round;
            if (quads < 16 * U * stride) stride = (quads + U * round - 1) / (U * round) * round;
            const size_t threads = (quads + U * stride - 1) / (U * stride) * stride;
            if (inner < 4)
                launch(flat_kernel<Op, U, 4, true>, threads, stride);
            else if constexpr (Op::kDivides)
                launch(flat_kernel<Op, U, 2, true>, threads, stride);
        } else {
            constexpr int U = Op::kMaxU < 4 ? Op::kMaxU : 4;
            const size_t threads = (quads + U - 1) / U;
            inner >= 4 ? launch(flat_kernel<Op, U, 2, false>, threads, 1) : launch(flat_kernel<Op, U, 4, false>, threads, 1);
        }
    } else {
        size_t blocks = (n + kThreads - 1) / kThreads;
        if (blocks > 262144) blocks = 262144;
        hipLaunchKernelGGL((generic_kernel<Op>), dim3(unsigned(blocks)), dim3(kThreads), 0, st, op, n, C,
                           inner, qp);
    }
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e, name);
    return LQ_OK;
}

int make_qparams(const float* scale, const float* zp, int on_host, size_t C, QParams* qp,
                 const char* name) {
    LQ_REQUIRE(scale && zp, LQ_ERR_VALUE, "%s: scale / zero_point is NULL", name);
    if (on_host) {
        LQ_REQUIRE(C == 1, LQ_ERR_VALUE, "%s: host qparams are per-tensor only (C = %zu)", name, C);
        *qp = QParams{nullptr, nullptr, scale[0], zp[0]};
    } else {
        *qp = QParams{scale, zp, 0.f, 0.f};
    }
    return LQ_OK;
}

// ---------------------------------------------------------------- min / max
struct MinMax {
    float lo, hi;
    int nan;
};

__device__ __forceinline__ void mm_update(MinMax& m, float v) {
    m.nan |= (v != v);
    m.lo = fminf(m.lo, v);  // fminf/fmaxf drop NaN; the flag carries it
    m.hi = fmaxf(m.hi, v);
}

__device__ __forceinline__ MinMax mm_block_reduce(MinMax m) {
    block_minmax(m.lo, m.hi, m.nan);
    return m;
}

__device__ __forceinline__ void mm_write(MinMax m, float* mn, float* mx, size_t idx) {
    const float qnan = __builtin_nanf("");
    mn[idx] = m.nan ? qnan : m.lo;
    mx[idx] = m.nan ? qnan : m.hi;
}

// Elements e .. e+3 at any float address
__device__ __forceinline__ float4 nt_load_any(const float* p) {
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));
    const f32x4u v = __builtin_nontemporal_load(reinterpret_cast<const f32x4u*>(p));
    return make_float4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ void mm_update(MinMax& m, float4 v) {
    mm_update(m, v.x), mm_update(m, v.y), mm_update(m, v.z), mm_update(m, v.w);
}

// Channel elements lie in `outer` contiguous runs of `inner`.  A channel has `splits`
// blocks, `run_splits` of them side by side in a run: block (c, split) scans its slice of each of
// its share of the runs.  Partials are laid out [split][c]; with splits == 1 they are the
// final answer.  The last quad of a run that is not whole quads begins at its fourth element from
// the end: the elements it takes twice change nothing.
// (8192 x 16 x 64, 16 channels: 77 us while the blocks of a channel shared out its runs only lengthwise, which
// runs of 64 do not allow.)
__global__ __launch_bounds__(kThreads) void minmax_seg_kernel(const float* __restrict__ x,
                                                              size_t runs_all, size_t C, size_t inner,
                                                              unsigned splits, unsigned run_splits, float* pmin,
                                                              float* pmax) {
    const size_t c = blockIdx.x / splits;
    const unsigned sp = blockIdx.x - unsigned(c * splits);
    const unsigned part = sp / run_splits, parts = splits / run_splits;
    const size_t per_part = (runs_all + parts - 1) / parts, first = part * per_part;
    const size_t outer = first + per_part < runs_all ? first + per_part : runs_all;  // (past `first` where a share is empty)
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    if (inner >= 4 && inner <= 2 * kThreads && runs_all > 1 && run_splits == 1) {
        // runs shorter than the block: a power of two of lanes per run, several runs at once
        const unsigned last = unsigned(inner) - 4, quads = unsigned(inner + 3) / 4;
        const unsigned shift = quads > 1 ? 32 - __builtin_clz(quads - 1) : 0, runs = kThreads >> shift;
        const unsigned i = threadIdx.x & ((1u << shift) - 1);
        const float* p = x + c * inner + (i * 4 < last ? i * 4 : last);  // lanes past the run read its end again
        const size_t run = C * inner;
        size_t o = first + (threadIdx.x >> shift);
        for (; o + 3 * runs < outer; o += 4 * runs) {
            const float4 a = nt_load_any(p + o * run), b = nt_load_any(p + (o + runs) * run),
                         d = nt_load_any(p + (o + 2 * runs) * run), e = nt_load_any(p + (o + 3 * runs) * run);
            mm_update(m, a), mm_update(m, b), mm_update(m, d), mm_update(m, e);
        }
        for (; o < outer; o += runs) mm_update(m, nt_load_any(p + o * run));
    } else if (inner >= 4) {
        const size_t inner4 = (inner + 3) / 4;
        const size_t per = (inner4 + run_splits - 1) / run_splits;
        const size_t lo4 = size_t(sp - part * run_splits) * per;
        const size_t hi4 = lo4 + per < inner4 ? lo4 + per : inner4;
        const size_t whole = hi4 < inner / 4 ? hi4 : inner / 4;
        for (size_t o = first; o < outer; ++o) {
            const float* p = x + (o * C + c) * inner;
            size_t i = lo4 + threadIdx.x;
            // four independent loads in flight per lane
            for (; i + 3 * kThreads < whole; i += 4 * kThreads) {
                const float4 a = nt_load_any(p + i * 4), b = nt_load_any(p + (i + kThreads) * 4),
                             d = nt_load_any(p + (i + 2 * kThreads) * 4), e = nt_load_any(p + (i + 3 * kThreads) * 4);
                mm_update(m, a), mm_update(m, b), mm_update(m, d), mm_update(m, e);
            }
            for (; i < hi4; i += kThreads) mm_update(m, nt_load_any(p + (i * 4 < inner - 4 ? i * 4 : inner - 4)));
        }
    } else {
        for (size_t o = first + threadIdx.x; o < outer; o += kThreads)
            for (size_t i = 0; i < inner; ++i) mm_update(m, x[(o * C + c) * inner + i]);
    }
    m = mm_block_reduce(m);
    if (threadIdx.x == 0) mm_write(m, pmin, pmax, size_t(sp) * C + c);
}

// Short runs (inner < 64, e.g. a channel-last tensor): view x as
// [outer][C*inner]; a thread owns one column and walks down a slice of rows,
// so a wavefront reads contiguous memory.  Partials [split][C*inner].
__global__ __launch_bounds__(kThreads) void minmax_col_kernel(const float* __restrict__ x,
                                                              size_t outer, size_t cols,
                                                              unsigned splits, float* pmin,
                                                              float* pmax) {
    const size_t col = size_t(blockIdx.x) * kThreads + threadIdx.x;
    const unsigned sp = blockIdx.y;
    if (col >= cols) return;
    const size_t per = (outer + splits - 1) / splits;
    const size_t lo = size_t(sp) * per;
    const size_t hi = lo + per < outer ? lo + per : outer;
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    size_t r = lo;
    for (; r + 8 <= hi; r += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = __builtin_nontemporal_load(&x[(r + u) * cols + col]);
#pragma unroll
        for (int u = 0; u < 8; ++u) mm_update(m, v[u]);
    }
    for (; r < hi; ++r) mm_update(m, x[r * cols + col]);
    mm_write(m, pmin, pmax, size_t(sp) * cols + col);
}

// The same for few columns, where a thread per column would leave most of a block's lanes idle: `lanes` threads,
// 4 * lanes a multiple of cols, read consecutive quads of x, so that each of a thread's four elements stays in
// one column; the rows a block has read at once are folded in LDS.  Block b takes steps b, b + blocks, ... of
// 4 * lanes elements.  Partials [block][cols].
__global__ __launch_bounds__(kThreads) void minmax_period_kernel(const float* __restrict__ x, size_t n, unsigned cols,
                                                                 unsigned lanes, float* pmin, float* pmax) {
    __shared__ float s_lo[4 * kThreads], s_hi[4 * kThreads];
    const unsigned tid = threadIdx.x, step = 4 * lanes;
    MinMax m[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) m[e] = MinMax{__builtin_inff(), -__builtin_inff(), 0};
    auto take = [&](float4 v) {
        mm_update(m[0], v.x), mm_update(m[1], v.y), mm_update(m[2], v.z), mm_update(m[3], v.w);
    };
    if (tid < lanes) {
        const size_t stride = size_t(gridDim.x) * step;
        size_t i = size_t(blockIdx.x) * step + tid * 4;
        for (; i + 3 * stride + 4 <= n; i += 4 * stride) {
            const float4 a = nt_load_any(x + i), b = nt_load_any(x + i + stride), c = nt_load_any(x + i + 2 * stride),
                         d = nt_load_any(x + i + 3 * stride);
            take(a), take(b), take(c), take(d);
        }
        for (; i + 4 <= n; i += stride) take(nt_load_any(x + i));
#pragma unroll
        for (int e = 0; e < 3; ++e)
            if (i + e < n) mm_update(m[e], x[i + e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            s_lo[tid * 4 + e] = m[e].nan ? __builtin_nanf("") : m[e].lo;
            s_hi[tid * 4 + e] = m[e].nan ? __builtin_nanf("") : m[e].hi;
        }
    }
    __syncthreads();
    for (unsigned rows = step / cols; rows > 1;) {  // entry row * cols + col; the upper rows into the lower ones
        const unsigned keep = (rows + 1) / 2;
        for (unsigned k = tid; k < (rows - keep) * cols; k += kThreads) {
            const float a = s_lo[k], b = s_lo[k + keep * cols], c = s_hi[k], d = s_hi[k + keep * cols];
            s_lo[k] = a != a || b < a ? a != a ? a : b : b != b ? b : a;
            s_hi[k] = c != c || d > c ? c != c ? c : d : d != d ? d : c;
        }
        __syncthreads();
        rows = keep;
    }
    for (unsigned k = tid; k < cols; k += kThreads) {
        pmin[size_t(blockIdx.x) * cols + k] = s_lo[k];
        pmax[size_t(blockIdx.x) * cols + k] = s_hi[k];
    }
}

// Folds partials [groups][C][inner_cols] into mn[C], mx[C]; one block per
// channel, four independent loads per thread in flight.
__global__ __launch_bounds__(256) void minmax_finalize_kernel(const float* __restrict__ pmin,
                                                              const float* __restrict__ pmax,
                                                              size_t C, unsigned groups,
                                                              unsigned inner_cols, float* mn,
                                                              float* mx) {
    const size_t c = blockIdx.x;
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    const size_t per_c = size_t(groups) * inner_cols;
    for (size_t t0 = threadIdx.x; t0 < per_c; t0 += 4 * 256) {
        float a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const size_t t = t0 + size_t(u) * 256;
            a[u] = __builtin_inff(), b[u] = -__builtin_inff();
            if (t < per_c) {
                const size_t g = t / inner_cols, i = t - g * inner_cols;
                const size_t idx = (g * C + c) * inner_cols + i;
                a[u] = pmin[idx], b[u] = pmax[idx];
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            m.nan |= (a[u] != a[u]) | (b[u] != b[u]);
            m.lo = fminf(m.lo, a[u]);
            m.hi = fmaxf(m.hi, b[u]);
        }
    }
    m = mm_block_reduce(m);
    if (threadIdx.x == 0) mm_write(m, mn, mx, c);
}

__global__ void minmax_identity_kernel(float* mn, float* mx, size_t C) {
    size_t c = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c < C) {
        mn[c] = __builtin_inff();
        mx[c] = -__builtin_inff();
    }
}

// ---------------------------------------------------------------- qparams
__global__ void calc_qparams_kernel(const float* __restrict__ mn, const float* __restrict__ mx,
                                    size_t C, int symmetric, int qmin, int qmax, int is_signed,
                                    float eps, float half_range, float* scale, float* zp) {
    size_t c = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (c >= C) return;
    qparams_of(mn[c], mx[c], symmetric, qmin, qmax, is_signed, eps, half_range, &scale[c], &zp[c]);
}

// Per-tensor qparams from a range kept by the producing kernel (one block):
// reduce the partial slots, then calculate_qparams; also writes the range
// itself when asked.
__global__ __launch_bounds__(1024) void calc_qparams_from_range_kernel(const float* __restrict__ range,
                                                                        int symmetric, int qmin, int qmax,
                                                                        int is_signed, float eps,
                                                                        float half_range, float* scale,
                                                                        float* zp, float* mn_out,
                                                                        float* mx_out) {
    float mn, mx;
    range_block_load<4>(range, mn, mx);
    if (threadIdx.x == 0) {
        if (mn_out) *mn_out = mn;
        if (mx_out) *mx_out = mx;
        qparams_of(mn, mx, symmetric, qmin, qmax, is_signed, eps, half_range, scale, zp);
    }
}

// The same and the codes of a tensor of up to kRangeTensor elements: every block reduces the slots (from the L2, under
// its loads of x), so that no launch of one block stands between the producing kernel and the codes.  Beyond, what the
// blocks read of the slots costs more than that launch: 38.7 M elements behind 1200 slots 34.8 us with blocks that stay
// for several chunks, against 31.7 + 4.6 under the tracer and the same in a graph.
constexpr int kRangeChunk = 2;  // float4 per thread
constexpr size_t kRangeTensor = size_t(1) << 22;
__global__ __launch_bounds__(1024) void quantize_range_kernel(QuantizeOp<int8_t> op, unsigned quads, unsigned tail,
                                                              const float* __restrict__ range, int symmetric, int qmin,
                                                              int qmax, int is_signed, float eps, float half_range,
                                                              float* scale, float* zp) {
    const unsigned at = blockIdx.x * 1024 * kRangeChunk + threadIdx.x;
    float4 v[kRangeChunk];
#pragma unroll
    for (int u = 0; u < kRangeChunk; ++u)
        if (at + u * 1024 < quads) v[u] = op.load(at + u * 1024);
    float mn, mx, s, z;
    range_block_load<1>(range, mn, mx);
    qparams_of(mn, mx, symmetric, qmin, qmax, is_signed, eps, half_range, &s, &z);
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) *scale = s, *zp = z;
        if (threadIdx.x < tail) op.scalar(quads * 4 + threadIdx.x, s, z);
    }
    const float r = 1.0f / s;
#pragma unroll
    for (int u = 0; u < kRangeChunk; ++u)
        if (at + u * 1024 < quads) op.store(at + u * 1024, v[u], splat(s), splat(z), splat(r));
}

// Elements e .. e+3 of x[0 .. n), zeros past n.  One unconditional 16-byte load (any float address) from where all
// four exist: a load under a condition would be waited for before the next one is issued.
__device__ __forceinline__ float4 load_quad(const float* x, size_t e, size_t n) {
    float4 v{0.f, 0.f, 0.f, 0.f};
    if (n < 4) {  // uniform
        if (e < n) v.x = x[e];
        if (e + 1 < n) v.y = x[e + 1];
        if (e + 2 < n) v.z = x[e + 2];
        return v;
    }
    const size_t at = e < n - 4 ? e : n - 4;
    __builtin_memcpy(&v, x + at, 16);
    return v;
}
// ... and, once it has arrived, the elements in place
__device__ __forceinline__ float4 place_quad(float4 v, size_t e, size_t n) {
    if (n < 4 || e + 4 <= n) return v;
    const size_t d = e - (n - 4);
    return d == 1 ? float4{v.y, v.z, v.w, 0.f}
                  : (d == 2 ? float4{v.z, v.w, 0.f, 0.f} : (d == 3 ? float4{v.w, 0.f, 0.f, 0.f} : float4{0.f, 0.f, 0.f, 0.f}));
}
__device__ __forceinline__ void mm_update_quad(MinMax& m, float4 v, size_t e, size_t n) {
    if (e + 4 <= n) {
        mm_update(m, v.x), mm_update(m, v.y), mm_update(m, v.z), mm_update(m, v.w);
    } else {
        if (e < n) mm_update(m, v.x);
        if (e + 1 < n) mm_update(m, v.y);
        if (e + 2 < n) mm_update(m, v.z);
    }
}

// Dynamic per-row quantization in one pass over x: a block holds one row in registers, takes
// its min / max (observer.py:634-653 with ch_axis = 0), turns them into the row's qparams
// (qparams_of) and writes the row's codes with QuantizeOp's arithmetic - the three separate
// launches' results, bit for bit, with x read once instead of twice.
// RAGGED: rows of any length at any float address, their codes at any byte address.  (1500 rows of 3333 in the four launches of the
// three calls 24.4 us, 2 of 7386 24.6; in one 10.2 and 10.6, of which the host takes most.)
template <int R, bool RAGGED>  // quads per lane: rows of up to 1024 * R floats
__global__ __launch_bounds__(256) void quantize_rows_dynamic_kernel(
    const float* __restrict__ x, int cols, int symmetric, int qmin, int qmax, int is_signed, float eps,
    float half_range, int off, float* __restrict__ scale, float* __restrict__ zp, float* __restrict__ mn_out,
    float* __restrict__ mx_out, int8_t* __restrict__ q) {
    __shared__ float s_sz[2];
    const size_t row = blockIdx.x;
    const float* xr = x + row * size_t(cols);
    float4 v[R];
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    if constexpr (RAGGED) {
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int e = (u * 256 + int(threadIdx.x)) * 4;
            if (e < cols) v[u] = load_quad(xr, e, cols);
        }
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int e = (u * 256 + int(threadIdx.x)) * 4;
            if (e < cols) v[u] = place_quad(v[u], e, cols), mm_update_quad(m, v[u], e, cols);
        }
    } else {
#pragma unroll
        for (int u = 0; u < R; ++u) {
            const int i = u * 256 + int(threadIdx.x);
            if (i * 4 < cols) {
                v[u] = nt_load(&reinterpret_cast<const float4*>(xr)[i]);
                mm_update(m, v[u].x), mm_update(m, v[u].y), mm_update(m, v[u].z), mm_update(m, v[u].w);
            }
        }
    }
    m = mm_block_reduce(m);
    // (one thread's division: other blocks have the SIMDs meanwhile, and would wait for everybody's)
    if (threadIdx.x == 0) {
        const float qnan = __builtin_nanf("");
        const float mn = m.nan ? qnan : m.lo, mx = m.nan ? qnan : m.hi;
        float s, z;
        qparams_of(mn, mx, symmetric, qmin, qmax, is_signed, eps, half_range, &s, &z);
        scale[row] = s, zp[row] = z;
        if (mn_out) mn_out[row] = mn;
        if (mx_out) mx_out[row] = mx;
        s_sz[0] = s, s_sz[1] = z;
    }
    __syncthreads();
    const float s = s_sz[0], z = s_sz[1], r = 1.0f / s;
    const QuantizeOp<int8_t> op{nullptr, nullptr, float(double(qmin)), float(double(qmax)), off};
    int8_t* qr = q + row * size_t(cols);
#pragma unroll
    for (int u = 0; u < R; ++u) {
        const int e = (u * 256 + int(threadIdx.x)) * 4;
        if (e >= cols) break;
        const Code8x4 c = op.pack(v[u], s, z, r);
        if (!RAGGED) {
            *reinterpret_cast<Code8x4*>(qr + e) = c;
        } else if (e + 4 <= cols) {
            __builtin_memcpy(qr + e, &c, 4);
        } else {  // (named one by one: an index would put the codes into LDS, at a place found in the dispatch packet)
            qr[e] = c.v[0];
            if (e + 1 < cols) qr[e + 1] = c.v[1];
            if (e + 2 < cols) qr[e + 2] = c.v[2];
        }
    }
}

// Dynamic per-tensor quantization: global min / max (observer.py:363-375), qparams, codes.  A block holds 8192
// elements in registers.
//
// Small tensors (up to kExchange blocks) in one launch, x read once: the blocks' ranges meet through a slot per
// block in device memory - written through, and polled by every block until it is filled - and each block then
// derives the qparams itself and writes its codes.  The last block to leave empties the slots for the next
// launch.  That is quick where all blocks are resident, and kExchange of them are a sixteenth of the device, less than the
// share of one of the hardware queues that streams have (exchange_blocks).  Nothing depends on it: kernels of other processes,
// or a stream that may not use every CU, can keep a block out for any time, so a block that has read a slot kExchangePolls
// times without finding a range (a few milliseconds) takes the range of x itself - the same minimum and maximum -, ends, and makes room.
//
// Beyond, and under capture (slots cleared inside a graph are unset until its replay), two launches: slices'
// ranges (minmax_seg_kernel), then this kernel with PARTS - every block reduces
// the slices' ranges itself, which saves the finalize and qparams launches between.
//
// Rows of `cols` elements go to rows of `ld` codes, zeros past `cols` (what a GEMM of ragged rows wants).
//
// 8192 elements 3.3 us, 65536 (8 blocks, the exchange) 5.7.  A slot is read first when most of them have been written, and
// not at once again.  In two launches 1 M elements take 7.5 us, 4 M 11.3, 16 M 30.8 (14.8, 22.9 and 41.2 while the codes of the
// last quads were picked by an index: the array lay in LDS, at a place that every wavefront computed from the dispatch
// packet, which is read from host memory; 262144 elements in one launch 8.9 -> 5.7).  Blocks that exchange and take that long to
// start were measured as: a dynamic Linear in two launches / in one 333 x 1000 -> 1001 (42 blocks) 16.6 / 13.6, with 128 blocks
// 25.7 / 24.9, with 256 32.7 / 30.7, too little for that much of the device.  Before either: one block on one CU for up to
// 262144 elements (61 us), five launches beyond (1 M elements: 12.3 us).
constexpr int kDynThreads = 512, kDynQuads = 4, kDynPerBlock = kDynThreads * kDynQuads * 4;
constexpr int kExchange = 64, kExchangePolls = 4096, kMaxParts = 512;
constexpr unsigned long long kSlotEmpty = ~0ull;  // NaNs that no range contains: mm_write's NaN is the canonical one
struct DynScratch {
    unsigned long long slot[kExchange];    // low word: the block's minimum, high word: its maximum
    unsigned left;                        // blocks that have read the slots
};

// RAGGED: rows of `cols` elements to rows of `ld` codes (a multiple of 4); the quads are those of the codes, so
// that every store is one aligned word.  Otherwise one run of n elements.
template <bool PARTS, bool RAGGED>
__global__ __launch_bounds__(kDynThreads) __attribute__((amdgpu_waves_per_eu(8)))
void quantize_tensor_dynamic_kernel(const float* __restrict__ x, size_t n, unsigned cols, unsigned ld, int symmetric,
                                    int qmin, int qmax, int is_signed, float eps, float half_range, int off,
                                    DynScratch* slots, int polls, const float* __restrict__ parts, int n_parts, float* scale,
                                    float* zp, float* mn_out, float* mx_out, int8_t* __restrict__ q) {
    __shared__ int s_last, s_missing;
    const int tid = threadIdx.x;
    if (tid == 0) s_missing = 0;  // (the first reduction's barrier is between this and the slots)
    const size_t first = size_t(blockIdx.x) * kDynPerBlock;
    const float qnan = __builtin_nanf("");
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    if (PARTS && tid < n_parts) m.lo = parts[tid], m.hi = parts[n_parts + tid];
    float4 v[kDynQuads];
    int count[kDynQuads];  // elements of the quad that exist
    auto at = [&](int u) { return first + size_t(u * kDynThreads + tid) * 4; };
    auto element = [&](int u) {
        if (!RAGGED) return at(u);
        const unsigned row = unsigned(at(u)) / ld;  // (fewer than 2^32 codes: see the launcher)
        return size_t(row) * cols + (unsigned(at(u)) - row * ld);
    };
#pragma unroll
    for (int u = 0; u < kDynQuads; ++u) {
        const size_t e = element(u);
        v[u] = load_quad(x, e, n);
        if (RAGGED) {
            const int left = int(cols) - int(unsigned(at(u)) % ld);
            count[u] = e >= n || left <= 0 ? 0 : (left < 4 ? left : 4);
        } else {
            count[u] = e + 4 <= n ? 4 : (e < n ? int(n - e) : 0);
        }
    }
    if (RAGGED || first + kDynPerBlock > n) {
#pragma unroll
        for (int u = 0; u < kDynQuads; ++u) v[u] = place_quad(v[u], element(u), n);
    }
    if (PARTS) {
        m.nan = (m.lo != m.lo) | (m.hi != m.hi);
    } else if (!RAGGED && first + kDynPerBlock <= n) {
#pragma unroll
        for (int u = 0; u < kDynQuads; ++u)
            mm_update(m, v[u].x), mm_update(m, v[u].y), mm_update(m, v[u].z), mm_update(m, v[u].w);
    } else {
#pragma unroll
        for (int u = 0; u < kDynQuads; ++u) mm_update_quad(m, v[u], 0, count[u]);
    }
    m = mm_block_reduce(m);
    if (!PARTS && gridDim.x > 1) {
        if (tid == 0) {
            const unsigned lo = __float_as_uint(m.nan ? qnan : m.lo), hi = __float_as_uint(m.nan ? qnan : m.hi);
            __hip_atomic_store(&slots->slot[blockIdx.x], (unsigned long long)hi << 32 | lo, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        m = MinMax{__builtin_inff(), -__builtin_inff(), 0};
        if (tid < int(gridDim.x)) {
            unsigned long long got = kSlotEmpty;
            __builtin_amdgcn_s_sleep(12);
            for (int spin = 0; got == kSlotEmpty && spin < polls; ++spin) {
                if (spin) __builtin_amdgcn_s_sleep(4);
                got = __hip_atomic_load(&slots->slot[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            m.lo = __uint_as_float(unsigned(got)), m.hi = __uint_as_float(unsigned(got >> 32));
            m.nan = (m.lo != m.lo) | (m.hi != m.hi);
            if (got == kSlotEmpty) s_missing = 1;
        }
        __syncthreads();  // every slot has been read (and the reduction may use its LDS again)
        if (s_missing) {  // a block that has not started: its elements and all others, read here
            m = MinMax{__builtin_inff(), -__builtin_inff(), 0};
            for (size_t e = size_t(tid) * 4; e < n; e += kDynThreads * 4)
                mm_update_quad(m, place_quad(load_quad(x, e, n), e, n), e, n);
        }
        if (tid == 0) {
            const unsigned before = __hip_atomic_fetch_add(&slots->left, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_last = before == gridDim.x - 1;
        }
        m = mm_block_reduce(m);
    }
    const float mn = m.nan ? qnan : m.lo, mx = m.nan ? qnan : m.hi;
    float s, z;
    qparams_of(mn, mx, symmetric, qmin, qmax, is_signed, eps, half_range, &s, &z);
    if (blockIdx.x == 0 && tid == 0) {
        *scale = s, *zp = z;
        if (mn_out) *mn_out = mn;
        if (mx_out) *mx_out = mx;
    }
    if (!PARTS && gridDim.x > 1 && s_last) {  // nobody reads the slots any more
        if (tid < kExchange) slots->slot[tid] = kSlotEmpty;
        if (tid == 0) slots->left = 0;
    }
    const float r = 1.0f / s;
    const QuantizeOp<int8_t> op{nullptr, nullptr, float(double(qmin)), float(double(qmax)), off};
#pragma unroll
    for (int u = 0; u < kDynQuads; ++u) {
        Code8x4 c = op.pack(v[u], s, z, r);
        if (RAGGED) {
            unsigned w;
            __builtin_memcpy(&w, &c, 4);
            w = count[u] >= 4 ? w : (count[u] <= 0 ? 0u : w & ((1u << (8 * count[u])) - 1u));  // zeros past the row
            if (at(u) < size_t(n / cols) * ld) __builtin_memcpy(q + at(u), &w, 4);
        } else if (count[u] == 4) {
            __builtin_memcpy(q + at(u), &c, 4);
        } else {  // (named one by one, as in quantize_rows_dynamic_kernel)
            if (count[u] > 0) q[at(u)] = c.v[0];
            if (count[u] > 1) q[at(u) + 1] = c.v[1];
            if (count[u] > 2) q[at(u) + 2] = c.v[2];
        }
    }
}

// One row: a whole dynamic-quantized Linear as a stream of the weight.  Every block needs the row's range and
// codes: it takes them itself (the row is at most 64 KiB of L2 reads per block) while its first weights are on
// the way - they are requested before the range is known -, so the layer costs what lq_qlinear_i8 of one row
// does (qgemv1_kernel: four weight rows per wavefront, a KiB of a row per load, v_dot4) plus the two block
// reductions.  4096 -> 11008: 24.2 us with the 16 x 16-tile kernel above (688 blocks of 1024 threads, each
// waiting for its range before its one weight fragment per wavefront), 11.5 when the weights had to arrive before the row's
// reductions could end (a barrier that waits for all loads, branches behind which the compiler does), now 10.4 with its
// launch (4.3 TB/s of weight).
// w rows are `ld` bytes apart, zeros past K; K <= 16384, ld % 16 == 0.
// ONE_ROUND: the block's registers hold the row (4 <= K <= 16 per thread).  Then nothing between the requests of the weights and
// their use branches or loops, so that what waits for the row waits for the row alone: loads past the row and the weight
// repeat their last ones (a range does not mind, and codes past K are zeros in LDS).
template <bool ONE_ROUND>
__global__ __launch_bounds__(512) void dynamic_gemv1_kernel(
    const float* __restrict__ x, int K, const int8_t* __restrict__ w, int ld, int N, const float* __restrict__ w_scale,
    const int32_t* __restrict__ wsum, const float* __restrict__ bias, int relu, int symmetric, int qmin, int qmax,
    int is_signed, float eps, float half_range, int off, float* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) int8_t dv_codes[];  // K bytes rounded up to a multiple of 4 KiB
    typedef int dv_v4i __attribute__((ext_vector_type(4)));
    constexpr int RW = 4, kKeep = 4;  // (with the weights' 64 registers: two blocks per CU)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, threads = blockDim.x, waves = threads >> 6;
    const int chunks = (K + 4095) / 4096;
    // threads x kKeep quads in registers; smaller blocks walk the row in several rounds (the last stays)
    const int quads = (K + 3) / 4, rounds = (quads + threads * kKeep - 1) / (threads * kKeep);
    float4 v[kKeep];
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    if constexpr (ONE_ROUND) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int e = (u * threads + tid) * 4;
            __builtin_memcpy(&v[u], x + (e < K - 4 ? e : K - 4), 16);
        }
    } else
    for (int rd = 0; rd < rounds; ++rd) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) v[u] = load_quad(x, size_t((rd * kKeep + u) * threads + tid) * 4, K);
        if (rounds > 1) {
#pragma unroll
            for (int u = 0; u < kKeep; ++u) {
                const int e = ((rd * kKeep + u) * threads + tid) * 4;
                v[u] = place_quad(v[u], e, K);
                mm_update_quad(m, v[u], e, K);
            }
        }
    }
    const int nb = (blockIdx.x * waves + wave) * RW;
    dv_v4i wv[RW][4];
    auto load_chunk = [&](int kc) {
#pragma unroll
        for (int r = 0; r < RW; ++r) {
            const int n = nb + r < N ? nb + r : N - 1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = kc * 4096 + i * 1024 + lane * 16;
                if constexpr (ONE_ROUND)
                    wv[r][i] = *reinterpret_cast<const dv_v4i*>(w + size_t(n) * ld + (k < ld ? k : 0));
                else
                    wv[r][i] = k < ld ? *reinterpret_cast<const dv_v4i*>(w + size_t(n) * ld + k) : dv_v4i{0, 0, 0, 0};
            }
        }
    };
    const int n_mine = nb + (lane < RW ? lane : 0);
    const bool mine = lane < RW && n_mine < N;
    const float c_ws = mine && w_scale ? w_scale[n_mine] : 1.0f;
    const int c_wsum = mine && wsum ? wsum[n_mine] : 0;
    const float c_bias = mine && bias ? bias[n_mine] : -0.0f;
    __builtin_amdgcn_sched_barrier(0);
    load_chunk(0);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (ONE_ROUND) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) mm_update(m, v[u]);
    } else if (rounds == 1) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int e = (u * threads + tid) * 4;
            v[u] = place_quad(v[u], e, K);
            mm_update_quad(m, v[u], e, K);
        }
    }
    m = mm_block_reduce(m);
    // (every thread derives the qparams: cheaper than one thread, a barrier and a read)
    const float qnan = __builtin_nanf("");
    float s, z;
    qparams_of(m.nan ? qnan : m.lo, m.nan ? qnan : m.hi, symmetric, qmin, qmax, is_signed, eps, half_range, &s, &z);
    const float rcp = 1.0f / s;
    const QuantizeOp<int8_t> op{nullptr, nullptr, float(double(qmin)), float(double(qmax)), off};
    if constexpr (ONE_ROUND) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int i = u * threads + tid, past = i * 4 - (K - 4);  // elements of the quad that lie in the one before
            const Code8x4 c = op.pack(v[u], s, z, rcp);
            unsigned word;
            __builtin_memcpy(&word, &c, 4);
            word = past <= 0 ? word : past < 4 ? word >> (8 * past) : 0u;
            if (i < chunks * 1024) *reinterpret_cast<unsigned*>(dv_codes + i * 4) = word;
        }
        for (int i = kKeep * threads + tid; i < chunks * 1024; i += threads) *reinterpret_cast<unsigned*>(dv_codes + i * 4) = 0u;
    } else
    for (int rd = rounds - 1; rd >= 0; --rd) {
        if (rd != rounds - 1) {
#pragma unroll
            for (int u = 0; u < kKeep; ++u) v[u] = load_quad(x, size_t((rd * kKeep + u) * threads + tid) * 4, K);
#pragma unroll
            for (int u = 0; u < kKeep; ++u) v[u] = place_quad(v[u], ((rd * kKeep + u) * threads + tid) * 4, K);
        }
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            // (whatever lies past K, stored or not, meets zeros of the weight)
            const int i = (rd * kKeep + u) * threads + tid;
            if (i < quads) *reinterpret_cast<Code8x4*>(dv_codes + i * 4) = op.pack(v[u], s, z, rcp);
        }
    }
    lds_barrier();  // (the weights are still on their way)
    int acc[RW] = {0, 0, 0, 0};
    for (int kc = 0; kc < chunks; ++kc) {
        if (kc) load_chunk(kc);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const dv_v4i av = *reinterpret_cast<const dv_v4i*>(dv_codes + kc * 4096 + i * 1024 + lane * 16);
#pragma unroll
            for (int r = 0; r < RW; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[r] = __builtin_amdgcn_sdot4(wv[r][i][e], av[e], acc[r], false);
        }
    }
    int sum = 0;
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        int t = acc[r];
        t += __builtin_amdgcn_update_dpp(0, t, 0x128, 0xf, 0xf, false);
        t += __builtin_amdgcn_update_dpp(0, t, 0x124, 0xf, 0xf, false);
        t += __builtin_amdgcn_update_dpp(0, t, 0x122, 0xf, 0xf, false);
        t += __builtin_amdgcn_update_dpp(0, t, 0x121, 0xf, 0xf, false);
        t = __builtin_amdgcn_readlane(t, 0) + __builtin_amdgcn_readlane(t, 16) + __builtin_amdgcn_readlane(t, 32) +
            __builtin_amdgcn_readlane(t, 48);
        if (lane == r) sum = t;
    }
    if (mine) {
        const int zi = int(z) + off;
        const int corr = (wsum != nullptr && zi != 0) ? zi * c_wsum : 0;
        float y = float(sum - corr) * (s * c_ws);
        y = y + c_bias;
        const float floor = relu ? 0.0f : -__builtin_inff();
        out[n_mine] = (y < floor) ? floor : y;
    }
}

// ---------------------------------------------------------------- static scratch (no-allocation entry point)
// lq_minmax_noalloc keeps the partial results of its two-stage reduction here instead of in
// the library's growable workspace, so that the call allocates nothing.  Each GPU holds its
// own copy of the array at its own address; the name below is only the host-side handle of
// the symbol, the device address comes from hipGetSymbolAddress, once per device.
constexpr size_t kNoAllocScratchBytes = size_t(1) << 20;
__device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];
void* g_scratch_ptr[16] = {nullptr};
std::mutex g_scratch_mutex;

int noalloc_scratch_ptr(void** out) {
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    LQ_REQUIRE(dev >= 0 && dev < 16, LQ_ERR_DEVICE, "device index %d out of range", dev);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void* p = nullptr;
        LQ_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        LQ_REQUIRE(p != nullptr, LQ_ERR_INTERNAL, "hipGetSymbolAddress returned a null address for the static scratch");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return LQ_OK;
}

// min / max launch sequence shared by lq_minmax and lq_minmax_noalloc.  `get_ws(nbytes, &ptr)`
// supplies the memory for the partial results of a two-stage reduction; `ws_limit` is the
// most it can supply: the number of slices per channel is cut down to fit (the result does
// not depend on it: min and max are exact in any order).
template <class GetWs>
int minmax_launch(const float* x, size_t outer, size_t C, size_t inner, float* mn, float* mx, hipStream_t st,
                  size_t ws_limit, GetWs get_ws) {
    LQ_REQUIRE(mn && mx, LQ_ERR_VALUE, "minmax: output pointer is NULL");
    LQ_REQUIRE(C >= 1, LQ_ERR_SHAPE, "minmax: C must be >= 1");
    const size_t per_channel = outer * inner;
    if (per_channel == 0) {  // empty reduction: identities (Reduce.cpp:95,107)
        hipLaunchKernelGGL(minmax_identity_kernel, dim3(unsigned((C + 255) / 256)), dim3(256), 0, st, mn,
                           mx, C);
        LQ_CHECK_LAUNCH("minmax_identity");
        return LQ_OK;
    }
    LQ_REQUIRE(x, LQ_ERR_VALUE, "minmax: x is NULL");
    LQ_REQUIRE(C <= 0x3fffffffull, LQ_ERR_SHAPE, "minmax: too many channels (%zu)", C);
    const bool folded = C == 1 && outer > 1;
    if (folded) inner *= outer, outer = 1;  // one run, whatever its shape

    if (inner < 64 && C > 1) {
        const size_t cols = C * inner;
        // enough row slices to occupy the chip, at least 32 rows each
        size_t col_blocks = (cols + kThreads - 1) / kThreads;
        size_t splits = 2048 / col_blocks;
        if (splits > outer / 32) splits = outer / 32;
        if (splits < 1) splits = 1;
        if (splits > 65535) splits = 65535;
        LQ_REQUIRE(2 * cols * sizeof(float) <= ws_limit, LQ_ERR_SHAPE,
                   "minmax: %zu channel-inner columns need %zu bytes of partial results, more than the %zu available",
                   cols, 2 * cols * sizeof(float), ws_limit);
        if (splits > ws_limit / (2 * cols * sizeof(float))) splits = ws_limit / (2 * cols * sizeof(float));
        void* ws = nullptr;
        int rc = get_ws(2 * splits * cols * sizeof(float), &ws);
        if (rc) return rc;
        float* pmin = static_cast<float*>(ws);
        float* pmax = pmin + splits * cols;
        // quads of one row of lanes keep their columns when 4 * lanes is a multiple of cols
        const size_t period = cols % 4 == 0 ? cols / 4 : (cols % 2 == 0 ? cols / 2 : cols);
        if (period <= kThreads) {
            const size_t lanes = kThreads / period * period;
            hipLaunchKernelGGL(minmax_period_kernel, dim3(unsigned(splits)), dim3(kThreads), 0, st, x, outer * cols,
                               unsigned(cols), unsigned(lanes), pmin, pmax);
            LQ_CHECK_LAUNCH("minmax_period");
        } else {
            hipLaunchKernelGGL(minmax_col_kernel, dim3(unsigned(col_blocks), unsigned(splits)),
                               dim3(kThreads), 0, st, x, outer, cols, unsigned(splits), pmin, pmax);
            LQ_CHECK_LAUNCH("minmax_col");
        }
        hipLaunchKernelGGL(minmax_finalize_kernel, dim3(unsigned(C)), dim3(256), 0, st, pmin, pmax, C,
                           unsigned(splits), unsigned(inner), mn, mx);
        LQ_CHECK_LAUNCH("minmax_finalize");
        return LQ_OK;
    }

    // contiguous runs: aim for ~2048 blocks, each with at least 4096 elements; side by side in a run first, then
    // each with a share of the runs where that pays for the second launch.  That launch takes the host 3.5 us; a block that has a
    // channel to itself takes 0.2 (lines in its L2) to 0.6 us per round trip.  us of one block per channel / shares, tensors in the
    // L2, then not: several runs per trip: 6 channels 115 x 93 (6 trips) 5.0 / 8.3, 6 x 512 x 64 (8) 6.2 / 7.8 and 7.8 / 7.3, 6 x 768 x 64
    // (12) 9.5 / 8.3 and 10.4 / 7.4; 300 channels 1024 x 64 (16) 17.0 / 17.3, 1536 x 64 (24) 23.9 / 22.6; 480 and more have the
    // memory busy by themselves: 655 x 443 x 64 13.6 / 15.7, 480 x 640 x 200 41 / 45.  Runs of more than 512, one after the other: 16
    // channels 3 x 2801 (9) 6.4 / 8.4, 20 channels 6 x 1500 (12) 7.4 / 7.8 and 8.7 / 8.2, 8 x 1500 (16) 9.5 / 8.7, 1000 channels
    // 6 x 1500 11.4 / 12.0.  One channel of 32768 in many runs 5.1 / 8.0 and 9.6 / 7.5, 65536 6.9 / 8.3 and 17.6 / 7.5.
    size_t run_splits = 1, splits = 1;
    if (C < 2048) {
        const size_t want = 2048 / C;
        run_splits = inner / 4096 < want ? inner / 4096 : want;
        if (run_splits < 1) run_splits = 1;
        size_t parts = want / run_splits, most = outer * (inner / run_splits) / 4096;
        if (parts > most) parts = most;
        if (parts > outer) parts = outer;
        if (parts < 1) parts = 1;
        if (run_splits == 1) {
            size_t trips = 0, few = 0;  // of a block alone; up to how many it stays alone
            if (inner <= 2 * kThreads) {
                size_t lanes = 1;
                while (lanes * 4 < inner) lanes *= 2;
                const size_t runs = kThreads / lanes;
                trips = outer / (4 * runs) + (outer % (4 * runs) + runs - 1) / runs;
                few = C < 250 ? 9 : C < 400 ? 16 : trips;
            } else {
                const size_t quads = (inner + 3) / 4;
                trips = outer * (quads / (4 * kThreads) + (quads % (4 * kThreads) + kThreads - 1) / kThreads);
                few = 12;
            }
            if (trips <= few) parts = 1;
        }
        if (folded && inner <= 32768) run_splits = parts = 1;
        splits = run_splits * parts;
    }
    float *pmin = mn, *pmax = mx;
    if (const size_t most = ws_limit / (2 * C * sizeof(float)); splits > most) {
        run_splits = run_splits < most ? run_splits : most;
        if (run_splits < 1) run_splits = 1;  // one block per channel writes mn / mx directly: no partials at all
        splits = most / run_splits * run_splits;
        if (splits < 1) splits = 1;
    }
    if (splits > 1) {
        void* ws = nullptr;
        int rc = get_ws(2 * splits * C * sizeof(float), &ws);
        if (rc) return rc;
        pmin = static_cast<float*>(ws);
        pmax = pmin + splits * C;
    }
    dim3 grid{unsigned(C * splits)}, block{kThreads};
    hipLaunchKernelGGL(minmax_seg_kernel, grid, block, 0, st, x, outer, C, inner, unsigned(splits), unsigned(run_splits), pmin,
                       pmax);
    LQ_CHECK_LAUNCH("minmax_seg");
    if (splits > 1) {
        hipLaunchKernelGGL(minmax_finalize_kernel, dim3(unsigned(C)), dim3(256), 0, st, pmin, pmax, C,
                           unsigned(splits), 1u, mn, mx);
        LQ_CHECK_LAUNCH("minmax_finalize");
    }
    return LQ_OK;
}

// What the kernels of small dynamic layers share: every block takes the min / max and qparams of all of x (at most 65536
// floats: repeating that per block costs less than a separate launch and its round trip), quantizes its own 16 rows
// m0 .. m0+15 into LDS and multiplies them with the 16 weight rows n0 .. n0+15: the 16 wavefronts split the k steps of
// v_mfma_i32_16x16x64_i8 (activation fragments from the LDS codes, weight rows from global memory) and meet through LDS
// atomics in `red` [4][64] (red[q * 64 + lane]: activation row m0 + 4 (lane / 16) + q, weight row n0 + lane % 16), which
// is complete when the function returns.  `ld` bytes separate rows of weight codes and of the codes in LDS: K where that is a
// multiple of 16, otherwise a multiple of 16 beyond it with zeros in the weight past K (RAGGED).  Quads of x then straddle
// rows, and every code is placed by itself; what LDS holds past K is multiplied by those zeros.
struct SmallTile {
    float s;        // the activation's scale
    int zp;         // and zero point, as stored
    float c_ws;     // output lanes (tid < 256): scale, code sum and bias of column n0 + tid % 16
    int c_wsum;
    float c_bias;
    // float(acc - zp * wsum[n]) * (s * w_scale[n]) + bias[n] and the optional ReLU, in the order of the GEMM's epilogue
    __device__ __forceinline__ float output(int acc, bool corrected, int relu) const {
        const int corr = (corrected && zp != 0) ? zp * c_wsum : 0;
        const float f = float(acc - corr);
        const float sc = s * c_ws;
        float y = f * sc;
        y = y + c_bias;
        const float floor = relu ? 0.0f : -__builtin_inff();
        return (y < floor) ? floor : y;
    }
};
typedef int dl_v4i __attribute__((ext_vector_type(4)));

template <bool RAGGED>
__device__ __forceinline__ SmallTile small_tile(const float* __restrict__ x, int M, int K, int ld, int8_t* codes, int* red,
                                                const int8_t* __restrict__ w, int N, const float* __restrict__ w_scale,
                                                const int32_t* __restrict__ wsum, const float* __restrict__ bias, int m0,
                                                int n0, int symmetric, int qmin, int qmax, int is_signed, float eps,
                                                float half_range, int off) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int kKeep = 16;
    const int n = M * K, quads = n >> 2;
    const float4* x4 = reinterpret_cast<const float4*>(x);
    // What does not depend on x is requested first, so that it arrives under the quantization: the
    // wavefront's first weight fragment and the output lane's column parameters.
    const int ln = lane & 15, lg = lane >> 4;
    // (requested with lane = 4 * row + chunk, so that four neighbouring lanes read 64 contiguous bytes,
    // and handed to the lane that multiplies it - row lane % 16, chunk lane / 16 - by dl_place)
    const int rq = lane >> 2, cq = lane & 3;
    const int8_t* wrow = w + size_t(n0 + rq < N ? n0 + rq : N - 1) * size_t(ld);
    auto dl_place = [&](dl_v4i f) {
        const int from = (4 * ln + lg) * 4;
        return dl_v4i{__builtin_amdgcn_ds_bpermute(from, f[0]), __builtin_amdgcn_ds_bpermute(from, f[1]),
                      __builtin_amdgcn_ds_bpermute(from, f[2]), __builtin_amdgcn_ds_bpermute(from, f[3])};
    };
    const int ksteps = (ld + 63) >> 6;
    const bool first_in_k = wave < ksteps && wave * 64 + cq * 16 < ld;
    const dl_v4i wf_first = first_in_k ? *reinterpret_cast<const dl_v4i*>(wrow + wave * 64 + cq * 16) : dl_v4i{0, 0, 0, 0};
    SmallTile t;
    const int out_n = n0 + (tid & 15);
    const bool out_lane = tid < 256 && out_n < N;
    t.c_ws = (out_lane && w_scale) ? w_scale[out_n] : 1.0f;
    t.c_wsum = (out_lane && wsum) ? wsum[out_n] : 0;
    t.c_bias = (out_lane && bias) ? bias[out_n] : -0.0f;
    MinMax m{__builtin_inff(), -__builtin_inff(), 0};
    float4 v[kKeep];
#pragma unroll
    for (int u = 0; u < kKeep; ++u) {
        const int i = u * 1024 + tid;
        if (i < quads) v[u] = x4[i];
    }
    const bool in_tail = RAGGED && tid < (n & 3);  // the elements behind the last quad
    float v_tail = 0.f;
    if (in_tail) v_tail = x[4 * quads + tid];
    if (tid < 256) red[tid] = 0;
    // the block's rows m0 .. m0+15 are a contiguous range of elements; rows past M (the last block's padding)
    // feed accumulator rows that are never stored
    const int rows = m0 + 16 < M ? 16 : M - m0;
    const int q_lo = (m0 * K) >> 2, q_hi = ((m0 + rows) * K) >> 2;
    for (int i = ((rows * ld) >> 2) + tid; i < 4 * ld; i += 1024) reinterpret_cast<unsigned*>(codes)[i] = 0u;
#pragma unroll
    for (int u = 0; u < kKeep; ++u)
        if (u * 1024 + tid < quads) mm_update(m, v[u]);
    if (in_tail) mm_update(m, v_tail);
    m = mm_block_reduce(m);
    // (every thread derives the qparams: cheaper than one thread, a barrier and a read)
    const float qnan = __builtin_nanf("");
    float s, z;
    qparams_of(m.nan ? qnan : m.lo, m.nan ? qnan : m.hi, symmetric, qmin, qmax, is_signed, eps, half_range, &s, &z);
    t.s = s, t.zp = int(z) + off;
    const float r = 1.0f / s;
    const QuantizeOp<int8_t> op{x4, reinterpret_cast<Code8x4*>(codes), float(double(qmin)), float(double(qmax)), off};
    if constexpr (!RAGGED) {
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int i = u * 1024 + tid;
            if (i >= q_lo && i < q_hi) op.q[i - q_lo] = op.pack(v[u], s, z, r);
        }
    } else {
        // (element e of the block's range is in row floor((e + 0.5) / K): e < 16 K <= 97 280, so the quotient's rounding, at
        // most 16 * 2^-22, stays below its distance from an integer, at least 0.5 / 6080)
        const float per_row = 1.0f / float(K);
        const int count = rows * K;
        auto put = [&](int e, int8_t code) {
            if (e >= 0 && e < count) {
                const int row = int((float(e) + 0.5f) * per_row);
                codes[row * ld + (e - row * K)] = code;
            }
        };
#pragma unroll
        for (int u = 0; u < kKeep; ++u) {
            const int i = u * 1024 + tid;
            if (i >= q_lo && i <= q_hi && i < quads) {
                const Code8x4 c = op.pack(v[u], s, z, r);
#pragma unroll
                for (int j = 0; j < 4; ++j) put(4 * i + j - m0 * K, c.v[j]);
            }
        }
        if (in_tail) put(4 * quads + tid - m0 * K, op.pack(splat(v_tail), s, z, r).v[0]);
    }
    lds_barrier();  // (the weights are still on their way)

    dl_v4i acc = dl_v4i{0, 0, 0, 0};
    for (int ks = wave; ks < ksteps; ks += 16) {
        const int k = ks * 64 + lg * 16;
        const bool in_k = k < ld;  // ld % 16 == 0: a 16-byte chunk is inside or outside as a whole
        const int kq = ks * 64 + cq * 16;
        const dl_v4i wf = dl_place(ks == wave ? wf_first
                                              : (kq < ld ? *reinterpret_cast<const dl_v4i*>(wrow + kq) : dl_v4i{0, 0, 0, 0}));
        const dl_v4i af = in_k ? *reinterpret_cast<const dl_v4i*>(codes + size_t(ln) * ld + k) : dl_v4i{0, 0, 0, 0};
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, wf, acc, 0, 0, 0);
    }
    if (wave < ksteps) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
            __hip_atomic_fetch_add(&red[q * 64 + lane], acc[q], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __syncthreads();
    return t;
}

// A whole dynamic-quantized Linear on a small activation in one launch
// (lucid/nn/quantized/dynamic/linear.py:87-99: x.min() / x.max(), calculate_qparams, quantize,
// dequantize-free integer GEMM, bias): a block per 16 x 16 outputs.  Same bits as lq_quantize_tensor_dynamic_i8
// followed by lq_qlinear_i8.
template <bool RAGGED>
__global__ __launch_bounds__(1024) void dynamic_linear_small_kernel(
    const float* __restrict__ x, int M, int K, const int8_t* __restrict__ w, int ld, int N, const float* __restrict__ w_scale,
    const int32_t* __restrict__ wsum, const float* __restrict__ bias, int relu, int symmetric, int qmin, int qmax,
    int is_signed, float eps, float half_range, int off, float* __restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) int8_t dl_smem[];
    int8_t* const codes = dl_smem;                                      // [16][ld]: the block's rows
    int* const red = reinterpret_cast<int*>(dl_smem + size_t(16) * ld);  // [4][64]
    const int tid = threadIdx.x, n0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
    const SmallTile t = small_tile<RAGGED>(x, M, K, ld, codes, red, w, N, w_scale, wsum, bias, m0, n0, symmetric, qmin, qmax,
                                           is_signed, eps, half_range, off);
    if (tid < 256) {
        const int q = tid >> 6, l = tid & 63;
        const int mm = m0 + 4 * (l >> 4) + q, nn = n0 + (l & 15);
        if (mm < M && nn < N) out[size_t(mm) * N + nn] = t.output(red[tid], wsum != nullptr, relu);
    }
}

// Two dynamic-quantized Linears with an optional ReLU after each, on a small activation, in ONE
// launch (the MLP Linear(784,256) -> ReLU -> Linear(256,10) at batch 64 is 0.43 MOP: three
// launches cost three round trips).  Layer 1 runs exactly as dynamic_linear_small_kernel runs it -
// a block per 16 x 16 tile of the hidden activation, so the 50 k inputs are quantized by 64 CUs
// at once - with each block's tile (ReLU applied) and its min / max written through to device
// scope; the block that arrives last (one counter, at most kMlpBlocks arrivals) then owns the whole
// hidden activation - 64 KB there, one round trip - and does for layer 2 what the separate operators
// do: the tensor's min / max (from the tiles'), calculate_qparams, the codes, the integer GEMM
// (one wavefront per 16 x 16 output tile), float(acc - zp * wsum[n]) * (s * w_scale[n]) + bias[n],
// ReLU.  Same bits as two lq_dynamic_linear_small_f32 calls (the ReLU between them folded into
// the first).  15.7 us for that MLP; with ONE block doing both layers it was 21 us (one CU's
// vector units quantized all 50 k inputs).  `hid`: [M][ld2] float32, then kMlpBlocks minima and as many maxima;
// `counter`: zero between launches (the last block resets it).  Columns of `hid` from N1 to ld2 hold anything: their codes
// meet the zeros of layer 2's padded weight rows.  KS2: steps of 64 k that ld2 takes at most, and quads of the hidden
// activation per thread of the last block: M * ld2 is at most 4096 KS2.  (More than 64 rows, which the last block's wavefronts
// take 64 at a time, in two calls of two launches 28.5 us, whatever their size: 148 rows of 32-48-15 14.0 in one, 256 of
// 256-128-64 18.1, 2048 of 32-16-8 24.9.)
constexpr int kMlpBlocks = 192, kMlpMaxHidden = 511;
template <bool RAGGED, int KS2>
__global__ __launch_bounds__(1024) void dynamic_mlp2_blocks_kernel(
    const float* __restrict__ x, int M, int K1, const int8_t* __restrict__ w1, int ld1, int N1, const float* __restrict__ ws1,
    const int32_t* __restrict__ wsum1, const float* __restrict__ b1, int relu1, const int8_t* __restrict__ w2, int ld2, int N2,
    const float* __restrict__ ws2, const int32_t* __restrict__ wsum2, const float* __restrict__ b2, int relu2,
    int symmetric, int qmin, int qmax, int is_signed, float eps, float half_range, int off, float* __restrict__ out,
    float* hid, int* counter) {
    extern __shared__ __attribute__((aligned(16))) int8_t mb_smem[];
    __shared__ int s_arrived;
    typedef unsigned mb_v4u __attribute__((ext_vector_type(4)));
    constexpr unsigned kScopeDevice = 16;  // "sc1" cache-policy bit of buffer accesses
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int8_t* const codes = mb_smem;                                       // [16][ld1]: the block's rows
    int* const red = reinterpret_cast<int*>(mb_smem + size_t(16) * ld1);  // [4][64]
    int8_t* const codes2 = mb_smem + size_t(16) * ld1 + 1024;             // [M rounded up to 16][ld2]: the last block's
    const float qnan = __builtin_nanf("");
    const int n0 = blockIdx.x * 16, m0 = blockIdx.y * 16;
    const int nblocks = gridDim.x * gridDim.y, bid = blockIdx.y * gridDim.x + blockIdx.x;
    const int ln = lane & 15, lg = lane >> 4;
    const int rq = lane >> 2, cq = lane & 3;
    auto place = [&](dl_v4i f) {
        const int from = (4 * ln + lg) * 4;
        return dl_v4i{__builtin_amdgcn_ds_bpermute(from, f[0]), __builtin_amdgcn_ds_bpermute(from, f[1]),
                      __builtin_amdgcn_ds_bpermute(from, f[2]), __builtin_amdgcn_ds_bpermute(from, f[3])};
    };
    const size_t hid_bytes = size_t(M) * ld2 * 4;
    const __amdgpu_buffer_rsrc_t hbuf = __builtin_amdgcn_make_buffer_rsrc(hid, 0, int(hid_bytes) + 8 * kMlpBlocks, 0x00020000);
    const SmallTile t = small_tile<RAGGED>(x, M, K1, ld1, codes, red, w1, N1, ws1, wsum1, b1, m0, n0, symmetric, qmin, qmax,
                                           is_signed, eps, half_range, off);
    MinMax hm{__builtin_inff(), -__builtin_inff(), 0};
    if (tid < 256) {
        const int q = tid >> 6, l = tid & 63;
        const int mm = m0 + 4 * (l >> 4) + q, nn = n0 + (l & 15);
        if (mm < M && nn < N1) {
            const float y = t.output(red[tid], wsum1 != nullptr, relu1);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(y), hbuf, unsigned(mm * ld2 + nn) * 4, 0, kScopeDevice);
            mm_update(hm, y);
        }
    }
    hm = mm_block_reduce(hm);
    if (tid == 0) {
        const float lo = hm.nan ? qnan : hm.lo, hi = hm.nan ? qnan : hm.hi;
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(lo), hbuf, unsigned(hid_bytes) + bid * 4, 0, kScopeDevice);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(hi), hbuf, unsigned(hid_bytes) + 4 * kMlpBlocks + bid * 4, 0,
                                              kScopeDevice);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this thread's part of the tile has been written through
    __syncthreads();
    if (tid == 0) s_arrived = __hip_atomic_fetch_add(counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (s_arrived != nblocks - 1) return;

    // ---- the last block: layer 2 on the whole hidden activation.  Everything it needs from
    // memory is requested together: the tiles' ranges, the activation, its weight fragments.
    float slot_lo = __builtin_inff(), slot_hi = -__builtin_inff();
    if (tid < nblocks) {
        slot_lo = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(hbuf, unsigned(hid_bytes) + tid * 4, 0, kScopeDevice));
        slot_hi = __uint_as_float(
            __builtin_amdgcn_raw_buffer_load_b32(hbuf, unsigned(hid_bytes) + 4 * kMlpBlocks + tid * 4, 0, kScopeDevice));
    }
    const int quads2 = (M * ld2) >> 2;  // at most KS2 per thread
    mb_v4u h[KS2];
#pragma unroll
    for (int u = 0; u < KS2; ++u) {
        const int i = u * 1024 + tid;
        h[u] = __builtin_amdgcn_raw_buffer_load_b128(hbuf, unsigned(i < quads2 ? i : 0) * 16, 0, kScopeDevice);
    }
    const int cb2 = wave >> 2;
    const int n2 = cb2 * 16 + ln, nc2 = n2 < N2 ? n2 : N2 - 1;
    dl_v4i w2f[KS2];
    {
        const int r2 = cb2 * 16 + rq;
        const int8_t* wrow2 = w2 + size_t(r2 < N2 ? r2 : N2 - 1) * size_t(ld2) + cq * 16;
#pragma unroll
        for (int ks = 0; ks < KS2; ++ks)
            w2f[ks] = ks * 64 + cq * 16 < ld2 ? *reinterpret_cast<const dl_v4i*>(wrow2 + ks * 64) : dl_v4i{0, 0, 0, 0};
    }
    SmallTile t2;
    t2.c_ws = ws2 ? ws2[nc2] : 1.0f;
    t2.c_wsum = wsum2 ? wsum2[nc2] : 0;
    t2.c_bias = b2 ? b2[nc2] : -0.0f;
    for (int i = quads2 + tid; i < ((M + 15) >> 4) * 4 * ld2; i += 1024) reinterpret_cast<unsigned*>(codes2)[i] = 0u;
    MinMax tm{slot_lo, slot_hi, int((slot_lo != slot_lo) | (slot_hi != slot_hi))};
    if (tm.nan) tm.lo = __builtin_inff(), tm.hi = -__builtin_inff();
    tm = mm_block_reduce(tm);
    if (tid == 0) *counter = 0;  // ready for the next launch
    float s2, z2;
    qparams_of(tm.nan ? qnan : tm.lo, tm.nan ? qnan : tm.hi, symmetric, qmin, qmax, is_signed, eps, half_range, &s2, &z2);
    t2.s = s2, t2.zp = int(z2) + off;
    {
        const float r2 = 1.0f / s2;
        const QuantizeOp<int8_t> op{nullptr, reinterpret_cast<Code8x4*>(codes2), float(double(qmin)), float(double(qmax)), off};
#pragma unroll
        for (int u = 0; u < KS2; ++u) {
            const int i = u * 1024 + tid;
            if (i < quads2) op.q[i] = op.pack(__builtin_bit_cast(float4, h[u]), s2, z2, r2);
        }
    }
    if (cb2 * 16 < N2) {
#pragma unroll
        for (int ks = 0; ks < KS2; ++ks) w2f[ks] = place(w2f[ks]);
    }
    __syncthreads();
    if (cb2 * 16 < N2) {
        for (int rb2 = wave & 3; rb2 * 16 < M; rb2 += 4) {
            dl_v4i acc2 = dl_v4i{0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < KS2; ++ks) {
                const int k = ks * 64 + lg * 16;
                if (ks * 64 < ld2) {  // uniform
                    const dl_v4i af = k < ld2 ? *reinterpret_cast<const dl_v4i*>(codes2 + size_t(16 * rb2 + ln) * ld2 + k)
                                              : dl_v4i{0, 0, 0, 0};
                    acc2 = __builtin_amdgcn_mfma_i32_16x16x64_i8(af, w2f[ks], acc2, 0, 0, 0);
                }
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int mm = 16 * rb2 + 4 * lg + q;
                if (mm < M && n2 < N2) out[size_t(mm) * N2 + n2] = t2.output(acc2[q], wsum2 != nullptr, relu2);
            }
        }
    }
}

// Blocks that may meet through the slots: no more than the share of the device that one hardware queue may have (with 32
// queues that is 32; 16 are far below any).
int exchange_blocks(int* most) {
    static DeviceOnce once;
    static int capacity[32] = {0};
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    const int rc = device_once(once, [&]() -> int {
        int flat = 0, ragged = 0, cus = 0;
        LQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&flat, quantize_tensor_dynamic_kernel<false, false>, kDynThreads, 0));
        LQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&ragged, quantize_tensor_dynamic_kernel<false, true>, kDynThreads, 0));
        LQ_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        capacity[dev] = (flat < ragged ? flat : ragged) * cus;
        return LQ_OK;
    });
    if (rc) return rc;
    const int share = capacity[dev] / hardware_queues();
    *most = share < 16 ? 16 : share < kExchange ? share : kExchange;
    return LQ_OK;
}

// Dynamic per-tensor quantization of n = rows * cols elements to rows of ld codes.
int quantize_tensor(const float* x, size_t n, unsigned cols, unsigned ld, int symmetric, int qmin, int qmax, int is_signed,
                    float eps, int off, float* scale, float* zp, float* mn, float* mx, int8_t* q, hipStream_t st,
                    int polls = kExchangePolls) {
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    const bool ragged = ld != cols;
    const size_t codes = ragged ? n / cols * ld : n;
    const size_t blocks = codes ? (codes + kDynPerBlock - 1) / kDynPerBlock : 1;
    LQ_REQUIRE((!ragged || blocks * kDynPerBlock < (size_t(1) << 32)) && blocks < 0x7fffffffull, LQ_ERR_SHAPE,
               "dynamic quantization of %zu elements", n);
    void* tmp = nullptr;
    int most = 1;
    if (blocks > 1 && blocks <= size_t(kExchange)) {
        if (const int rc = exchange_blocks(&most)) return rc;
    }
    bool exchange = blocks <= size_t(most);
    size_t fresh = 0;
    std::unique_lock<std::recursive_mutex> lock;
    if (blocks > 1) {
        lock = scratch_lock(st);
        if (exchange) {
            // not in a graph: slots first cleared there would be unset until its replay, and replays on
            // another stream would share them with this one
            hipStreamCaptureStatus capturing = hipStreamCaptureStatusNone;
            if (st) LQ_HIP(hipStreamIsCapturing(st, &capturing));  // (see lq_stream_is_capturing)
            exchange = capturing == hipStreamCaptureStatusNone;
        }
        const int rc = exchange ? stream_buffer(7, sizeof(DynScratch), 0, st, &tmp, &fresh)
                                : call_buffer(5, 2 * kMaxParts * sizeof(float), st, &tmp);
        if (rc) return rc;
    }
    DynScratch* d = exchange ? static_cast<DynScratch*>(tmp) : nullptr;
    float* parts = static_cast<float*>(tmp);
    if (fresh) {
        int rc = lq_fill_bytes(d, 0xff, sizeof(d->slot), reinterpret_cast<lq_stream>(st));
        if (!rc) rc = lq_fill_bytes(&d->left, 0, sizeof(d->left), reinterpret_cast<lq_stream>(st));
        if (rc) return rc;
    }
    auto launch = [&](auto kernel, const float* ranges, int n_ranges) {
        hipLaunchKernelGGL(kernel, dim3(unsigned(blocks)), dim3(kDynThreads), 0, st, x, n, cols, ld, symmetric, qmin, qmax,
                           is_signed, eps, half_range, off, d, polls, ranges, n_ranges, scale, zp, mn, mx, q);
    };
    if (exchange) {
        ragged ? launch(quantize_tensor_dynamic_kernel<false, true>, nullptr, 0)
               : launch(quantize_tensor_dynamic_kernel<false, false>, nullptr, 0);
        LQ_CHECK_LAUNCH("quantize_tensor_dynamic");
        return LQ_OK;
    }
    // slices of at least 4096 elements
    const unsigned splits = n < 4096 ? 1u : (n / 4096 < size_t(kMaxParts) ? unsigned(n / 4096) : unsigned(kMaxParts));
    hipLaunchKernelGGL(minmax_seg_kernel, dim3(splits), dim3(kThreads), 0, st, x, size_t(1), size_t(1), n, splits, splits, parts,
                       parts + splits);
    LQ_CHECK_LAUNCH("minmax_seg");
    ragged ? launch(quantize_tensor_dynamic_kernel<true, true>, parts, int(splits))
           : launch(quantize_tensor_dynamic_kernel<true, false>, parts, int(splits));
    LQ_CHECK_LAUNCH("quantize_tensor_parts");
    return LQ_OK;
}

int dynamic_mlp2(int max_rows, const float* x, int M, int K1, const int8_t* w1, int ldw1, int N1, const float* w1_scale,
                 const int32_t* w1sum, const float* bias1, int relu1, const int8_t* w2, int ldw2, int N2,
                 const float* w2_scale, const int32_t* w2sum, const float* bias2, int relu2,
                 int symmetric, int qmin, int qmax, int is_signed, float eps, int code_offset,
                 float* out, lq_stream stream) {
    if (M == 0 || N2 == 0) return LQ_OK;
    LQ_REQUIRE(x && w1 && w2 && out, LQ_ERR_VALUE, "dynamic_mlp2_small: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "dynamic_mlp2_small: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    // a block holds 16 rows of x's codes; the last one also the hidden activation's codes, in rows of ldw2 bytes
    LQ_REQUIRE(M > 0 && M <= max_rows && K1 > 0 && ldw1 >= K1 && ldw1 % 16 == 0 && ldw1 <= 1024 && N1 > 0 && N1 <= kMlpMaxHidden &&
                   ldw2 >= N1 && ldw2 % 16 == 0 && ldw2 <= 512 && N2 > 0 && N2 <= 64 && aligned16(x) && aligned16(w1) &&
                   aligned16(w2) && long(M) * K1 <= 65536 && long(M) * ldw2 <= 32768 &&
                   ((M + 15) / 16) * ((N1 + 15) / 16) <= kMlpBlocks,
               LQ_ERR_NOT_IMPLEMENTED,
               "dynamic_mlp2_small: takes up to %d rows, weight rows of a multiple of 16 bytes (K1 up to 1024, a hidden width "
               "up to %d), up to 64 outputs, 65536 inputs, 32768 hidden values in 192 tiles and 16-byte aligned operands (got "
               "M = %d, K1 = %d in rows of %d, N1 = %d in rows of %d, N2 = %d); use two lq_dynamic_linear_f32 calls", max_rows, kMlpMaxHidden, M, K1, ldw1, N1, ldw2, N2);
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    // the hidden activation and the tiles' ranges pass through the stream's split-K scratch
    SkScratch sk;
    const auto lock = scratch_lock(as_stream(stream));
    const size_t hid_bytes = size_t(M) * ldw2 * 4;
    if (int rc = sk_scratch(1, hid_bytes + 8 * kMlpBlocks, as_stream(stream), &sk)) return rc;
    const size_t lds = size_t(16) * ldw1 + 1024 + size_t((M + 15) / 16 * 16) * ldw2;  // at most 16 + 1 + 32 + 7.5 KiB
    static DeviceOnce attr_once[4];
    auto launch = [&](auto kernel, int form) -> int {
        if (int rc = allow_dynamic_lds(attr_once[form], reinterpret_cast<const void*>(kernel), 64 * 1024)) return rc;
        hipLaunchKernelGGL(kernel, dim3(unsigned((N1 + 15) / 16), unsigned((M + 15) / 16)), dim3(1024), lds,
                           as_stream(stream), x, M, K1, w1, ldw1, N1, w1_scale, w1sum, bias1, relu1, w2, ldw2, N2, w2_scale,
                           w2sum, bias2, relu2, symmetric, qmin, qmax, is_signed, eps, half_range, code_offset, out,
                           reinterpret_cast<float*>(sk.slabs), sk.counters);
        LQ_CHECK_LAUNCH("dynamic_mlp2_small");
        return LQ_OK;
    };
    const bool ragged = ldw1 != K1, wide = ldw2 > 256 || M * ldw2 > 16384;
    return ragged ? (wide ? launch(dynamic_mlp2_blocks_kernel<true, 8>, 0) : launch(dynamic_mlp2_blocks_kernel<true, 4>, 1))
                  : (wide ? launch(dynamic_mlp2_blocks_kernel<false, 8>, 2) : launch(dynamic_mlp2_blocks_kernel<false, 4>, 3));
}

int quantize_rows(const float* x, size_t rows, size_t cols, bool ragged, int symmetric, int qmin, int qmax, int is_signed,
                  float eps, int off, float* scale, float* zp, float* mn, float* mx, int8_t* q, hipStream_t st) {
    if (rows == 0) return LQ_OK;
    LQ_REQUIRE(x && q && scale && zp, LQ_ERR_VALUE, "quantize_rows_dynamic: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + off >= -128 && qmax + off <= 127, LQ_ERR_VALUE,
               "quantize_rows_dynamic: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, off);
    LQ_REQUIRE(ragged || (cols >= 4 && cols % 4 == 0 && cols <= 16384 && aligned16(x) &&
                          (reinterpret_cast<uintptr_t>(q) & 3u) == 0),
               LQ_ERR_NOT_IMPLEMENTED,
               "quantize_rows_dynamic: rows of %zu floats (a multiple of 4, at most 16384, 16-byte aligned) are what this call "
               "takes; use lq_quantize_rows_dynamic_ragged_i8, or lq_minmax + lq_calc_qparams + lq_quantize", cols);
    LQ_REQUIRE(cols >= 1 && cols <= 16384 && rows <= 0x7fffffffull, LQ_ERR_NOT_IMPLEMENTED,
               "quantize_rows_dynamic: %zu rows of %zu floats (1 to 16384); use lq_minmax + lq_calc_qparams + lq_quantize", rows, cols);
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(unsigned(rows)), dim3(256), 0, st, x, int(cols), symmetric, qmin, qmax, is_signed, eps,
                           half_range, off, scale, zp, mn, mx, q);
    };
    auto of_length = [&](auto r) {
        constexpr int R = decltype(r)::value;
        ragged ? launch(quantize_rows_dynamic_kernel<R, true>) : launch(quantize_rows_dynamic_kernel<R, false>);
    };
    if (cols <= 1024) of_length(std::integral_constant<int, 1>{});
    else if (cols <= 4096) of_length(std::integral_constant<int, 4>{});
    else if (cols <= 8192) of_length(std::integral_constant<int, 8>{});
    else of_length(std::integral_constant<int, 16>{});
    LQ_CHECK_LAUNCH("quantize_rows_dynamic");
    return LQ_OK;
}

}  // namespace

namespace lq {
int minmax_noalloc_init() {
    void* p = nullptr;
    return noalloc_scratch_ptr(&p);
}
}  // namespace lq

extern "C" {

int lq_quantize_tensor_dynamic_i8(const float* x, size_t n, int symmetric, int qmin, int qmax, int is_signed,
                                  float eps, int code_offset, float* scale, float* zp, float* mn_out,
                                  float* mx_out, int8_t* q, lq_stream stream) {
    LQ_REQUIRE(scale && zp && (n == 0 || (x && q)), LQ_ERR_VALUE, "quantize_tensor_dynamic: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "quantize_tensor_dynamic: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    LQ_REQUIRE(n <= (size_t(1) << 18), LQ_ERR_NOT_IMPLEMENTED,
               "quantize_tensor_dynamic: the one-launch form is for tensors of up to 262144 elements (got %zu); "
               "use lq_minmax + lq_calc_qparams + lq_quantize", n);
    return quantize_tensor(x, n, unsigned(n ? n : 1), unsigned(n ? n : 1), symmetric, qmin, qmax, is_signed, eps,
                           code_offset, scale, zp, mn_out, mx_out, q, as_stream(stream));
}

int lq_quantize_tensor_dynamic_polls_i8(const float* x, size_t rows, unsigned cols, unsigned ld, int symmetric, int qmin,
                                        int qmax, int is_signed, float eps, int code_offset, float* scale, float* zp,
                                        float* mn_out, float* mx_out, int8_t* q, int polls, lq_stream stream) {
    LQ_REQUIRE(scale && zp && x && q, LQ_ERR_VALUE, "quantize_tensor_dynamic: NULL pointer");
    LQ_REQUIRE(rows > 0 && cols > 0 && ld >= cols && (ld == cols || ld % 4 == 0) && ld <= 0x7fffffffu &&
                   rows <= (size_t(1) << 32) / ld,
               LQ_ERR_SHAPE, "quantize_tensor_dynamic: %zu rows of %u elements and %u codes", rows, cols, ld);
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "quantize_tensor_dynamic: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    LQ_REQUIRE(polls >= 0, LQ_ERR_VALUE, "quantize_tensor_dynamic: %d polls", polls);
    return quantize_tensor(x, rows * cols, cols, ld, symmetric, qmin, qmax, is_signed, eps, code_offset, scale, zp, mn_out,
                           mx_out, q, as_stream(stream), polls < kExchangePolls ? polls : kExchangePolls);
}

int lq_dynamic_linear_f32(const float* x, int M, int K, const int8_t* w, int ldw, int N, const float* w_scale,
                          const int32_t* wsum, const float* bias, int relu, int symmetric, int qmin, int qmax,
                          int is_signed, float eps, int code_offset, float* out, lq_stream stream) {
    LQ_REQUIRE(M >= 0 && N >= 0 && K >= 0, LQ_ERR_SHAPE, "dynamic_linear: negative extent");
    if (M == 0 || N == 0) return LQ_OK;
    LQ_REQUIRE(out && w_scale && wsum && (K == 0 || (x && w)), LQ_ERR_VALUE, "dynamic_linear: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "dynamic_linear: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    LQ_REQUIRE(ldw >= K && ldw % 16 == 0 && (K == 0 || aligned16(w)), LQ_ERR_VALUE,
               "dynamic_linear: weight rows of %d bytes for K = %d (a multiple of 16, zeros past K, 16-byte aligned)", ldw, K);
    LQ_REQUIRE(ldw <= 131071, LQ_ERR_SHAPE, "dynamic_linear: K = %d overflows the int32 accumulator", K);
    hipStream_t st = as_stream(stream);
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    const size_t n = size_t(M) * K;
    if (M == 1 && K > 0 && K <= 16384) {
        // every block quantizes the whole row: eight wavefronts, or four where that leaves CUs without a block
        const int waves = (N + 31) / 32 < 256 ? 4 : 8;
        const auto kernel = K >= 4 && K <= waves * 64 * 16 ? dynamic_gemv1_kernel<true> : dynamic_gemv1_kernel<false>;
        hipLaunchKernelGGL(kernel, dim3(unsigned((N + 4 * waves - 1) / (4 * waves))), dim3(waves * 64),
                           size_t((K + 4095) / 4096) * 4096, st, x, K, w, ldw, N, w_scale, wsum, bias, relu, symmetric, qmin,
                           qmax, is_signed, eps, half_range, code_offset, out);
        LQ_CHECK_LAUNCH("dynamic_gemv1");
        return LQ_OK;
    }
    // codes (rows as long as the weight's), scale and zero point, then the GEMM
    const size_t code_bytes = (size_t(M) * ldw + 255) / 256 * 256;
    void* tmp = nullptr;
    const auto lock = scratch_lock(st);
    int rc = call_buffer(6, code_bytes + 256, st, &tmp);
    if (rc) return rc;
    int8_t* codes = static_cast<int8_t*>(tmp);
    float* qp = reinterpret_cast<float*>(codes + code_bytes);
    rc = quantize_tensor(x, n, unsigned(K ? K : 1), unsigned(ldw ? ldw : 1), symmetric, qmin, qmax, is_signed, eps,
                         code_offset, qp, qp + 1, qp + 2, qp + 3, codes, st);
    if (rc) return rc;
    GemmArgs g{};
    g.a = codes, g.w = w, g.M = M, g.N = N, g.K = ldw;
    g.wsum = wsum, g.a_zp = code_offset, g.a_zp_dev = qp + 1, g.a_scale = qp, g.w_scale = w_scale;
    g.bias = bias, g.bias_dtype = LQ_F32, g.relu = relu, g.out_mode = OUT_F32, g.out = out, g.ldo = N, g.ldr = N;
    return run_gemm(g, 0, 0, st);
}

int lq_dynamic_mlp2_small_f32(const float* x, int M, int K1, const int8_t* w1, int N1, const float* w1_scale,
                              const int32_t* w1sum, const float* bias1, int relu1, const int8_t* w2, int N2,
                              const float* w2_scale, const int32_t* w2sum, const float* bias2, int relu2, int symmetric,
                              int qmin, int qmax, int is_signed, float eps, int code_offset, float* out,
                              lq_stream stream) {
    if (M == 0 || N2 == 0) return LQ_OK;
    LQ_REQUIRE(K1 >= 16 && K1 % 16 == 0 && long(M) * K1 <= 65536 && N1 >= 16 && N1 % 16 == 0 && N1 <= 256,
               LQ_ERR_NOT_IMPLEMENTED,
               "dynamic_mlp2_small: takes K1 %% 16 == 0 and a hidden width that is a multiple of 16 up to 256 (got M = %d, "
               "K1 = %d, N1 = %d); use lq_dynamic_mlp2_small_rows_f32 or two lq_dynamic_linear_f32 calls", M, K1, N1);
    return lq_dynamic_mlp2_small_rows_f32(x, M, K1, w1, K1, N1, w1_scale, w1sum, bias1, relu1, w2, N1, N2, w2_scale, w2sum,
                                          bias2, relu2, symmetric, qmin, qmax, is_signed, eps, code_offset, out, stream);
}

int lq_dynamic_mlp2_small_rows_f32(const float* x, int M, int K1, const int8_t* w1, int ldw1, int N1, const float* w1_scale,
                                   const int32_t* w1sum, const float* bias1, int relu1, const int8_t* w2, int ldw2, int N2,
                                   const float* w2_scale, const int32_t* w2sum, const float* bias2, int relu2,
                                   int symmetric, int qmin, int qmax, int is_signed, float eps, int code_offset,
                                   float* out, lq_stream stream) {
    return dynamic_mlp2(64, x, M, K1, w1, ldw1, N1, w1_scale, w1sum, bias1, relu1, w2, ldw2, N2, w2_scale, w2sum, bias2, relu2,
                        symmetric, qmin, qmax, is_signed, eps, code_offset, out, stream);
}

int lq_dynamic_mlp2_rows_f32(const float* x, int M, int K1, const int8_t* w1, int ldw1, int N1, const float* w1_scale,
                             const int32_t* w1sum, const float* bias1, int relu1, const int8_t* w2, int ldw2, int N2,
                             const float* w2_scale, const int32_t* w2sum, const float* bias2, int relu2,
                             int symmetric, int qmin, int qmax, int is_signed, float eps, int code_offset,
                             float* out, lq_stream stream) {
    return dynamic_mlp2(2048, x, M, K1, w1, ldw1, N1, w1_scale, w1sum, bias1, relu1, w2, ldw2, N2, w2_scale, w2sum, bias2, relu2,
                        symmetric, qmin, qmax, is_signed, eps, code_offset, out, stream);
}

int lq_dynamic_linear_small_f32(const float* x, int M, int K, const int8_t* w, int N, const float* w_scale,
                                const int32_t* wsum, const float* bias, int relu, int symmetric, int qmin, int qmax,
                                int is_signed, float eps, int code_offset, float* out, lq_stream stream) {
    if (M == 0 || N == 0) return LQ_OK;
    LQ_REQUIRE(K >= 16 && K % 16 == 0 && K <= 6080, LQ_ERR_NOT_IMPLEMENTED,
               "dynamic_linear_small: takes K %% 16 == 0 and K <= 6080 (got K = %d); use lq_dynamic_linear_small_rows_f32 or "
               "lq_quantize_tensor_dynamic_i8 + lq_qlinear_i8", K);
    return lq_dynamic_linear_small_rows_f32(x, M, K, w, K, N, w_scale, wsum, bias, relu, symmetric, qmin, qmax, is_signed, eps,
                                            code_offset, out, stream);
}

int lq_dynamic_linear_small_rows_f32(const float* x, int M, int K, const int8_t* w, int ldw, int N, const float* w_scale,
                                     const int32_t* wsum, const float* bias, int relu, int symmetric, int qmin, int qmax,
                                     int is_signed, float eps, int code_offset, float* out, lq_stream stream) {
    if (M == 0 || N == 0) return LQ_OK;
    LQ_REQUIRE(x && w && out, LQ_ERR_VALUE, "dynamic_linear_small: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "dynamic_linear_small: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    // 16 rows of codes (16 ldw bytes) + 1 KiB of reduction scratch have to fit the 96 KiB of dynamic
    // LDS the kernel is allowed: ldw <= 6080
    LQ_REQUIRE(M > 0 && M <= 64 && K > 0 && ldw >= K && ldw % 16 == 0 && long(M) * K <= 65536 && ldw <= 6080 && N > 0 &&
                   aligned16(x) && aligned16(w),
               LQ_ERR_NOT_IMPLEMENTED,
               "dynamic_linear_small: takes up to 64 rows, weight rows of a multiple of 16 bytes up to 6080, at most 65536 "
               "activations and 16-byte aligned operands (got M = %d, K = %d in rows of %d); use "
               "lq_quantize_tensor_dynamic_i8 + lq_qlinear_i8", M, K, ldw);
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    const int tiles = (M + 15) / 16;
    const size_t lds = size_t(16) * ldw + 256 * sizeof(int);
    static DeviceOnce attr_once[2];
    auto launch = [&](auto kernel, int form) -> int {
        if (int rc = allow_dynamic_lds(attr_once[form], reinterpret_cast<const void*>(kernel), 96 * 1024)) return rc;
        hipLaunchKernelGGL(kernel, dim3(unsigned((N + 15) / 16), unsigned(tiles)), dim3(1024), lds, as_stream(stream), x, M, K,
                           w, ldw, N, w_scale, wsum, bias, relu, symmetric, qmin, qmax, is_signed, eps, half_range,
                           code_offset, out);
        LQ_CHECK_LAUNCH("dynamic_linear_small");
        return LQ_OK;
    };
    return ldw != K ? launch(dynamic_linear_small_kernel<true>, 0) : launch(dynamic_linear_small_kernel<false>, 1);
}

int lq_quantize_rows_dynamic_i8(const float* x, size_t rows, size_t cols, int symmetric, int qmin, int qmax,
                                int is_signed, float eps, int code_offset, float* scale, float* zp,
                                float* mn_out, float* mx_out, int8_t* q, lq_stream stream) {
    return quantize_rows(x, rows, cols, false, symmetric, qmin, qmax, is_signed, eps, code_offset, scale, zp, mn_out, mx_out, q,
                         as_stream(stream));
}

int lq_quantize_rows_dynamic_ragged_i8(const float* x, size_t rows, size_t cols, int symmetric, int qmin, int qmax,
                                       int is_signed, float eps, int code_offset, float* scale, float* zp,
                                       float* mn_out, float* mx_out, int8_t* q, lq_stream stream) {
    return quantize_rows(x, rows, cols, true, symmetric, qmin, qmax, is_signed, eps, code_offset, scale, zp, mn_out, mx_out, q,
                         as_stream(stream));
}

int lq_minmax(const float* x, size_t outer, size_t C, size_t inner, float* mn, float* mx,
              lq_stream stream) {
    hipStream_t st = as_stream(stream);
    const auto lock = scratch_lock(st);
    return minmax_launch(x, outer, C, inner, mn, mx, st, ~size_t(0),
                         [st](size_t nbytes, void** ws) {
                             return recording_graph() ? call_buffer(5, nbytes, st, ws) : workspace(nbytes, st, ws);
                         });
}

int lq_minmax_noalloc(const float* x, size_t outer, size_t C, size_t inner, float* mn, float* mx,
                      lq_stream stream) {
    void* scratch = nullptr;
    int rc = noalloc_scratch_ptr(&scratch);
    if (rc) return rc;
    return minmax_launch(x, outer, C, inner, mn, mx, as_stream(stream), kNoAllocScratchBytes,
                         [scratch](size_t nbytes, void** ws) {
                             // minmax_launch sizes its partials to the limit it was given
                             LQ_REQUIRE(nbytes <= kNoAllocScratchBytes, LQ_ERR_SHAPE,
                                        "minmax_noalloc: %zu bytes of partials exceed the %zu-byte static scratch",
                                        nbytes, kNoAllocScratchBytes);
                             *ws = scratch;
                             return int(LQ_OK);
                         });
}

int lq_calc_qparams(const float* mn, const float* mx, size_t C, int symmetric, int qmin, int qmax,
                    int is_signed, float eps, float* scale, float* zp, lq_stream stream) {
    if (C == 0) return LQ_OK;
    LQ_REQUIRE(mn && mx && scale && zp, LQ_ERR_VALUE, "calc_qparams: NULL pointer");
    LQ_REQUIRE(qmax > qmin, LQ_ERR_VALUE, "calc_qparams: empty grid [%d,%d]", qmin, qmax);
    // (quant_max - quant_min) / 2.0 is a Python float promoted to float32
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    hipLaunchKernelGGL(calc_qparams_kernel, dim3(unsigned((C + 255) / 256)), dim3(256), 0,
                       as_stream(stream), mn, mx, C, symmetric, qmin, qmax, is_signed, eps, half_range,
                       scale, zp);
    LQ_CHECK_LAUNCH("calc_qparams");
    return LQ_OK;
}

size_t lq_range_buffer_bytes(void) { return size_t(kRangeWords) * 4; }

int lq_calc_qparams_from_range(const float* range, int symmetric, int qmin, int qmax, int is_signed,
                               float eps, float* scale, float* zp, float* mn_out, float* mx_out,
                               lq_stream stream) {
    LQ_REQUIRE(range && scale && zp, LQ_ERR_VALUE, "calc_qparams_from_range: NULL pointer");
    LQ_REQUIRE(qmax > qmin, LQ_ERR_VALUE, "calc_qparams_from_range: empty grid [%d,%d]", qmin, qmax);
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    hipLaunchKernelGGL(calc_qparams_from_range_kernel, dim3(1), dim3(1024), 0, as_stream(stream), range,
                       symmetric, qmin, qmax, is_signed, eps, half_range, scale, zp, mn_out, mx_out);
    LQ_CHECK_LAUNCH("calc_qparams_from_range");
    return LQ_OK;
}

int lq_quantize_from_range_i8(const float* x, size_t n, const float* range, int symmetric, int qmin, int qmax, int is_signed,
                              float eps, int code_offset, float* scale, float* zp, int8_t* q, lq_stream stream) {
    LQ_REQUIRE(range && scale && zp && (n == 0 || (x && q)), LQ_ERR_VALUE, "quantize_from_range: NULL pointer");
    LQ_REQUIRE(qmax > qmin && qmin + code_offset >= -128 && qmax + code_offset <= 127, LQ_ERR_VALUE,
               "quantize_from_range: grid [%d,%d] + offset %d does not fit int8", qmin, qmax, code_offset);
    // (a handful of elements, and addresses that vectors cannot take: the two steps as well)
    if (n < 4 || n > kRangeTensor || !aligned16(x) || (reinterpret_cast<uintptr_t>(q) & 3u) != 0) {
        const int rc = lq_calc_qparams_from_range(range, symmetric, qmin, qmax, is_signed, eps, scale, zp, nullptr, nullptr, stream);
        return rc ? rc : lq_quantize(x, q, LQ_I8, code_offset, 1, 1, n, scale, zp, 0, qmin, qmax, stream);
    }
    const float half_range = float((double(qmax) - double(qmin)) / 2.0);
    const QuantizeOp<int8_t> op{reinterpret_cast<const float4*>(x), reinterpret_cast<Code8x4*>(q), float(double(qmin)),
                                float(double(qmax)), code_offset};
    const unsigned quads = unsigned(n / 4), blocks = (quads + 1024 * kRangeChunk - 1) / (1024 * kRangeChunk);
    hipLaunchKernelGGL(quantize_range_kernel, dim3(blocks), dim3(1024), 0, as_stream(stream), op, quads,
                       unsigned(n % 4), range, symmetric, qmin, qmax, is_signed, eps, half_range, scale, zp);
    LQ_CHECK_LAUNCH("quantize_from_range");
    return LQ_OK;
}

int lq_quantize(const float* x, void* q, int q_dtype, int code_offset, size_t outer, size_t C,
                size_t inner, const float* scale, const float* zp, int qparams_on_host, int qmin,
                int qmax, lq_stream stream) {
    if (outer * C * inner == 0) return LQ_OK;
    LQ_REQUIRE(x && q, LQ_ERR_VALUE, "quantize: NULL tensor pointer");
    LQ_REQUIRE(q_dtype == LQ_I8 || q_dtype == LQ_I16, LQ_ERR_DTYPE,
               "quantize: code storage must be int8 or int16 (got dtype %d)", q_dtype);
    const int lim_lo = q_dtype == LQ_I8 ? -128 : -32768, lim_hi = q_dtype == LQ_I8 ? 127 : 32767;
    LQ_REQUIRE(qmin <= qmax && qmin + code_offset >= lim_lo && qmax + code_offset <= lim_hi,
               LQ_ERR_VALUE, "quantize: grid [%d,%d] + offset %d does not fit the code storage", qmin,
               qmax, code_offset);
    QParams qp;
    int rc = make_qparams(scale, zp, qparams_on_host, C, &qp, "quantize");
    if (rc) return rc;
    const float lo = float(double(qmin)), hi = float(double(qmax));
    if (q_dtype == LQ_I8) {
        QuantizeOp<int8_t> op{reinterpret_cast<const float4*>(x), reinterpret_cast<Code8x4*>(q), lo, hi,
                              code_offset};
        return launch_elementwise(op, outer, C, inner, qp, aligned16(x) && aligned16(q),
                                  as_stream(stream), "quantize");
    }
    QuantizeOp<int16_t> op{reinterpret_cast<const float4*>(x), reinterpret_cast<Code16x4*>(q), lo, hi,
                           code_offset};
    return launch_elementwise(op, outer, C, inner, qp, aligned16(x) && aligned16(q), as_stream(stream),
                              "quantize");
}

int lq_dequantize(const void* q, int q_dtype, int code_offset, float* out, size_t outer, size_t C,
                  size_t inner, const float* scale, const float* zp, int qparams_on_host,
                  lq_stream stream) {
    if (outer * C * inner == 0) return LQ_OK;
    LQ_REQUIRE(q && out, LQ_ERR_VALUE, "dequantize: NULL tensor pointer");
    LQ_REQUIRE(q_dtype == LQ_I8 || q_dtype == LQ_I16, LQ_ERR_DTYPE,
               "dequantize: code storage must be int8 or int16 (got dtype %d)", q_dtype);
    QParams qp;
    int rc = make_qparams(scale, zp, qparams_on_host, C, &qp, "dequantize");
    if (rc) return rc;
    if (q_dtype == LQ_I8) {
        DequantizeOp<int8_t> op{reinterpret_cast<const Code8x4*>(q), reinterpret_cast<float4*>(out),
                                code_offset};
        return launch_elementwise(op, outer, C, inner, qp, aligned16(q) && aligned16(out),
                                  as_stream(stream), "dequantize");
    }
    DequantizeOp<int16_t> op{reinterpret_cast<const Code16x4*>(q), reinterpret_cast<float4*>(out),
                             code_offset};
    return launch_elementwise(op, outer, C, inner, qp, aligned16(q) && aligned16(out),
                              as_stream(stream), "dequantize");
}

int lq_fake_quantize(const float* x, float* out, size_t outer, size_t C, size_t inner,
                     const float* scale, const float* zp, int qparams_on_host, int qmin, int qmax,
                     lq_stream stream) {
    if (outer * C * inner == 0) return LQ_OK;
    LQ_REQUIRE(x && out, LQ_ERR_VALUE, "fake_quantize: NULL tensor pointer");
    LQ_REQUIRE(qmin <= qmax, LQ_ERR_VALUE, "fake_quantize: empty grid [%d,%d]", qmin, qmax);
    QParams qp;
    int rc = make_qparams(scale, zp, qparams_on_host, C, &qp, "fake_quantize");
    if (rc) return rc;
    FakeQuantizeOp op{reinterpret_cast<const float4*>(x), reinterpret_cast<float4*>(out),
                      float(double(qmin)), float(double(qmax))};
    return launch_elementwise(op, outer, C, inner, qp, aligned16(x) && aligned16(out),
                              as_stream(stream), "fake_quantize");
}

}  // extern "C"
