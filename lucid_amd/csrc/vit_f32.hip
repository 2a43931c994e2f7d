// float32 companions of the int8 Linear path: what a ViT block does between its
// quantized Linears.  Lucid's dynamic-quantized ViT keeps LayerNorm, attention,
// GELU, the residual adds and the patch embedding in float32
// (lucid/models/vision/vit/_model.py:132-161,202-204,275-278,449-458); these kernels
// are those steps on gfx950, in float32 end to end:
//
//   lq_layernorm_f32        lucid/_C/backend/cpu/Norm.cpp:35-65
//   lq_gelu_f32             lucid/nn/functional/activations.py:219 (approximate="none", erf)
//   lq_add_f32              residual add
//   lq_attention_f32        scaled dot-product attention, CpuBackend.h:7603-7730,
//                           read straight from the packed qkv activation
//   lq_patchify_f32 + lq_sgemm_nt_f32   the stride = kernel patch convolution as a GEMM
//   lq_assemble_tokens_f32  class token + position table
//   lq_patch_embed_f32      the three above in one launch: the GEMM gathers the patches itself
//
// Matrix products use the float32 MFMA instructions; results agree with a CPU
// float32 evaluation to rounding-order differences (tested to 1e-4 relative).
#include "common.hpp"
#include "qepilogue.hpp"
#include "range_slots.hpp"

using namespace lq;

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

// The sum over the 64 lanes, in every lane: lane l adds lane l ^ 32's value, then l ^ 16's, 8, 4, 2, 1.  (Rows of 16 lanes are
// rotated by 8, 4, 2, 1: once a value is the same in lanes that differ in bit 3, lane l + 4 has what lane l ^ 4 has, and so
// on.  As six ds_bpermute the two sums of a LayerNorm row were a chain of 1200 cycles.)
__device__ __forceinline__ float wave_sum(float v) {
    typedef unsigned pair __attribute__((ext_vector_type(2)));
    pair p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v = __uint_as_float(p.x) + __uint_as_float(p.y);
    p = __builtin_bit_cast(pair, __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false));
    v = __uint_as_float(p.x) + __uint_as_float(p.y);
#define LQ_ROW_ROR(n) __uint_as_float(unsigned(__builtin_amdgcn_update_dpp(0, int(__float_as_uint(v)), 0x120 + n, 0xf, 0xf, false)))
    v += LQ_ROW_ROR(8);
    v += LQ_ROW_ROR(4);
    v += LQ_ROW_ROR(2);
    v += LQ_ROW_ROR(1);
#undef LQ_ROW_ROR
    return v;
}

// ---------------------------------------------------------------- LayerNorm
// One wavefront per row; the row (a few KiB) is re-read from cache for the
// variance and the output pass.  mean, centred values, var = dot(c,c)/N,
// rstd = 1/sqrt(var+eps), y = (c*rstd)*gamma + beta: the reference's steps.
constexpr int LN_ROWS_PER_WAVE = 1;
constexpr int LN_KEEP = 8;  // float4 per lane held in registers: rows of up to 2048 floats

__global__ __launch_bounds__(256) void layernorm_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ gamma,
                                                        const float* __restrict__ beta,
                                                        float* __restrict__ out, long rows, int cols,
                                                        float eps, float* range) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const bool vec = (cols % 4 == 0) && aligned16(x) && aligned16(out) && aligned16(gamma) && aligned16(beta);
    const float inv_n = 1.0f / float(cols);
    RangeKeep kept;
    auto track = [&](float y) { kept.add(y); };
    for (int rr = 0; rr < LN_ROWS_PER_WAVE; ++rr) {
        const long row = (long(blockIdx.x) * 4 + wave) * LN_ROWS_PER_WAVE + rr;
        if (row >= rows) break;
        const float* xr = x + row * cols;
        float* yr = out + row * cols;
        if (vec && cols <= LN_KEEP * 256) {
            // the row stays in registers (one trip to memory instead of three); the sums run
            // over the same values in the same order as below
            float4 v[LN_KEEP];
#pragma unroll
            for (int u = 0; u < LN_KEEP; ++u) {
                const int c = lane * 4 + u * 256;
                if (c < cols) v[u] = *reinterpret_cast<const float4*>(xr + c);
            }
            float s = 0.0f;
#pragma unroll
            for (int u = 0; u < LN_KEEP; ++u)
                if (lane * 4 + u * 256 < cols) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
            const float mean = wave_sum(s) * inv_n;
            float q = 0.0f;
#pragma unroll
            for (int u = 0; u < LN_KEEP; ++u)
                if (lane * 4 + u * 256 < cols) {
                    const float a = v[u].x - mean, b = v[u].y - mean, cc = v[u].z - mean, d = v[u].w - mean;
                    q += (a * a + b * b) + (cc * cc + d * d);
                }
            const float var = wave_sum(q) * inv_n;
            const float rstd = 1.0f / sqrtf(var + eps);
#pragma unroll
            for (int u = 0; u < LN_KEEP; ++u) {
                const int c = lane * 4 + u * 256;
                if (c < cols) {
                    const float4 g = *reinterpret_cast<const float4*>(gamma + c);
                    const float4 b = *reinterpret_cast<const float4*>(beta + c);
                    float4 y;
                    y.x = ((v[u].x - mean) * rstd) * g.x + b.x;
                    y.y = ((v[u].y - mean) * rstd) * g.y + b.y;
                    y.z = ((v[u].z - mean) * rstd) * g.z + b.z;
                    y.w = ((v[u].w - mean) * rstd) * g.w + b.w;
                    *reinterpret_cast<float4*>(yr + c) = y;
                    track(y.x), track(y.y), track(y.z), track(y.w);
                }
            }
            continue;
        }
        float s = 0.0f;
        if (vec) {
            for (int c = lane * 4; c < cols; c += 256) {
                const float4 v = *reinterpret_cast<const float4*>(xr + c);
                s += (v.x + v.y) + (v.z + v.w);
            }
        } else {
            for (int c = lane; c < cols; c += 64) s += xr[c];
        }
        const float mean = wave_sum(s) * inv_n;
        float q = 0.0f;
        if (vec) {
            for (int c = lane * 4; c < cols; c += 256) {
                const float4 v = *reinterpret_cast<const float4*>(xr + c);
                const float a = v.x - mean, b = v.y - mean, cc = v.z - mean, d = v.w - mean;
                q += (a * a + b * b) + (cc * cc + d * d);
            }
        } else {
            for (int c = lane; c < cols; c += 64) {
                const float a = xr[c] - mean;
                q += a * a;
            }
        }
        const float var = wave_sum(q) * inv_n;
        const float rstd = 1.0f / sqrtf(var + eps);
        if (vec) {
            for (int c = lane * 4; c < cols; c += 256) {
                const float4 v = *reinterpret_cast<const float4*>(xr + c);
                const float4 g = *reinterpret_cast<const float4*>(gamma + c);
                const float4 b = *reinterpret_cast<const float4*>(beta + c);
                float4 y;
                y.x = ((v.x - mean) * rstd) * g.x + b.x;
                y.y = ((v.y - mean) * rstd) * g.y + b.y;
                y.z = ((v.z - mean) * rstd) * g.z + b.z;
                y.w = ((v.w - mean) * rstd) * g.w + b.w;
                *reinterpret_cast<float4*>(yr + c) = y;
                track(y.x), track(y.y), track(y.z), track(y.w);
            }
        } else {
            for (int c = lane; c < cols; c += 64) {
                const float y = ((xr[c] - mean) * rstd) * gamma[c] + beta[c];
                yr[c] = y;
                track(y);
            }
        }
    }
    if (range) kept.store(range);
}

// LayerNorm feeding a dynamic quantizer without ever storing its float32 output: the first
// kernel takes each row's mean and 1/sqrt(var + eps) and the range of the normalized values, the
// second (after the qparams have been derived from that range) normalizes again - the same
// expressions on the same inputs, so the same bits - and writes int8 codes.  x is read twice
// and 1 byte per element written, where LayerNorm + quantize read it twice, write it once as
// float32 and read that back.  Rows of up to 2048 floats, vector-aligned.
template <int KEEP>  // float4 per lane held in registers: 4 for rows of up to 1024 floats, else KEEP
__global__ __launch_bounds__(256) void layernorm_stats_kernel(const float* __restrict__ x,
                                                              const float* __restrict__ gamma,
                                                              const float* __restrict__ beta, long rows, int cols,
                                                              float eps, float* __restrict__ stats, float* range) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const float inv_n = 1.0f / float(cols);
    RangeKeep kept;
    auto track = [&](float y) { kept.add(y); };
    const long row = long(blockIdx.x) * 4 + wave;
    if (row < rows) {
        const float* xr = x + row * cols;
        float4 v[KEEP], gv[KEEP], bv[KEEP];
#pragma unroll
        for (int u = 0; u < KEEP; ++u) {
            const int c = lane * 4 + u * 256;
            if (c < cols) v[u] = *reinterpret_cast<const float4*>(xr + c);
        }
        // gamma and beta are needed after the two reductions: requested now, they arrive under them
#pragma unroll
        for (int u = 0; u < KEEP; ++u) {
            const int c = lane * 4 + u * 256;
            if (c < cols) {
                gv[u] = *reinterpret_cast<const float4*>(gamma + c);
                bv[u] = *reinterpret_cast<const float4*>(beta + c);
            }
        }
        float s = 0.0f;
#pragma unroll
        for (int u = 0; u < KEEP; ++u)
            if (lane * 4 + u * 256 < cols) s += (v[u].x + v[u].y) + (v[u].z + v[u].w);
        const float mean = wave_sum(s) * inv_n;
        float q = 0.0f;
#pragma unroll
        for (int u = 0; u < KEEP; ++u)
            if (lane * 4 + u * 256 < cols) {
                const float a = v[u].x - mean, b = v[u].y - mean, cc = v[u].z - mean, d = v[u].w - mean;
                q += (a * a + b * b) + (cc * cc + d * d);
            }
        const float var = wave_sum(q) * inv_n;
        const float rstd = 1.0f / sqrtf(var + eps);
        if (lane == 0) stats[2 * row] = mean, stats[2 * row + 1] = rstd;
#pragma unroll
        for (int u = 0; u < KEEP; ++u) {
            const int c = lane * 4 + u * 256;
            if (c < cols) {
                const float4 g = gv[u], b = bv[u];
                track(((v[u].x - mean) * rstd) * g.x + b.x);
                track(((v[u].y - mean) * rstd) * g.y + b.y);
                track(((v[u].z - mean) * rstd) * g.z + b.z);
                track(((v[u].w - mean) * rstd) * g.w + b.w);
            }
        }
    }
    kept.store(range);
}

// four codes of normalized values
__device__ __forceinline__ uint32_t layernorm_codes(float4 v, float4 g, float4 b, float mean, float rstd, const QGrid& G, int off) {
    const float y[4] = {((v.x - mean) * rstd) * g.x + b.x, ((v.y - mean) * rstd) * g.y + b.y,
                        ((v.z - mean) * rstd) * g.z + b.z, ((v.w - mean) * rstd) * g.w + b.w};
    float c[4];
    quant_fast<false>(y, G, c);
    const int c0 = int(c[0]) + off, c1 = int(c[1]) + off, c2 = int(c[2]) + off, c3 = int(c[3]) + off;
    return uint32_t(c0 & 0xff) | (uint32_t(c1 & 0xff) << 8) | (uint32_t(c2 & 0xff) << 16) | (uint32_t(c3) << 24);
}

constexpr long kRangeRows = 2048;  // rows whose blocks reduce the kept range themselves
// One wavefront per row.  RANGE: the grid is that of the kept range, which every block reduces while its rows are on
// their way; the first block hands it out.
struct LnGrid {
    const float* range;
    int symmetric, qmin, qmax, is_signed;
    float eps, half_range;
};
template <int KEEP, bool RANGE>
__global__ __launch_bounds__(256) void layernorm_quantize_kernel(const float* __restrict__ x,
                                                                 const float* __restrict__ gamma,
                                                                 const float* __restrict__ beta,
                                                                 const float* __restrict__ stats, long rows, int cols,
                                                                 float* scale, float* zp, LnGrid grid, int off,
                                                                 int8_t* __restrict__ q) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const long row = long(blockIdx.x) * 4 + wave;
    const long at = row < rows ? row : 0;
    const float* xr = x + at * cols;
    float4 v[KEEP], g[KEEP], b[KEEP];
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
        const int c = lane * 4 + u * 256;
        if (c < cols) {
            v[u] = *reinterpret_cast<const float4*>(xr + c);
            g[u] = *reinterpret_cast<const float4*>(gamma + c);
            b[u] = *reinterpret_cast<const float4*>(beta + c);
        }
    }
    const float mean = stats[2 * at], rstd = stats[2 * at + 1];
    float s, z;
    if constexpr (RANGE) {
        float mn, mx;
        range_block_load<2>(grid.range, mn, mx);
        qparams_of(mn, mx, grid.symmetric, grid.qmin, grid.qmax, grid.is_signed, grid.eps, grid.half_range, &s, &z);
        if (blockIdx.x == 0 && threadIdx.x == 0) *scale = s, *zp = z;
    } else {
        s = *scale, z = *zp;
    }
    if (row >= rows) return;
    const QGrid G = make_qgrid(s, z, float(grid.qmin), float(grid.qmax), true);
    int8_t* qr = q + row * cols;
#pragma unroll
    for (int u = 0; u < KEEP; ++u) {
        const int c = lane * 4 + u * 256;
        if (c < cols) *reinterpret_cast<uint32_t*>(qr + c) = layernorm_codes(v[u], g[u], b[u], mean, rstd, G, off);
    }
}

// ---------------------------------------------------------------- elementwise
// Four float4 per thread (block-strided, so each access of a wavefront is
// contiguous); the optional range costs one partial slot per block.
constexpr int GELU_PER_THREAD = 4;

__global__ __launch_bounds__(256) void gelu_kernel(const float* __restrict__ x, float* __restrict__ out,
                                                   size_t n, int vec, float* range) {
    RangeKeep kept;
    auto track = [&](float y) { kept.add(y); };
    const size_t base = size_t(blockIdx.x) * (256 * GELU_PER_THREAD) + threadIdx.x;
    if (vec) {
        float4 v[GELU_PER_THREAD];
#pragma unroll
        for (int u = 0; u < GELU_PER_THREAD; ++u) {
            const size_t i = base + size_t(u) * 256;
            if (i * 4 < n) v[u] = reinterpret_cast<const float4*>(x)[i];
        }
#pragma unroll
        for (int u = 0; u < GELU_PER_THREAD; ++u) {
            const size_t i = base + size_t(u) * 256;
            if (i * 4 < n) {
                float4 y = {gelu_erf(v[u].x), gelu_erf(v[u].y), gelu_erf(v[u].z), gelu_erf(v[u].w)};
                reinterpret_cast<float4*>(out)[i] = y;
                track(y.x), track(y.y), track(y.z), track(y.w);
            }
        }
    } else {
#pragma unroll
        for (int u = 0; u < GELU_PER_THREAD; ++u) {
            const size_t i = base + size_t(u) * 256;
            if (i < n) {
                const float y = gelu_erf(x[i]);
                out[i] = y;
                track(y);
            }
        }
    }
    if (range) kept.store(range);
}

// dst[r, :] = src[r * src_row_stride : r * src_row_stride + cols]
__global__ __launch_bounds__(256) void gather_rows_kernel(const float* __restrict__ src, size_t src_row_stride,
                                                          float* __restrict__ dst, size_t rows, size_t cols) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= rows * cols) return;
    const size_t r = i / cols, c = i - r * cols;
    dst[i] = src[r * src_row_stride + c];
}

__global__ __launch_bounds__(256) void add_kernel(const float* __restrict__ a, const float* __restrict__ b,
                                                  float* __restrict__ out, size_t n, int vec) {
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (vec) {
        if (i * 4 >= n) return;
        const float4 u = reinterpret_cast<const float4*>(a)[i];
        const float4 v = reinterpret_cast<const float4*>(b)[i];
        float4 y = {u.x + v.x, u.y + v.y, u.z + v.z, u.w + v.w};
        reinterpret_cast<float4*>(out)[i] = y;
    } else if (i < n) {
        out[i] = a[i] + b[i];
    }
}

// image [B,C,H,W] -> patch rows [B*(H/p)*(W/p), C*p*p], column order (c, ph, pw):
// the im2col of a convolution whose stride equals its kernel
__global__ __launch_bounds__(256) void patchify_kernel(const float* __restrict__ img, float* __restrict__ out,
                                                       int B, int C, int H, int W, int p) {
    const int gh = H / p, gw = W / p, K = C * p * p;
    const size_t total = size_t(B) * gh * gw * K;
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= total) return;
    const int k = int(i % K);
    const size_t row = i / K;
    const int pw = k % p, ph = (k / p) % p, c = k / (p * p);
    const int gx = int(row % gw), gy = int((row / gw) % gh), b = int(row / (size_t(gw) * gh));
    out[i] = img[((size_t(b) * C + c) * H + (gy * p + ph)) * W + (gx * p + pw)];
}

// tokens[b,0,:] = cls + pos[0]; tokens[b,1+i,:] = patches[b,i,:] + pos[1+i]
__global__ __launch_bounds__(256) void assemble_tokens_kernel(const float* __restrict__ patches,
                                                              const float* __restrict__ cls,
                                                              const float* __restrict__ pos,
                                                              float* __restrict__ out, int B, int T, int D) {
    const size_t total = size_t(B) * T * D;
    const size_t i = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (i >= total) return;
    const int d = int(i % D);
    const int t = int((i / D) % T);
    const size_t b = i / (size_t(D) * T);
    const float v = t == 0 ? cls[d] : patches[(b * (T - 1) + (t - 1)) * D + d];
    out[i] = v + pos[size_t(t) * D + d];
}

// (e0, e1) = h + m + l part by part, each part a pair of bfloat16 (e0's in the low half): the
// packed conversion rounds to nearest, the remainders are exact (8 + 8 + 8 significant bits with
// signed remainders).  A NaN stays a NaN in every part; an infinity turns into a NaN in the
// lower parts, so a non-finite input gives a non-finite output.
typedef __bf16 at_bf2 __attribute__((ext_vector_type(2)));
typedef float at_f2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t at_pk(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(at_f2{a, b}, at_bf2));
}
__device__ __forceinline__ void at_split3x2(float e0, float e1, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = at_pk(e0, e1);
    e0 -= __uint_as_float(h << 16), e1 -= __uint_as_float(h & 0xffff0000u);
    m = at_pk(e0, e1);
    e0 -= __uint_as_float(m << 16), e1 -= __uint_as_float(m & 0xffff0000u);
    l = at_pk(e0, e1);
}

typedef __bf16 sg_v8bf __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------- float32 GEMM, out = a . w^T + bias
// float32 operands on the bfloat16 matrix instruction: both operands are split into three
// bfloat16 parts when a tile is written to LDS (at_split3x2), and six part products per k step
// (hi.hi, hi.mid, mid.hi, hi.lo, lo.hi, mid.mid, smallest first, accumulated in float32) give
// every product 2^-24 relative accuracy - a float32 GEMM at six instructions of
// v_mfma_f32_32x32x16_bf16 per 16 k, against eight of v_mfma_f32_32x32x2_f32 at four times the
// cycles each.
//
// 128 x 128 x 32 block tile, 4 wavefronts of 64 x 64; BLOCKS of them per CU; the next tile's operands wait in registers
// while the current one is multiplied.  LDS: per part 256 rows (A's 128, then W's) of 32
// bfloat16 = 64 bytes; the 16-byte chunk k of row r sits at chunk k ^ ((r / 4) % 4), which puts
// the 16 rows of a fragment pass on 16 different bank groups.
constexpr int SG_BM = 128, SG_BN = 128, SG_BK = 32, SG_ROWS = SG_BM + SG_BN;

__device__ __forceinline__ int sg_index(int row, int k) {  // k a multiple of 4
    return row * SG_BK + ((((k >> 3) ^ ((row >> 2) & 3)) << 3) | (k & 7));
}

// PATCH: the A operand is an image [B,C,H,W] read as the rows of its p x p patches (row = (b, gy,
// gx), column = (c, ph, pw): four consecutive columns are four consecutive pixels of one image
// row when p is a multiple of 4), and the result row (b, i) lands on token row 1 + i of image b
// with the position table added; the blocks of the first row tile also write the class-token rows.
struct PatchForm {
    int C, H, W, p, gw, per_image;  // per_image = (H/p) * (W/p) patches
    int B, log2p;                   // log2p = -1 when p is not a power of two
    const float* cls;  // [N]
    const float* pos;  // [(1 + per_image), N]
};

// NU rows of A and as many of W for a thread, RS apart from row `a_row` / `w_row` on: groups of four consecutive k.
// PATCH 0: a is a plain [M,K] matrix.  1: patch rows with p a power of two and every group of
// four columns one aligned 16-byte load (no branch and no division in the loop).  2: patch rows
// of any geometry, element by element.
// VEC: groups of four k of both operands are whole, aligned 16 bytes (known to the compiler: where the two ways to load meet,
// the registers of one are copied, and a copy waits for the load).
template <int PATCH, bool VEC, int RS, int NU>
struct SgLoader {
    const float* __restrict__ a;
    const float* __restrict__ w;
    int M, N, K, a_row, w_row;
    const PatchForm& pf;
    size_t patch_at[NU];  // PATCH: where the patch of row u starts in the image
    __device__ __forceinline__ SgLoader(const float* a_, const float* w_, int M_, int N_, int K_, int a_row_, int w_row_,
                                        const PatchForm& pf_)
        : a(a_), w(w_), M(M_), N(N_), K(K_), a_row(a_row_), w_row(w_row_), pf(pf_) {
        if constexpr (PATCH != 0) {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const int row = min(a_row + RS * u, M - 1);
                const int b = row / pf.per_image, i = row - b * pf.per_image;
                const int gy = i / pf.gw, gx = i - gy * pf.gw;
                patch_at[u] = (size_t(b) * pf.C * pf.H + size_t(gy) * pf.p) * pf.W + size_t(gx) * pf.p;
            }
        }
    }
    __device__ __forceinline__ float4 any_row(const float* base, int row, int rows, int k) const {
        float4 v = {0.f, 0.f, 0.f, 0.f};
        if (row < rows) {
            const float* p = base + size_t(row) * K + k;
            if (k < K) v.x = p[0];
            if (k + 1 < K) v.y = p[1];
            if (k + 2 < K) v.z = p[2];
            if (k + 3 < K) v.w = p[3];
        }
        return v;
    }
    // PATCH: column k of a patch row is pixel (c, ph, pw) of the patch.  Loads go to clamped (always valid) addresses: what
    // a row past M gives is never stored, what lies past K is zeroed when it is stashed (zeroed here, every load would be
    // waited for where it is issued).
    __device__ __forceinline__ void patches(int k, float4 (&ra)[NU]) const {
        if constexpr (PATCH == 1) {
            const int kk = min(k, K - 4);
            const int pw = kk & (pf.p - 1), ph = (kk >> pf.log2p) & (pf.p - 1), c = kk >> (2 * pf.log2p);
            const size_t pixel = (size_t(c) * pf.H + ph) * pf.W + pw;
#pragma unroll
            for (int u = 0; u < NU; ++u) ra[u] = *reinterpret_cast<const float4*>(a + patch_at[u] + pixel);
        } else {
            const int pp = pf.p * pf.p;
            size_t pixel[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int kk = min(k + e, K - 1);
                const int c = kk / pp, r = kk - c * pp;
                const int ph = r / pf.p, pw = r - ph * pf.p;
                pixel[e] = (size_t(c) * pf.H + ph) * pf.W + pw;
            }
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                const float* p = a + patch_at[u];
                ra[u] = float4{p[pixel[0]], p[pixel[1]], p[pixel[2]], p[pixel[3]]};
            }
        }
    }
    // plain rows in the aligned case
    __device__ __forceinline__ void rows_vec(const float* base, int row0, int rows, int k, float4 (&r)[NU]) const {
        const int kk = min(k, K - 4);
#pragma unroll
        for (int u = 0; u < NU; ++u)
            r[u] = *reinterpret_cast<const float4*>(base + size_t(min(row0 + RS * u, rows - 1)) * K + kk);
    }
    __device__ __forceinline__ void operator()(int k, float4 (&ra)[NU], float4 (&rb)[NU]) const {
        if constexpr (PATCH != 0) patches(k, ra);
        if constexpr (VEC) {
            if constexpr (PATCH == 0) rows_vec(a, a_row, M, k, ra);
            rows_vec(w, w_row, N, k, rb);
        } else {
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                if constexpr (PATCH == 0) ra[u] = any_row(a, a_row + RS * u, M, k);
                rb[u] = any_row(w, w_row + RS * u, N, k);
            }
        }
    }
};

// a tile that reaches past K: zeros there
template <int NU>
__device__ __forceinline__ void sg_inside(float4 (&r)[NU], int k, int K) {
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        r[u].x = k < K ? r[u].x : 0.f, r[u].y = k + 1 < K ? r[u].y : 0.f;
        r[u].z = k + 2 < K ? r[u].z : 0.f, r[u].w = k + 3 < K ? r[u].w : 0.f;
    }
}

// four consecutive k of a row, as three parts, into an image of rows of SG_BK bfloat16 per part
template <int LEN>
__device__ __forceinline__ void sg_stash(uint16_t (&sp)[3][LEN], int row, int k, float4 v) {
    uint32_t lo[3], hi[3];
    at_split3x2(v.x, v.y, lo[0], lo[1], lo[2]);
    at_split3x2(v.z, v.w, hi[0], hi[1], hi[2]);
    const int at = sg_index(row, k);
#pragma unroll
    for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(&sp[p][at]) = uint2{lo[p], hi[p]};
}

template <int PATCH, bool VEC, int BLOCKS>
__global__ __launch_bounds__(256, BLOCKS) void sgemm_nt_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                               const float* __restrict__ bias, float* __restrict__ out,
                                                               int M, int N, int K, PatchForm pf) {
    __shared__ __attribute__((aligned(16))) uint16_t sp[3][SG_ROWS * SG_BK];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * SG_BM, n0 = blockIdx.x * SG_BN;
    // loader: row tid / 8 (+ 32 u) of either operand, four consecutive k at 4 * (tid % 8)
    const int lrow = tid >> 3, lk = (tid & 7) * 4;
    const SgLoader<PATCH, VEC, 32, 4> fetch(a, w, M, N, K, m0 + lrow, n0 + lrow, pf);
    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;

    float4 ra[4], rb[4];
    const int nk = (K + SG_BK - 1) / SG_BK;
    const int fr = lane & 31, kg = lane >> 5;
    fetch(lk, ra, rb);
    for (int t = 0; t < nk; ++t) {
        if ((t + 1) * SG_BK > K) sg_inside(ra, t * SG_BK + lk, K), sg_inside(rb, t * SG_BK + lk, K);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            sg_stash(sp, lrow + 32 * u, lk, ra[u]);
            sg_stash(sp, SG_BM + lrow + 32 * u, lk, rb[u]);
        }
        lds_barrier();
        if (t + 1 < nk) fetch((t + 1) * SG_BK + lk, ra, rb);
#pragma unroll
        for (int ks = 0; ks < SG_BK / 16; ++ks) {
            uint4 fa[2][3], fb[2][3];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int at = sg_index(wm * 64 + i * 32 + fr, 16 * ks + 8 * kg);
#pragma unroll
                for (int p = 0; p < 3; ++p) fa[i][p] = *reinterpret_cast<const uint4*>(&sp[p][at]);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int at = sg_index(SG_BM + wn * 64 + j * 32 + fr, 16 * ks + 8 * kg);
#pragma unroll
                for (int p = 0; p < 3; ++p) fb[j][p] = *reinterpret_cast<const uint4*>(&sp[p][at]);
            }
            auto mm = [&](int pa, int pb) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sg_v8bf, fa[i][pa]),
                                                                            __builtin_bit_cast(sg_v8bf, fb[j][pb]),
                                                                            acc[i][j], 0, 0, 0);
            };
            mm(1, 1), mm(0, 2), mm(2, 0), mm(0, 1), mm(1, 0), mm(0, 0);
        }
        lds_barrier();  // the tile has been read: the next one may be written (what was requested is still on its way)
    }
    // result layout of the 32x32 MFMA: column = lane % 32, row = 8*(r/4) + 4*(lane/32) + r%4
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int n = n0 + wn * 64 + j * 32 + (lane & 31);
            if (n >= N) continue;
            const float bv = bias ? bias[n] : 0.0f;
            if constexpr (PATCH != 0) {
                // the sixteen position values are requested before the first store: a store
                // between two loads would make each load wait for the one before it
                float pv[16];
                size_t at[16];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int mq = m0 + wm * 64 + i * 32 + 8 * q + 4 * (lane >> 5);
                    int b = mq / pf.per_image, t = mq - b * pf.per_image;
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        at[4 * q + r] = (size_t(b) * (pf.per_image + 1) + 1 + t) * N + n;
                        pv[4 * q + r] = mq + r < M ? pf.pos[size_t(1 + t) * N + n] : 0.0f;
                        if (++t == pf.per_image) t = 0, ++b;
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m < M) out[at[r]] = (acc[i][j][r] + bv) + pv[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                    if (m < M) out[size_t(m) * N + n] = acc[i][j][r] + bv;
                }
            }
        }
    if constexpr (PATCH != 0) {
        // class-token rows: token 0 of every image, this block's 128 columns
        if (blockIdx.y == 0) {
            const int n = n0 + (tid & 127);
            if (n < N) {
                const float v = pf.cls[n] + pf.pos[n];
                for (int b = tid >> 7; b < pf.B; b += 2) out[size_t(b) * (pf.per_image + 1) * N + n] = v;
            }
        }
    }
}


// The same product for few tiles: 32 x 32 outputs per block, K dealt to its four wavefronts in turns of SG_BK, each of which
// stages its own rows in LDS of its own (no barrier in the loop) and keeps two sums per element (even and odd halves of a
// turn, so that consecutive MFMAs do not wait for each other); the eight sums are added once, in a fixed order.  A 128 x 128
// tile is a chain of K / 32 turns of 2.2 us (split, barrier, LDS reads, MFMAs, barrier) however few of them there are:
// patches of ViT-B/16, K = N = 768, us: 196 rows 55 -> 9, 784 55 -> 17, 1568 61 -> 27, 3136 62 -> 52.  Beyond
// SG_SMALL_BLOCKS blocks the larger tiles win, whose operands are split less often (4704 rows 69 against 58, 2048 x 2048 x 512
// 52 against 42).  Operands that are no whole, aligned 16 bytes are read float by float, more often here: us of small / large tiles,
// 2592 tiles 2301 x 1147 x 1155 139 / 108, 2304 x 770 82.5 / 77.5, 2025 x 3001 272 / 264, 2000 x 770 75 / 77, 1600 x 1155 94 / 107; at
// addresses between 16 bytes rows of K = 768 and 3072 are slower still: 1920 x 768 90 / 74, 1600 x 3072 300 / 256, 1536 x 768 70 / 72
// (K = 1156 as 1155).  Root mean square of the error against float64 6.4e-8 of the result's (1.6e-7 for the large tiles, whose
// sums are longer).
constexpr int SG_SMALL = 32;
constexpr long SG_SMALL_BLOCKS = 2600, SG_SMALL_RAGGED = 2000, SG_SMALL_UNALIGNED = 1500;

template <int PATCH, bool VEC>
__global__ __launch_bounds__(256, 3) void sgemm_nt_small_kernel(const float* __restrict__ a, const float* __restrict__ w,
                                                                const float* __restrict__ bias, float* __restrict__ out,
                                                                int M, int N, int K, PatchForm pf) {
    __shared__ __attribute__((aligned(16))) union {
        uint16_t parts[4][3][2 * SG_SMALL * SG_BK];
        float sums[4][SG_SMALL][SG_SMALL + 4];
    } lds;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = blockIdx.y * SG_SMALL, n0 = blockIdx.x * SG_SMALL;
    const int lrow = lane >> 3, lk = (lane & 7) * 4;
    const SgLoader<PATCH, VEC, 8, 4> fetch(a, w, M, N, K, m0 + lrow, n0 + lrow, pf);
    uint16_t(&sp)[3][2 * SG_SMALL * SG_BK] = lds.parts[wave];
    v16f acc[2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;
    const int nk = (K + SG_BK - 1) / SG_BK;
    const int fr = lane & 31, kg = lane >> 5;
    float4 ra[4], rb[4];
    if (wave < nk) fetch(wave * SG_BK + lk, ra, rb);
    for (int t = wave; t < nk; t += 4) {
        if ((t + 1) * SG_BK > K) sg_inside(ra, t * SG_BK + lk, K), sg_inside(rb, t * SG_BK + lk, K);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            sg_stash(sp, lrow + 8 * u, lk, ra[u]);
            sg_stash(sp, SG_SMALL + lrow + 8 * u, lk, rb[u]);
        }
        // (the wavefront's own LDS: its instructions execute in order, the fence is for the compiler)
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (t + 4 < nk) fetch((t + 4) * SG_BK + lk, ra, rb);
        uint4 fa[2][3], fb[2][3];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int at = sg_index(fr, 16 * ks + 8 * kg), bt = sg_index(SG_SMALL + fr, 16 * ks + 8 * kg);
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                fa[ks][p] = *reinterpret_cast<const uint4*>(&sp[p][at]);
                fb[ks][p] = *reinterpret_cast<const uint4*>(&sp[p][bt]);
            }
        }
        auto mm = [&](int pa, int pb) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
                acc[ks] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sg_v8bf, fa[ks][pa]),
                                                                  __builtin_bit_cast(sg_v8bf, fb[ks][pb]), acc[ks], 0, 0, 0);
        };
        mm(1, 1), mm(0, 2), mm(2, 0), mm(0, 1), mm(1, 0), mm(0, 0);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 16; ++r) lds.sums[wave][8 * (r >> 2) + 4 * kg + (r & 3)][fr] = acc[0][r] + acc[1][r];
    __syncthreads();
    // row tid / 8, four columns from 4 * (tid % 8)
    const int row = tid >> 3, col = (tid & 7) * 4, m = m0 + row;
    if (m < M) {
        float4 v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const float4*>(&lds.sums[i][row][col]);
        const float y[4] = {(v[0].x + v[1].x) + (v[2].x + v[3].x), (v[0].y + v[1].y) + (v[2].y + v[3].y),
                            (v[0].z + v[1].z) + (v[2].z + v[3].z), (v[0].w + v[1].w) + (v[2].w + v[3].w)};
        size_t at = size_t(m) * N;
        const float* pos = nullptr;
        if constexpr (PATCH != 0) {
            const int b = m / pf.per_image, t = m - b * pf.per_image;
            at = (size_t(b) * (pf.per_image + 1) + 1 + t) * N;
            pos = pf.pos + size_t(1 + t) * N;
        }
        float bv[4], pv[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = min(n0 + col + e, N - 1);
            bv[e] = bias ? bias[n] : 0.0f;
            pv[e] = PATCH != 0 ? pos[n] : 0.0f;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int n = n0 + col + e;
            if (n < N) out[at + n] = PATCH != 0 ? (y[e] + bv[e]) + pv[e] : y[e] + bv[e];
        }
    }
    if constexpr (PATCH != 0) {
        if (blockIdx.y == 0) {
            // class-token rows: token 0 of every image, this block's columns
            const int n = n0 + (tid & 31);
            if (n < N) {
                const float v = pf.cls[n] + pf.pos[n];
                for (int b = tid >> 5; b < pf.B; b += 8) out[size_t(b) * (pf.per_image + 1) * N + n] = v;
            }
        }
    }
}

// (by M, N, K and whether operands are aligned: a matrix and the image whose patches are its rows get the same sums)
template <int PATCH, bool VEC>
int launch_sgemm(const float* a, const float* w, const float* bias, float* out, int M, int N, int K, const PatchForm& pf,
                 hipStream_t st, bool large) {
    const long tiles_m = (long(M) + SG_SMALL - 1) / SG_SMALL, tiles_n = (long(N) + SG_SMALL - 1) / SG_SMALL;
    const long most = VEC ? SG_SMALL_BLOCKS : K % 4 != 0 ? SG_SMALL_RAGGED : SG_SMALL_UNALIGNED;
    if (!large && tiles_m * tiles_n <= most) {
        const dim3 grid{unsigned(tiles_n), unsigned(tiles_m)};
        sgemm_nt_small_kernel<PATCH, VEC><<<grid, 256, 0, st>>>(a, w, bias, out, M, N, K, pf);
    } else {
        const dim3 grid{(unsigned(N) + SG_BN - 1) / SG_BN, (unsigned(M) + SG_BM - 1) / SG_BM};
        const long tiles = long(grid.x) * grid.y;
        // three blocks per CU (168 registers, up to 4 % slower) where they are one round and two per CU are a second, nearly
        // empty one: 12 544 rows of ViT-B/16's patches, 588 tiles, 134 -> 106 us; 441 tiles 78 with two, 82 with three.  (Float by float
        // too, where two to six registers go to scratch: 588 tiles with K = 770 165 us, with two 175; 520 x 333 73 and 79.)
        if (tiles > 512 && tiles <= 768)
            sgemm_nt_kernel<PATCH, VEC, 3><<<grid, 256, 0, st>>>(a, w, bias, out, M, N, K, pf);
        else
            sgemm_nt_kernel<PATCH, VEC, 2><<<grid, 256, 0, st>>>(a, w, bias, out, M, N, K, pf);
    }
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

// ---------------------------------------------------------------- attention
// Head dim 64, at most 208 tokens.  qkv is the packed activation [B, T, 3, H, 64] of the qkv
// Linear; out is [B, T, H*64].
//
// float32 operands on the bfloat16 matrix instruction.  A float32 is the exact sum of three
// bfloat16 values (8 + 8 + 8 significant bits: at_split3x2), and a product a * b keeps 2^-24
// relative accuracy with six of the nine part products (hi.hi, hi.mid, mid.hi, hi.lo, lo.hi,
// mid.mid; the three left out are below 2^-24 of |a b|).  Part products are exact in float32
// and accumulate in float32, so each dot product is as accurate as a float32 one, and
// v_mfma_f32_16x16x32_bf16 runs sixteen times the rate of v_mfma_f32_16x16x4_f32: six
// instructions of the one replace eight of the other at a sixth of the time each.
//
// A head's queries are dealt to `parts` blocks of four wavefronts; a wavefront takes up to QT
// tiles of 16 queries and reads each fragment of K and V once for all of them.  The three parts
// of K, and after the scores those of V^T in their place, are the block's 80 KB of LDS, so that
// two blocks share a CU.  What is read from memory is requested a phase ahead (V under the scores,
// the next head's K and queries under the products with V), fragments a step ahead, and the
// exponentials and splits of the probabilities are issued between the products with V.
//
// Bound by the matrix pipe and the vector unit together: of the about 36 000 cycles that two blocks of
// a CU take for a head of 197 tokens, the products are 16 800 of every SIMD, splits, exponentials and
// LDS writes about as much, and at 64 x 12 heads the power limit holds the clock near 1.7 GHz.
// 12 heads of 197 tokens 18.3 -> 10.5 us, 96 heads 20.1 -> 14.9, 384 46.4 -> 34.5, 768 77.4 -> 67.6
// against attention_head_kernel below, a block of 16 wavefronts per head with K and V side by side (all K and V fragments
// read once per 16 queries, the softmax a phase of its own), which is kept for the counts of heads that give every CU one.
//
// Per wavefront: S^T = K . Q^T as 13 tiles of 16 keys x 16 queries (accumulators stay in
// registers), softmax over the keys of each query (a lane holds 52 of a query's keys, the other
// three lane groups the rest), then O = P . V where the S^T accumulators ARE the A operand:
// register r of tile t holds P[query = lane%16][key = 16t + 4*(lane/16) + r], so two tiles give
// a lane the eight k slots of an instruction, which is a valid k-slice assignment as long as V
// is read with the same one ([column][key] keeps a lane's four keys of a tile in 8 contiguous
// bytes); the thirteenth tile goes through the 16-key form of the instruction alone.
constexpr int AT_D = 64, AT_TMAX = 208, AT_NT = AT_TMAX / 16, AT_WAVES = 4;
// K: rows of 64 bfloat16 = 128 bytes = half of the 64 banks; the 16-byte chunk k of row r sits at chunk
// k ^ (r / 2 % 8), so the 16 rows of a fragment (same logical chunk) cover every bank once.
// V^T: 106 dwords per row = 10 mod 32: the 16 rows a fragment reads (8 bytes each) fall on 16
// different bank pairs
constexpr int AT_VLD = AT_TMAX + 4;
constexpr int AT_PART_K = AT_TMAX * AT_D, AT_PART_V = AT_D * AT_VLD;  // elements of one part
constexpr size_t AT_SMEM = size_t(3) * (AT_PART_V > AT_PART_K ? AT_PART_V : AT_PART_K) * 2;
static_assert(2 * (AT_SMEM + 208) <= 160 * 1024, "two blocks per CU, with a flag and the range reduction's few words");

typedef __bf16 at_v8bf __attribute__((ext_vector_type(8)));
typedef short at_v4s __attribute__((ext_vector_type(4)));

__device__ __forceinline__ int at_k_index(int row, int col) {  // col a multiple of 4
    return row * AT_D + ((((col >> 3) ^ (row >> 1 & 7)) << 3) | (col & 7));
}
// V^T's row of a column: tile j of the output is columns 4 i + j, i = 0..15, so that a lane has four consecutive floats of a
// query at the end
__device__ __forceinline__ int at_v_index(int j, int i, int key) { return (16 * j + i) * AT_VLD + key; }
// P is up to 1 for every key until the division by its sum, so that 208 keys of one score add up to 208 max |V| on the way to a
// result of max |V| at most.  For a head with values of V beyond AT_VMAX, whose sums could be infinite, P is 2^-8 of that: the
// subtraction S - (max + 8) then rounds what S - max has exactly near the maximum, and scores close to each other give results
// 2.9e-7 from float64 instead of 2.2e-7, which is why other heads do without.  (V times 2^-8 instead: the matrix instruction
// takes the subnormal parts of |V| < 1e-31 for zero, and 768 heads take 68.0 us where they take 67.3 with V's maximum, 66.2 without.)
constexpr float AT_VMAX = 0x1p119f;
static_assert(AT_TMAX < 256, "AT_TMAX * AT_VMAX and 2^-8 * AT_TMAX * FLT_MAX are finite");
// f over the four lanes of one number in the four rows of 16 lanes; every lane gets it
template <class F>
__device__ __forceinline__ float at_rows4(float v, F f) {
    auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    v = f(__uint_as_float(x[0]), __uint_as_float(x[1]));
    x = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return f(__uint_as_float(x[0]), __uint_as_float(x[1]));
}

// acc[q] += a[q] . b from the parts, smallest terms first.  16 bytes a lane: 32 k slots; 8 bytes: 16.
constexpr int kAtPa[6] = {1, 0, 2, 0, 1, 0}, kAtPb[6] = {1, 2, 0, 1, 0, 0};
__device__ __forceinline__ v4f at_mm(const uint4& x, const uint4& y, v4f acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(at_v8bf, x), __builtin_bit_cast(at_v8bf, y), acc, 0,
                                                   0, 0);
}
__device__ __forceinline__ v4f at_mm(const uint2& x, const uint2& y, v4f acc) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(at_v4s, x), __builtin_bit_cast(at_v4s, y), acc, 0,
                                                     0, 0);
}

// WIDE: offsets within 32 token rows take more than 32 bits
template <int QT, bool WIDE>
__global__ __launch_bounds__(64 * AT_WAVES, 2) void attention_kernel(const float* __restrict__ qkv,
                                                                     float* __restrict__ out, int T, int H, int heads,
                                                                     int parts, int out_vec, float scale,
                                                                     float* range) {
    extern __shared__ __attribute__((aligned(16))) uint16_t at_smem[];  // K's parts, then V^T's
    __shared__ int s_large;  // V has values beyond AT_VMAX
    constexpr int THREADS = 64 * AT_WAVES, ROW4 = AT_D / 4;
    constexpr int KP = AT_TMAX * ROW4 / THREADS;  // 16-byte pieces of K per thread: one of every 16 rows
    constexpr int VP = (AT_TMAX + 31) / 32;       // pairs of such pieces of V: one of every 32 rows
    static_assert(AT_TMAX * ROW4 % THREADS == 0 && THREADS / ROW4 == 16 && AT_D == 64, "");
    const size_t tok_stride = size_t(3) * H * AT_D;
    using Offset = std::conditional_t<WIDE, size_t, unsigned>;
    const Offset row_bytes = Offset(tok_stride) * 4u;
    const int tiles = (T + 15) / 16;
    // Blocks are dealt to the 8 XCDs in turn: the parts of a head follow each other on one of them, where
    // the second finds the first one's K and V in the L2.
    const int items = (heads + 7) / 8 * 8 * parts;
    float4 kheld[KP], qheld[QT][2 * (AT_D / 32)];
    // Four floats of token row row0 + r (row0 the same in the whole wavefront; past the last token: a row of the
    // tokens there are - such a key's probability is 0, such a query is not stored), as a scalar base and
    // an offset per lane.
    auto fetch = [&](const float* head_base, int which, int row0, int r, int col) {
        const int rb = row0 < T ? row0 : 0;
        const float* p = head_base + size_t(rb) * tok_stride + size_t(which) * H * AT_D;
        const Offset off = (rb + r < T ? Offset(r) * row_bytes : Offset(0)) + Offset(col) * 4u;
        return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(p) + off);
    };
    struct Item {
        const float* base;
        int head, t0, nq;  // this wavefront's queries are tiles t0 .. t0 + nq - 1
    };
    auto item_of = [&](int item, int wave_id) {
        Item it;
        const int part = item / 8 % parts;
        it.head = item / (8 * parts) * 8 + item % 8;
        const int b = it.head / H;
        it.base = qkv + size_t(b) * T * tok_stride + size_t(it.head - b * H) * AT_D;
        // Tiles [first, end) are the part's.  Which wavefronts get fewer than QT changes from block to block: those of
        // one number mostly share a SIMD.
        const int first = tiles * part / parts, n = tiles * (part + 1) / parts - first;
        const int wave = (wave_id + item / 8) % AT_WAVES;
        it.t0 = first + n * wave / AT_WAVES;
        it.nq = first + n * (wave + 1) / AT_WAVES - it.t0;
        return it;
    };
    // piece x of what a wavefront has of an item before its scores: K, then the lane's slice of its query rows
    // (Q[16 tile + c][32 u + 8 g + 0..7])
    constexpr int PIECES = KP + QT * 2 * (AT_D / 32);
    auto request = [&](const Item& it, int x, int tid) {
        if (x < KP) {
            kheld[x] = fetch(it.base, 1, x * (THREADS / ROW4), tid / ROW4, tid % ROW4 * 4);
        } else {
            const int q = (x - KP) / 4, e = (x - KP) % 4, lane = tid & 63;
            qheld[q][e] = fetch(it.base, 0, (it.t0 + q) * 16, lane & 15, 32 * (e / 2) + 8 * (lane >> 4) + 4 * (e % 2));
        }
    };
    const int wave_id = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
    RangeKeep kept;
    int next = blockIdx.x;
    while (next < items && item_of(next, 0).head >= heads) next += gridDim.x;
    if (next < items) {
        const Item it = item_of(next, wave_id);
#pragma unroll
        for (int x = 0; x < PIECES; ++x) request(it, x, threadIdx.x);
    }
    while (next < items) {
        const Item it = item_of(next, wave_id);
        do next += gridDim.x;
        while (next < items && item_of(next, 0).head >= heads);
        // behind the last item it is requested again, rather than leaving the registers' old values alive through the loop
        const Item after = next < items ? item_of(next, wave_id) : it;
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));  // what follows from the lane is computed per item: kept across items, it would be spilled
        const int lane = tid & 63, g = lane >> 4, c = lane & 15;
        if (tid == 0) s_large = 0;  // between the barrier at the end of the item before, past which nobody reads it, and the next
        // K rows into LDS as three bfloat16 parts
#pragma unroll
        for (int u = 0; u < KP; ++u) {
            const int i = tid + u * THREADS, row = i / ROW4, c4 = (i % ROW4) * 4;
            uint32_t d0[3], d1[3];
            at_split3x2(kheld[u].x, kheld[u].y, d0[0], d0[1], d0[2]);
            at_split3x2(kheld[u].z, kheld[u].w, d1[0], d1[1], d1[2]);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<uint2*>(at_smem + p * AT_PART_K + at_k_index(row, c4)) = uint2{d0[p], d1[p]};
        }
        // B operand of S^T, pre-scaled so that S = scale * log2(e) * Q.K^T (the scores are kept in the
        // base-2 domain, so that the softmax numerators are one v_exp_f32 each)
        uint4 qf[QT][AT_D / 32][3];
        const float qs = scale * 1.4426950408889634f;
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int u = 0; u < AT_D / 32; ++u) {
                const float4 a = qheld[q][2 * u], bq = qheld[q][2 * u + 1];
                const float v[8] = {a.x * qs, a.y * qs, a.z * qs, a.w * qs, bq.x * qs, bq.y * qs, bq.z * qs, bq.w * qs};
                uint32_t d[3][4];
#pragma unroll
                for (int e = 0; e < 4; ++e) at_split3x2(v[2 * e], v[2 * e + 1], d[0][e], d[1][e], d[2][e]);
#pragma unroll
                for (int p = 0; p < 3; ++p) qf[q][u][p] = uint4{d[p][0], d[p][1], d[p][2], d[p][3]};
            }
        __syncthreads();  // K is in LDS
        // Pairs of consecutive keys of V at the same four columns (V^T keeps a column's keys contiguous, so a pair of
        // keys is one dword of each part).  Four lanes cover 64 bytes of a row and 16 pairs follow each other, so that
        // the dwords of a write fall on all banks evenly.
        const int vpair = tid / 4 % 16, vcol = (tid / 64 * 4 + tid % 4) * 4;
        float4 vheld[VP][2];
        auto request_v = [&](int u, int e) { vheld[u][e] = fetch(it.base, 2, 32 * u, 2 * vpair + e, vcol); };
        // st[q][t][r] = S[query 16 (t0 + q) + c][key 16t + 4g + r]
        v4f st[QT][AT_NT];
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int t = 0; t < AT_NT; ++t) st[q][t] = v4f{0.f, 0.f, 0.f, 0.f};
        // A step is a tile of keys and half of the head's columns; the next step's fragments are read ahead of its
        // products.  V is requested a piece per step when half of the queries' fragments are done with.
        auto scores = [&](auto n) {
            constexpr int NQ = decltype(n)::value, STEPS = AT_NT * (AT_D / 32);
            uint4 kf[2][3];
            auto read = [&](int s) {
                const int at = at_k_index(16 * (s % AT_NT) + c, 32 * (s / AT_NT) + 8 * g);
#pragma unroll
                for (int p = 0; p < 3; ++p) kf[s & 1][p] = *reinterpret_cast<const uint4*>(at_smem + p * AT_PART_K + at);
            };
            read(0);
#pragma unroll
            for (int s = 0; s < STEPS; ++s) {
                const int u = s / AT_NT, t = s % AT_NT;
                if (s + 1 < STEPS) read(s + 1);
                if (s >= AT_NT) request_v((s - AT_NT) / 2, (s - AT_NT) % 2);
                if (s == STEPS - 1) request_v(VP - 1, 1);
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) st[q][t] = at_mm(kf[s & 1][kAtPa[x]], qf[q][u][kAtPb[x]], st[q][t]);
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);  // the reads first
                __builtin_amdgcn_sched_group_barrier(0x008, 6 * NQ, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        if (QT == 2 && it.nq == 2)
            scores(std::integral_constant<int, QT>{});
        else if (it.nq > 0)
            scores(std::integral_constant<int, 1>{});
        else
#pragma unroll
            for (int u = 0; u < 2 * VP; ++u) request_v(u / 2, u % 2);
        static_assert(AT_NT == 2 * VP - 1, "a piece of V per step, two in the last");
        __syncthreads();  // nobody reads K any more
        float vmax = 0.0f;  // a NaN stays
#pragma unroll
        for (int u = 0; u < VP; ++u) {
            if (32 * u + 32 > AT_TMAX && 32 * u + 2 * vpair >= AT_TMAX) continue;
            const float4 v0 = vheld[u][0], v1 = vheld[u][1];
            const float a[4] = {v0.x, v0.y, v0.z, v0.w}, bb[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                vmax = __builtin_elementwise_maximum(__builtin_elementwise_maximum(vmax, __builtin_fabsf(a[e])), __builtin_fabsf(bb[e]));
                uint32_t d[3];
                at_split3x2(a[e], bb[e], d[0], d[1], d[2]);
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    *reinterpret_cast<uint32_t*>(at_smem + p * AT_PART_V + at_v_index(e, vcol / 4, 32 * u + 2 * vpair)) = d[p];
            }
        }
        if (!(vmax <= AT_VMAX)) s_large = 1;
        float mx[QT], sum[QT][4];  // four sums of every fourth key each: shorter chains round less
        auto mask = [&](int t) {  // keys past the last token
#pragma unroll
            for (int q = 0; q < QT; ++q)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (16 * t + 4 * g + r >= T) st[q][t][r] = -__builtin_inff();
        };
        mask(AT_NT - 1);
        if (T <= 16 * (AT_NT - 1)) {
#pragma unroll
            for (int t = 0; t < AT_NT - 1; ++t) mask(t);
        }
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            mx[q] = -__builtin_inff(), sum[q][0] = sum[q][1] = sum[q][2] = sum[q][3] = 0.0f;
#pragma unroll
            for (int t = 0; t < AT_NT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) mx[q] = __builtin_elementwise_maximum(mx[q], st[q][t][r]);
            mx[q] = at_rows4(mx[q], [](float a, float b) { return __builtin_elementwise_maximum(a, b); });
        }
        __syncthreads();  // V^T is in LDS
        if (s_large) {
#pragma unroll
            for (int q = 0; q < QT; ++q) mx[q] += 8.0f;
        }

        // O[q][n] = sum_key P[q][key] V[key][n] with P = 2^(S - max), or 2^(S - max - 8) (AT_VMAX), divided by P's sum at the
        // end, in four tiles of 16 columns
        static_assert(AT_NT % 2 == 1, "tile pairs and one single tile");
        constexpr int NJ = AT_D / 16;
        v4f o[QT][NJ];
#pragma unroll
        for (int q = 0; q < QT; ++q)
#pragma unroll
            for (int j = 0; j < NJ; ++j) o[q][j] = v4f{0.f, 0.f, 0.f, 0.f};
        auto values = [&](auto n) {
            constexpr int NQ = decltype(n)::value, PAIRS = AT_NT / 2;
            // Parts of the probabilities of tiles 2 tp and 2 tp + 1: the eight k slots of this lane are keys
            // 32 tp + 4 g + 0..3 and 32 tp + 16 + 4 g + 0..3.  Pair e is slots 2 e and 2 e + 1.
            uint32_t pd[2][NQ][3][4];
            auto probs = [&](int tp, int q, int e) {
                const int t = 2 * tp + e / 2, r = e % 2 * 2;
                const float a = __builtin_amdgcn_exp2f(st[q][t][r] - mx[q]);  // 2^(-inf) = 0 for the padded keys
                const float b = __builtin_amdgcn_exp2f(st[q][t][r + 1] - mx[q]);
                sum[q][r] += a;
                sum[q][r + 1] += b;
                auto& d = pd[tp & 1][q];
                at_split3x2(a, b, d[0][e], d[1][e], d[2][e]);
            };
            uint4 vf[2][3];
            auto read = [&](int s) {
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    const uint16_t* vpart = at_smem + p * AT_PART_V;
                    const int key = 32 * (s / NJ) + 4 * g;
                    const uint2 x = *reinterpret_cast<const uint2*>(vpart + at_v_index(s % NJ, c, key));
                    uint2 y = {0, 0};
                    if (s / NJ < PAIRS) y = *reinterpret_cast<const uint2*>(vpart + at_v_index(s % NJ, c, key + 16));
                    vf[s & 1][p] = uint4{x.x, x.y, y.x, y.y};
                }
            };
            read(0);
#pragma unroll
            for (int q = 0; q < NQ; ++q)
#pragma unroll
                for (int e = 0; e < 4; ++e) probs(0, q, e);
            // a step is a pair of key tiles and 16 columns; under its products the vector unit makes a fourth of the
            // next pair's probabilities, and the last steps request the next item
#pragma unroll
            for (int s = 0; s < PAIRS * NJ; ++s) {
                const int tp = s / NJ, j = s % NJ;
                read(s + 1);
                constexpr int FROM = PAIRS * NJ * 3 / 4, N = PAIRS * NJ - FROM;
                if (QT == 2 && s >= FROM) {
#pragma unroll
                    for (int x = (s - FROM) * PIECES / N; x < (s - FROM + 1) * PIECES / N; ++x) request(after, x, tid);
                }
#pragma unroll
                for (int q = 0; q < NQ; ++q)
                    if (tp + 1 < PAIRS || j < 2) probs(tp + 1, q, j);
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        const auto& d = pd[tp & 1][q][kAtPa[x]];
                        o[q][j] = at_mm(uint4{d[0], d[1], d[2], d[3]}, vf[s & 1][kAtPb[x]], o[q][j]);
                    }
                __builtin_amdgcn_sched_group_barrier(0x100, 3, 0);
#pragma unroll
                for (int x = 0; x < 6 * NQ; ++x) {
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x402, 3, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            // the last tile: keys 16 (AT_NT - 1) + 4 g + 0..3, four k slots per lane
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int s = PAIRS * NJ + j;
                if (j + 1 < NJ) read(s + 1);
#pragma unroll
                for (int x = 0; x < 6; ++x)
#pragma unroll
                    for (int q = 0; q < NQ; ++q) {
                        const auto& d = pd[PAIRS & 1][q][kAtPa[x]];
                        const uint4& v = vf[s & 1][kAtPb[x]];
                        o[q][j] = at_mm(uint2{d[0], d[1]}, uint2{v.x, v.y}, o[q][j]);
                    }
            }
        };
        if (QT == 2 && it.nq == 2)
            values(std::integral_constant<int, QT>{});
        else if (it.nq > 0)
            values(std::integral_constant<int, 1>{});
        else if (QT == 2)
#pragma unroll
            for (int x = 0; x < PIECES; ++x) request(after, x, tid);
        if (QT == 1) {  // mostly one item per block: nothing to request
#pragma unroll
            for (int x = 0; x < KP; ++x) kheld[x] = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int x = 0; x < 2 * (AT_D / 32); ++x) qheld[0][x] = float4{0.f, 0.f, 0.f, 0.f};
            if (next < items) {
#pragma unroll
                for (int x = 0; x < PIECES; ++x) request(after, x, tid);
            }
        }
        // result layout of the 16x16 MFMA: column slot = lane % 16, row = 4*(lane/16) + r; the 16 lanes
        // of a row store 256 consecutive bytes
        const int b = it.head / H, h = it.head - b * H;
#pragma unroll
        for (int q = 0; q < QT; ++q) {
            if (q >= it.nq) continue;
            const float total = at_rows4((sum[q][0] + sum[q][1]) + (sum[q][2] + sum[q][3]), [](float a, float b) { return a + b; });
            const float inv = total > 0.0f ? 1.0f / total : 0.0f;
            const int row0 = (it.t0 + q) * 16;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float by = __shfl(inv, 4 * g + r, 64);  // of query row0 + 4 g + r
                const int row = row0 + 4 * g + r;
                if (row < T) {
                    float v[NJ];
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        v[j] = o[q][j][r] * by;
                        kept.add(v[j]);
                    }
                    float* at = out + (size_t(b) * T + row) * (size_t(H) * AT_D) + size_t(h) * AT_D + 4 * c;
                    if (out_vec)
                        *reinterpret_cast<float4*>(at) = float4{v[0], v[1], v[2], v[3]};
                    else
                        at[0] = v[0], at[1] = v[1], at[2] = v[2], at[3] = v[3];
                }
            }
        }
        __syncthreads();  // V^T has been read: the next item's K may be written
    }
    if (range) kept.store(range);
}

// One block per head, one wavefront per tile of 16 queries, K's parts and V^T's side by side in LDS: after the one barrier
// that follows the splits a wavefront runs scores, softmax and P . V on its own.  K and V are split once per head where the
// kernel above splits them once per part, which is what counts while every CU has one head (see lq_attention_f32 for the line
// and both sides' times); each fragment serves 16 queries.  The probabilities are normalized before P . V.
constexpr size_t AT_HEAD_SMEM = size_t(3) * (AT_PART_K + AT_PART_V) * 2;
static_assert(AT_HEAD_SMEM + 1024 <= 160 * 1024, "LDS of a CU, with the range reduction's few words");

// acc += a . b from the parts, smallest terms first
template <class V>
__device__ __forceinline__ v4f at_mma6(const V (&a)[3], const V (&b)[3], v4f acc) {
#pragma unroll
    for (int x = 0; x < 6; ++x) acc = at_mm(a[kAtPa[x]], b[kAtPb[x]], acc);
    return acc;
}

__global__ __launch_bounds__(1024) void attention_head_kernel(const float* __restrict__ qkv, float* __restrict__ out, int T,
                                                             int H, float scale, float* range) {
    extern __shared__ __attribute__((aligned(16))) uint16_t at_smem[];
    uint16_t* const k_lds = at_smem;
    uint16_t* const v_lds = at_smem + 3 * AT_PART_K;
    const int b = blockIdx.x / H, h = blockIdx.x % H;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const size_t tok_stride = size_t(3) * H * AT_D;
    const float* base = qkv + size_t(b) * T * tok_stride + size_t(h) * AT_D;
    // K and V are requested before anything is used (a block of 13 wavefronts holds all of both: four
    // 16-byte pieces of each per thread).  A thread's V pieces are two pairs of consecutive keys at the
    // same four columns: V^T keeps a column's keys contiguous, so a pair of keys is one dword of each part
    constexpr int kPieces = AT_TMAX * (AT_D / 4), kHeld = 4;
    constexpr int kPairs = (AT_TMAX / 2) * (AT_D / 4);
    float4 kheld[kHeld], vheld[kHeld];
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int i = tid + u * int(blockDim.x), row = i / (AT_D / 4), c4 = (i % (AT_D / 4)) * 4;
        kheld[u] = float4{0.f, 0.f, 0.f, 0.f};
        if (i < kPieces && row < T) kheld[u] = *reinterpret_cast<const float4*>(base + size_t(row) * tok_stride + size_t(H) * AT_D + c4);
    }
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int i = tid + (u >> 1) * int(blockDim.x), row = 2 * (i / (AT_D / 4)) + (u & 1), c4 = (i % (AT_D / 4)) * 4;
        vheld[u] = float4{0.f, 0.f, 0.f, 0.f};
        if (i < kPairs && row < T) vheld[u] = *reinterpret_cast<const float4*>(base + size_t(row) * tok_stride + size_t(2) * H * AT_D + c4);
    }
    // One wavefront per tile of 16 queries.  With 4 n + 1 tiles one SIMD would hold a wavefront more
    // than the others and everybody would wait for it: the launch then has three more wavefronts,
    // and the last tile's four each compute its scores but only one 16-column tile of its output.
    const int tiles = (T + 15) / 16;
    const bool shared_last = int(blockDim.x) > tiles * 64;
    const int q0 = (wave < tiles ? wave : tiles - 1) * 16;
    const int only_j = (shared_last && wave >= tiles - 1) ? wave - (tiles - 1) : -1;  // wavefront-uniform
    const int g = lane >> 4, c = lane & 15;
    // the lane's slice of its query row: Q[q0 + c][32 u + 8 g + 0..7]
    float4 qheld[2 * (AT_D / 32)];
    {
        const int q = q0 + c;
        const float* qp = base + size_t(q < T ? q : T - 1) * tok_stride;
#pragma unroll
        for (int u = 0; u < AT_D / 32; ++u) {
            qheld[2 * u] = *reinterpret_cast<const float4*>(qp + 32 * u + 8 * g);
            qheld[2 * u + 1] = *reinterpret_cast<const float4*>(qp + 32 * u + 8 * g + 4);
        }
    }
    // K rows into LDS as three bfloat16 parts (rows past T are zero)
    auto place_k = [&](int i, float4 kv) {
        const int row = i / (AT_D / 4), c4 = (i % (AT_D / 4)) * 4;
        uint32_t lo[3], hi[3];
        at_split3x2(kv.x, kv.y, lo[0], lo[1], lo[2]);
        at_split3x2(kv.z, kv.w, hi[0], hi[1], hi[2]);
        const int at = at_k_index(row, c4);
#pragma unroll
        for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(k_lds + p * AT_PART_K + at) = uint2{lo[p], hi[p]};
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int i = tid + u * int(blockDim.x);
        if (i < kPieces) place_k(i, kheld[u]);
    }
    for (int i = tid + kHeld * int(blockDim.x); i < kPieces; i += blockDim.x) {  // fewer than 13 wavefronts
        const int row = i / (AT_D / 4), c4 = (i % (AT_D / 4)) * 4;
        float4 kv = {0.f, 0.f, 0.f, 0.f};
        if (row < T) kv = *reinterpret_cast<const float4*>(base + size_t(row) * tok_stride + size_t(H) * AT_D + c4);
        place_k(i, kv);
    }
    // V^T's parts: keys 2 pair and 2 pair + 1 at columns c4 .. c4 + 3 (keys past T are zero)
    auto place_v = [&](int i, float4 v0, float4 v1) {
        const int pair = i / (AT_D / 4), c4 = (i % (AT_D / 4)) * 4;
        const float a[4] = {v0.x, v0.y, v0.z, v0.w}, bb[4] = {v1.x, v1.y, v1.z, v1.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t d[3];
            at_split3x2(a[e], bb[e], d[0], d[1], d[2]);
#pragma unroll
            for (int p = 0; p < 3; ++p)
                *reinterpret_cast<uint32_t*>(v_lds + p * AT_PART_V + (c4 + e) * AT_VLD + 2 * pair) = d[p];
        }
    };
#pragma unroll
    for (int u = 0; u < kHeld / 2; ++u) {
        const int i = tid + u * int(blockDim.x);
        if (i < kPairs) place_v(i, vheld[2 * u], vheld[2 * u + 1]);
    }
    for (int i = tid + (kHeld / 2) * int(blockDim.x); i < kPairs; i += blockDim.x) {  // fewer than 13 wavefronts
        const int pair = i / (AT_D / 4), c4 = (i % (AT_D / 4)) * 4;
        float4 v0 = {0.f, 0.f, 0.f, 0.f}, v1 = {0.f, 0.f, 0.f, 0.f};
        const float* vp = base + size_t(2) * H * AT_D + c4;
        if (2 * pair < T) v0 = *reinterpret_cast<const float4*>(vp + size_t(2 * pair) * tok_stride);
        if (2 * pair + 1 < T) v1 = *reinterpret_cast<const float4*>(vp + size_t(2 * pair + 1) * tok_stride);
        place_v(i, v0, v1);
    }
    // B operand of S^T, pre-scaled so that S = scale * log2(e) * Q.K^T (the scores are kept in the
    // base-2 domain, so that the softmax numerators are one v_exp_f32 each)
    uint4 qf[AT_D / 32][3];
    {
        const float qs = scale * 1.4426950408889634f;
#pragma unroll
        for (int u = 0; u < AT_D / 32; ++u) {
            const float4 a = qheld[2 * u], bq = qheld[2 * u + 1];
            const float v[8] = {a.x * qs, a.y * qs, a.z * qs, a.w * qs, bq.x * qs, bq.y * qs, bq.z * qs, bq.w * qs};
            uint32_t d[3][4];
#pragma unroll
            for (int e = 0; e < 4; ++e) at_split3x2(v[2 * e], v[2 * e + 1], d[0][e], d[1][e], d[2][e]);
#pragma unroll
            for (int p = 0; p < 3; ++p) qf[u][p] = uint4{d[p][0], d[p][1], d[p][2], d[p][3]};
        }
    }
    __syncthreads();  // the only one before the range reduction: from here on a wavefront is on its own
    v4f st[AT_NT];
#pragma unroll
    for (int t = 0; t < AT_NT; ++t) st[t] = v4f{0.f, 0.f, 0.f, 0.f};
    // k slice outermost: the 13 tiles' accumulators are independent chains
#pragma unroll
    for (int u = 0; u < AT_D / 32; ++u)
#pragma unroll
        for (int t = 0; t < AT_NT; ++t) {
            uint4 kf[3];
            const int at = at_k_index(16 * t + c, 32 * u + 8 * g);
#pragma unroll
            for (int p = 0; p < 3; ++p) kf[p] = *reinterpret_cast<const uint4*>(k_lds + p * AT_PART_K + at);
            st[t] = at_mma6(kf, qf[u], st[t]);
        }
    // st[t][r] = S[query q0 + c][key 16t + 4g + r]
    float mx = -__builtin_inff();
#pragma unroll
    for (int t = 0; t < AT_NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int key = 16 * t + 4 * g + r;
            if (key >= T) st[t][r] = -__builtin_inff();
            mx = fmaxf(mx, st[t][r]);
        }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < AT_NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float e = __builtin_amdgcn_exp2f(st[t][r] - mx);  // 2^(-inf) = 0 for the padded keys
            st[t][r] = e;
            sum += e;
        }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    const float inv = sum > 0.0f ? 1.0f / sum : 0.0f;

    // O[q][n] = sum_key P[q][key] V[key][n], four 16-wide column tiles; tile j of the output holds
    // head-dim columns 16 j + c: the 16 lanes of a fragment read consecutive V^T rows (rows 4 c + j,
    // which would let a lane store four consecutive floats, fall on four bank pairs only)
    static_assert(AT_NT % 2 == 1, "tile pairs and one single tile");
    v4f o[AT_D / 16];
#pragma unroll
    for (int j = 0; j < AT_D / 16; ++j) o[j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int tp = 0; tp < AT_NT / 2; ++tp) {
        // the eight k slots of this lane: keys 32 tp + 4 g + 0..3 and 32 tp + 16 + 4 g + 0..3
        float pv[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            pv[r] = st[2 * tp][r] * inv;
            pv[4 + r] = st[2 * tp + 1][r] * inv;
        }
        uint32_t d[3][4];
#pragma unroll
        for (int e = 0; e < 4; ++e) at_split3x2(pv[2 * e], pv[2 * e + 1], d[0][e], d[1][e], d[2][e]);
        uint4 pf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) pf[p] = uint4{d[p][0], d[p][1], d[p][2], d[p][3]};
#pragma unroll
        for (int j = 0; j < AT_D / 16; ++j) {
            if (only_j >= 0 && only_j != j) continue;
            uint4 vf[3];
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                const uint16_t* vrow = v_lds + p * AT_PART_V + (16 * j + c) * AT_VLD + 32 * tp + 4 * g;
                const uint2 lo = *reinterpret_cast<const uint2*>(vrow), hi = *reinterpret_cast<const uint2*>(vrow + 16);
                vf[p] = uint4{lo.x, lo.y, hi.x, hi.y};
            }
            o[j] = at_mma6(pf, vf, o[j]);
        }
    }
    {
        // the last tile: keys 16 (AT_NT - 1) + 4 g + 0..3, four k slots per lane
        float pv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) pv[r] = st[AT_NT - 1][r] * inv;
        uint32_t d[3][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) at_split3x2(pv[2 * e], pv[2 * e + 1], d[0][e], d[1][e], d[2][e]);
        uint2 pf[3];
#pragma unroll
        for (int p = 0; p < 3; ++p) pf[p] = uint2{d[p][0], d[p][1]};
#pragma unroll
        for (int j = 0; j < AT_D / 16; ++j) {
            if (only_j >= 0 && only_j != j) continue;
            uint2 vf[3];
#pragma unroll
            for (int p = 0; p < 3; ++p)
                vf[p] = *reinterpret_cast<const uint2*>(v_lds + p * AT_PART_V + (16 * j + c) * AT_VLD + 16 * (AT_NT - 1) + 4 * g);
            o[j] = at_mma6(pf, vf, o[j]);
        }
    }
    // result layout of the 16x16 MFMA: column slot = lane % 16, row = 4*(lane/16) + r; the 16 lanes
    // of a row store 64 consecutive bytes
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int q = q0 + 4 * g + r;
        if (q < T) {
            float* orow = out + (size_t(b) * T + q) * (size_t(H) * AT_D) + size_t(h) * AT_D + c;
#pragma unroll
            for (int j = 0; j < AT_D / 16; ++j)
                if (only_j < 0 || only_j == j) orow[16 * j] = o[j][r];
        }
    }
    if (range) {
        RangeKeep kept;
#pragma unroll
        for (int j = 0; j < AT_D / 16; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if (q0 + 4 * g + r < T && (only_j < 0 || only_j == j)) kept.add(o[j][r]);
        kept.store(range);
    }
}

unsigned blocks_for(size_t n) { return unsigned((n + 255) / 256); }

}  // namespace

namespace lq {
int sgemm_nt(const float* a, const float* w, const float* bias, float* out, int M, int N, int K, bool large, hipStream_t st) {
    LQ_REQUIRE(a && w && out, LQ_ERR_VALUE, "sgemm: null pointer");
    LQ_REQUIRE(M >= 0 && N >= 0 && K > 0, LQ_ERR_SHAPE, "sgemm: bad shape (%d, %d, %d)", M, N, K);
    if (M == 0 || N == 0) return LQ_OK;
    LQ_REQUIRE(M <= 65535 * SG_BM, LQ_ERR_SHAPE, "sgemm: M too large");
    const bool vec = K % 4 == 0 && aligned16(a) && aligned16(w);
    return (vec ? launch_sgemm<0, true> : launch_sgemm<0, false>)(a, w, bias, out, M, N, K, PatchForm{}, st, large);
}
}  // namespace lq

extern "C" {

int lq_layernorm_f32(const float* x, const float* gamma, const float* beta, float* out, long rows, int cols,
                     float eps, float* range, void* stream) {
    LQ_REQUIRE(x && gamma && beta && out, LQ_ERR_VALUE, "layernorm: null pointer");
    LQ_REQUIRE(rows >= 0 && cols > 0, LQ_ERR_SHAPE, "layernorm: bad shape (%ld, %d)", rows, cols);
    if (rows == 0) return LQ_OK;
    const long per_block = 4L * LN_ROWS_PER_WAVE;
    LQ_REQUIRE((rows + per_block - 1) / per_block < 0x7fffffffL, LQ_ERR_SHAPE, "layernorm: too many rows");
    LQ_REQUIRE(range == nullptr || (rows + per_block - 1) / per_block <= kRangeSlots, LQ_ERR_SHAPE,
               "layernorm: %ld rows are too many for a kept range (at most %ld)", rows,
               long(kRangeSlots) * per_block);
    layernorm_kernel<<<unsigned((rows + per_block - 1) / per_block), 256, 0, as_stream(stream)>>>(
        x, gamma, beta, out, rows, cols, eps, range);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_layernorm_stats_f32(const float* x, const float* gamma, const float* beta, long rows, int cols, float eps,
                           float* stats, float* range, void* stream) {
    LQ_REQUIRE(x && gamma && beta && stats && range, LQ_ERR_VALUE, "layernorm_stats: null pointer");
    LQ_REQUIRE(rows >= 0 && cols > 0, LQ_ERR_SHAPE, "layernorm_stats: bad shape (%ld, %d)", rows, cols);
    LQ_REQUIRE(cols % 4 == 0 && cols <= LN_KEEP * 256 && aligned16(x) && aligned16(gamma) && aligned16(beta),
               LQ_ERR_NOT_IMPLEMENTED,
               "layernorm_stats: rows of %d floats; the fused form takes vector-aligned rows of a multiple of 4, "
               "at most %d (use lq_layernorm_f32 + lq_quantize)", cols, LN_KEEP * 256);
    if (rows == 0) return LQ_OK;
    const long blocks = (rows + 3) / 4;
    LQ_REQUIRE(blocks <= kRangeSlots, LQ_ERR_SHAPE, "layernorm_stats: %ld rows are too many for a kept range", rows);
    if (cols <= 4 * 256)
        layernorm_stats_kernel<4><<<unsigned(blocks), 256, 0, as_stream(stream)>>>(x, gamma, beta, rows, cols, eps, stats, range);
    else
        layernorm_stats_kernel<LN_KEEP><<<unsigned(blocks), 256, 0, as_stream(stream)>>>(x, gamma, beta, rows, cols, eps, stats,
                                                                                          range);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

namespace {
int launch_layernorm_quantize(const float* x, const float* gamma, const float* beta, const float* stats, long rows, int cols,
                              float* scale, float* zp, const LnGrid& grid, int code_offset, int8_t* q, void* stream) {
    LQ_REQUIRE(x && gamma && beta && stats && scale && zp && q, LQ_ERR_VALUE, "layernorm_quantize: null pointer");
    LQ_REQUIRE(rows >= 0 && cols > 0, LQ_ERR_SHAPE, "layernorm_quantize: bad shape (%ld, %d)", rows, cols);
    LQ_REQUIRE(cols % 4 == 0 && cols <= LN_KEEP * 256 && aligned16(x) && aligned16(gamma) && aligned16(beta) &&
                   (reinterpret_cast<uintptr_t>(q) & 3u) == 0,
               LQ_ERR_NOT_IMPLEMENTED, "layernorm_quantize: rows of %d floats are not what the fused form takes", cols);
    LQ_REQUIRE(grid.qmax > grid.qmin && grid.qmin + code_offset >= -128 && grid.qmax + code_offset <= 127, LQ_ERR_VALUE,
               "layernorm_quantize: grid [%d,%d] + offset %d does not fit int8", grid.qmin, grid.qmax, code_offset);
    if (rows == 0) return LQ_OK;
    const long blocks = (rows + 3) / 4;
    LQ_REQUIRE(blocks < 0x7fffffffL, LQ_ERR_SHAPE, "layernorm_quantize: too many rows");
#define LQ_LN_QUANTIZE(KEEP, RANGE) \
    layernorm_quantize_kernel<KEEP, RANGE><<<unsigned(blocks), 256, 0, as_stream(stream)>>>(x, gamma, beta, stats, rows, \
                                                                                                  cols, scale, zp, grid, code_offset, q)
    if (cols <= 4 * 256 && grid.range)
        LQ_LN_QUANTIZE(4, true);
    else if (cols <= 4 * 256)
        LQ_LN_QUANTIZE(4, false);
    else if (grid.range)
        LQ_LN_QUANTIZE(LN_KEEP, true);
    else
        LQ_LN_QUANTIZE(LN_KEEP, false);
#undef LQ_LN_QUANTIZE
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}
}  // namespace

int lq_layernorm_quantize_i8(const float* x, const float* gamma, const float* beta, const float* stats, long rows,
                             int cols, const float* scale, const float* zp, int qmin, int qmax, int code_offset,
                             int8_t* q, void* stream) {
    const LnGrid grid{nullptr, 0, qmin, qmax, 0, 0.0f, 0.0f};
    return launch_layernorm_quantize(x, gamma, beta, stats, rows, cols, const_cast<float*>(scale), const_cast<float*>(zp), grid,
                                     code_offset, q, stream);
}

int lq_layernorm_quantize_from_range_i8(const float* x, const float* gamma, const float* beta, const float* stats, long rows,
                                        int cols, const float* range, int symmetric, int qmin, int qmax, int is_signed,
                                        float eps, int code_offset, float* scale, float* zp, int8_t* q, void* stream) {
    LQ_REQUIRE(range && scale && zp, LQ_ERR_VALUE, "layernorm_quantize: null pointer");
    // Every block of the one launch reads a slot per block of the statistics: up to 2048 rows that is less than the launch it
    // saves (12 608 rows of 768: 16.6 us against 8.3 + 4.6).
    // No rows have no block that hands out the qparams.
    if (rows > kRangeRows || rows == 0) {
        const int rc = lq_calc_qparams_from_range(range, symmetric, qmin, qmax, is_signed, eps, scale, zp, nullptr, nullptr, stream);
        return rc ? rc : lq_layernorm_quantize_i8(x, gamma, beta, stats, rows, cols, scale, zp, qmin, qmax, code_offset, q, stream);
    }
    const LnGrid grid{range, symmetric, qmin, qmax, is_signed, eps, float((double(qmax) - double(qmin)) / 2.0)};
    return launch_layernorm_quantize(x, gamma, beta, stats, rows, cols, scale, zp, grid, code_offset, q, stream);
}

int lq_gelu_f32(const float* x, float* out, size_t n, float* range, void* stream) {
    LQ_REQUIRE(x && out, LQ_ERR_VALUE, "gelu: null pointer");
    if (n == 0) return LQ_OK;
    const int vec = (n % 4 == 0) && aligned16(x) && aligned16(out);
    const size_t units = vec ? n / 4 : n;
    const size_t blocks = (units + 256 * GELU_PER_THREAD - 1) / (256 * GELU_PER_THREAD);
    LQ_REQUIRE(blocks < 0x7fffffffull, LQ_ERR_SHAPE, "gelu: tensor too large");
    LQ_REQUIRE(range == nullptr || blocks <= size_t(kRangeSlots), LQ_ERR_SHAPE,
               "gelu: %zu elements are too many for a kept range (at most %zu)", n,
               size_t(kRangeSlots) * 256 * GELU_PER_THREAD * 4);
    gelu_kernel<<<unsigned(blocks), 256, 0, as_stream(stream)>>>(x, out, n, vec, range);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_add_f32(const float* a, const float* b, float* out, size_t n, void* stream) {
    LQ_REQUIRE(a && b && out, LQ_ERR_VALUE, "add: null pointer");
    if (n == 0) return LQ_OK;
    const int vec = (n % 4 == 0) && aligned16(a) && aligned16(b) && aligned16(out);
    add_kernel<<<blocks_for(vec ? n / 4 : n), 256, 0, as_stream(stream)>>>(a, b, out, n, vec);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_patchify_f32(const float* img, float* out, int B, int C, int H, int W, int patch, void* stream) {
    LQ_REQUIRE(img && out, LQ_ERR_VALUE, "patchify: null pointer");
    LQ_REQUIRE(B >= 0 && C > 0 && H > 0 && W > 0 && patch > 0 && H % patch == 0 && W % patch == 0, LQ_ERR_SHAPE,
               "patchify: image %dx%dx%dx%d is not a whole number of %d-pixel patches", B, C, H, W, patch);
    const size_t total = size_t(B) * C * H * W;
    if (total == 0) return LQ_OK;
    patchify_kernel<<<blocks_for(total), 256, 0, as_stream(stream)>>>(img, out, B, C, H, W, patch);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_assemble_tokens_f32(const float* patches, const float* cls, const float* pos, float* out, int B, int T,
                           int D, void* stream) {
    LQ_REQUIRE(patches && cls && pos && out, LQ_ERR_VALUE, "assemble_tokens: null pointer");
    LQ_REQUIRE(B >= 0 && T >= 1 && D > 0, LQ_ERR_SHAPE, "assemble_tokens: bad shape");
    const size_t total = size_t(B) * T * D;
    if (total == 0) return LQ_OK;
    assemble_tokens_kernel<<<blocks_for(total), 256, 0, as_stream(stream)>>>(patches, cls, pos, out, B, T, D);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_sgemm_nt_f32(const float* a, const float* w, const float* bias, float* out, int M, int N, int K,
                    void* stream) {
    return sgemm_nt(a, w, bias, out, M, N, K, false, as_stream(stream));
}

int lq_patch_embed_f32(const float* img, const float* w, const float* bias, const float* cls, const float* pos,
                       float* out, int B, int C, int H, int W, int patch, int D, void* stream) {
    LQ_REQUIRE(img && w && cls && pos && out, LQ_ERR_VALUE, "patch_embed: null pointer");
    LQ_REQUIRE(B >= 0 && C > 0 && H > 0 && W > 0 && D > 0 && patch > 0 && H % patch == 0 && W % patch == 0,
               LQ_ERR_SHAPE, "patch_embed: image %dx%dx%dx%d is not a whole number of %d-pixel patches", B, C, H, W,
               patch);
    const int per_image = (H / patch) * (W / patch);
    const size_t rows = size_t(B) * per_image, K = size_t(C) * patch * patch;
    LQ_REQUIRE(rows < (size_t(1) << 31) && K < (size_t(1) << 31), LQ_ERR_SHAPE, "patch_embed: too many patch rows");
    if (B == 0) return LQ_OK;
    LQ_REQUIRE(rows <= size_t(65535) * SG_BM, LQ_ERR_SHAPE, "patch_embed: too many patch rows");
    int log2p = -1;
    for (int e = 0; e < 15; ++e)
        if ((1 << e) == patch) log2p = e;
    const PatchForm pf{C, H, W, patch, W / patch, per_image, B, log2p, cls, pos};
    const bool vec = K % 4 == 0 && aligned16(w);
    const auto launch = vec && log2p >= 2 && W % 4 == 0 && aligned16(img) ? launch_sgemm<1, true>
                        : vec                                             ? launch_sgemm<2, true>
                                                                          : launch_sgemm<2, false>;
    return launch(img, w, bias, out, int(rows), D, int(K), pf, as_stream(stream), false);
}

int lq_gather_rows_f32(const float* src, size_t src_row_stride, float* dst, size_t rows, size_t cols,
                       void* stream) {
    LQ_REQUIRE(src && dst, LQ_ERR_VALUE, "gather_rows: null pointer");
    LQ_REQUIRE(src_row_stride >= cols, LQ_ERR_SHAPE, "gather_rows: row stride smaller than the row");
    if (rows * cols == 0) return LQ_OK;
    gather_rows_kernel<<<blocks_for(rows * cols), 256, 0, as_stream(stream)>>>(src, src_row_stride, dst, rows, cols);
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

int lq_attention_f32(const float* qkv, float* out, int B, int T, int H, int D, float scale, float* range,
                     void* stream) {
    LQ_REQUIRE(qkv && out, LQ_ERR_VALUE, "attention: null pointer");
    LQ_REQUIRE(B >= 0 && T >= 1 && H >= 1, LQ_ERR_SHAPE, "attention: bad shape");
    LQ_REQUIRE(D == AT_D && T <= AT_TMAX, LQ_ERR_NOT_IMPLEMENTED,
               "attention: head dim %d / %d tokens; this kernel handles head dim 64 and up to 208 tokens", D, T);
    LQ_REQUIRE(aligned16(qkv), LQ_ERR_VALUE, "attention: qkv must be 16-byte aligned");
    if (B == 0) return LQ_OK;
    // (the call's limit: the kernels here use a slot per block and at most 512 of them, a slot per head would take one each)
    LQ_REQUIRE(range == nullptr || long(B) * H <= kRangeSlots, LQ_ERR_SHAPE,
               "attention: a kept range is limited to %d (batch, head) pairs, got %ld", kRangeSlots, long(B) * H);
    const int heads = B * H, tiles = (T + 15) / 16;
    constexpr long kSlots = 512;  // two blocks of attention_kernel on each of 256 CUs, which take further items in turn
    const auto blocks = [&](int qt) { return (long(heads) + 7) / 8 * 8 * ((tiles + qt * AT_WAVES - 1) / (qt * AT_WAVES)); };
    const auto launch = [&](auto qt, auto wide) -> int {
        constexpr int QT = decltype(qt)::value;
        const auto kernel = attention_kernel<QT, decltype(wide)::value>;
        static DeviceOnce attr_once;
        if (int rc = allow_dynamic_lds(attr_once, reinterpret_cast<const void*>(kernel), int(AT_SMEM))) return rc;
        const long items = blocks(QT);
        kernel<<<unsigned(items < kSlots ? items : kSlots), 64 * AT_WAVES, AT_SMEM, as_stream(stream)>>>(
            qkv, out, T, H, heads, int(items / ((long(heads) + 7) / 8 * 8)), aligned16(out), scale, range);
        return LQ_OK;
    };
    // One tile of queries per wavefront while that makes no more blocks than have a place at once, or no more than two tiles
    // would (up to 64 tokens: 1100 heads of 64 tokens 32.2 us against 34.6 with two): 64 heads of 197 tokens 10.5 (15.0 with
    // two, 17.7 in one block per head), 160 heads of 160 tokens 15.6 (20.5, 17.5), 768 heads of 193 tokens 73.6 (59.1, 66.4).
    // One block per head while every CU has one head and either of the others would give it two blocks: 192 heads of 130
    // tokens 15.4 (20.4 with one tile per wavefront, 20.2 with two), 192 of 65 tokens 12.3 (14.7, 15.0), 192 of 193 tokens 19.2
    // (20.9, 21.0).  With two blocks the CU does two thirds more for them than one block does, which longer heads
    // earn back from about 2912 tiles on: 224 heads of 208 tokens 21.1 (26.8, 21.9), 256 of them 24.1 (27.0, 22.6).
    using One = std::integral_constant<int, 1>;
    int rc;
    if (size_t(H) * 3 * AT_D * 4 * 32 > UINT32_MAX) {
        rc = launch(One{}, std::true_type{});
    } else if (tiles <= AT_WAVES || blocks(1) <= (tiles <= 2 * AT_WAVES ? kSlots / 2 : kSlots)) {
        rc = launch(One{}, std::false_type{});
    } else if (heads <= 256 && heads * tiles <= 2912) {
        static DeviceOnce attr_once;
        rc = allow_dynamic_lds(attr_once, reinterpret_cast<const void*>(attention_head_kernel), int(AT_HEAD_SMEM));
        const int waves = tiles + (tiles % 4 == 1 ? 3 : 0);  // see the kernel: the last tile shared by four
        if (rc == LQ_OK)
            attention_head_kernel<<<unsigned(heads), waves * 64, AT_HEAD_SMEM, as_stream(stream)>>>(qkv, out, T, H, scale, range);
    } else {
        rc = launch(std::integral_constant<int, 2>{}, std::false_type{});
    }
    if (rc) return rc;
    LQ_CHECK_LAUNCH();
    return LQ_OK;
}

}  // extern "C"
