// Group-wise affine weight-only quantization (int4 / int8 codes packed in 32-bit
// words) and the matmul that decodes it on the fly - the operator set Lucid binds
// as engine.quantized.{quantize, dequantize, quantized_matmul}
// (lucid/_C/ops/quantized/QuantizedMatmul.cpp:47-115, lucid/quantization/_qgemm.py:69-320)
// on top of MLX.  MLX is not part of the Lucid checkout; this follows the published
// contract (mlx.core.quantize documentation, restated in _qgemm.py:84-97,167-171):
//
//   per row, per group of `group_size` consecutive elements:
//     s = (max - min) / (2^bits - 1),  beta = min
//     c_i = clip(round((w_i - beta) / s), 0, 2^bits - 1)      w_i ~ c_i * s + beta
//   codes little-endian inside a word: code j of a word sits at bits [j*bits, (j+1)*bits)
//   y = x . w_hat^T, float32
//
// A constant group (max == min) gets s = 1e-7-floored, so its codes are 0 and it
// decodes to beta exactly.  The decode side takes scales and biases as given (any
// sign), so weights packed elsewhere under the same contract load unchanged.
#include "wq_pack.hpp"

using namespace lq;

namespace {

__device__ __forceinline__ float wave_min(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fminf(v, __shfl_xor(v, d, 64));
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

// One wavefront per group.  Lane l owns elements l, l + 64 (group_size 128) of the group.
__global__ __launch_bounds__(256) void wq_quantize_kernel(const float* __restrict__ w, size_t groups, int gs,
                                                          int bits, uint32_t* __restrict__ packed,
                                                          float* __restrict__ scales, float* __restrict__ biases) {
    const size_t g = size_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (g >= groups) return;
    const int lane = threadIdx.x & 63;
    const float* src = w + g * gs;
    const int per_word = 32 / bits;
    const float nmax = float((1 << bits) - 1);
    float lo = __builtin_inff(), hi = -__builtin_inff();
    for (int i = lane; i < gs; i += 64) {
        const float v = src[i];
        lo = fminf(lo, v);
        hi = fmaxf(hi, v);
    }
    lo = wave_min(lo);
    hi = wave_max(hi);
    float s = (hi - lo) / nmax;
    s = s < 1e-7f ? 1e-7f : s;
    if (lane == 0) scales[g] = s, biases[g] = lo;
    // one lane per output word
    uint32_t* dst = packed + g * (gs / per_word);
    for (int wd = lane; wd < gs / per_word; wd += 64) {
        uint32_t word = 0;
        for (int j = 0; j < per_word; ++j) {
            float q = __builtin_rintf((src[wd * per_word + j] - lo) / s);
            q = q < 0.0f ? 0.0f : (q > nmax ? nmax : q);
            word |= uint32_t(q) << (j * bits);
        }
        dst[wd] = word;
    }
}

__global__ __launch_bounds__(256) void wq_dequantize_kernel(const uint32_t* __restrict__ packed,
                                                            const float* __restrict__ scales,
                                                            const float* __restrict__ biases, size_t words, int gs,
                                                            int bits, float* __restrict__ out) {
    const size_t wd = size_t(blockIdx.x) * 256 + threadIdx.x;
    if (wd >= words) return;
    const int per_word = 32 / bits;
    const uint32_t mask = (1u << bits) - 1u;
    const size_t first = wd * per_word, g = first / gs;
    const float s = scales[g], b = biases[g];
    const uint32_t word = packed[wd];
    for (int j = 0; j < per_word; ++j) out[first + j] = float((word >> (j * bits)) & mask) * s + b;
}

constexpr int WQ_ROWS = 16;  // output columns per block, four per wavefront

// One activation row (decode): y[n] = sum_k x[k] * (c[n, k] * s[n, g(k)] + b[n, g(k)]), per group
// acc += s * sum(c*x) + b * sum(x).  A block stages the row in LDS once; a lane takes 16 bytes of codes
// (32 int4 or 16 int8 codes, never straddling a group) per step, so a wavefront streams 1 KiB of
// contiguous weight per load.  The weight stream is software-pipelined:
// a wavefront owns four weight rows and walks K in steps of 64 * CODES; the 16-byte code
// loads (and scale / bias) of all four rows for the next step are in flight while the current
// step is multiplied, and the first step's loads are issued before x is staged (behind the requests of x itself), so the only
// exposed memory latency is the first one.  K need not fill the last step: its lanes past K read
// the row's last 16 bytes against zeros of x.
template <int BITS>
__global__ __launch_bounds__(256) void wq_gemv1_kernel(const float* x, const uint32_t* packed, const float* scales,
                                                       const float* biases, int N, int K, int gs, float* out) {
    extern __shared__ __attribute__((aligned(16))) float sx[];
    constexpr int CODES = 128 / BITS, QUADS = CODES / 4, RW = WQ_ROWS / 4;
    constexpr uint32_t MASK = (1u << BITS) - 1u;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int last_chunk = K / CODES - 1, steps = last_chunk / 64 + 1, chunks = steps * 64;  // (chunks: those of whole steps)
    const int gs_shift = 31 - __builtin_clz(gs);
    const int words_per_row = K * BITS / 32, groups_per_row = K >> gs_shift;
    const uint4* wrow[RW];
    const float* srow[RW];
    const float* brow[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        int n = blockIdx.x * WQ_ROWS + wave * RW + r;
        n = n < N ? n : N - 1;  // clamped rows are computed and dropped at the store
        wrow[r] = reinterpret_cast<const uint4*>(packed + size_t(n) * words_per_row);
        srow[r] = scales + size_t(n) * groups_per_row;
        brow[r] = biases + size_t(n) * groups_per_row;
    }
    struct Operands {
        uint4 w[RW];
        float s[RW], b[RW];
    };
    // Scales and biases of the wavefront's rows.  With at most 64 groups per row (and RW = 4) they
    // come in two wavefront-wide direct loads into LDS - 16 lanes x 16 bytes per row and array -
    // instead of two 4-byte loads per row and step: a load instruction costs the memory pipeline
    // about the same whatever it carries.  Layout: sb[wave][array][row][64].
    const bool sb_lds = RW == 4 && groups_per_row <= 64 && groups_per_row % 4 == 0 &&
                        ((reinterpret_cast<uintptr_t>(scales) | reinterpret_cast<uintptr_t>(biases)) & 15u) == 0;
    float* const sb = sx + chunks * CODES + wave * 512;
    auto fetch = [&](int step, Operands& o) {
        int L = step * 64 + lane;
        L = L < last_chunk ? L : last_chunk;
        const int g = (L * CODES) >> gs_shift;  // group sizes are powers of two
#pragma unroll
        for (int r = 0; r < RW; ++r) o.w[r] = wrow[r][L];
        if (!sb_lds) {
#pragma unroll
            for (int r = 0; r < RW; ++r) o.s[r] = srow[r][g], o.b[r] = brow[r][g];
        }
    };
    auto pin = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    Operands o0, o1;
    // Loads return in the order they were requested: the first 4096 of x, which every block finds in its L2, before the scales
    // and the weights, so that x is in LDS by the time the first codes arrive.
    constexpr int kAhead = 4;
    float4 xv[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
        const int i = (u * 256 + tid) * 4;
        xv[u] = *reinterpret_cast<const float4*>(x + (i < K ? i : 0));
    }
    pin();
    if (sb_lds) {
        const int r = lane >> 4;
        int part = (lane & 15) * 4;
        part = part < groups_per_row ? part : groups_per_row - 4;  // lanes past the row's groups repeat its last four
        typedef __attribute__((address_space(1))) void* gptr;
        typedef __attribute__((address_space(3))) void* lptr;
        __builtin_amdgcn_global_load_lds((gptr)(srow[r % RW] + part), (lptr)(sb), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((gptr)(brow[r % RW] + part), (lptr)(sb + 256), 16, 0, 0);
    }
    pin();
    fetch(0, o0);
    pin();
    // (in LDS the lanes of a wavefront read consecutive 16-byte slots: lane L of a step, quad j of its chunk)
    auto stage = [&](int i, float4 v) {
        const int L = i / CODES, j = (i % CODES) / 4;
        *reinterpret_cast<float4*>(sx + (j * chunks + L) * 4) = v;
    };
    const float4 zero{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kAhead; ++u) {
        const int i = (u * 256 + tid) * 4;
        if (i < chunks * CODES) stage(i, i < K ? xv[u] : zero);
    }
    for (int i = (kAhead * 256 + tid) * 4; i < chunks * CODES; i += 256 * 4)
        stage(i, i < K ? *reinterpret_cast<const float4*>(x + i) : zero);
    // the direct loads are older than the RW weight loads, which may still be on their way
    static_assert(RW == 4, "the count below");
    __builtin_amdgcn_s_waitcnt(0x0074 | (0xF << 8));  // vmcnt(4)
    lds_barrier();
    float acc[RW];
#pragma unroll
    for (int r = 0; r < RW; ++r) acc[r] = 0.0f;
    auto compute = [&](int step, Operands& o) {
        const int L = step * 64 + lane;
        if (sb_lds) {
            const int g = ((L < last_chunk ? L : last_chunk) * CODES) >> gs_shift;
#pragma unroll
            for (int r = 0; r < RW; ++r) o.s[r] = sb[r * 64 + g], o.b[r] = sb[256 + r * 64 + g];
        }
        float dot[RW], sum = 0.0f;
#pragma unroll
        for (int r = 0; r < RW; ++r) dot[r] = 0.0f;
#pragma unroll
        for (int quad = 0; quad < QUADS; ++quad) {
            const float4 xv = *reinterpret_cast<const float4*>(sx + (quad * chunks + L) * 4);
            sum += (xv.x + xv.y) + (xv.z + xv.w);
#pragma unroll
            for (int r = 0; r < RW; ++r) {
                const uint32_t words[4] = {o.w[r].x, o.w[r].y, o.w[r].z, o.w[r].w};
                float c[4];
                if (BITS == 4) {
                    // the even nibbles of a word as the bytes of `lo`, the odd ones as the bytes of `hi`
                    // (three instructions per eight codes), then one byte-to-float conversion per code:
                    // five instructions less per word than a bit-field extract and a conversion per code
                    const uint32_t word = words[quad >> 1];
                    const uint32_t lo = word & 0x0f0f0f0fu, hi = (word >> 4) & 0x0f0f0f0fu;
                    const int sh = (quad & 1) * 16;  // a constant once the quad loop is unrolled
                    c[0] = float((lo >> sh) & 0xffu), c[1] = float((hi >> sh) & 0xffu);
                    c[2] = float((lo >> (sh + 8)) & 0xffu), c[3] = float((hi >> (sh + 8)) & 0xffu);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int j = quad * 4 + e;  // code index inside the 16-byte load
                        c[e] = float((words[j * BITS / 32] >> ((j * BITS) % 32)) & MASK);
                    }
                }
                // fused multiply-adds by name (contraction is off for this library): the decode
                // loop is bound by vector instructions, not by memory
                dot[r] = __builtin_fmaf(c[0], xv.x, dot[r]);
                dot[r] = __builtin_fmaf(c[1], xv.y, dot[r]);
                dot[r] = __builtin_fmaf(c[2], xv.z, dot[r]);
                dot[r] = __builtin_fmaf(c[3], xv.w, dot[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < RW; ++r) acc[r] += o.s[r] * dot[r] + o.b[r] * sum;
    };
    const int last = steps - 1;
    int step = 0;
    for (;;) {
        fetch(step + 1 < steps ? step + 1 : last, o1);
        pin();
        compute(step, o0);
        pin();
        if (++step >= steps) break;
        fetch(step + 1 < steps ? step + 1 : last, o0);
        pin();
        compute(step, o1);
        pin();
        if (++step >= steps) break;
    }
#pragma unroll
    for (int r = 0; r < RW; ++r) {
        float v = acc[r];
#pragma unroll
        for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d, 64);
        const int n = blockIdx.x * WQ_ROWS + wave * RW + r;
        if (lane == 0 && n < N) out[n] = v;
    }
}

constexpr int kGemv1MaxLds = 160 * 1024;
// x of whole steps, then scales / biases per wavefront
size_t wq_gemv1_lds(int K, int bits) {
    const size_t step = 64 * 128 / bits;
    return (size_t(K) + step - 1) / step * step * sizeof(float) + 4 * 512 * sizeof(float);
}

template <int BITS>
int launch_gemv1(const float* x, const uint32_t* packed, const float* scales, const float* biases, int N, int K,
                 int gs, float* out, hipStream_t st) {
    const size_t smem = wq_gemv1_lds(K, BITS);
    static DeviceOnce once;
    if (const int rc = allow_dynamic_lds(once, reinterpret_cast<const void*>(wq_gemv1_kernel<BITS>), kGemv1MaxLds)) return rc;
    hipLaunchKernelGGL((wq_gemv1_kernel<BITS>), dim3(unsigned((N + WQ_ROWS - 1) / WQ_ROWS)), dim3(256), smem, st, x,
                       packed, scales, biases, N, K, gs, out);
    LQ_CHECK_LAUNCH("wq_gemv1");
    return LQ_OK;
}

// Small-batch matmul on the matrix cores (16 activation rows per block row; up to about a hundred rows, more
// where the weight is small: wq_gemm_beats_small_batch).
//
// y[m, n] = sum over groups g of  s[n, g] * (sum_{k in g} c[n, k] x[m, k])  +  b[n, g] * (sum_{k in g} x[m, k]):
// the inner sums run on v_mfma_f32_16x16x32_bf16 with the codes themselves as one operand -
// a code c enters exactly as c - 2^(bits-1), or 128 + c (wq_codes), which goes into the bias term - and x as the
// other, split into three bfloat16 parts x = hi + mid + lo (exact: 8 + 8 + 8 significant
// bits, wq_split3x2), one MFMA each.  Products are exact and accumulate in float32, so nothing of x or
// of the weight is rounded before the sums.
//
// Operand layout of the instruction: lane = (row % 16) + 16 * quarter holds eight k of its
// row, quarter q the k slots 8q .. 8q+7 of the instruction's 32.  x is the A operand (rows
// m) and the codes the B operand (rows n), so an accumulator lane holds column n = lane % 16
// and rows m = 4 * quarter + 0..3, and s, b are one value per lane.
//
// A lane streams its weight row with 16-byte loads (32 int4 / 16 int8 codes; the four
// quarters of a row take consecutive loads: a "window" of 128 / 64 k, 1 KiB per wavefront
// load over 16 rows).  An instruction must stay inside one group, because the scale is
// applied to its sum.  With group_size >= the window that holds as loaded (register j of
// every quarter feeds instruction j).  With two groups per window the registers are
// exchanged between lane halves (v_permlane32_swap: instructions 0, 1 then hold the first
// two quarters' k, instructions 2, 3 the last two), with four groups the 4 x 4 (register,
// quarter) matrix is transposed (v_permlane32_swap + v_permlane16_swap), so instruction i
// holds the k of quarter i.  Which k a slot of an instruction ends up with does not matter
// as long as x follows: the block writes the three parts of its x range into LDS in exactly
// that order.  The threads that split x also add it up per group segment, in float32
// pair by pair, and leave the sums in LDS (as one more accumulator tile against a row of ones, which the calls with 128 + c
// keep, they take a third of the matrix instructions).
//
// Every block needs the x of its k range next to its weights (64 bytes of x per k against
// rows / 2 or rows bytes of codes), and every block converts it again.  So a block takes
// many rows (one to three 16-row tiles per wavefront, wq_form) and a short k range (512 or 1024),
// keeps that range's fragments in LDS for all its wavefronts, and requests its first weights
// when it starts.  The k ranges of a row tile are blocks of their own (grid.y); each
// writes its partial sums to a slab, and the last one to arrive (an arrival counter per row
// tile, reset by that block) adds the slabs in index order - the result does not depend on
// the order of arrival - and stores.  One launch, no workspace besides the slabs.
//
// Handing slabs on is a third of the time where the weight is a few ten MB (16 x 11008 x 4096 int8, 384 rows x 512 k per block: 4.4 us
// until the first window, 6.8 us for all of them, 2.3 us for the slab to be written through, 4.1 us for the last block of a row tile
// to fetch eight).  So a block may also take 1024 k in four parts, four of its sixteen wavefronts for each, and add the parts in
// LDS: half the slabs, and four wavefronts per SIMD to wait with (20.1 -> 18.4 us; int4 18.9 -> 16.8, 16 x 1033 x 4608 int8
// 9.8 -> 9.2, 4 x 1024 x 1024 int8 8.3 -> 7.0).  All of K in a block needs no slabs, but every block then fetches and splits all
// of x: 18.9 us, 18.3, 11.0, 5.3.

// a block of one part is eight wavefronts with all of its k range, one of four sixteen with a quarter each
constexpr int wq_waves(int parts) { return parts == 4 ? 16 : 8; }
constexpr int wq_slice(int parts) { return parts == 4 ? 1024 : 512; }  // k
// weight rows, with `rb` tiles of 16 per wavefront
constexpr int wq_rows(int rb, int parts) { return wq_waves(parts) / parts * rb * 16; }
// LDS: 48 or 96 KiB of x fragments, the sums of x per group segment, the tables of the rows
constexpr size_t wq_lds_bytes(int rb, int parts, int gs) {
    return size_t(wq_slice(parts) / 32) * 3 * 64 * 16 + (wq_slice(parts) / 32) * 16 * 4 +
           size_t(2) * wq_rows(rb, parts) * (wq_slice(parts) / gs + 1) * 4;
}

// Where the A fragment of row m, lane quarter qd of instruction block `blk` sits among the block's
// 64 16-byte slots.  The threads of a wavefront that write the fragments share one m and differ in
// (block, quarter): with the plain slot m + 16 qd they would all hit the same four banks (a
// 64-way conflict: the writes took a tenth of the kernel); rotating m by 4 qd + blk spreads them
// evenly over the 16 bank groups.  A bijection within the block, so the reads of a whole block
// stay conflict-free.
__device__ __forceinline__ int wq_x_slot(int m, int qd, int blk) { return ((m + 4 * qd + blk) & 15) + 16 * qd; }

// lanes of a group of N neighbours (4, 8 or 16): everyone gets the sum
template <int N>
__device__ __forceinline__ float wq_neighbour_sum(float v) {
    auto moved = [&](auto ctrl) { return __uint_as_float(unsigned(__builtin_amdgcn_mov_dpp(int(__float_as_uint(v)), ctrl(), 0xf, 0xf, true))); };
    v += moved(std::integral_constant<int, 0xb1>());  // the other of the pair
    v += moved(std::integral_constant<int, 0x4e>());  // the other pair of the quad
    if (N >= 8) v += moved(std::integral_constant<int, 0x141>());   // the other quad (lanes 0..7 mirrored)
    if (N >= 16) v += moved(std::integral_constant<int, 0x140>());  // the other eight (lanes 0..15 mirrored)
    return v;
}

template <int BITS, int SW, int RB, int KP, bool PATTERN>
__global__ __launch_bounds__(64 * wq_waves(KP)) __attribute__((amdgpu_waves_per_eu((RB <= 2 && KP == 1) || KP == 4 ? 4 : 2, (RB <= 2 && KP == 1) || KP == 4 ? 4 : 2))) void wq_mfma_kernel(
    const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N, int K,
    int gs_shift, float* out, float* slabs, int* counters) {
    using G = WqGeom<BITS>;
    constexpr int CODES = G::CODES, WK = G::WK, NI = G::NI;
    constexpr int GW = 1 << SW, SEG = WK / GW;  // group segments per window and their length
    constexpr int IPS = NI / GW;                // instructions per segment
    constexpr int THREADS = 64 * wq_waves(KP), SLICE = wq_slice(KP);
    constexpr int WAVES = wq_waves(KP) / KP, WPW = SLICE / KP / WK;  // wavefronts of a k range; windows of a wavefront: 4 or 8
    constexpr int WPS = KP * WPW;                               // windows of the block
    constexpr int kWqRows = wq_rows(RB, KP);
    constexpr int UNITS = WPS * NI * 64;                    // (window, instruction, lane) triples of the block's x
    constexpr int AHEAD = RB == 1 || WPW < 2 ? WPW : 2;                // windows of weights a wavefront has requested and not used
    static_assert(IPS >= 1, "a segment is at least one instruction");
    static_assert(UNITS % THREADS == 0, "");
    // Dynamic LDS: the x fragments of the block's windows ([window][instruction][part][lane],
    // 16 bytes each), then the block's rows of scales and of biases for the groups of those
    // windows - each row padded by one float: lanes of a quarter read 16 different rows at the
    // same group, and the odd stride spreads them over the banks.
    extern __shared__ __attribute__((aligned(16))) uint4 wq_lds[];
    __shared__ int s_arrived;
    // the wavefront index as a scalar, so that branches on it are uniform
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, q = lane >> 4;
    // the k ranges of a row tile are neighbours in the grid: they are dispatched together, so the pieces of a
    // weight row (one per k range) are requested at about the same time
    const int tile = blockIdx.y, ks = blockIdx.x, mb = blockIdx.z, slices = gridDim.x;
    // the wavefront's columns and its part of the k range (one part: a constant, or its loops and stores test for it: 33 x 14336
    // x 4096 int4 of 64 43.6 us, 42.0 with the constant, and 64 x 11008 x 4096 of 128 43.2 and 42.2)
    const int wc = KP == 1 ? wave : wave % WAVES, part = KP == 1 ? 0 : wave / WAVES;
    const int n_base = tile * kWqRows + wc * (RB * 16), m0 = mb * 16;
    const int words_per_row = K * BITS / 32, groups_per_row = K >> gs_shift;
    const int windows = (K + WK - 1) / WK;  // the last one may be partial (K is a multiple of 32: whole 16-byte loads)
    const int w0 = ks * WPS;
    const int nw = windows - w0 < WPS ? windows - w0 : WPS;  // at least 1: the host sizes grid.y so
    const int w_first = part * WPW, w_end = nw < w_first + WPW ? nw : w_first + WPW;  // the wavefront's (none in a short last range)
    // groups of this block's windows, and the row stride of the tables
    const int g0 = (w0 * WK) >> gs_shift;
    const int k_end = (w0 + nw) * WK < K ? (w0 + nw) * WK : K;
    const int ng = ((k_end - 1) >> gs_shift) - g0 + 1;
    const int gmax = SLICE >> gs_shift, gp = (gmax < 1 ? 1 : gmax) + 1;

    // Every global load of the block is requested before anything is consumed, in the order of
    // consumption (the wait counter retires loads in order): the scale / bias tables (short, from
    // the L2), x, the weights.
    // Tables: kWqRows rows x gcap slots (gcap = the groups of a full k range of 512 or 1024: 4, 8, 16 or 32), four slots per
    // 16-byte load where the rows allow it (a dword per lane costs the vector cache as many cycles
    // as 16 bytes per lane do).
    constexpr int kTabVec = (kWqRows * (SLICE / 32) + 4 * THREADS - 1) / 4 / THREADS;  // 16-byte loads per thread and table, in groups of 32
    const int gcap = gp - 1, gsh = 31 - __builtin_clz(unsigned(gcap));  // a power of two: shifts, no division
    const bool tab_vec = ng == gcap && (groups_per_row & 3) == 0 && aligned16(scales) && aligned16(biases);
    // (No branch between these requests and none that gives a register another value: the compiler would wait for each load
    // where the two meet - a memory trip per table and row of x before the first weight was asked for.)
    float4 tab_s[kTabVec], tab_b[kTabVec];
    const int row_first = tile * kWqRows;
    auto table_at = [&](int i) {
        const int n = row_first + (i >> gsh) < N ? row_first + (i >> gsh) : N - 1;
        return size_t(n) * groups_per_row + g0 + (i & (gcap - 1));
    };
    if (tab_vec) {
#pragma unroll
        for (int u = 0; u < kTabVec; ++u) {
            const int i = (threadIdx.x + u * THREADS) * 4;
            const size_t at = table_at(i < kWqRows * gcap ? i : 0);
            tab_s[u] = *reinterpret_cast<const float4*>(scales + at);
            tab_b[u] = *reinterpret_cast<const float4*>(biases + at);
        }
    }
    // x of the block's windows: a thread takes eight consecutive k of one row (a wavefront reads
    // 2 KiB of a row)
    constexpr int OCTS = SLICE / 8;  // per row
    static_assert(16 * OCTS == UNITS, "");
    float4 raw[UNITS / THREADS][2];
#pragma unroll
    for (int u = 0; u < UNITS / THREADS; ++u) {
        const int unit = u * THREADS + threadIdx.x, m = m0 + unit / OCTS, kl = (unit % OCTS) * 8;
        // (K is a multiple of 32; what lies past M and K becomes zero below)
        const float* src = x + size_t(m < M ? m : M - 1) * K + (w0 * WK + kl < k_end ? w0 * WK + kl : 0);
        raw[u][0] = *reinterpret_cast<const float4*>(src);
        raw[u][1] = *reinterpret_cast<const float4*>(src + 4);
    }
    // The weights of the first windows are requested now (of all of them where a wavefront has one tile; more tiles keep
    // enough bytes in flight with two, in a loop of a third of the code).  For the request a lane takes quarter lane % 4 of row lane / 4 - four neighbouring lanes read 64
    // contiguous bytes, where the operand layout (row lane % 16, quarter lane / 16) would make
    // every lane a cache access of its own -; a lane permutation below puts each 16 bytes
    // where the instruction wants them.
    const uint32_t* row[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) {
        int n = n_base + rb * 16 + (lane >> 2);
        n = n < N ? n : N - 1;  // clamped rows are computed and dropped at the store
        row[rb] = packed + size_t(n) * words_per_row + (lane & 3) * (CODES * BITS / 32);
    }
    auto fetch = [&](uint4 (&w)[RB], int wi) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            // past K every lane reads the same 16 bytes: one cache line, dropped later or multiplied by zeros of x
            w[rb] = *reinterpret_cast<const uint4*>(
                (w0 + wi) * WK + (lane & 3) * CODES < k_end ? row[rb] + (w0 + wi) * (WK * BITS / 32) : packed);
    };
    uint4 ahead[AHEAD][RB];
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(ahead[j], w_first + j);
    // The tables go to LDS, then x, split and laid out as fragments by the block itself: a thread
    // finds the (instruction, quarter) that holds its eight k - the exchange of registers is its
    // own inverse.
    uint4* x_lds = wq_lds;
    float* sum_lds = reinterpret_cast<float*>(wq_lds + WPS * NI * 3 * 64);  // of x: [segment][row]
    float* s_lds = sum_lds + SLICE / 32 * 16;
    float* b_lds = s_lds + kWqRows * gp;
    if (tab_vec) {
#pragma unroll
        for (int u = 0; u < kTabVec; ++u) {
            const int i = (threadIdx.x + u * THREADS) * 4, row = i >> gsh, g = i & (gcap - 1);
            if (i < kWqRows * gcap) {
                float* sd = s_lds + row * gp + g;
                float* bd = b_lds + row * gp + g;
                sd[0] = tab_s[u].x, sd[1] = tab_s[u].y, sd[2] = tab_s[u].z, sd[3] = tab_s[u].w;
                bd[0] = tab_b[u].x, bd[1] = tab_b[u].y, bd[2] = tab_b[u].z, bd[3] = tab_b[u].w;
            }
        }
    } else {  // the last k range of a K that is not a multiple of the block's, or rows that vectors cannot take
        for (int i = threadIdx.x; i < kWqRows * gcap; i += THREADS) {
            const int row = i >> gsh, g = i & (gcap - 1);
            // (zeros past the row's groups: a partial window's segments past K read them)
            s_lds[row * gp + g] = g < ng ? scales[table_at(i)] : 0.0f;
            b_lds[row * gp + g] = g < ng ? biases[table_at(i)] : 0.0f;
        }
    }
    {
#pragma unroll
        for (int u = 0; u < UNITS / THREADS; ++u) {
            const int unit = u * THREADS + threadIdx.x, ml = unit / OCTS, kl = (unit % OCTS) * 8;
            const int wi = kl / WK, off = kl % WK, qs = off / CODES, js = (off % CODES) / (32 / BITS);
            int qd, rho;
            wq_source(SW, js, qs, qd, rho);
            const int i = BITS == 4 ? rho : rho / 2;
            float v[8] = {raw[u][0].x, raw[u][0].y, raw[u][0].z, raw[u][0].w,
                          raw[u][1].x, raw[u][1].y, raw[u][1].z, raw[u][1].w};
            const bool there = m0 + ml < M && w0 * WK + kl < k_end;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = there ? v[e] : 0.0f;
            // a wavefront has one row of x: the segments' sums, in float32, pair by pair
            if constexpr (!PATTERN) {
                const float sum = wq_neighbour_sum<SEG / 8>(((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7])));
                if (lane % (SEG / 8) == 0) sum_lds[kl / SEG * 16 + ml] = sum;
            }
            uint32_t d3[3][4];
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                // slots 2d, 2d+1: the 4-bit decode pairs nibble d with nibble d + 4
                const float e0 = BITS == 4 ? v[d] : v[2 * d], e1 = BITS == 4 ? v[d + 4] : v[2 * d + 1];
                wq_split3x2(e0, e1, d3[0][d], d3[1][d], d3[2][d]);
            }
            if (wi < nw) {
#pragma unroll
                for (int p = 0; p < 3; ++p)
                    x_lds[((wi * NI + i) * 3 + p) * 64 + wq_x_slot(ml, qd, wi * NI + i)] = uint4{d3[p][0], d3[p][1], d3[p][2], d3[p][3]};
            }
        }
    }
    lds_barrier();  // (the weights are still on their way)

    // (one part of one tile, which has all its windows at once: four sums, a quarter as long; error of 51 x 92 x 3072 int8 against
    // float64 1.33e-7 of the result with one sum, 1.25e-7 in four parts, 1.24e-7 so.  128 + c have more to round than that: one sum.)
    constexpr int SUMS = KP == 1 && RB == 1 && !PATTERN ? 4 : 1;
    v4f ys[SUMS][RB];
#pragma unroll
    for (int i = 0; i < SUMS; ++i)
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) ys[i][rb] = v4f{0.f, 0.f, 0.f, 0.f};
    const int row_in_tile = wc * (RB * 16) + r;
    auto window = [&](int wi, const uint4 (&wv)[RB], v4f (&y)[RB]) {
        uint32_t wd[RB][4];
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            // lane (row r, quarter q) takes what lane 4 r + q loaded
            const int from = (4 * r + q) * 4;
            wd[rb][0] = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(wv[rb].x)));
            wd[rb][1] = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(wv[rb].y)));
            wd[rb][2] = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(wv[rb].z)));
            wd[rb][3] = uint32_t(__builtin_amdgcn_ds_bpermute(from, int(wv[rb].w)));
            wq_exchange<SW>(wd[rb]);
        }
#pragma unroll
        for (int e = 0; e < GW; ++e) {
            const int g = (((w0 + wi) * WK + e * SEG) >> gs_shift) - g0;
            // (PATTERN: acc[RB] is the segment's sum of x, from the same fragments against ones: what of its rounding the
            // codes' sums share, the bias takes out again)
            constexpr int ACC = PATTERN ? RB + 1 : RB;
            const uint4 ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // eight times 1.0
            v4f acc[ACC];
#pragma unroll
            for (int rb = 0; rb < ACC; ++rb) acc[rb] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int ii = 0; ii < IPS; ++ii) {
                const int i = e * IPS + ii;
                uint4 cf[RB];
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) cf[rb] = wq_codes<BITS, PATTERN>(wd[rb], i);
#pragma unroll
                for (int p = 0; p < 3; ++p) {
                    const v8bf xf = __builtin_bit_cast(v8bf, x_lds[((wi * NI + i) * 3 + p) * 64 + wq_x_slot(lane & 15, lane >> 4, wi * NI + i)]);
#pragma unroll
                    for (int rb = 0; rb < RB; ++rb)
                        acc[rb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, __builtin_bit_cast(v8bf, cf[rb]),
                                                                          acc[rb], 0, 0, 0);
                    if constexpr (PATTERN)
                        acc[RB] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf, __builtin_bit_cast(v8bf, ones), acc[RB], 0, 0, 0);
                }
            }
            // the sums of the lane's rows m
            const v4f sums = PATTERN ? acc[ACC - 1] : *reinterpret_cast<const v4f*>(sum_lds + (wi * GW + e) * 16 + 4 * q);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
                const float sc = s_lds[(row_in_tile + rb * 16) * gp + g];
                const float bi = b_lds[(row_in_tile + rb * 16) * gp + g];
                if constexpr (PATTERN) {
                    y[rb] = y[rb] + (acc[rb] * sc + sums * (bi - 128.0f * sc));
                } else {
                    // the codes entered as (c + centre) / unit
                    const float bz = bi - float(kWqCentre<BITS>) * sc;
#pragma unroll
                    for (int t = 0; t < 4; ++t)
                        y[rb][t] = __builtin_fmaf(acc[rb][t], kWqUnit<BITS> * sc, __builtin_fmaf(sums[t], bz, y[rb][t]));
                }
            }
        }
    };
#pragma unroll 1
    for (int w = w_first; w < w_end; w += AHEAD)
#pragma unroll
        for (int j = 0; j < AHEAD; ++j) {
            if (w + j < w_end) window(w + j, ahead[j], ys[j % SUMS]);
            if (AHEAD < WPW) fetch(ahead[j], w + j + AHEAD);
        }
    v4f(&y)[RB] = ys[0];
    if constexpr (SUMS == 4) y[0] = (ys[0][0] + ys[1][0]) + (ys[2][0] + ys[3][0]);
    if constexpr (KP > 1) {  // the parts of the range meet where x was
        v4f* const parts = reinterpret_cast<v4f*>(wq_lds) + lane;
        lds_barrier();
        if (part > 0) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) parts[((part - 1) * WAVES + wc) * (RB * 64) + rb * 64] = y[rb];
        }
        lds_barrier();
        if (part == 0) {
#pragma unroll
            for (int p = 1; p < KP; ++p)
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) y[rb] = y[rb] + parts[((p - 1) * WAVES + wc) * (RB * 64) + rb * 64];
        }
    }

    // accumulator element t of a lane: row m = 4 * quarter + t, column n = lane % 16
    auto store_out = [&](const v4f (&v)[RB]) {
#pragma unroll
        for (int rb = 0; rb < RB; ++rb) {
            const int n = n_base + rb * 16 + r;
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int mm = m0 + 4 * q + t;
                if (n < N && mm < M) out[size_t(mm) * N + n] = v[rb][t];
            }
        }
    };
    if (slices == 1) {
        if (part == 0) store_out(y);
        return;
    }
    // slab of (row tile, k range): [wavefront][tile of 16 rows][lane] x 16 bytes, written through to
    // device scope; then the arrival counter of the row tile
    constexpr unsigned kScopeDevice = 16;  // "sc1" cache-policy bit of buffer accesses
    constexpr unsigned kSlabBytes = WAVES * RB * 64 * 16;
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    const size_t tile_index = size_t(mb) * gridDim.y + tile;
    float* first_slab = slabs + tile_index * slices * (kSlabBytes / 4);
    const unsigned my_off = unsigned((wc * RB) * 64 + lane) * 16;
    if (part == 0) {
        const __amdgpu_buffer_rsrc_t mine =
            __builtin_amdgcn_make_buffer_rsrc(first_slab + size_t(ks) * (kSlabBytes / 4), 0, kSlabBytes, 0x00020000);
#pragma unroll
        for (int rb = 0; rb < RB; ++rb)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, y[rb]), mine, my_off + unsigned(rb * 64 * 16), 0,
                                                   kScopeDevice);
    }
    __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0): this wavefront's partial sums have been written through
    __syncthreads();                      // ... and so have the other wavefronts'
    if (threadIdx.x == 0)
        s_arrived = __hip_atomic_fetch_add(&counters[tile_index], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_arrived) != slices - 1 || part > 0) return;
    v4f total[RB];
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) total[rb] = v4f{0.f, 0.f, 0.f, 0.f};
    // eight slabs are requested together (one memory round trip, not eight); a slot past the
    // last slab re-reads the last one and is not added, so that the loads stay unconditional
    constexpr int kBatch = 8;
    for (int k0 = 0; k0 < slices; k0 += kBatch) {
        v4u part[kBatch][RB];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int k = k0 + j < slices ? k0 + j : slices - 1;
            const __amdgpu_buffer_rsrc_t other =
                __builtin_amdgcn_make_buffer_rsrc(first_slab + size_t(k) * (kSlabBytes / 4), 0, kSlabBytes, 0x00020000);
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
                part[j][rb] = __builtin_amdgcn_raw_buffer_load_b128(other, my_off + unsigned(rb * 64 * 16), 0, kScopeDevice);
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j)
            if (k0 + j < slices) {
#pragma unroll
                for (int rb = 0; rb < RB; ++rb) total[rb] = total[rb] + __builtin_bit_cast(v4f, part[j][rb]);
            }
    }
    store_out(total);
    if (threadIdx.x == 0) counters[tile_index] = 0;  // ready for the next launch
}


// Tiles of 16 weight rows per wavefront and parts of a block's k range.  Four parts of 1024 k (a CU per block) with as many
// tiles as give every block a CU at once; where the blocks are too many for that, one part of 512 k, of which a CU
// has two blocks, one starting or adding slabs while the other streams: with two tiles per wavefront, in groups of 32 one (the tables of
// two do not leave a CU room for a second block).  One part of one tile is also the better one where K is no multiple of 1024 and
// half of the second range would be empty, and where K is short.
// us of 1 / 2 / 3 tiles of four parts, then of one part of one and of two: groups of 64, 128 alike: 16 x 11008 x 4096 int8 (688 / 344 / 232
// blocks) 25.5 / 23.7 / 17.9, - / 19.7 (344); the same int4 22.4 / 21.0 / 15.9, - / 19.3; 33 x 4096 x 4096 int4 (768 / 384 / 264) 21.8 / 19.9 / 21.9,
// - / 17.7 (384); 33 x 4096 x 11008 int4 (2112 / 1056 / 726) 61.4 / 49.4 / 45.8, - / 39.8 (1056); 38 x 2767 x 1536 int4 (264 / 132 / 90) 14.2 / 9.9 /
// 12.1, 8.7 (198) / 10.9; 31 x 10765 x 320 int8 (338 / 170 / 114) 9.5 / 7.1 / 8.4, 6.0 (170) / 7.5; 4 x 3092 x 3904 int8 (196 / 100 / 68) 9.4 / 11.5 /
// 14.2, 10.0 (200) / 12.8; 51 x 92 x 3072 int8 (24 / 12 / 12) 8.5 / 10.7 / 13.1, 8.0 (24) / 10.9;
// groups of 32: 33 x 4096 x 4096 int4 (768 / 384 / 264) 23.3 / 21.8 / 24.5, 19.5 (768) / 23.2 (384); 33 x 8192 x 2048 int8 24.8 / 22.3 / 28.8, 20.1
// / 23.7; 64 x 8192 x 8192 int4 (4096 / 2048 / 1376) 111 / 83.5 / 84.0, 83.5 (4096) / 97.9; 33 x 3529 x 1280 int8 (336 / 168 / 114) 16.0 / 11.6 / 15.5,
// 9.3 (252) / 12.7; 62 x 3817 x 3360 int4 34.1 / 27.1 / 34.5, 28.5 / 33.8.
// The costs below follow 1850 shapes timed in every form (2 to 64 rows, and more where this kernel takes them; 64 to 16384 columns, K
// from 32 to 12288), in us behind what all have in common: what they choose is the fastest or within 3 % but for 49 shapes, 0.3 % off
// on average and 13 % at most.
struct WqForm {
    int tiles, parts;
};
WqForm wq_form(int M, int N, int K, int gs) {
    auto ranges = [&](int kp) { return (K + wq_slice(kp) - 1) / wq_slice(kp); };
    auto blocks = [&](int rb, int kp) { return long((M + 15) / 16) * ((N + wq_rows(rb, kp) - 1) / wq_rows(rb, kp)) * ranges(kp); };
    // handing slabs on: the last block fetches eight at a time
    auto slabs = [&](int kp) { return ranges(kp) == 1 ? 0.0 : 1.5 + 1.5 * ((ranges(kp) + 7) / 8); };
    WqForm best{1, 4};
    double least = 1e30;
    auto take = [&](int rb, int kp, double cost) {
        if (cost < least) least = cost, best = WqForm{rb, kp};
    };
    // one part: alone on a CU, or two blocks at once, of which the last round of 512 may leave one
    const double short1 = 0.35 + 0.65 * (K < 512 ? K : 512) / 512;
    auto one_part = [&](int rb, double alone, double round) {
        const long n = blocks(rb, 1);
        const double last = n > 512 && n % 512 > 0 && n % 512 <= 256 ? 2.4 : 0.0;
        take(rb, 1, (n <= 256 ? alone : round * (n > 512 ? double(n) / 512 : 1.0) + last) * short1 + slabs(1));
    };
    one_part(1, gs == 32 ? 6.8 : 6.3, gs == 32 ? 9.3 : 10.1);
    if (gs > 32) one_part(2, ranges(1) == 1 ? 9.5 : 11.0, 15.3);
    // four parts: rounds of 256 blocks, and what each range of K adds to one
    constexpr double kRound[4] = {0.0, 6.3, 9.0, 11.8}, kRange[4] = {0.0, 0.08, 0.06, 0.2};
    const double short4 = 0.62 + 0.38 * (K < 1024 ? K : 1024) / 1024;
    for (int rb = 1; rb <= 3; ++rb)
        take(rb, 4, double((blocks(rb, 4) + 255) / 256) * (kRound[rb] * short4 + kRange[rb] * ranges(4)) + slabs(4));
    return best;
}

template <int BITS, int SW, int RB, int KP, bool PATTERN>
int launch_wq_mfma_form(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N,
                        int K, int gs, float* out, hipStream_t st) {
    using G = WqGeom<BITS>;
    constexpr int WPS = wq_slice(KP) / G::WK;
    const int mblocks = (M + 15) / 16, windows = (K + G::WK - 1) / G::WK;
    const int tiles = (N + wq_rows(RB, KP) - 1) / wq_rows(RB, KP), slices = (windows + WPS - 1) / WPS;
    static DeviceOnce attr_once;
    if (const int rc = allow_dynamic_lds(attr_once, reinterpret_cast<const void*>(wq_mfma_kernel<BITS, SW, RB, KP, PATTERN>),
                                         int(wq_lds_bytes(RB, KP, 32))))
        return rc;
    SkScratch sk;
    const auto lock = scratch_lock(st);
    if (slices > 1) {
        const int rc = sk_scratch(size_t(mblocks) * tiles, size_t(mblocks) * tiles * slices * (wq_waves(KP) / KP * RB * 64 * 16), st, &sk);
        if (rc) return rc;
    }
    hipLaunchKernelGGL((wq_mfma_kernel<BITS, SW, RB, KP, PATTERN>), dim3(unsigned(slices), unsigned(tiles), unsigned(mblocks)), dim3(64 * wq_waves(KP)),
                       wq_lds_bytes(RB, KP, gs), st, x, packed, scales, biases, M, N, K, 31 - __builtin_clz(unsigned(gs)), out,
                       reinterpret_cast<float*>(sk.slabs), sk.counters);
    LQ_CHECK_LAUNCH("wq_mfma");
    return LQ_OK;
}

template <int BITS>
int launch_wq_mfma(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N,
                   int K, int gs, float* out, hipStream_t st) {
    const int sw = wq_swap_mode(BITS, gs);
    const WqForm form = wq_form(M, N, K, gs);
    const bool pattern = BITS == 4 && M > 1 && M <= 64 && K % WqGeom<BITS>::WK == 0;
#define LQ_WQ_FORM(SWM, RBS, KPS)                                                                                            \
    if (sw == SWM && form.tiles == RBS && form.parts == KPS)                                                                 \
        return pattern ? launch_wq_mfma_form<BITS, SWM, RBS, KPS, BITS == 4>(x, packed, scales, biases, M, N, K, gs, out, st) \
                       : launch_wq_mfma_form<BITS, SWM, RBS, KPS, false>(x, packed, scales, biases, M, N, K, gs, out, st)
#define LQ_WQ_FORMS(SWM) LQ_WQ_FORM(SWM, 1, 1); LQ_WQ_FORM(SWM, 1, 4); LQ_WQ_FORM(SWM, 2, 4); LQ_WQ_FORM(SWM, 3, 4)
    LQ_WQ_FORMS(0);
    LQ_WQ_FORM(0, 2, 1);
    LQ_WQ_FORMS(1);
    if constexpr (BITS == 4) {  // (the last swap mode of either width: groups of 32)
        LQ_WQ_FORM(1, 2, 1);
        LQ_WQ_FORMS(2);
    }
#undef LQ_WQ_FORMS
#undef LQ_WQ_FORM
    return fail(LQ_ERR_VALUE, "wq_matmul: group_size %d, bits %d", gs, BITS);
}

int check_group(const char* who, int K, int gs, int bits) {
    LQ_REQUIRE(bits == 4 || bits == 8, LQ_ERR_VALUE, "%s: bits must be 4 or 8 (got %d)", who, bits);
    LQ_REQUIRE(gs == 32 || gs == 64 || gs == 128, LQ_ERR_VALUE, "%s: group_size must be 32, 64 or 128 (got %d)", who,
               gs);
    LQ_REQUIRE(K > 0 && K % gs == 0, LQ_ERR_SHAPE, "%s: the quantized axis (%d) must be a multiple of group_size %d",
               who, K, gs);
    return LQ_OK;
}

}  // namespace

extern "C" {

int lq_wq_quantize(const float* w, int N, int K, int group_size, int bits, uint32_t* packed, float* scales,
                   float* biases, lq_stream stream) {
    int rc = check_group("wq_quantize", K, group_size, bits);
    if (rc) return rc;
    LQ_REQUIRE(N >= 0, LQ_ERR_SHAPE, "wq_quantize: negative row count");
    if (N == 0) return LQ_OK;
    LQ_REQUIRE(w && packed && scales && biases, LQ_ERR_VALUE, "wq_quantize: NULL pointer");
    const size_t groups = size_t(N) * (K / group_size);
    LQ_REQUIRE((groups + 3) / 4 < 0x7fffffffull, LQ_ERR_SHAPE, "wq_quantize: tensor too large");
    hipLaunchKernelGGL(wq_quantize_kernel, dim3(unsigned((groups + 3) / 4)), dim3(256), 0, as_stream(stream), w,
                       groups, group_size, bits, packed, scales, biases);
    LQ_CHECK_LAUNCH("wq_quantize");
    return LQ_OK;
}

int lq_wq_dequantize(const uint32_t* packed, const float* scales, const float* biases, int N, int K, int group_size,
                     int bits, float* out, lq_stream stream) {
    int rc = check_group("wq_dequantize", K, group_size, bits);
    if (rc) return rc;
    LQ_REQUIRE(N >= 0, LQ_ERR_SHAPE, "wq_dequantize: negative row count");
    if (N == 0) return LQ_OK;
    LQ_REQUIRE(packed && scales && biases && out, LQ_ERR_VALUE, "wq_dequantize: NULL pointer");
    const size_t words = size_t(N) * K * bits / 32;
    LQ_REQUIRE((words + 255) / 256 < 0x7fffffffull, LQ_ERR_SHAPE, "wq_dequantize: tensor too large");
    hipLaunchKernelGGL(wq_dequantize_kernel, dim3(unsigned((words + 255) / 256)), dim3(256), 0, as_stream(stream),
                       packed, scales, biases, words, group_size, bits, out);
    LQ_CHECK_LAUNCH("wq_dequantize");
    return LQ_OK;
}

int lq_wq_matmul(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N, int K,
                 int group_size, int bits, float* out, lq_stream stream) {
    int rc = check_group("wq_matmul", K, group_size, bits);
    if (rc) return rc;
    LQ_REQUIRE(M >= 0 && N >= 0, LQ_ERR_SHAPE, "wq_matmul: negative extent");
    if (M == 0 || N == 0) return LQ_OK;
    LQ_REQUIRE(x && packed && scales && biases && out, LQ_ERR_VALUE, "wq_matmul: NULL pointer");
    hipStream_t st = as_stream(stream);
    if (aligned16(x) && aligned16(packed)) {
        // one row is a stream of the weight; more rows go to the matrix cores: 16 rows x 512 or 1024 k of
        // wq_rows(tiles, parts) columns per block, or (wq_gemm.hip) tiles over all of K
        if (M == 1 && wq_gemv1_lds(K, bits) <= size_t(kGemv1MaxLds))
            return bits == 4 ? launch_gemv1<4>(x, packed, scales, biases, N, K, group_size, out, st)
                             : launch_gemv1<8>(x, packed, scales, biases, N, K, group_size, out, st);
        if (wq_gemm_beats_small_batch(M, N, K, group_size, bits))
            return launch_wq_gemm(x, packed, scales, biases, M, N, K, group_size, bits, out, st);
        // (its slabs grow with M x N x K: not for the weights of 2 GiB that the large-batch kernel leaves)
        if (M <= 64 || size_t(N) * K * bits / 8 < 0x7fffffffull)
            return bits == 4 ? launch_wq_mfma<4>(x, packed, scales, biases, M, N, K, group_size, out, st)
                             : launch_wq_mfma<8>(x, packed, scales, biases, M, N, K, group_size, out, st);
    }
    // operands that are not 16-byte aligned, large batches on such a weight: decode once into the workspace, then the float32 MFMA GEMM
    void* ws = nullptr;
    const auto lock = scratch_lock(st);
    rc = workspace(size_t(N) * K * sizeof(float), st, &ws);
    if (rc) return rc;
    rc = lq_wq_dequantize(packed, scales, biases, N, K, group_size, bits, static_cast<float*>(ws), stream);
    if (rc) return rc;
    // (its large tiles whatever the size: a rare route, and the one that the products without a decoded weight are measured against)
    return sgemm_nt(x, static_cast<const float*>(ws), nullptr, out, M, N, K, true, st);
}

}  // extern "C"
