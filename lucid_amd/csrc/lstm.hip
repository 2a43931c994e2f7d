// Weight-only int8 LSTM layers over a whole sequence, in one launch.
//
//   raw[t] = x[t] W_ih^T + h[t-1] W_hh^T + (b_ih + b_hh)        gates i, f, g, o
//   c[t] = sigmoid(f) c[t-1] + sigmoid(i) tanh(g),  h[t] = sigmoid(o) tanh(c[t])
//
// (lucid/nn/quantized/dynamic/rnn.py:66-84, CpuBackend.h:13394-13519).  A chain of `steps` small
// dependent products: the time is the number of steps times the latency of one.
//
// Split.  A block keeps the recurrent weights of 16 hidden units (64 gate rows x hidden codes) in
// registers for the whole sequence, as bfloat16 matrix operands: an int8 code is exact in bfloat16,
// and h is split into three bfloat16 parts (exact: 8 + 8 + 8 significant bits), so every product is
// exact and accumulates in float32; the row's scale is applied to the sum.  The wavefronts of a
// block divide the hidden axis between them: each loads its own columns of h[t-1] straight into
// operand layout (16 batch rows x 32 columns per instruction), multiplies them with all four gate
// tiles, and the partial sums meet in LDS; wavefront w of the first four then finishes batch rows
// 4 j + w of the 16 units, with c in registers.  ceil(hidden / 16) blocks serve 16 batch rows of one
// direction; other rows and the other direction are independent groups in the same grid.
//
// Input.  Up to 512 columns a block also keeps the input weights of its units and takes the input product
// of the next step while its h travels to the other blocks, where it costs nothing.  Stacked layers then
// share the launch: layer k reads h[t] of layer k - 1 from that one's output as it appears, so L layers
// take steps + L - 1 step times in place of L * steps.  The registers of the second weight halve the blocks
// per CU; where that would mean more launches than it saves (lq_lstm_fused_layers), or beyond 512 columns,
// the input products of all steps are taken beforehand (`gx`) and a layer is a launch of its own.
//
// Exchange.  h[t] is the layer's output, so the blocks of a group hand it to each other through y
// itself: y is filled with a bit pattern no h can have (all ones, a NaN) before the launch, h is
// written through to device scope, and a wavefront re-reads its columns of h[t-1] until every word is
// there - no flags, no barrier, one memory trip each way per step.
//
// Progress.  A block waits only for blocks of its own launch, so all of them have to be resident: the
// launcher bounds the grid by what the device holds of this kernel over the number of hardware queues
// that streams share (four unless GPU_MAX_HW_QUEUES says more; a queue starts a launch only after the one
// before it is fully placed), and larger batches run as several launches.  A wait is bounded besides:
// after kSpinLimit reads the block stops waiting for the rest of the sequence and the output keeps its NaNs.
//
// hidden 512, 16 rows: 3.4 us per step with gx, 3.8 with the input product; two such layers of 64 steps
// 272 us per call, against 580 us as two launches with a GEMM (43 us with the decoding of its weight) each
// and 4.67 ms with a float32 GEMM, a gate kernel and the host's share of their launches per step.
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include "common.hpp"

using namespace lq;

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kUnits = 16, kRows = 16;     // hidden units of a block, batch rows of a group
constexpr unsigned kEmpty = 0xffffffffu;   // a word of y that has not been written
constexpr int kSpinLimit = 1 << 20;        // about a second of waiting for one step
constexpr int kScopeDevice = 16;           // "sc1" cache-policy bit of buffer accesses

constexpr int kParts = LQ_LSTM_PARTS;      // grid z: the directions of one layer, or stacked layers

struct LstmArgs {
    const float* gx[2];
    const float* x;              // input of part 0 (of every direction) where the kernel takes the input product
    const int8_t* wx[kParts];
    const float* wx_scale[kParts];
    const int8_t* w[kParts];
    const float* w_scale[kParts];
    const float* b_ih[kParts];
    const float* b_hh[kParts];
    const float* h0;   // [parts][B][H] or null (zeros), likewise c0
    const float* c0;
    float* h_n;        // [parts][B][H]
    float* c_n;
    float* y[kParts];  // element (t, b, col + j) at t * y_step + b * y_row + col + j; col = d * H in direction d
    long y_step, y_row, gx_step, gx_row, x_step, x_row;
    long y_elems, x_elems;
    int T, B, H, I, row0, dir0, stacked;
};

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v2f{a, b}, v2bf));
}
// (a, b) = h + m + l, each part a pair of bfloat16; the remainders are exact
__device__ __forceinline__ void split3(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    h = pk_bf16(a, b);
    a -= __uint_as_float(h << 16), b -= __uint_as_float(h & 0xffff0000u);
    m = pk_bf16(a, b);
    a -= __uint_as_float(m << 16), b -= __uint_as_float(m & 0xffff0000u);
    l = pk_bf16(a, b);
}
// two int8 codes as a pair of bfloat16 (their floats have zeros below bit 16)
__device__ __forceinline__ uint32_t codes_bf16(int c0, int c1) {
    return __builtin_amdgcn_perm(__float_as_uint(float(c1)), __float_as_uint(float(c0)), 0x07060302u);
}
__device__ __forceinline__ float sigmoid(float x) { return 1.0f / (1.0f + expf(-x)); }

// the codes of one row of a weight at this lane's eight columns of an instruction, as bfloat16
__device__ __forceinline__ v8bf load_codes(const int8_t* row, int k, int K) {
    int c[8];
    if (k + 8 <= K) {
        uint64_t raw;
        __builtin_memcpy(&raw, row + k, 8);
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = int(int8_t(raw >> (8 * e)));
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) c[e] = k + e < K ? int(row[k + e]) : 0;
    }
    return __builtin_bit_cast(v8bf, v4u{codes_bf16(c[0], c[1]), codes_bf16(c[2], c[3]), codes_bf16(c[4], c[5]),
                                        codes_bf16(c[6], c[7])});
}
// device-scope access to what follows element `at` of an array of `elems` floats
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words_from(const float* base, long at, long elems) {
    const long bytes = (elems - at) * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + at, 0,
                                             bytes < 0x7fffffffl ? int(bytes) : 0x7fffffff, 0x00020000);
}
template <int KP>
__device__ __forceinline__ void load_columns(v4u (&raw)[KP][2], __amdgpu_buffer_rsrc_t src, unsigned off) {
#pragma unroll
    for (int i = 0; i < KP; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
            raw[i][j] = __builtin_amdgcn_raw_buffer_load_b128(src, off + unsigned(i * 32 + j * 4) * 4, 0, kScopeDevice);
}
// columns from `left` on (of another direction, row or step) become zero; the largest word left
template <int KP>
__device__ __forceinline__ unsigned mask_columns(v4u (&raw)[KP][2], int left) {
    unsigned worst = 0;
#pragma unroll
    for (int i = 0; i < KP; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (i * 32 + e >= left) raw[i][e >> 2][e & 3] = 0u;
            worst = worst > raw[i][e >> 2][e & 3] ? worst : raw[i][e >> 2][e & 3];
        }
    return worst;
}
// acc[g] += columns . codes of gate g: three exact part products each
template <int KP>
__device__ __forceinline__ void multiply(v4f (&acc)[4], const v4u (&raw)[KP][2], const v8bf (&wf)[4][KP]) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
        v4u part3[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const v4u r = raw[i][e >> 1];
            uint32_t hh, mm, ll;
            split3(__uint_as_float(r[(2 * e) & 3]), __uint_as_float(r[(2 * e + 1) & 3]), hh, mm, ll);
            part3[0][e] = hh, part3[1][e] = mm, part3[2][e] = ll;
        }
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, part3[q]), wf[g][i], acc[g], 0, 0, 0);
    }
}

// W wavefronts, each with KPW instructions of 32 hidden columns (hidden <= 32 W KPW) and KX of 32 input
// columns; KX = 0 reads the input products from gx.  The weights take 16 (KPW + KX) registers, which
// decides how many wavefronts a SIMD holds.
template <int W, int KPW, int KX>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(KX == 0 && KPW <= 2 ? 4 : 2, KX == 0 && KPW <= 2 ? 4 : 2)))
void lstm_sequence_kernel(LstmArgs p) {
    __shared__ float part[2][W][4][4][64];  // [step parity][wavefront][gate][row of the quad][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ln = lane & 15, lq4 = lane >> 4;
    const int z = p.dir0 + blockIdx.z, d = p.stacked ? 0 : z, H = p.H;
    const int u0 = blockIdx.x * kUnits, m0 = p.row0 + blockIdx.y * kRows;
    float* const y = p.y[z];

    // ---- the block's weights: tile g = gate g of units u0 .. u0+15, this wavefront's columns
    v8bf wf[4][KPW], wxf[4][KX > 0 ? KX : 1];
    float scale_h[4], scale_x[4];  // of the unit whose products this lane accumulates
    // ---- the input of this part: x, or the output of the layer below
    const bool above = p.stacked && z > 0;
    const float* const in = above ? p.y[above ? z - 1 : 0] : p.x;
    const int I = above ? H : p.I;
    const long in_step = above ? p.y_step : p.x_step, in_row = above ? p.y_row : p.x_row;
    const long in_elems = above ? p.y_elems : p.x_elems;
    const int kx_lane = wave * KX * 32 + lq4 * 8;
    {
        const int unit = u0 + ln < H ? u0 + ln : H - 1;  // units past H are computed and never stored
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int i = 0; i < KPW; ++i)
                wf[g][i] = load_codes(p.w[z] + (size_t(g) * H + unit) * H, (wave * KPW + i) * 32 + lq4 * 8, H);
            if constexpr (KX > 0) {
#pragma unroll
                for (int i = 0; i < KX; ++i)
                    wxf[g][i] = load_codes(p.wx[z] + (size_t(g) * H + unit) * I, kx_lane + i * 32, I);
                scale_h[g] = p.w_scale[z][g * H + unit], scale_x[g] = p.wx_scale[z][g * H + unit];
            }
        }
    }
    // ---- the element this lane finishes (wavefronts 0..3)
    const int unit = u0 + ln, row = m0 + 4 * lq4 + wave;
    const bool mine = wave < 4 && unit < H && row < p.B;
    float ws[4], bias[4], c = 0.0f;
    const size_t state = (size_t(z) * p.B + (row < p.B ? row : 0)) * H + unit;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        ws[g] = KX > 0 ? 1.0f : mine ? p.w_scale[z][g * H + unit] : 0.0f;
        bias[g] = mine && p.b_ih[z] ? p.b_ih[z][g * H + unit] + p.b_hh[z][g * H + unit] : 0.0f;
    }
    if (mine && p.c0) c = p.c0[state];
    const float* gx_lane = KX > 0 ? nullptr : p.gx[d] + size_t(mine ? row : 0) * p.gx_row + (mine ? unit : 0);
    // ---- the row whose h this lane reads; rows past the batch repeat the last one
    const int hrow = m0 + ln < p.B ? m0 + ln : p.B - 1;
    const int k_lane = wave * KPW * 32 + lq4 * 8;
    const int left = H - k_lane;  // columns of this wavefront's first step from k_lane on that exist
    bool waiting = true;
    float hv = 0.0f;

    // The input product of a step needs nothing of the step before it, so it is taken while the h of that
    // step is on its way to the other blocks; its first read is issued before the gates are computed.
    const unsigned x_off = unsigned(hrow * in_row + kx_lane) * 4;
    v4u rx[KX > 0 ? KX : 1][2];
    v4f accx[4];  // scaled
    auto input_words = [&](int t) { return words_from(in, long(t) * in_step, in_elems); };
    auto input_product = [&](int t) {
        if constexpr (KX > 0) {
            for (int spin = 0;; ++spin) {
                const unsigned worst = mask_columns<KX>(rx, I - kx_lane);
                if (!above || !waiting || __builtin_amdgcn_ballot_w64(worst == kEmpty) == 0) break;
                if (spin >= kSpinLimit) waiting = false;
                asm volatile("" ::: "memory");
                load_columns<KX>(rx, input_words(t), x_off);
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) accx[g] = v4f{0.f, 0.f, 0.f, 0.f};
            multiply<KX>(accx, rx, wxf);
#pragma unroll
            for (int g = 0; g < 4; ++g) accx[g] *= scale_x[g];
        }
    };
    if constexpr (KX > 0) {
        const int t = d ? p.T - 1 : 0;
        load_columns<KX>(rx, input_words(t), x_off);
        input_product(t);
    }

    for (int s = 0; s < p.T; ++s) {
        const int t = d ? p.T - 1 - s : s;
        const int t_next = d ? t - 1 : t + 1;  // of the next step, if there is one
        float gx[4];
        if (KX == 0 && mine) {
#pragma unroll
            for (int g = 0; g < 4; ++g) gx[g] = gx_lane[size_t(t) * p.gx_step + size_t(g) * H];
        }
        v4u raw[KPW][2];
        if (s == 0) {
#pragma unroll
            for (int i = 0; i < KPW; ++i)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const int k = k_lane + i * 32 + e;
                    raw[i][e >> 2][e & 3] =
                        p.h0 && k < H ? __float_as_uint(p.h0[(size_t(z) * p.B + hrow) * H + k]) : 0u;
                }
        } else {
            const __amdgpu_buffer_rsrc_t src =
                words_from(y, long(d ? t + 1 : t - 1) * p.y_step + long(d) * H, p.y_elems);
            const unsigned off = unsigned(hrow * p.y_row + k_lane) * 4;
            for (int spin = 0;; ++spin) {
                asm volatile("" ::: "memory");  // read again: the words change under the loop
                load_columns<KPW>(raw, src, off);
                const unsigned worst = mask_columns<KPW>(raw, left);
                if (!waiting || __builtin_amdgcn_ballot_w64(worst == kEmpty) == 0) break;
                if (spin >= kSpinLimit) waiting = false;
            }
        }
        if constexpr (KX > 0) {
            if (s + 1 < p.T) load_columns<KX>(rx, input_words(t_next), x_off);
        }
        v4f acc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
        multiply<KPW>(acc, raw, wf);
        if constexpr (KX > 0) {
#pragma unroll
            for (int g = 0; g < 4; ++g) acc[g] = acc[g] * scale_h[g] + accx[g];
        }
        float(*const mine_part)[4][64] = part[s & 1][wave];
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) mine_part[g][r][lane] = acc[g][r];
        // (a buffer is written again two steps later, after the next step's barrier: by then it has been read)
        __syncthreads();
        if (wave < 4) {
            float raw4[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float sum = part[s & 1][0][g][wave][lane];
#pragma unroll
                for (int w = 1; w < W; ++w) sum += part[s & 1][w][g][wave][lane];
                raw4[g] = mine ? (KX > 0 ? sum : gx[g] + sum * ws[g]) + bias[g] : 0.0f;
            }
            const float ig = sigmoid(raw4[0]), fg = sigmoid(raw4[1]), gg = tanhf(raw4[2]), og = sigmoid(raw4[3]);
            c = fg * c + ig * gg;
            hv = og * tanhf(c);
            if (mine) {
                unsigned bits = __float_as_uint(hv);
                bits = bits == kEmpty ? 0x7fc00000u : bits;  // a NaN, but not the one that means "not written"
                const __amdgpu_buffer_rsrc_t dst = words_from(y, long(t) * p.y_step + long(d) * H, p.y_elems);
                __builtin_amdgcn_raw_buffer_store_b32(bits, dst, unsigned(row * p.y_row + unit) * 4, 0, kScopeDevice);
            }
        }
        if (KX > 0 && s + 1 < p.T) input_product(t_next);
    }
    if (mine) {
        p.h_n[state] = hv;
        p.c_n[state] = c;
    }
}

// every word of the outputs "not written yet"
__global__ __launch_bounds__(256) void lstm_empty_kernel(LstmArgs p) {
    float* const y = p.y[blockIdx.y];
    const long stride = long(gridDim.x) * 256;
    for (long i = long(blockIdx.x) * 256 + threadIdx.x; i < p.y_elems; i += stride) y[i] = __uint_as_float(kEmpty);
}

// Launches that may be placed at once: the hardware queues of the process, which HIP takes from the environment.
int hardware_queues() {
    static const int n = [] {
        const char* v = std::getenv("GPU_MAX_HW_QUEUES");
        const long q = v ? std::strtol(v, nullptr, 10) : 0;
        return q > 4 ? int(q < 1024 ? q : 1024) : 4;
    }();
    return n;
}

// Launches of one kernel form: 16-row groups of one direction or of one stack, as many at once as may be.
struct LstmSplit {
    int per_group, groups, at_once, both;  // blocks of a group; groups; groups of a launch; its parts
    int launches;
};

template <int W, int KPW, int KX>
int split_lstm(int B, int H, int parts, bool stacked, LstmSplit* out) {
    static DeviceOnce once;
    static int capacity[32] = {0};  // blocks of this kernel the device holds at once
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    const int rc = device_once(once, [&]() -> int {
        int per_cu = 0;
        hipDeviceProp_t prop;
        LQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lstm_sequence_kernel<W, KPW, KX>, W * 64, 0));
        LQ_HIP(hipGetDeviceProperties(&prop, dev));
        capacity[dev] = per_cu * prop.multiProcessorCount;
        return LQ_OK;
    });
    if (rc) return rc;
    LstmSplit s;
    s.per_group = (H + kUnits - 1) / kUnits;
    s.groups = (B + kRows - 1) / kRows;
    const int fit = capacity[dev] / hardware_queues() / s.per_group;
    s.both = stacked || fit >= parts ? parts : 1;
    s.at_once = fit / s.both < s.groups ? fit / s.both : s.groups;
    s.launches = s.at_once < 1 ? 0 : (parts / s.both) * ((s.groups + s.at_once - 1) / s.at_once);
    *out = s;
    return LQ_OK;
}

template <int W, int KPW, int KX>
int launch_lstm(LstmArgs p, int parts, hipStream_t st) {
    LstmSplit s;
    if (int rc = split_lstm<W, KPW, KX>(p.B, p.H, parts, p.stacked != 0, &s)) return rc;
    LQ_REQUIRE(s.launches >= 1, LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: %d x hidden %d do not fit the device at once",
               p.stacked ? parts : 1, p.H);
    const int n_y = p.stacked ? parts : 1;
    const long fill_blocks = (p.y_elems + 1023) / 1024;
    hipLaunchKernelGGL(lstm_empty_kernel, dim3(unsigned(fill_blocks < 2048 ? fill_blocks : 2048), unsigned(n_y)), dim3(256),
                       0, st, p);
    LQ_CHECK_LAUNCH("lstm_empty");
    for (p.dir0 = 0; p.dir0 < parts; p.dir0 += s.both)
        for (int g = 0; g < s.groups; g += s.at_once) {
            p.row0 = g * kRows;
            const int n = s.groups - g < s.at_once ? s.groups - g : s.at_once;
            hipLaunchKernelGGL((lstm_sequence_kernel<W, KPW, KX>), dim3(unsigned(s.per_group), unsigned(n), unsigned(s.both)),
                               dim3(W * 64), 0, st, p);
            LQ_CHECK_LAUNCH("lstm_sequence");
        }
    return LQ_OK;
}

// f(W, KPW, KX) for the form that serves `hidden` columns and `inputs` (0: gates_x).  More wavefronts
// before more columns each: a wavefront's loads, splits and products are a serial chain.
template <typename F>
int with_form(int hidden, int inputs, F f) {
    const int ks = (hidden + 31) / 32, kx = (inputs + 31) / 32;
    using std::integral_constant;
    if (kx == 0) {
        if (ks <= 4) return f(integral_constant<int, 4>(), integral_constant<int, 1>(), integral_constant<int, 0>());
        if (ks <= 8) return f(integral_constant<int, 8>(), integral_constant<int, 1>(), integral_constant<int, 0>());
        if (ks <= 16) return f(integral_constant<int, 8>(), integral_constant<int, 2>(), integral_constant<int, 0>());
        return f(integral_constant<int, 8>(), integral_constant<int, 4>(), integral_constant<int, 0>());
    }
    if (ks <= 4 && kx <= 4) return f(integral_constant<int, 4>(), integral_constant<int, 1>(), integral_constant<int, 1>());
    if (ks <= 8)
        return kx <= 8 ? f(integral_constant<int, 8>(), integral_constant<int, 1>(), integral_constant<int, 1>())
                       : f(integral_constant<int, 8>(), integral_constant<int, 1>(), integral_constant<int, 2>());
    return kx <= 8 ? f(integral_constant<int, 8>(), integral_constant<int, 2>(), integral_constant<int, 1>())
                   : f(integral_constant<int, 8>(), integral_constant<int, 2>(), integral_constant<int, 2>());
}
constexpr int kMaxFused = 512;  // hidden and input columns of a form that takes the input product
constexpr int kMaxHidden = 1024;

// A step of all rows: one launch of the recurrence per rows that fit the device, or a float32 GEMM and a gate kernel
// (lq_lstm_cell_f32) on decoded weights, issued from Python.  Measured, us per step of both: hidden 64, 8192 rows 25.7 /
// 32.9; 128, 4096 rows 25.6 / 35.4, 8192 rows 46.9 / 47.2; 256, 1024 rows 29.6 / 37.4, 2048 rows 57.9 / 43.1; 512, 512
// rows 37 / 49, 1024 rows 73 / 56; 768, 128 rows 41 / 58, 256 rows 80 / 60; 1024, 128 rows 46 / 71, 256 rows 89 / 73,
// 4096 rows 1399 / 289; 1024 in two directions, 16 rows 15 / 130, 256 rows 180 / 146.  The estimates are within 20 %.
double sequence_step_us(int hidden) { return 2.9 + 0.0026 * hidden; }
double gemm_step_us(int batch, int hidden) {
    const double least = 17.0 + 0.05 * hidden, rows = batch * (2.8e-5 * hidden + 3.8e-8 * hidden * hidden);
    return std::sqrt(least * least + rows * rows);
}

}  // namespace

extern "C" {

int lq_lstm_sequence_pays(int batch, int hidden, int directions, int* pays) {
    LQ_REQUIRE(pays, LQ_ERR_VALUE, "lstm_sequence_pays: NULL pointer");
    LQ_REQUIRE(batch >= 0 && hidden > 0, LQ_ERR_SHAPE, "lstm_sequence_pays: bad extent (%d, %d)", batch, hidden);
    LQ_REQUIRE(directions == 1 || directions == 2, LQ_ERR_VALUE, "lstm_sequence_pays: directions must be 1 or 2");
    *pays = 0;
    if (batch == 0 || hidden > kMaxHidden) return LQ_OK;
    LstmSplit s;
    const int rc = with_form(hidden, 0, [&](auto w, auto k, auto x) {
        return split_lstm<w(), k(), x()>(batch, hidden, directions, false, &s);
    });
    if (rc) return rc;
    *pays = s.launches > 0 && s.launches * sequence_step_us(hidden) <= directions * gemm_step_us(batch, hidden);
    return LQ_OK;
}

int lq_lstm_fused_layers(int steps, int batch, int inputs, int hidden, int layers, int directions, int* fused) {
    LQ_REQUIRE(fused, LQ_ERR_VALUE, "lstm_fused_layers: NULL pointer");
    LQ_REQUIRE(steps >= 0 && batch >= 0 && inputs > 0 && hidden > 0 && layers > 0, LQ_ERR_SHAPE,
               "lstm_fused_layers: bad extent (%d, %d, %d, %d, %d)", steps, batch, inputs, hidden, layers);
    LQ_REQUIRE(directions == 1 || directions == 2, LQ_ERR_VALUE, "lstm_fused_layers: directions must be 1 or 2");
    *fused = 0;
    if (steps == 0 || batch == 0 || hidden > kMaxFused || inputs > kMaxFused) return LQ_OK;
    // Costs per layer in steps of the recurrence.  An input product in a GEMM of its own, with the decoded
    // weight it reads, is worth twelve (43 us at 1024 x 2048 x 512, a step 3.4).
    constexpr long kGemm = 12;
    LstmSplit s;
    int rc = with_form(hidden, 0, [&](auto w, auto k, auto x) { return split_lstm<w(), k(), x()>(batch, hidden, directions, false, &s); });
    if (rc) return rc;
    double best = s.launches ? double(s.launches) * steps + kGemm * directions : 1e30;
    for (int n = 1; n <= (directions == 1 ? (layers < kParts ? layers : kParts) : 1); ++n) {
        const int columns = n > 1 && hidden > inputs ? hidden : inputs;
        rc = with_form(hidden, columns, [&](auto w, auto k, auto x) {
            return split_lstm<w(), k(), x()>(batch, hidden, directions == 2 ? 2 : n, n > 1, &s);
        });
        if (rc) return rc;
        const double cost = double(s.launches) * (steps + n - 1) / n;
        if (s.launches && cost < best) best = cost, *fused = n;
    }
    return LQ_OK;
}

int lq_lstm_sequence_f32(const lq_lstm_args* a, lq_stream stream) {
    LQ_REQUIRE(a, LQ_ERR_VALUE, "lstm_sequence: args is NULL");
    LQ_REQUIRE(a->steps >= 0 && a->batch >= 0 && a->hidden > 0, LQ_ERR_SHAPE, "lstm_sequence: bad extent (%d, %d, %d)",
               a->steps, a->batch, a->hidden);
    LQ_REQUIRE(a->directions == 1 || a->directions == 2, LQ_ERR_VALUE, "lstm_sequence: directions must be 1 or 2");
    LQ_REQUIRE(a->layers >= 1 && a->layers <= kParts && (a->layers == 1 || (a->directions == 1 && a->x)), LQ_ERR_VALUE,
               "lstm_sequence: %d layers, 1 or (one direction, input product taken here) at most %d", a->layers, kParts);
    LQ_REQUIRE(a->hidden <= kMaxHidden, LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: hidden %d, at most %d", a->hidden, kMaxHidden);
    LQ_REQUIRE(!a->x || (a->inputs > 0 && a->inputs <= kMaxFused && a->hidden <= kMaxFused), LQ_ERR_NOT_IMPLEMENTED,
               "lstm_sequence: input product of %d columns for hidden %d, at most %d", a->inputs, a->hidden, kMaxFused);
    if (a->steps == 0 || a->batch == 0) return LQ_OK;
    LQ_REQUIRE(a->h_n && a->c_n, LQ_ERR_VALUE, "lstm_sequence: NULL output pointer");
    LstmArgs p{};
    p.stacked = a->layers > 1;
    const int parts = p.stacked ? a->layers : a->directions;
    for (int z = 0; z < parts; ++z) {
        if (!a->x) {
            LQ_REQUIRE(a->gates_x[z], LQ_ERR_VALUE, "lstm_sequence: NULL operand");
            p.gx[z] = a->gates_x[z];
        } else {
            LQ_REQUIRE(a->w_ih[z] && a->w_ih_scale[z], LQ_ERR_VALUE, "lstm_sequence: NULL operand");
        }
        LQ_REQUIRE(a->w_hh[z] && a->w_hh_scale[z], LQ_ERR_VALUE, "lstm_sequence: NULL operand");
        LQ_REQUIRE((a->bias_ih[z] == nullptr) == (a->bias_hh[z] == nullptr), LQ_ERR_VALUE,
                   "lstm_sequence: one of the two biases is NULL");
        p.y[z] = a->y[p.stacked ? z : 0];
        LQ_REQUIRE(p.y[z], LQ_ERR_VALUE, "lstm_sequence: NULL output pointer");
        p.wx[z] = a->w_ih[z], p.wx_scale[z] = a->w_ih_scale[z];
        p.w[z] = a->w_hh[z], p.w_scale[z] = a->w_hh_scale[z];
        p.b_ih[z] = a->bias_ih[z], p.b_hh[z] = a->bias_hh[z];
    }
    p.x = a->x, p.I = a->inputs;
    p.h0 = a->h0, p.c0 = a->c0, p.h_n = a->h_n, p.c_n = a->c_n;
    p.T = a->steps, p.B = a->batch, p.H = a->hidden;
    const long width = long(a->directions) * p.H, gates = 4L * p.H;
    p.y_step = a->batch_first ? width : p.B * width, p.y_row = a->batch_first ? p.T * width : width;
    p.gx_step = a->batch_first ? gates : p.B * gates, p.gx_row = a->batch_first ? p.T * gates : gates;
    p.x_step = a->batch_first ? p.I : long(p.B) * p.I, p.x_row = a->batch_first ? long(p.T) * p.I : p.I;
    p.y_elems = long(p.T) * p.B * width, p.x_elems = long(p.T) * p.B * p.I;
    // an element is addressed as a 32-bit byte offset from its step's first
    LQ_REQUIRE((p.B - 1) * p.y_row + width < 0x7fffffffL / 4 &&
                   (!a->x || (p.B - 1) * p.x_row + p.I < 0x7fffffffL / 4),
               LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: %ld outputs or %ld inputs are too many", p.y_elems, p.x_elems);
    const int columns = !a->x ? 0 : p.stacked && p.H > p.I ? p.H : p.I;
    return with_form(p.H, columns, [&](auto w, auto k, auto x) { return launch_lstm<w(), k(), x()>(p, parts, as_stream(stream)); });
}

}  // extern "C"
