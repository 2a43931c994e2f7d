// The recurrence of a weight-only int8 LSTM layer over a whole sequence, in one launch.
//
//   raw[t] = x[t] W_ih^T + h[t-1] W_hh^T + (b_ih + b_hh)        gates i, f, g, o
//   c[t] = sigmoid(f) c[t-1] + sigmoid(i) tanh(g),  h[t] = sigmoid(o) tanh(c[t])
//
// (lucid/nn/quantized/dynamic/rnn.py:66-84, CpuBackend.h:13394-13519).  The input products of all
// steps are taken beforehand (`gx`); what is left is a chain of `steps` small dependent products,
// so the time is the number of steps times the latency of one.
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
// Exchange.  h[t] is the layer's output, so the blocks of a group hand it to each other through y
// itself: y is filled with a bit pattern no h can have (all ones, a NaN) before the launch, h is
// written through to device scope, and a wavefront re-reads its columns of h[t-1] until every word is
// there - no flags, no barrier, one memory trip each way per step.
//
// Progress.  A block waits only for blocks of its own launch, so all of them have to be resident: the
// launcher bounds the grid by a quarter of what the device holds of this kernel (streams share four
// hardware queues, and a queue starts a launch only after the one before it is fully placed), and
// larger batches run as several launches.  A wait is bounded besides: after kSpinLimit reads the
// block stops waiting for the rest of the sequence and the output keeps its NaNs.
//
// hidden 512, 16 rows: 3.4 us per step on the MI355X, against 36 us for a float32 GEMM, a gate kernel and
// the host's share of their launches per step.
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

struct LstmArgs {
    const float* gx[2];
    const int8_t* w[2];
    const float* w_scale[2];
    const float* b_ih[2];
    const float* b_hh[2];
    const float* h0;   // [dirs][B][H] or null (zeros), likewise c0
    const float* c0;
    float* h_n;        // [dirs][B][H]
    float* c_n;
    float* y;          // element (t, b, d * H + j) at t * y_step + b * y_row + d * H + j
    long y_step, y_row, gx_step, gx_row;
    long y_elems;
    int T, B, H, row0, dir0;
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

// W wavefronts, each with KPW steps of 32 hidden columns: hidden <= 32 W KPW.  The weights take 16 KPW
// registers: KPW <= 2 fits four wavefronts per SIMD, KPW = 4 (hidden > 512) two.
template <int W, int KPW>
__global__ __launch_bounds__(W * 64) __attribute__((amdgpu_waves_per_eu(KPW <= 2 ? 4 : 2, KPW <= 2 ? 4 : 2)))
void lstm_sequence_kernel(LstmArgs p) {
    __shared__ float part[2][W][4][4][64];  // [step parity][wavefront][gate][row of the quad][lane]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ln = lane & 15, lq4 = lane >> 4;
    const int d = p.dir0 + blockIdx.z, H = p.H;
    const int u0 = blockIdx.x * kUnits, m0 = p.row0 + blockIdx.y * kRows;

    // ---- the block's weights: tile g = gate g of units u0 .. u0+15, this wavefront's hidden columns
    v8bf wf[4][KPW];
    {
        const int unit = u0 + ln < H ? u0 + ln : H - 1;  // units past H are computed and never stored
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int8_t* row = p.w[d] + (size_t(g) * H + unit) * H;
#pragma unroll
            for (int i = 0; i < KPW; ++i) {
                const int k = (wave * KPW + i) * 32 + lq4 * 8;
                int c[8];
                if (k + 8 <= H) {
                    uint64_t raw;
                    __builtin_memcpy(&raw, row + k, 8);
#pragma unroll
                    for (int e = 0; e < 8; ++e) c[e] = int(int8_t(raw >> (8 * e)));
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e) c[e] = k + e < H ? int(row[k + e]) : 0;
                }
                wf[g][i] = __builtin_bit_cast(v8bf, v4u{codes_bf16(c[0], c[1]), codes_bf16(c[2], c[3]),
                                                        codes_bf16(c[4], c[5]), codes_bf16(c[6], c[7])});
            }
        }
    }
    // ---- the element this lane finishes (wavefronts 0..3)
    const int unit = u0 + ln, row = m0 + 4 * lq4 + wave;
    const bool mine = wave < 4 && unit < H && row < p.B;
    float ws[4], bias[4], c = 0.0f;
    const size_t state = (size_t(d) * p.B + (row < p.B ? row : 0)) * H + unit;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        ws[g] = mine ? p.w_scale[d][g * H + unit] : 0.0f;
        bias[g] = mine && p.b_ih[d] ? p.b_ih[d][g * H + unit] + p.b_hh[d][g * H + unit] : 0.0f;
    }
    if (mine && p.c0) c = p.c0[state];
    const float* gx_lane = p.gx[d] + size_t(mine ? row : 0) * p.gx_row + (mine ? unit : 0);
    // ---- the row whose h this lane reads; rows past the batch repeat the last one
    const int hrow = m0 + ln < p.B ? m0 + ln : p.B - 1;
    const int k_lane = wave * KPW * 32 + lq4 * 8;
    const int left = H - k_lane;  // columns of this wavefront's first step from k_lane on that exist
    bool waiting = true;
    float hv = 0.0f;

    for (int s = 0; s < p.T; ++s) {
        const int t = d ? p.T - 1 - s : s;
        float gx[4];
        if (mine) {
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
                        p.h0 && k < H ? __float_as_uint(p.h0[(size_t(d) * p.B + hrow) * H + k]) : 0u;
                }
        } else {
            const long at = long(d ? t + 1 : t - 1) * p.y_step + long(d) * H;
            const long bytes = (p.y_elems - at) * 4;
            const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
                p.y + at, 0, bytes < 0x7fffffffl ? int(bytes) : 0x7fffffff, 0x00020000);
            const unsigned off = unsigned(hrow * p.y_row + k_lane) * 4;
            for (int spin = 0;; ++spin) {
                asm volatile("" ::: "memory");  // read again: the words change under the loop
#pragma unroll
                for (int i = 0; i < KPW; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        raw[i][j] = __builtin_amdgcn_raw_buffer_load_b128(src, off + unsigned(i * 32 + j * 4) * 4, 0, kScopeDevice);
                unsigned worst = 0;
#pragma unroll
                for (int i = 0; i < KPW; ++i)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        // columns past H (of another direction, row or step) count as zero
                        if (i * 32 + e >= left) raw[i][e >> 2][e & 3] = 0u;
                        worst = worst > raw[i][e >> 2][e & 3] ? worst : raw[i][e >> 2][e & 3];
                    }
                if (!waiting || __builtin_amdgcn_ballot_w64(worst == kEmpty) == 0) break;
                if (spin >= kSpinLimit) waiting = false;
            }
        }
        v4f acc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < KPW; ++i) {
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
                raw4[g] = mine ? (gx[g] + sum * ws[g]) + bias[g] : 0.0f;
            }
            const float ig = sigmoid(raw4[0]), fg = sigmoid(raw4[1]), gg = tanhf(raw4[2]), og = sigmoid(raw4[3]);
            c = fg * c + ig * gg;
            hv = og * tanhf(c);
            if (mine) {
                unsigned bits = __float_as_uint(hv);
                bits = bits == kEmpty ? 0x7fc00000u : bits;  // a NaN, but not the one that means "not written"
                const long at = long(t) * p.y_step + long(d) * H;
                const long bytes = (p.y_elems - at) * 4;
                const __amdgpu_buffer_rsrc_t dst = __builtin_amdgcn_make_buffer_rsrc(
                    p.y + at, 0, bytes < 0x7fffffffl ? int(bytes) : 0x7fffffff, 0x00020000);
                __builtin_amdgcn_raw_buffer_store_b32(bits, dst, unsigned(row * p.y_row + unit) * 4, 0, kScopeDevice);
            }
        }
    }
    if (mine) {
        p.h_n[state] = hv;
        p.c_n[state] = c;
    }
}

template <int W, int KPW>
int launch_lstm(LstmArgs p, int dirs, hipStream_t st) {
    static DeviceOnce once;
    static int capacity[32] = {0};  // blocks of this kernel the device holds at once
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    const int rc = device_once(once, [&]() -> int {
        int per_cu = 0;
        hipDeviceProp_t prop;
        LQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, lstm_sequence_kernel<W, KPW>, W * 64, 0));
        LQ_HIP(hipGetDeviceProperties(&prop, dev));
        capacity[dev] = per_cu * prop.multiProcessorCount;
        return LQ_OK;
    });
    if (rc) return rc;
    const int per_group = (p.H + kUnits - 1) / kUnits;
    const int groups = (p.B + kRows - 1) / kRows;
    int at_once = capacity[dev] / 4 / per_group;  // groups (16 rows of one direction) of a launch
    LQ_REQUIRE(at_once >= 1, LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: hidden %d does not fit the device at once", p.H);
    const int both = at_once >= dirs ? dirs : 1;
    at_once = at_once / both < groups ? at_once / both : groups;
    for (p.dir0 = 0; p.dir0 < dirs; p.dir0 += both)
        for (int g = 0; g < groups; g += at_once) {
            p.row0 = g * kRows;
            const int n = groups - g < at_once ? groups - g : at_once;
            hipLaunchKernelGGL((lstm_sequence_kernel<W, KPW>), dim3(unsigned(per_group), unsigned(n), unsigned(both)),
                               dim3(W * 64), 0, st, p);
            LQ_CHECK_LAUNCH("lstm_sequence");
        }
    return LQ_OK;
}

}  // namespace

extern "C" {

int lq_lstm_sequence_f32(const lq_lstm_args* a, lq_stream stream) {
    LQ_REQUIRE(a, LQ_ERR_VALUE, "lstm_sequence: args is NULL");
    LQ_REQUIRE(a->steps >= 0 && a->batch >= 0 && a->hidden > 0, LQ_ERR_SHAPE, "lstm_sequence: bad extent (%d, %d, %d)",
               a->steps, a->batch, a->hidden);
    LQ_REQUIRE(a->directions == 1 || a->directions == 2, LQ_ERR_VALUE, "lstm_sequence: directions must be 1 or 2");
    LQ_REQUIRE(a->hidden <= 1024, LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: hidden %d, at most 1024", a->hidden);
    if (a->steps == 0 || a->batch == 0) return LQ_OK;
    LQ_REQUIRE(a->y && a->h_n && a->c_n, LQ_ERR_VALUE, "lstm_sequence: NULL output pointer");
    LstmArgs p{};
    for (int d = 0; d < a->directions; ++d) {
        LQ_REQUIRE(a->gates_x[d] && a->w_hh[d] && a->w_hh_scale[d], LQ_ERR_VALUE, "lstm_sequence: NULL operand");
        LQ_REQUIRE((a->bias_ih[d] == nullptr) == (a->bias_hh[d] == nullptr), LQ_ERR_VALUE,
                   "lstm_sequence: one of the two biases is NULL");
        p.gx[d] = a->gates_x[d], p.w[d] = a->w_hh[d], p.w_scale[d] = a->w_hh_scale[d];
        p.b_ih[d] = a->bias_ih[d], p.b_hh[d] = a->bias_hh[d];
    }
    p.h0 = a->h0, p.c0 = a->c0, p.h_n = a->h_n, p.c_n = a->c_n, p.y = a->y;
    p.T = a->steps, p.B = a->batch, p.H = a->hidden;
    const long width = long(a->directions) * p.H, gates = 4L * p.H;
    p.y_step = a->batch_first ? width : p.B * width, p.y_row = a->batch_first ? p.T * width : width;
    p.gx_step = a->batch_first ? gates : p.B * gates, p.gx_row = a->batch_first ? p.T * gates : gates;
    p.y_elems = long(p.T) * p.B * width;
    // an element is addressed as a 32-bit byte offset from its step's first
    LQ_REQUIRE((p.B - 1) * p.y_row + width < 0x7fffffffL / 4, LQ_ERR_NOT_IMPLEMENTED,
               "lstm_sequence: output of %ld elements is too large", p.y_elems);
    hipStream_t st = as_stream(stream);
    const int rc = lq_fill_bytes(a->y, 0xff, size_t(p.y_elems) * 4, stream);
    if (rc) return rc;
    const int ksteps = (p.H + 31) / 32;
    // more wavefronts before more columns each: a wavefront's loads, splits and products are a serial chain
    if (ksteps <= 4) return launch_lstm<4, 1>(p, a->directions, st);
    if (ksteps <= 8) return launch_lstm<8, 1>(p, a->directions, st);
    if (ksteps <= 16) return launch_lstm<8, 2>(p, a->directions, st);
    return launch_lstm<8, 4>(p, a->directions, st);
}

}  // extern "C"
