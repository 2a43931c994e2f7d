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
// operand layout (16 batch rows x 16 columns per load), multiplies them with all four gate
// tiles, and the partial sums meet in LDS; wavefront w of the first four then finishes units 4 w .. 4 w + 3
// of the 16 rows, with c in registers.  ceil(hidden / 16) blocks serve 16 batch rows of one
// direction; other rows and the other direction are independent groups in the same grid.
//
// Input.  Up to 512 columns a block also keeps the input weights of its units, in wavefronts of their own: they
// take the input product of the next step while h travels to the other blocks.  Stacked layers then
// share the launch: layer k reads h[t] of layer k - 1 from that one's output as it appears, so L layers
// take little more than the steps of one.  The second weight halves the blocks
// per CU; where that would mean more launches than it saves (lq_lstm_fused_layers), or beyond 512 columns,
// the input products of all steps are taken beforehand (`gx`) and a layer is a launch of its own.
//
// Exchange.  The blocks of a group hand h[t] to each other through a ring of four steps in device memory, laid out as
// the loads read it: a block writes eight whole 128-byte lines, a load is 1 KiB in a row.  Empty words hold a bit pattern no h
// can have (all ones, a NaN); h is written through to device scope, and a wavefront re-reads what is missing of h[t-1]
// until every word is there - no flags, no barrier, one memory trip each way per step.  A block empties its slot again two
// steps before it is written.  Layers above read their input from the output y of the layer below, emptied before the launch.
//
// Order of the loads.  A CU returns loads in the order they were issued, so an input load that misses the L2 ahead of the
// loads of h holds those up: input loads are issued when h has arrived (a barrier tells), for the step after
// the next one.
//
// Progress.  A block waits only for blocks of its own launch, so all of them have to be resident: the
// launcher bounds the grid by what the device holds of this kernel over the number of hardware queues
// that streams share (four unless GPU_MAX_HW_QUEUES says more; a queue starts a launch only after the one
// before it is fully placed), and larger batches run as several launches.  A wait is bounded besides:
// after kSpinLimit reads a wavefront gives up for the rest of the sequence.  It is out of step with the others then, and the ring may
// hold any step of theirs, so its sums are NaN from there on, and with them all that the block computes and hands out.
//
// hidden 512, 512 inputs, 16 rows, 64 steps: the kernel takes 157 us, 2.45 per step (1.9 at hidden 256, 1.56 at 128).  Of a step's
// 5700 cycles (timestamps) 780 pass before the first read, 1650 with the 32 KiB of h that a CU reads past its L2 (940 at hidden
// 128), 2040 in splits and products, 80 at the barrier, 1130 with sums and gates.  A second such layer adds 11 us (168): two steps,
// and what its input wavefronts wait for on each of the others, y of the layer below, which they read row by row.  It was 272 when h
// was read from y's rows too (every line twice), the input loads stood between h and its products, and one set of wavefronts took
// both products.  Placing a group's blocks on one XCD and exchanging through its L2 instead measured 150 against 153 us for one
// layer (sums in one chain then): not worth the placement.
#include <cmath>
#include <cstdlib>
#include <type_traits>
#include "common.hpp"
#include "lstm_gates.hpp"

using namespace lq;

namespace {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef float v2f __attribute__((ext_vector_type(2)));

constexpr int kUnits = 16, kRows = 16;     // hidden units of a block, batch rows of a group
constexpr unsigned kEmpty = 0xffffffffu;   // a word of h that has not been written
constexpr unsigned kNan = 0x7fc00000u;
constexpr int kSpinLimit = 1 << 20;        // about a second of waiting for one step
constexpr int kScopeDevice = 16;           // "sc1" cache-policy bit of buffer accesses
constexpr int kSlots = 4;                  // steps of h that a ring holds
constexpr int kSlotWords = kUnits * kRows; // of one block's h of one step
// partial sums of a gate tile in LDS: four rows of 64 lanes, the rows 4 banks apart (read four units x 16 rows at a time)
constexpr int kGateRow = 68, kGateFloats = 4 * kGateRow;

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
    unsigned* rings;             // [part][group][slot][block of units][kSlotWords]
    long ring_words;             // of all of them
    int T, B, H, I, row0, dir0, stacked, spins;
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
// Columns of a wavefront.  An instruction's 32 columns are two runs of 16, of which the lane's quarter has four each
// (`kRun` apart): a lane's 16-byte loads then lie beside those of the other quarters, 64 bytes of a row per load.  Which
// column is which k of the instruction does not matter as long as the weight is held in the same order.
constexpr int kRun = 16;

// Gate tiles of a weight [4 H][K] as bfloat16 operands: rows `unit` + g H, this lane's eight columns per instruction, all
// of them requested before the first is used (columns past K are zero: four codes that end with the row are shifted).
template <int KP>
__device__ __forceinline__ void load_weights(v8bf (&wf)[4][KP], const int8_t* w, int H, int unit, int k_lane, int K) {
    uint32_t raw[4][KP][2];
    if (K >= 4) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int8_t* const row = w + (size_t(g) * H + unit) * K;
#pragma unroll
            for (int i = 0; i < 2 * KP; ++i) {
                const int k = k_lane + i * kRun;
                __builtin_memcpy(&raw[g][i >> 1][i & 1], row + (k < K - 4 ? k : K - 4), 4);
            }
        }
#pragma unroll
        for (int i = 0; i < 2 * KP; ++i) {
            const int past = k_lane + i * kRun - (K - 4);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint32_t four = raw[g][i >> 1][i & 1];
                raw[g][i >> 1][i & 1] = past <= 0 ? four : past < 4 ? four >> (8 * past) : 0u;
            }
        }
    } else {
        for (int g = 0; g < 4; ++g)
            for (int i = 0; i < 2 * KP; ++i) {
                uint32_t four = 0;
                for (int e = 0; e < 4; ++e)
                    if (k_lane + i * kRun + e < K)
                        four |= uint32_t(uint8_t(w[(size_t(g) * H + unit) * K + k_lane + i * kRun + e])) << (8 * e);
                raw[g][i >> 1][i & 1] = four;
            }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
#pragma unroll
        for (int i = 0; i < KP; ++i) {
            v4u pairs;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t two = raw[g][i][e >> 1] >> (16 * (e & 1));
                pairs[e] = codes_bf16(int(int8_t(two)), int(int8_t(two >> 8)));
            }
            wf[g][i] = __builtin_bit_cast(v8bf, pairs);
        }
}
// device-scope access to what follows element `at` of an array of `elems` floats
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words_from(const float* base, long at, long elems) {
    const long bytes = (elems - at) * 4;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base) + at, 0,
                                             bytes < 0x7fffffffl ? int(bytes) : 0x7fffffff, 0x00020000);
}
template <int KP, int SCOPE>
__device__ __forceinline__ void load_columns(v4u (&raw)[KP][2], __amdgpu_buffer_rsrc_t src, unsigned off, unsigned missing = ~0u) {
#pragma unroll
    for (int i = 0; i < 2 * KP; ++i)
        if (missing >> i & 1)
            raw[i >> 1][i & 1] = __builtin_amdgcn_raw_buffer_load_b128(src, off + unsigned(i * kRun) * 4, 0, SCOPE);
}
// columns from `left` on (of another direction, row or step) become zero
template <int KP>
__device__ __forceinline__ void mask_columns(v4u (&raw)[KP][2], int left) {
#pragma unroll
    for (int i = 0; i < 2 * KP; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (i * kRun + e >= left) raw[i >> 1][i & 1][e] = 0u;
}
// the loads of which some lane has words that have not been written
template <int KP>
__device__ __forceinline__ unsigned missing_words(const v4u (&raw)[KP][2]) {
    unsigned missing = 0;
#pragma unroll
    for (int i = 0; i < 2 * KP; ++i) {
        const v4u r = raw[i >> 1][i & 1];
        const unsigned a = r[0] > r[1] ? r[0] : r[1], b = r[2] > r[3] ? r[2] : r[3];
        if (__builtin_amdgcn_ballot_w64((a > b ? a : b) == kEmpty)) missing |= 1u << i;
    }
    return missing;
}
// eight columns as three operands, whose sum they are
__device__ __forceinline__ void split_columns(v4u (&parts)[3], const v4u (&raw)[2]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const v4u r = raw[e >> 1];
        uint32_t hh, mm, ll;
        split3(__uint_as_float(r[(2 * e) & 3]), __uint_as_float(r[(2 * e + 1) & 3]), hh, mm, ll);
        parts[0][e] = hh, parts[1][e] = mm, parts[2][e] = ll;
    }
}
// acc[g] += columns . codes of gate g: three exact part products each, the smaller ones added up among themselves first
// (against float64, outputs of eight sizes: 0.9 to 1.3e-7, 1.1 to 1.7e-7 as one chain in two halves; 2 % of a step).  The splits of an instruction's columns come
// before the products of the one before, which they do not wait for.
template <int KP>
__device__ __forceinline__ void multiply(v4f (&acc)[4], const v4u (&raw)[KP][2], const v8bf (&wf)[4][KP]) {
    v4u parts[2][3];
    v4f low[4];  // of the two smaller parts: their sums are rounded at their own size
#pragma unroll
    for (int g = 0; g < 4; ++g) low[g] = v4f{0.f, 0.f, 0.f, 0.f};
    split_columns(parts[0], raw[0]);
#pragma unroll
    for (int i = 0; i < KP; ++i) {
        if (i + 1 < KP) split_columns(parts[(i + 1) & 1], raw[i + 1]);
#pragma unroll
        for (int q = 2; q >= 0; --q)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                v4f& to = q == 0 ? acc[g] : low[g];
                to = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, parts[i & 1][q]), wf[g][i], to, 0, 0, 0);
            }
    }
    // (every product is issued before the first sum waits: for a few registers less the compiler would go gate by gate)
    if (KP == 1) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[g] += low[g];
}

// W wavefronts for h, each with KPW instructions of 32 hidden columns (hidden <= 32 W KPW), and XW for the
// input, each with KX of 32 input columns; XW = 0 reads the input products from gx.
//
// The two roles meet at one barrier a step.  An h wavefront waits for its columns of h[t-1], multiplies them, adds the
// input product its partner left in LDS and puts its partial sums there; behind the barrier the first four finish the
// gates.  An input wavefront is a step ahead and off the chain: x[t+1] arrives while it multiplies x[t].
template <int W, int KPW, int XW, int KX>
struct LstmForm {
    static constexpr int kThreads = (W + XW) * 64;
    static constexpr int kPartFloats = W * 4 * kGateFloats, kInputFloats = XW * 4 * 4 * 64;
    static constexpr int kLdsBytes = 2 * (kPartFloats + kInputFloats) * 4;
    // wavefronts of a SIMD: the weights take 16 registers per instruction, the rest about 100.  At most as many as the
    // registers used leave room for: the compiler keeps further ones out by allotting more registers, which the occupancy query of
    // split_lstm does not see (two per SIMD at hidden 128, 114 registers: it counted on two blocks per CU where one fitted).
    static constexpr int kPerSimd = XW == 0 && KPW <= 2 ? 4 : 2;
    static constexpr int kMostPerSimd = KPW == 1 && KX == 1 ? 4 : kPerSimd;
};

template <int W, int KPW, int XW, int KX>
__global__ __launch_bounds__((W + XW) * 64)
    __attribute__((amdgpu_waves_per_eu(LstmForm<W, KPW, XW, KX>::kPerSimd, LstmForm<W, KPW, XW, KX>::kMostPerSimd)))
void lstm_sequence_kernel(LstmArgs p) {
    using Form = LstmForm<W, KPW, XW, KX>;
    extern __shared__ __align__(16) float lds[];
    // partial sums [step parity][wavefront][gate][kGateFloats]; scaled input products [parity][wavefront][gate][lane][row]
    float* const part = lds;
    float* const inputs = lds + 2 * Form::kPartFloats;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ln = lane & 15, lq4 = lane >> 4;
    const int z = p.dir0 + blockIdx.z, d = p.stacked ? 0 : z, H = p.H;
    const int u0 = blockIdx.x * kUnits, m0 = p.row0 + blockIdx.y * kRows;
    float* const y = p.y[z];
    // the row whose h and x this lane reads; rows past the batch repeat the last one
    const int in_batch = m0 + ln < p.B ? m0 + ln : p.B - 1;
    const int tile_unit = u0 + ln < H ? u0 + ln : H - 1;  // units past H are computed and never stored

    if constexpr (XW > 0) {
        if (wave >= W) {
            // ---- the input of this part: x, or the output of the layer below
            const int w = wave - W;
            const bool above = p.stacked && z > 0;
            const float* const in = above ? p.y[above ? z - 1 : 0] : p.x;
            const int I = above ? H : p.I;
            const long in_step = above ? p.y_step : p.x_step, in_row = above ? p.y_row : p.x_row;
            const long in_elems = above ? p.y_elems : p.x_elems;
            const int k_lane = w * KX * 32 + lq4 * 4;
            const bool whole = (w + 1) * KX * 32 <= I;
            v8bf wf[4][KX];
            float scale[4];
            load_weights<KX>(wf, p.wx[z], H, tile_unit, k_lane, I);
#pragma unroll
            for (int g = 0; g < 4; ++g) scale[g] = p.wx_scale[z][g * H + tile_unit];
            const unsigned off = unsigned(in_batch * in_row + k_lane) * 4;
            bool waiting = above;
            v4u raw[KX][2], next[KX][2];  // of the step to multiply and of the one after
            auto request = [&](v4u (&raw)[KX][2], int s, unsigned missing) {
                const __amdgpu_buffer_rsrc_t src = words_from(in, long(d ? p.T - 1 - s : s) * in_step, in_elems);
                if (above) load_columns<KX, kScopeDevice>(raw, src, off, missing);
                else load_columns<KX, 0>(raw, src, off);
            };
            auto product = [&](v4u (&raw)[KX][2], int s) {
                for (int spin = 0;; ++spin) {
                    if (!whole) mask_columns<KX>(raw, I - k_lane);
                    const unsigned missing = waiting ? missing_words<KX>(raw) : 0;
                    if (!missing) break;
                    if (spin >= p.spins) waiting = false;  // (what is not written is NaN, what is written is right)
                    asm volatile("" ::: "memory");  // read again: the words change under the loop
                    request(raw, s, missing);
                }
                v4f acc[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
                multiply<KX>(acc, raw, wf);
                v4f* const out = reinterpret_cast<v4f*>(inputs + (s & 1) * Form::kInputFloats) + w * 4 * 64 + lane;
#pragma unroll
                for (int g = 0; g < 4; ++g) out[g * 64] = acc[g] * scale[g];
            };
            auto step = [&](v4u (&raw)[KX][2], v4u (&next)[KX][2], int s) {
                lds_barrier();  // h[s - 1] is there: until the next wait for h the loads are the input's
                request(next, s + 2 < p.T ? s + 2 : p.T - 1, ~0u);
                lds_barrier();  // the products of step s are done: the matrix unit is the input's
                if (s + 1 < p.T) product(raw, s + 1);  // (this half of `inputs` was read at step s - 1)
            };
            request(raw, 0, ~0u);
            product(raw, 0);
            request(raw, 1 < p.T ? 1 : 0, ~0u);
            for (int s = 0; s < p.T; s += 2) {
                step(raw, next, s);
                if (s + 1 < p.T) step(next, raw, s + 1);
            }
            return;
        }
    }

    // ---- the block's weights: tile g = gate g of units u0 .. u0+15, this wavefront's columns
    const int k_lane = wave * KPW * 32 + lq4 * 4;
    v8bf wf[4][KPW];
    float scale_h[4];  // of the unit whose products this lane accumulates
    load_weights<KPW>(wf, p.w[z], H, tile_unit, k_lane, H);
#pragma unroll
    for (int g = 0; g < 4; ++g) scale_h[g] = p.w_scale[z][g * H + tile_unit];
    // ---- the element this lane finishes (wavefronts 0..3)
    const int tile_row = lane >> 2, unit = u0 + 4 * wave + (lane & 3), row = m0 + tile_row;
    const bool mine = wave < 4 && unit < H && row < p.B;
    float bias[4], c = 0.0f, hv = 0.0f;
    const size_t state = (size_t(z) * p.B + (row < p.B ? row : 0)) * H + unit;
#pragma unroll
    for (int g = 0; g < 4; ++g) bias[g] = mine && p.b_ih[z] ? p.b_ih[z][g * H + unit] + p.b_hh[z][g * H + unit] : 0.0f;
    if (mine && p.c0) c = p.c0[state];
    const float* const gx_lane = XW > 0 ? nullptr : p.gx[d] + size_t(mine ? row : 0) * p.gx_row + (mine ? unit : 0);
    float gx[4], gx_next[4];
    auto request_gx = [&](int s) {
        const float* const at = gx_lane + size_t(d ? p.T - 1 - s : s) * p.gx_step;
#pragma unroll
        for (int g = 0; g < 4; ++g) gx_next[g] = at[size_t(g) * H];
    };
    if (XW == 0 && wave < 4) request_gx(0);
    // ---- the ring of this group
    const unsigned slot_bytes = unsigned(gridDim.x) * kSlotWords * 4;
    const long group = long(z) * ((p.B + kRows - 1) / kRows) + m0 / kRows;
    const __amdgpu_buffer_rsrc_t ring = __builtin_amdgcn_make_buffer_rsrc(
        p.rings + group * kSlots * gridDim.x * kSlotWords, 0, int(slot_bytes * kSlots), 0x00020000);
    const unsigned h_off = unsigned(wave * 2 * KPW * kSlotWords + lane * 4) * 4;
    // the loads behind which there is a block; the columns of the others stay zero
    const int blocks_left = int(gridDim.x) - wave * 2 * KPW;
    const unsigned present = blocks_left <= 0 ? 0u : blocks_left >= 2 * KPW ? ~0u : (1u << blocks_left) - 1u;
    const unsigned own_off = (blockIdx.x * kSlotWords + wave * 64 + lane) * 4;  // four units of a row side by side
    const int own_sum = (tile_row & 3) * kGateRow + (tile_row >> 2) * 16 + 4 * wave + (lane & 3);
    bool waiting = true;
    unsigned bits = 0;
    auto store_y = [&](int s) {
        const int t = d ? p.T - 1 - s : s;
        const __amdgpu_buffer_rsrc_t dst = words_from(y, long(t) * p.y_step + long(d) * H, p.y_elems);
        __builtin_amdgcn_raw_buffer_store_b32(bits, dst, unsigned(row * p.y_row + unit) * 4, 0, kScopeDevice);
    };
    v4u raw[KPW][2];
#pragma unroll
    for (int i = 0; i < KPW; ++i) raw[i][0] = raw[i][1] = v4u{0u, 0u, 0u, 0u};
    if (p.h0) {
#pragma unroll
        for (int i = 0; i < KPW; ++i)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int k = k_lane + (i * 2 + (e >> 2)) * kRun + (e & 3);
                const float v = p.h0[(size_t(z) * p.B + in_batch) * H + (k < H ? k : 0)];
                raw[i][e >> 2][e & 3] = k < H ? __float_as_uint(v) : 0u;
            }
    }
    for (int s = 0; s < p.T; ++s) {
        v4f in_acc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) in_acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
        if (s > 0) {
            const unsigned slot = unsigned((s - 1) % kSlots) * slot_bytes;
            // A read that meets the writes of the same line delays both, and one that comes too early costs a whole trip
            // more: the first is issued when most of h has arrived.  Steps of hidden 512 / 256 / 128, 16 rows, in us: at
            // once 2.75 / 2.05 / 1.6, after 448 cycles 2.25 / 1.7 / 1.5, after 576 2.2 / 1.7 / 1.45, after 896 2.3 / 1.8 / 1.55
            // (sums and gates of then; now 64 cycles either way are within 2 %, and 128 late costs 1 to 2 %).
            if (gridDim.x > 16) __builtin_amdgcn_s_sleep(8);
            else __builtin_amdgcn_s_sleep(5);
            unsigned missing = present;
            for (int spin = 0;; ++spin) {
                asm volatile("" ::: "memory");  // read again: the words change under the loop
#pragma unroll
                for (int i = 0; i < 2 * KPW; ++i)
                    if (missing >> i & 1)
                        raw[i >> 1][i & 1] =
                            __builtin_amdgcn_raw_buffer_load_b128(ring, h_off + unsigned(i * kSlotWords) * 4, slot, kScopeDevice);
                missing = waiting ? missing_words<KPW>(raw) : 0;
                if (!missing) break;
                if (spin >= p.spins) waiting = false;
            }
            // What this wavefront stored in the last step is there before it hands out more (see where a slot is emptied).
            // The loads above have waited for it; a wavefront whose columns no block has made none.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        if constexpr (XW > 0) {
            lds_barrier();
            if (wave < XW) {
                const v4f* const left = reinterpret_cast<const v4f*>(inputs + (s & 1) * Form::kInputFloats) + wave * 4 * 64 + lane;
#pragma unroll
                for (int g = 0; g < 4; ++g) in_acc[g] = left[g * 64];
            }
        }
        if (XW == 0 && wave < 4) {
#pragma unroll
            for (int g = 0; g < 4; ++g) gx[g] = gx_next[g];
            request_gx(s + 1 < p.T ? s + 1 : s);
        }
        v4f acc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[g] = v4f{0.f, 0.f, 0.f, 0.f};
        multiply<KPW>(acc, raw, wf);
        float* const parts = part + (s & 1) * Form::kPartFloats;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            acc[g] = acc[g] * scale_h[g] + in_acc[g];
#pragma unroll
            for (int r = 0; r < 4; ++r) parts[(wave * 4 + g) * kGateFloats + r * kGateRow + lane] = acc[g][r];
        }
        if (!waiting)  // (once more, and not in place of the sums: what gives them another value here costs a step 3 %)
            for (int i = lane; i < 4 * kGateFloats; i += 64) parts[wave * 4 * kGateFloats + i] = __uint_as_float(kNan);
        // (a buffer is written again two steps later, after the next step's barrier: by then it has been read)
        lds_barrier();
        if (wave < 4) {
            float raw4[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float sum = parts[g * kGateFloats + own_sum];
#pragma unroll
                for (int w = 1; w < W; ++w) sum += parts[(w * 4 + g) * kGateFloats + own_sum];
                raw4[g] = (XW > 0 ? sum : gx[g] + sum) + bias[g];
            }
            const float ig = sigmoid(raw4[0]), fg = sigmoid(raw4[1]), gg = tanh_gate(raw4[2]), og = sigmoid(raw4[3]);
            c = fg * c + ig * gg;
            hv = og * tanh_gate(c);
            bits = __float_as_uint(hv);
            bits = bits == kEmpty ? kNan : bits;  // a NaN, but not the one that means "not written"
            if (s + 1 < p.T) {
                __builtin_amdgcn_raw_buffer_store_b32(unit < H ? bits : 0u, ring, own_off, unsigned(s % kSlots) * slot_bytes,
                                                      kScopeDevice);
                // Every block has taken h[s - 2], or it would not have handed out h[s - 1]: its slot is for h[s + 2].  The
                // next step waits for this store before it hands out h[s + 1], so nobody who has that still finds h[s - 2] here.
                if (s >= 2)
                    __builtin_amdgcn_raw_buffer_store_b32(kEmpty, ring, own_off, unsigned((s + 2) % kSlots) * slot_bytes,
                                                          kScopeDevice);
            }
            if (mine) store_y(s);
        }
    }
    if (mine) {
        p.h_n[state] = hv;
        p.c_n[state] = c;
    }
}

// every word that is handed from block to block "not written yet": the rings, and the outputs of the layers below others
__global__ __launch_bounds__(256) void lstm_empty_kernel(LstmArgs p) {
    unsigned* const words = blockIdx.y ? reinterpret_cast<unsigned*>(p.y[blockIdx.y - 1]) : p.rings;
    const long n = blockIdx.y ? p.y_elems : p.ring_words, stride = long(gridDim.x) * 256;
    for (long i = long(blockIdx.x) * 256 + threadIdx.x; i < n; i += stride) words[i] = kEmpty;
}

// Launches of one kernel form: 16-row groups of one direction or of one stack, as many at once as may be.
struct LstmSplit {
    int per_group, groups, at_once, both;  // blocks of a group; groups; groups of a launch; its parts
    int launches;
};

template <int W, int KPW, int XW, int KX>
int split_lstm(int B, int H, int parts, bool stacked, LstmSplit* out) {
    static DeviceOnce once;
    static int capacity[32] = {0};  // blocks of this kernel the device holds at once
    int dev = 0;
    LQ_HIP(hipGetDevice(&dev));
    const int rc = device_once(once, [&]() -> int {
        using Form = LstmForm<W, KPW, XW, KX>;
        int per_cu = 0;
        hipDeviceProp_t prop;
        const auto kernel = lstm_sequence_kernel<W, KPW, XW, KX>;
        LQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   Form::kLdsBytes));
        LQ_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, Form::kThreads, Form::kLdsBytes));
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

template <int W, int KPW, int XW, int KX>
int launch_lstm(LstmArgs p, int parts, hipStream_t st) {
    LstmSplit s;
    if (int rc = split_lstm<W, KPW, XW, KX>(p.B, p.H, parts, p.stacked != 0, &s)) return rc;
    LQ_REQUIRE(s.launches >= 1, LQ_ERR_NOT_IMPLEMENTED, "lstm_sequence: %d x hidden %d do not fit the device at once",
               p.stacked ? parts : 1, p.H);
    p.ring_words = long(parts) * s.groups * kSlots * s.per_group * kSlotWords;
    const auto lock = scratch_lock(st);
    void* tmp = nullptr;
    if (int rc = call_buffer(8, size_t(p.ring_words) * 4, st, &tmp)) return rc;
    p.rings = static_cast<unsigned*>(tmp);
    const int below = p.stacked ? parts - 1 : 0;
    const long most = below && p.y_elems > p.ring_words ? p.y_elems : p.ring_words, fill_blocks = (most + 1023) / 1024;
    hipLaunchKernelGGL(lstm_empty_kernel, dim3(unsigned(fill_blocks < 2048 ? fill_blocks : 2048), unsigned(below + 1)),
                       dim3(256), 0, st, p);
    LQ_CHECK_LAUNCH("lstm_empty");
    for (p.dir0 = 0; p.dir0 < parts; p.dir0 += s.both)
        for (int g = 0; g < s.groups; g += s.at_once) {
            p.row0 = g * kRows;
            const int n = s.groups - g < s.at_once ? s.groups - g : s.at_once;
            hipLaunchKernelGGL((lstm_sequence_kernel<W, KPW, XW, KX>),
                               dim3(unsigned(s.per_group), unsigned(n), unsigned(s.both)),
                               dim3(unsigned(LstmForm<W, KPW, XW, KX>::kThreads)), unsigned(LstmForm<W, KPW, XW, KX>::kLdsBytes),
                               st, p);
            LQ_CHECK_LAUNCH("lstm_sequence");
        }
    return LQ_OK;
}

template <int N>
using Int = std::integral_constant<int, N>;

// f(W, KPW, XW, KX) for the form that serves `hidden` columns and `inputs` (0: gates_x).
template <typename F>
int with_form(int hidden, int inputs, F f) {
    const int ks = (hidden + 31) / 32, kx = (inputs + 31) / 32;
    if (kx == 0) {
        if (ks <= 4) return f(Int<4>(), Int<1>(), Int<0>(), Int<0>());
        if (ks <= 8) return f(Int<8>(), Int<1>(), Int<0>(), Int<0>());
        if (ks <= 16) return f(Int<8>(), Int<2>(), Int<0>(), Int<0>());
        return f(Int<8>(), Int<4>(), Int<0>(), Int<0>());
    }
    if (ks <= 4 && kx <= 4) return f(Int<4>(), Int<1>(), Int<4>(), Int<1>());
    if (ks <= 8) return kx <= 8 ? f(Int<4>(), Int<2>(), Int<4>(), Int<2>()) : f(Int<4>(), Int<2>(), Int<4>(), Int<4>());
    return kx <= 8 ? f(Int<4>(), Int<4>(), Int<4>(), Int<2>()) : f(Int<4>(), Int<4>(), Int<4>(), Int<4>());
}
constexpr int kMaxFused = 512;  // hidden and input columns of a form that takes the input product
constexpr int kMaxHidden = 1024;

// A step of all rows: one launch of the recurrence per rows that fit the device, or a float32 GEMM and a gate kernel
// (lq_lstm_cell_f32) on decoded weights, issued from Python.  Measured, us per step of both: hidden 64, 8192 rows 19.0 /
// 23.6; 128, 4096 rows 19.7 / 25.8, 8192 rows 45.6 / 35.4; 256, 1024 rows 19.0 / 28.7, 1500 rows 28.0 / 31.0, 2048 rows 39.5 /
// 34.0; 512, 512 rows 27.2 / 41.3, 768 rows 40.3 / 43.4, 1024 rows 54.8 / 45.2; 768, 128 rows 25.4 / 51.8, 256 rows 50.5 / 53.6,
// 384 rows 76.0 / 54.6; 1024, 128 rows 26.6 / 64.8, 256 rows 54.2 / 66.6, 384 rows 80.9 / 67.7; 1024 in two directions, 256 rows
// 111 / 131.  The estimates below are those of an earlier recurrence, a fifth to two thirds above these (a launch's step is 2.4 up
// to hidden 256, 3.3 beyond), and 3 to 17 % above for the GEMM.  So the line lies low: of the sizes here hidden 256 with 1500 rows,
// 512 with 768, 768 and 1024 with 256 go to the GEMM for 6 to 23 % more.
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
    const int rc = with_form(hidden, 0, [&](auto w, auto k, auto xw, auto x) {
        return split_lstm<w(), k(), xw(), x()>(batch, hidden, directions, false, &s);
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
    // Costs per layer in steps of the recurrence.  An input product in a GEMM of its own, with the decoded weight it reads, is worth
    // twelve and, where inputs and hidden are 512, up to 24.  us of the device with the GEMM / with more launches: 512 -> 512, 64
    // rows, 16 steps 111 / 101, 24 139 / 139, 32 167 / 174; 256 -> 256, 128 rows, 16 steps 78 / 76, 24 97 / 106; 128 -> 512, 64
    // rows, 12 steps 76 / 76; 128 -> 128, 400 rows, 12 steps 58 / 51, 24 86 / 89; 200 -> 300 in two directions, 33 rows, 10 steps
    // 98 / 88, 20 135 / 154.
    constexpr long kGemm = 12;
    LstmSplit s;
    int rc = with_form(hidden, 0, [&](auto w, auto k, auto xw, auto x) { return split_lstm<w(), k(), xw(), x()>(batch, hidden, directions, false, &s); });
    if (rc) return rc;
    double best = s.launches ? double(s.launches) * steps + kGemm * directions : 1e30;
    for (int n = 1; n <= (directions == 1 ? (layers < kParts ? layers : kParts) : 1); ++n) {
        const int columns = n > 1 && hidden > inputs ? hidden : inputs;
        rc = with_form(hidden, columns, [&](auto w, auto k, auto xw, auto x) {
            return split_lstm<w(), k(), xw(), x()>(batch, hidden, directions == 2 ? 2 : n, n > 1, &s);
        });
        if (rc) return rc;
        const double cost = double(s.launches) * (steps + n - 1) / n;
        if (s.launches && cost < best) best = cost, *fused = n;
    }
    return LQ_OK;
}

int lq_lstm_sequence_f32(const lq_lstm_args* a, lq_stream stream) { return lq_lstm_sequence_spins_f32(a, kSpinLimit, stream); }

int lq_lstm_sequence_spins_f32(const lq_lstm_args* a, int spins, lq_stream stream) {
    LQ_REQUIRE(spins >= 0, LQ_ERR_VALUE, "lstm_sequence: %d spins", spins);
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
    p.T = a->steps, p.B = a->batch, p.H = a->hidden, p.spins = spins < kSpinLimit ? spins : kSpinLimit;
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
    return with_form(p.H, columns, [&](auto w, auto k, auto xw, auto x) { return launch_lstm<w(), k(), xw(), x()>(p, parts, as_stream(stream)); });
}

}  // extern "C"
