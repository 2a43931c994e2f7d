// Weight-only int4 / int8 product for large batches, the codes decoded inside the product:
//
//   y[m, n] = sum over groups g of  s[n, g] * (sum_{k in g} c[n, k] x[m, k])  +  b[n, g] * (sum_{k in g} x[m, k])
//
// (lucid/quantization/_qgemm.py:167-171).  As in the small-batch kernel the codes are one operand of
// v_mfma_f32_16x16x32_bf16, exactly, and x the other as three bfloat16 parts (exact), so a product of
// float32 accuracy costs three instructions where two float32 operands split the same way cost six.
//
// Bound: the matrix cores, 3 x 2 M N K operations; beside them each 64 k of a wavefront's tile take
// one fused multiply-add per element and term for the scales and biases, and the decoding of the codes.
//
// wq_prepare_kernel lays the operands of the epilogue-in-the-loop out once per call: x as its three parts
// in operand order (a fragment = 16 rows x 32 k of one part = 1 KiB, the lanes' 16 bytes in lane order), a
// stage of 64 k of all rows after the other; the sums of x over each segment of 64 (or 32) k; and the
// scale and bias of each segment as pairs, column after column.  Every block of the product would
// otherwise split its rows again (N / 256 times) and gather scales a cache line apart.
//
// wq_gemm_kernel: a block of eight wavefronts takes 32 MT rows x 64 NT columns, wavefront (i, j) the
// rows 16 MT i .. and the columns 16 NT j ..  Everything a stage needs - x fragments, packed codes, sums
// and scales - goes from memory straight into LDS in pieces of 1 KiB per wavefront and instruction, in a
// ring of RING stages: every wavefront issues the same number of loads per stage, so "stage s has
// arrived" is a count of outstanding loads and RING - 1 stages of them hide the latency (with one stage
// in flight a 64-k step took 2.8 us, of which 0.7 us were matrix instructions).  The segment sums stay
// in accumulators of their own until their group's scale has been applied: 8 MT NT registers per lane in
// all, which with two wavefronts per SIMD (one hides the other's scaling and LDS reads) caps MT NT at 12.
//
// The sums of a group are scaled while the next group is multiplied (two sets of accumulators take turns).
// 333 x 11008 x 4096, int4, groups of 128: 112 us, 0.80 PFLOP/s in bfloat16 terms (a library product of plain
// bfloat16 operands reaches 1.18 on the card); decoding to float32 (109 us) and a float32 GEMM (286 us) before.
// Of the 112, 11 are for centred codes (wq_codes): their decode is vector work that the matrix instructions do not
// hide.  (Interleaving the two by scheduling groups, two or three vector instructions per matrix one: 114.)
//
// The codes' 16-byte chunks are placed in LDS at chunk ^ (row / 4) (int8) or chunk ^ (row / 8) (int4), which
// spreads the 16 rows of an operand read over all banks; the permutation is applied on the global side.
#include "wq_pack.hpp"

using namespace lq;

namespace {

typedef unsigned v2u __attribute__((ext_vector_type(2)));

constexpr int kPiece = 1024;  // bytes one wavefront moves into LDS with one instruction

// One launch, two kinds of blocks.  The first `split_blocks`: one thread = eight consecutive k of one
// row; a block = 16 rows x two stages.  The others: 32 groups of 64 columns, read row by row and turned in LDS.
// 333 x 11008 x 4096 int4 of 128 10.4 -> 8.8 us, 100 x 11008 x 4096 of 32 21.0 -> 11.5: a thread that took four groups of a column for itself
// read 16 bytes of a line that the blocks of the next groups, on other XCDs, fetched again.  Few groups are not worth the turn, a row is
// a line or two: there a thread takes up to four consecutive groups of a column as before (the whole call, turned / not: 88 x 10080 x
// 640 int4 of 128 15.0 / 13.7, 198 x 5378 x 384 of 32 14.9 / 13.6, 351 x 4212 x 512 of 32 17.8 / 17.1; equal at 24 groups).
constexpr int kSbGroups = 32, kSbColumns = 64, kSbFew = 24;
template <int BITS>
__global__ __launch_bounds__(256) void wq_prepare_kernel(const float* __restrict__ x, const float* __restrict__ scales,
                                                         const float* __restrict__ biases, int M, int N, int K,
                                                         int gs_shift, int mtiles, int bm, int n_pad, int stages,
                                                         int segs, unsigned split_blocks, uint4* __restrict__ parts,
                                                         float* __restrict__ xsum, float2* __restrict__ sb) {
    if (blockIdx.x >= split_blocks && stages * segs < kSbFew * (segs == 2 ? 1 : (1 << gs_shift) / 64)) {
        const int groups = K >> gs_shift;
        const int per = segs == 2 ? 1 : (1 << gs_shift) / 64;  // segments per group
        const unsigned idx = (blockIdx.x - split_blocks) * 256 + threadIdx.x;
        const unsigned quad = idx / unsigned(n_pad), n = idx - quad * unsigned(n_pad);
        const int g0 = int(quad) * 4;
        float s[4] = {0.f, 0.f, 0.f, 0.f}, b[4] = {0.f, 0.f, 0.f, 0.f};
        if (n < unsigned(N)) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (g0 + e < groups) s[e] = scales[size_t(n) * groups + g0 + e], b[e] = biases[size_t(n) * groups + g0 + e];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
            for (int r = 0; r < per; ++r)
                if ((g0 + e) * per + r < stages * segs)
                    sb[size_t((g0 + e) * per + r) * n_pad + n] = float2{kWqUnit<BITS> * s[e], b[e] - float(kWqCentre<BITS>) * s[e]};
        return;
    }
    if (blockIdx.x >= split_blocks) {
        __shared__ float2 tile[kSbGroups][kSbColumns + 1];
        const int groups = K >> gs_shift;
        const int per = segs == 2 ? 1 : (1 << gs_shift) / 64;  // segments per group
        const unsigned idx = blockIdx.x - split_blocks, across = unsigned(n_pad) / kSbColumns;
        const int n0 = int(idx % across) * kSbColumns, first = int(idx / across) * kSbGroups;
        const int all = stages * segs / per, here = all - first < kSbGroups ? all - first : kSbGroups;  // groups, past K too
        // four groups per lane, and of a row's 32 side by side; the last four of a row where those asked for run past it
        float4 sv[2], bv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int n = n0 + u * 32 + int(threadIdx.x >> 3), g0 = first + int(threadIdx.x & 7) * 4;
            const size_t row = size_t(n < N ? n : N - 1) * groups;
            if (groups >= 4) {
                const size_t from = row + (g0 + 4 <= groups ? g0 : groups - 4);
                __builtin_memcpy(&sv[u], scales + from, 16);
                __builtin_memcpy(&bv[u], biases + from, 16);
            } else {  // uniform
                sv[u] = float4{scales[row], scales[row + groups / 2], scales[row + groups - 1], 0.f};
                bv[u] = float4{biases[row], biases[row + groups / 2], biases[row + groups - 1], 0.f};
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int c = u * 32 + int(threadIdx.x >> 3), q0 = int(threadIdx.x & 7) * 4, g0 = first + q0;
            const bool column = n0 + c < N;
            const float s4[4] = {sv[u].x, sv[u].y, sv[u].z, sv[u].w}, b4[4] = {bv[u].x, bv[u].y, bv[u].z, bv[u].w};
            // element e of the load is group `at + e`: what is past the row is zeros
            const int at = groups < 4 || g0 + 4 <= groups ? g0 : groups - 4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int g = groups < 4 ? (e < groups ? first + e : first + kSbGroups) : at + e, slot = g - first;
                if (column && slot >= q0 && slot < q0 + 4 && slot < here && (groups >= 4 || q0 == 0))
                    tile[slot][c] = float2{kWqUnit<BITS> * s4[e], b4[e] - float(kWqCentre<BITS>) * s4[e]};
            }
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (q0 + e < here && (!column || g0 + e >= groups)) tile[q0 + e][c] = float2{0.f, 0.f};
        }
        __syncthreads();
        for (int i = threadIdx.x; i < here * kSbColumns; i += 256) {
            const int g = i / kSbColumns, c = i % kSbColumns;
            const float2 v = tile[g][c];
            for (int r = 0; r < per; ++r)
                if ((first + g) * per + r < stages * segs) sb[size_t((first + g) * per + r) * n_pad + n0 + c] = v;
        }
        return;
    }
    const unsigned pairs = unsigned(stages + 1) / 2;
    const int mt = int(blockIdx.x / pairs);
    const int stage = int(blockIdx.x - unsigned(mt) * pairs) * 2 + (threadIdx.x >> 7);
    if (stage >= stages) return;
    const int row = (threadIdx.x >> 3) & 15, oct = threadIdx.x & 7;
    const int m = mt * 16 + row, k = stage * 64 + oct * 8;
    float4 a{0.f, 0.f, 0.f, 0.f}, b = a;
    if (m < M && k < K) {  // K is a multiple of 32
        const float* src = x + size_t(m) * K + k;
        __builtin_memcpy(&a, src, 16);
        __builtin_memcpy(&b, src + 4, 16);
    }
    const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
    sum += __shfl_xor(sum, 1, 64);
    sum += __shfl_xor(sum, 2, 64);
    if (segs == 1) sum += __shfl_xor(sum, 4, 64);
    // the sums of a row tile of the product: [stage][tile][segment][bm]
    const int tile = m / bm;
    if ((oct & (segs == 1 ? 7 : 3)) == 0)
        xsum[((size_t(stage) * (mtiles * 16 / bm) + tile) * segs + (segs == 1 ? 0 : oct >> 2)) * bm + (m - tile * bm)] = sum;
    uint32_t d3[3][4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
        wq_split3x2(BITS == 4 ? v[d] : v[2 * d], BITS == 4 ? v[d + 4] : v[2 * d + 1], d3[0][d], d3[1][d], d3[2][d]);
#pragma unroll
    for (int p = 0; p < 3; ++p)
        parts[(((size_t(stage) * mtiles + mt) * 2 + (oct >> 2)) * 3 + p) * 64 + row + 16 * (oct & 3)] =
            uint4{d3[p][0], d3[p][1], d3[p][2], d3[p][3]};
}

// What a stage of one block is made of, in pieces.
template <int BITS, int SEGS, int MT, int NT>
struct WqStage {
    static constexpr int X = 12 * MT;                     // fragments
    static constexpr int SUMS = 1;                        // SEGS x 32 MT floats
    static constexpr int SB1 = (NT + 1) / 2;              // 64 NT pairs of one segment
    static constexpr int SB = SEGS * SB1;
    static constexpr int W = NT * BITS / 2;               // 64 NT rows of 8 BITS bytes
    static constexpr int PIECES = X + SUMS + SB + W;
    static constexpr int PER_WAVE = (PIECES + 7) / 8;
    // as many stages as one block's share of the 160 KiB allows, up to four (two blocks per CU for small tiles)
    static constexpr int FIT = (PIECES <= 26 ? 80 : 160) / PIECES;
    static constexpr int RING = FIT > 4 ? 4 : FIT;
    static_assert(RING >= 2 && PER_WAVE * (RING - 2) <= 63, "");
};

// Scale applications per stage of 64 k; stages per turn of the main loop (an even number of groups: two sets
// of accumulators take turns, and which one is a compile-time matter); stages of a K, whole turns (what
// lies past K is zeros of x).
__host__ __device__ constexpr int wq_segs(int gs) { return gs == 32 ? 2 : 1; }
__host__ __device__ constexpr int wq_unroll(int gs) { return gs == 128 ? 4 : (gs == 64 ? 2 : 1); }
__host__ __device__ constexpr int wq_stages(int K, int gs) {
    return ((K + 63) / 64 + wq_unroll(gs) - 1) / wq_unroll(gs) * wq_unroll(gs);
}

// s_waitcnt immediate for vmcnt <= n and every LDS read done
constexpr int wq_vmcnt_lds(int n) { return (n & 0xF) | ((n >> 4) << 14) | (0x7 << 4); }

template <int BITS, int GS, int MT, int NT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
void wq_gemm_kernel(const char* __restrict__ parts, const char* __restrict__ xsum, const char* __restrict__ packed,
                    const char* __restrict__ sb, int M, int N, int K, int mtiles, int n_pad, float* __restrict__ out) {
    constexpr int SEGS = wq_segs(GS), UNROLL = wq_unroll(GS);
    using S = WqStage<BITS, SEGS, MT, NT>;
    extern __shared__ __attribute__((aligned(1024))) char wq_smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm = wave >> 2, wn = wave & 3, ln = lane & 15, q = lane >> 4;
    // every XCD gets a contiguous range of tiles, row tiles first: its L2 then reads a weight row once
    const int tiles_m = mtiles / (2 * MT), nblk = gridDim.x;
    const int xcd = blockIdx.x & 7, quot = nblk >> 3, rem = nblk & 7;
    const int lid = xcd * quot + (xcd < rem ? xcd : rem) + (int(blockIdx.x) >> 3);
    const int tn = lid / tiles_m, tm = lid - tn * tiles_m;
    const int stages = wq_stages(K, GS);

    // ---- the loads of a stage: piece u * 8 + wave (the last round repeats pieces: the counts stay equal)
    constexpr int ROW = 8 * BITS;  // bytes of codes per row and stage
    const unsigned row_bytes = unsigned(K) * BITS / 8, w_last = unsigned(N) * row_bytes - 16;
    const char* src[S::PER_WAVE];
    unsigned step[S::PER_WAVE], off[S::PER_WAVE];
#pragma unroll
    for (int u = 0; u < S::PER_WAVE; ++u) {
        int at = u * 8 + wave;
        at = at < S::PIECES ? at : at - 8;
        unsigned lane_off = unsigned(lane) * 16;
        if (at < S::X) {
            src[u] = parts + size_t(tm) * (S::X * kPiece) + at * kPiece;
            step[u] = unsigned(mtiles) * (6 * kPiece);
        } else if (at < S::X + S::SUMS) {
            src[u] = xsum + size_t(tm) * (SEGS * 32 * MT * 4);
            step[u] = unsigned(mtiles) * (16 * 4 * SEGS);
        } else if (at < S::X + S::SUMS + S::SB) {
            const int i = at - (S::X + S::SUMS), seg = i / S::SB1;
            src[u] = sb + (size_t(seg) * n_pad + tn * (64 * NT)) * 8 + (i - seg * S::SB1) * kPiece;
            step[u] = unsigned(n_pad) * (8 * SEGS);
        } else {
            constexpr int CH = ROW / 16;  // 16-byte chunks per row: 2 or 4
            const int i = at - (S::X + S::SUMS + S::SB), r = i * (64 / CH) + lane / CH;
            const int n = tn * (64 * NT) + r < N ? tn * (64 * NT) + r : N - 1;
            src[u] = packed;
            step[u] = ROW;
            lane_off = unsigned(n) * row_bytes + unsigned((lane % CH) ^ ((r / (16 / CH)) % CH)) * 16;
        }
        off[u] = lane_off;
    }
    auto load_stage = [&](int s, int slot) {
        const int sc = s < stages ? s : stages - 1;  // past the end: any stage, to keep the count
#pragma unroll
        for (int u = 0; u < S::PER_WAVE; ++u) {
            int at = u * 8 + wave;
            at = at < S::PIECES ? at : at - 8;
            const char* base = src[u] + size_t(sc) * step[u];
            unsigned o = off[u];
            if (u * 8 + 7 >= S::X + S::SUMS + S::SB) {  // (a round that may hold codes)
                // a stage past K runs past its row: into the next ones, or at the end of the weight onto its last
                // bytes (its x is zero).  Taken from the start of the weight: the last row may be the first one.
                if (at >= S::X + S::SUMS + S::SB) {
                    const unsigned from = unsigned(sc) * ROW + o;
                    base = packed, o = from < w_last ? from : w_last;
                }
            }
            __builtin_amdgcn_global_load_lds((__attribute__((address_space(1))) void*)(base + o),
                                             (__attribute__((address_space(3))) void*)(wq_smem + (slot * S::PIECES + at) * kPiece),
                                             16, 0, 0);
        }
    };

    v4f y[MT][NT], acc[2][MT][NT], xs[2][MT];
    wq_f2 sc[2][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) y[i][j] = acc[1][i][j] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MT; ++i) xs[1][i] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NT; ++j) sc[1][j] = wq_f2{0.f, 0.f};
    auto apply = [&](int b) {
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    y[i][j][r] = __builtin_fmaf(sc[b][j][0], acc[b][i][j][r], __builtin_fmaf(sc[b][j][1], xs[b][i][r], y[i][j][r]));
    };
#pragma unroll
    for (int s = 0; s < S::RING - 1; ++s) load_stage(s, s);
    int slot = 0;
    for (int s0 = 0; s0 < stages; s0 += UNROLL) {
#pragma unroll
        for (int u = 0; u < UNROLL; ++u) {
            // (the sums and scales read in the stage before may not be needed until after the barrier, which opens
            // their slot to the next loads: they are waited for here)
            __builtin_amdgcn_s_waitcnt(wq_vmcnt_lds(S::PER_WAVE * (S::RING - 2)));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // (the slot that everybody has just left)
            load_stage(s0 + u + S::RING - 1, slot == 0 ? S::RING - 1 : slot - 1);
            const char* base = wq_smem + slot * (S::PIECES * kPiece);
            slot = slot + 1 == S::RING ? 0 : slot + 1;
            const char* frag = base + (wm * MT * 6) * kPiece + lane * 16;
            const char* codes = base + (S::X + S::SUMS + S::SB) * kPiece;
            v8bf xf[2][MT][3];
            v2u wd[2][NT];
            auto read = [&](int ii) {
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int r = (wn * NT + j) * 16 + ln;
                    if constexpr (BITS == 4)
                        wd[ii][j][0] = *reinterpret_cast<const uint32_t*>(codes + r * 32 + (ii ^ ((r >> 3) & 1)) * 16 + q * 4);
                    else
                        wd[ii][j] = *reinterpret_cast<const v2u*>(
                            codes + r * 64 + ((ii * 2 + (q >> 1)) ^ ((r >> 2) & 3)) * 16 + (q & 1) * 8);
                }
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int p = 0; p < 3; ++p)
                        xf[ii][i][p] = *reinterpret_cast<const v8bf*>(frag + ((i * 2 + ii) * 3 + p) * kPiece);
            };
            read(0);
            __builtin_amdgcn_sched_barrier(0);
            read(1);
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) {
                // the group these 32 k belong to, counted from the start of the unrolled stages
                const int k = u * 64 + ii * 32, cur = (k / GS) & 1;
                if (k % GS == 0) {
                    apply(cur ^ 1);
                    const int e = SEGS == 2 ? ii : 0;
                    const char* pairs = base + (S::X + S::SUMS + e * S::SB1) * kPiece + (wn * 16 * NT + ln) * 8;
#pragma unroll
                    for (int j = 0; j < NT; ++j) sc[cur][j] = *reinterpret_cast<const wq_f2*>(pairs + j * 128);
                }
                if (k % (GS < 64 ? GS : 64) == 0) {
                    const int e = SEGS == 2 ? ii : 0;
                    const char* sums = base + S::X * kPiece + (e * 32 * MT + wm * 16 * MT + q * 4) * 4;
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const v4f part = *reinterpret_cast<const v4f*>(sums + i * 64);
                        xs[cur][i] = k % GS == 0 ? part : xs[cur][i] + part;
                    }
                }
                v8bf cf[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const uint32_t w4[4] = {wd[ii][j][0], wd[ii][j][1], 0u, 0u};
                    cf[j] = __builtin_bit_cast(v8bf, wq_codes<BITS>(w4, 0));
                }
#pragma unroll
                for (int i = 0; i < MT; ++i)
#pragma unroll
                    for (int p = 0; p < 3; ++p)
#pragma unroll
                        for (int j = 0; j < NT; ++j)
                            acc[cur][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                                xf[ii][i][p], cf[j], k % GS == 0 && p == 0 ? v4f{0.f, 0.f, 0.f, 0.f} : acc[cur][i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    apply(1);
    __builtin_amdgcn_s_waitcnt(wq_vmcnt_lds(0));  // the loads past the end have landed before the LDS is given up
    // accumulator element r of a lane: row 4 * quarter + r, column lane % 16
    const int m_base = (tm * 2 + wm) * MT * 16 + q * 4, n_base = (tn * 4 + wn) * (NT * 16) + ln;
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m_base + i * 16 + r;
            if (m < M) {
#pragma unroll
                for (int j = 0; j < NT; ++j)
                    if (n_base + j * 16 < N) out[size_t(m) * N + n_base + j * 16] = y[i][j][r];
            }
        }
}

struct Tile {
    int mt, nt;
    float us;  // estimated time of the product
};
// The block tile whose blocks take the least time: rounds of 256 blocks times a stage of 64 k, which is
// 0.38 us (barrier, LDS reads, loads) + 0.125 us per 16 x 16 x 8 tiles of a block.  Measured at K = 4096:
// 32 x 128 tiles 0.63 us per stage, 64 x 128 and 32 x 256 0.95, 64 x 256 1.45, 96 x 192 1.5, 96 x 256 1.95
// (8-bit codes; centred 4-bit ones take about a tenth more in every shape, which changes no choice).
Tile wq_gemm_tile(int M, int N, int stages) {
    static const int tiles[][2] = {{3, 4}, {3, 3}, {2, 4}, {2, 2}, {1, 4}, {1, 2}};
    Tile best{0, 0, 0.0f};
    for (const auto& t : tiles) {
        const int mt = t[0], nt = t[1];
        const long blocks = long((M + 32 * mt - 1) / (32 * mt)) * ((N + 64 * nt - 1) / (64 * nt));
        const float us = float((blocks + 255) / 256) * float(stages) * (0.38f + 0.125f * float(mt * nt));
        if (best.mt == 0 || us < best.us) best = Tile{mt, nt, us};
    }
    return best;
}

// One chunk of rows: prepare, product.
template <int BITS, int GS, int MT, int NT>
int launch_rows(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N, int K,
                float* out, hipStream_t st) {
    constexpr int SEGS = wq_segs(GS);
    using S = WqStage<BITS, SEGS, MT, NT>;
    constexpr int bm = 32 * MT, bn = 64 * NT;
    const int tiles_m = (M + bm - 1) / bm, mtiles = tiles_m * 2 * MT, tiles_n = (N + bn - 1) / bn, n_pad = tiles_n * bn;
    const int stages = wq_stages(K, GS), gs_shift = 31 - __builtin_clz(unsigned(GS));
    // each part is read in whole pieces: a piece of slack behind it
    const size_t part_bytes = size_t(stages) * mtiles * (6 * kPiece);
    const size_t sum_bytes = size_t(stages) * SEGS * mtiles * 16 * 4 + kPiece;
    const size_t sb_bytes = size_t(stages) * SEGS * n_pad * 8 + kPiece;
    void* ws = nullptr;
    const auto lock = scratch_lock(st);
    const int rc = workspace(part_bytes + sum_bytes + sb_bytes, st, &ws);
    if (rc) return rc;
    char* parts = static_cast<char*>(ws);
    char* xsum = parts + part_bytes;
    char* sb = xsum + sum_bytes;
    const unsigned split_blocks = unsigned((stages + 1) / 2) * unsigned(mtiles);
    // (groups of the stages, past K too)
    const int sb_groups = SEGS == 2 ? stages * 2 : stages / (GS / 64);
    static_assert(bn % kSbColumns == 0, "");
    const unsigned sb_blocks = sb_groups < kSbFew ? unsigned((size_t((sb_groups + 3) / 4) * n_pad + 255) / 256)
                                                  : unsigned((sb_groups + kSbGroups - 1) / kSbGroups) * unsigned(n_pad / kSbColumns);
    hipLaunchKernelGGL((wq_prepare_kernel<BITS>), dim3(split_blocks + sb_blocks), dim3(256), 0, st, x, scales, biases, M, N,
                       K, gs_shift, mtiles, bm, n_pad, stages, SEGS, split_blocks, reinterpret_cast<uint4*>(parts),
                       reinterpret_cast<float*>(xsum), reinterpret_cast<float2*>(sb));
    LQ_CHECK_LAUNCH("wq_prepare");
    static DeviceOnce once;
    constexpr int smem = S::RING * S::PIECES * kPiece;
    const int arc = allow_dynamic_lds(once, reinterpret_cast<const void*>(wq_gemm_kernel<BITS, GS, MT, NT>), smem);
    if (arc) return arc;
    hipLaunchKernelGGL((wq_gemm_kernel<BITS, GS, MT, NT>), dim3(unsigned(tiles_m) * unsigned(tiles_n)), dim3(512), smem,
                       st, parts, xsum, reinterpret_cast<const char*>(packed), sb, M, N, K, mtiles, n_pad, out);
    LQ_CHECK_LAUNCH("wq_gemm");
    return LQ_OK;
}

// The kernel's strides from stage to stage are 32-bit, and the prepared rows take half as much again as x: rows are
// taken in chunks of at most kMaxParts of them (43 thousand rows at K = 4096, far more than fill the chip).  Chunks
// are whole row tiles, so the bits do not depend on the split.
constexpr size_t kMaxParts = size_t(1) << 30;
template <int BITS, int GS, int MT, int NT>
int launch_tile(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N, int K,
                float* out, hipStream_t st) {
    constexpr int bm = 32 * MT;
    const size_t tile_bytes = size_t(wq_stages(K, GS)) * (2 * MT) * (6 * kPiece);
    const size_t tiles = tile_bytes < kMaxParts ? kMaxParts / tile_bytes : 1;
    const int rows = tiles * bm < size_t(M) ? int(tiles * bm) : M;
    for (int m0 = 0; m0 < M; m0 += rows) {
        const int rc = launch_rows<BITS, GS, MT, NT>(x + size_t(m0) * K, packed, scales, biases, M - m0 < rows ? M - m0 : rows,
                                                     N, K, out + size_t(m0) * N, st);
        if (rc || M - m0 <= rows) return rc;
    }
    return LQ_OK;
}

template <int BITS, int GS>
int launch(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N, int K,
           float* out, hipStream_t st) {
    const Tile t = wq_gemm_tile(M, N, wq_stages(K, GS));
#define LQ_WQ_GEMM(MT, NT) \
    if (t.mt == MT && t.nt == NT) return launch_tile<BITS, GS, MT, NT>(x, packed, scales, biases, M, N, K, out, st)
    LQ_WQ_GEMM(3, 4);
    LQ_WQ_GEMM(3, 3);
    LQ_WQ_GEMM(2, 4);
    LQ_WQ_GEMM(2, 2);
    LQ_WQ_GEMM(1, 4);
    LQ_WQ_GEMM(1, 2);
#undef LQ_WQ_GEMM
    return fail(LQ_ERR_VALUE, "wq_gemm: no tile %d x %d", t.mt, t.nt);
}

}  // namespace

namespace lq {

// The small-batch kernel splits K between its blocks (512 k each), so it fills the chip where M x N alone
// does not, but reads and decodes the weight once per 16 rows: 6.5 us + 30 ns (int4) or 35 ns (int8) per 256 rows x 512 k.
// This one prepares its operands first (7 us).  Both timed over 17 .. 512 rows, N 300 .. 32000, K 1024 .. 11008 and
// every group size: what this picks is 0.7 % slower than the better one on average; from 65 rows 1.6 x at worst (512 x
// 1000 x 1024: 12.7 / 20.1 us), 3 % of the problems by more than 5 %.  Up to 64 rows the estimates are closer together,
// so it has to be a tenth the faster one (0.4 % on average, 1.2 x at worst; with the small-batch kernel for all of them
// 11 % and 2.6 x; all of this with 8 us + 31 or 38 ns per block, before the small-batch kernel was a fifth faster).  us, small
// batch / this: 64 x 32000 x 4096 int4 groups of 128 131 / 74, int8 of 64 156 / 98;
// 64 x 11008 x 4096 int4 of 64 46 / 56.
bool wq_gemm_beats_small_batch(int M, int N, int K, int gs, int bits) {
    if (size_t(N) * K * bits / 8 >= 0x7fffffffull) return false;  // its weight offsets are 32-bit
    const double blocks = double((M + 15) / 16) * ((N + 255) / 256) * ((K + 511) / 512);
    // (up to 64 rows of 4 bits the two round differently, 128 + c there and centred codes here: the line stays where it was)
    const double small = bits == 4 && M <= 64 ? 8.0 + blocks * 0.031 : 6.5 + blocks * (bits == 4 ? 0.030 : 0.035);
    return 7.0 + wq_gemm_tile(M, N, wq_stages(K, gs)).us < (M <= 64 ? 0.9 : 1.0) * small;
}

int launch_wq_gemm(const float* x, const uint32_t* packed, const float* scales, const float* biases, int M, int N,
                   int K, int gs, int bits, float* out, hipStream_t st) {
#define LQ_WQ_GEMM(BITS, GS) \
    if (bits == BITS && gs == GS) return launch<BITS, GS>(x, packed, scales, biases, M, N, K, out, st)
    LQ_WQ_GEMM(4, 32);
    LQ_WQ_GEMM(4, 64);
    LQ_WQ_GEMM(4, 128);
    LQ_WQ_GEMM(8, 32);
    LQ_WQ_GEMM(8, 64);
    LQ_WQ_GEMM(8, 128);
#undef LQ_WQ_GEMM
    return fail(LQ_ERR_VALUE, "wq_gemm: group_size %d, bits %d", gs, bits);
}

}  // namespace lq
