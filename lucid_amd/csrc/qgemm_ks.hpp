// Small tiles of the int8 GEMM / implicit-GEMM convolution with K dealt to the wavefronts of a block.
//
// For problems of fewer tiles than the chip has places for, where a tile's time is a chain of memory round trips and not its
// arithmetic: small batches in the late layers of a network, long K under few outputs, up to 16 rows.  What a CU gets from memory
// then is bounded by the lines it can have on their way, so the tile is small (with 32 x 32 four times as many CUs fetch as with
// 64 x 64) and a line is asked for once, whole.  Each of W wavefronts has the whole tile over a share of K of its own:
//  * its rows go to a ring in LDS of its own by direct loads (an instruction is 8 whole 128-byte lines, or 16 of 64 bytes where
//    the channels of a convolution are no multiple of 128), and it waits for nobody: no barrier in the loop;
//  * the weight is the MFMA's first operand, so that a lane holds four consecutive columns of a row, and the wavefronts'
//    sums meet in LDS as 16-byte vectors, once;
//  * behind that one barrier a thread finishes whole groups of four columns, whose parameters, residual or join operand
//    were requested before the loop.
// (The first form loaded fragments straight into registers, 16 rows of 64 bytes per instruction: 49 x 512 x 4608 in 64 x 64 tiles
// 19 us and in 32 x 32 11, where four wavefronts that share stages and barriers take 11.3.)
//
// us, those four wavefronts on 64 x 64 tiles / this, replayed from a graph with operands out of the last-level cache:
// 49 x 512 x 4608 (3x3 gather) 11.3 / 6.4, 196 x 256 x 2304 8.4 / 5.2, 784 x 128 x 1152 7.0 / 4.8, 3136 x 64 x 576 6.1 / 4.3,
// 197 x 768 x 3072 8.7 / 5.6, 60 x 92 x 6624 12.4 / 6.4; 64 x 32 tiles: 784 x 512 x 4608 12.5 / 9.0, 1568 x 256 x 2304
// 8.7 / 7.0.  Two tiles per CU are slower than four wavefronts on larger ones: 392 x 512 x 1024 in 208 tiles 5.4 / 4.1,
// 3136 x 128 x 1152 in 392 tiles 7.3 / 7.9.  16-row tiles against the kernel whose wavefronts load fragments straight into registers: 16 x
// 11008 x 4096 10.9 / 9.5, 16 x 4096 x 4096 7.8 / 5.7, 16 x 1024 x 4096 6.9 / 3.8, 2 x 12000 x 1024 5.6 / 4.9.  Several rounds of tiles of 64
// columns, which have one stage each and nothing on its way during the products (other blocks of the CU have): 16 x 14336 x 4096
// 16.7 / 14.7, 16 x 16384 x 4096 17.1 / 15.7, 16 x 32000 x 4096 32.6 / 29.9 (weights in the last-level cache 25.2 / 20.4), 2 x 32000 x 4096
// 30.4 / 29.0, 16 x 151936 x 4096 142 / 111, 16 x 65536 x 1024 23.3 / 16.0.
#pragma once
#include "qgemm_tile.hpp"

namespace lq {
namespace {

// FM x FN MFMA tiles of 16 x 16 per wavefront, W wavefronts, NST stages of 128 bytes of k in a wavefront's ring
template <int FM_, int FN_, int W_, int NST_>
struct KsCfg {
    static constexpr int FM = FM_, FN = FN_, W = W_;
    static constexpr int BM = 16 * FM, BN = 16 * FN, THREADS = 64 * W;
    static constexpr int RING = NST_ * (BM + BN) * 128;  // bytes of a wavefront's ring
    static constexpr int LD = BN + 4;                    // words of a row of sums: 16 rows on different banks
    static constexpr int SMEM = W * RING;
    static constexpr int QROW = BN / 4;                  // groups of four columns in a row
    static constexpr int QPT = BM * QROW > THREADS ? BM * QROW / THREADS : 1;
    static_assert(BM * LD * 4 <= RING, "a wavefront's sums take the place of its ring");
    static_assert(SMEM <= 160 * 1024 && (QPT == 1 || (THREADS % QROW == 0 && BM * QROW % THREADS == 0)), "");
};

struct KsConv {
    FastDiv pix, ow;  // by cOH * cOW and cOW
};

// BK: bytes of k per stage (64 or 128)
template <class Cfg, int BK, int MODE, int CONV>
__global__ __launch_bounds__(Cfg::THREADS, Cfg::W / 4) void qgemm_ks_kernel(GemmArgs g, KsConv cv) {
    constexpr int FM = Cfg::FM, FN = Cfg::FN, W = Cfg::W, BM = Cfg::BM, BN = Cfg::BN, LD = Cfg::LD, QPT = Cfg::QPT;
    constexpr int C = BK / 16, RPI = 64 / C;       // 16-byte chunks of a row, rows of an instruction
    constexpr int NA = BM / RPI, NB = BN / RPI;    // instructions per operand and stage
    constexpr int STAGE = (BM + BN) * BK, NST = Cfg::RING / STAGE;
    extern __shared__ __attribute__((aligned(1024))) int8_t ks_smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ln = lane & 15, lg = lane >> 4;
    const int tiles_m = (g.M + BM - 1) / BM, tiles_n = (g.N + BN - 1) / BN;
    int tm, tn;
    tile_coords(blockIdx.x, gridDim.x, tiles_m, tiles_n, &tm, &tn);
    const int n_base = int(blockIdx.y) * g.N, n_limit = n_base + g.N;
    const int m0 = tm * BM, n0 = n_base + tn * BN;

    // this wavefront's stages
    const int stages = (g.K + BK - 1) / BK;
    const int per = (stages + W - 1) / W;
    const int first = wave * per;
    const int n_st = first >= stages ? 0 : (stages - first < per ? stages - first : per);
    const int parts = (stages + per - 1) / per;  // wavefronts with a share

    // Loader: instruction i moves rows RPI * i + lane / C of an operand; a lane fetches the chunk that belongs in its slot: chunk kc
    // of row r sits at kc ^ (r / 2 or / 4, the rows of 256 bytes) % C, which spreads the 16 rows of a fragment over all banks.
    const int lrow = lane / C;
    constexpr int RB = 256 / BK;  // rows of 256 bytes
    auto chunk_of = [&](int row) { return ((lane % C) ^ ((row / RB) % C)) * 16; };
    const int8_t *a_src[NA], *b_src[NB];
    int a_hw[CONV ? NA : 1], a_step[CONV ? NA : 1];
    unsigned a_off[CONV ? NA : 1];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
        const int n = n0 + RPI * i + lrow;  // (rows past the end repeat the last one: they are masked at the store)
        b_src[i] = g.w + size_t(n < n_limit ? n : n_limit - 1) * size_t(g.K) + (first * BK + chunk_of(RPI * i + lrow));
    }
    int u_ci = 0, u_kh = 0, u_kw = 0;  // CONV: the filter position of the next stage (uniform: Cg % BK == 0)
    auto enter_tap = [&] {
        const int dh = u_kh * g.cdh, dw = u_kw * g.cdw;
        const unsigned delta = unsigned(dh * g.cW + dw) * unsigned(g.cCin) + unsigned(u_ci);
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int ih = (a_hw[i] >> 16) + dh, iw = int(short(a_hw[i] & 0xffff)) + dw;
            const bool ok = unsigned(ih) < unsigned(g.cH) && unsigned(iw) < unsigned(g.cW);
            a_src[i] = ok ? g.cx + (a_off[i] + delta + unsigned(chunk_of(RPI * i + lrow))) : g.pad_src;
            a_step[i] = ok ? BK : 0;  // outside the image the bytes of the zero point are read again
        }
    };
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        int m = m0 + RPI * i + lrow;
        m = m < g.M ? m : g.M - 1;
        if constexpr (CONV != 0) {
            const unsigned b = cv.pix(unsigned(m)), rem = unsigned(m) - b * cv.pix.d;
            const unsigned oh = cv.ow(rem), ow = rem - oh * cv.ow.d;
            const int ih0 = int(oh) * g.csh - g.cph, iw0 = int(ow) * g.csw - g.cpw;
            a_hw[i] = (ih0 << 16) | (iw0 & 0xffff);
            // (may wrap for a tap outside the image; used after the bounds check only)
            a_off[i] = unsigned((int(b) * g.cH + ih0) * g.cW + iw0) * unsigned(g.cCin) + unsigned(int(blockIdx.y) * g.cCg);
        } else {
            a_src[i] = g.a + size_t(m) * size_t(g.K) + (first * BK + chunk_of(RPI * i + lrow));
        }
    }
    if constexpr (CONV != 0) {
        const int tap = first * BK / g.cCg;
        u_ci = first * BK - tap * g.cCg;
        u_kh = tap / g.cKW, u_kw = tap - u_kh * g.cKW;
        enter_tap();
    }
    int8_t* const ring = ks_smem + wave * Cfg::RING;
    const bool whole = g.K % BK == 0;  // otherwise the last stage's chunks past K are zeros
    auto load = [&](int t) {
        int8_t* sa = ring + (t % NST) * STAGE;
        if constexpr (CONV != 0) {
            if (u_ci == g.cCg) {
                u_ci = 0;
                if (++u_kw == g.cKW) u_kw = 0, ++u_kh;
                enter_tap();
            }
            u_ci += BK;
        }
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            const int8_t* src = (CONV || whole || (first + t) * BK + chunk_of(RPI * i + lrow) < g.K) ? a_src[i] : g.zeros;
            __builtin_amdgcn_global_load_lds(LQ_GPTR(src), LQ_LPTR(sa + i * 1024), 16, 0, 0);
            a_src[i] += CONV ? a_step[CONV ? i : 0] : BK;
        }
#pragma unroll
        for (int i = 0; i < NB; ++i) {
            const int8_t* src = (CONV || whole || (first + t) * BK + chunk_of(RPI * i + lrow) < g.K) ? b_src[i] : g.zeros;
            __builtin_amdgcn_global_load_lds(LQ_GPTR(src), LQ_LPTR(sa + BM * BK + i * 1024), 16, 0, 0);
            b_src[i] += BK;
        }
    };
    // What the thread's group of four columns needs is requested first: loads are counted off in order, so that a wait for a stage of the
    // ring never waits for these alone.
    constexpr bool kFloatOut = MODE == OUT_F32 || MODE == OUT_F16 || MODE == OUT_F32X;
    // Group tid % QROW of rows tid / QROW + i * ROWS.
    constexpr int ROWS = Cfg::THREADS / Cfg::QROW;
    const bool finisher = QPT > 1 || tid < BM * Cfg::QROW;
    const int row0 = tid / Cfg::QROW, nq = n0 + (tid % Cfg::QROW) * 4;
    const bool vec = nq + 4 <= n_limit;
    ColParams cp[4];
    float as[QPT];
    float4u res[kFloatOut ? QPT : 1];
    uint32_t jv[MODE == OUT_REQUANT_JOIN ? QPT : 1];
    if (finisher) {
        const int nc[4] = {nq < n_limit ? nq : n_limit - 1, nq + 1 < n_limit ? nq + 1 : n_limit - 1,
                           nq + 2 < n_limit ? nq + 2 : n_limit - 1, nq + 3 < n_limit ? nq + 3 : n_limit - 1};
        load_cols(g, nc, cp);
#pragma unroll
        for (int i = 0; i < QPT; ++i) {
            const int m = m0 + row0 + i * ROWS;
            as[i] = g.a_scale ? g.a_scale[(g.a_scale_per_row && m < g.M) ? m : 0] : 1.0f;
            if (vec && m < g.M) {
                if (kFloatOut && g.residual != nullptr)
                    res[i] = *reinterpret_cast<const float4u*>(g.residual + size_t(m) * size_t(g.ldr) + size_t(nq));
                if (MODE == OUT_REQUANT_JOIN)
                    jv[i] = *reinterpret_cast<const unaligned_codes4*>(g.join_q + size_t(m) * size_t(g.join_ld) + size_t(nq));
            }
        }
    }
    for (int s = 0; s < NST; ++s)
        if (s < n_st) load(s);

    v4i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) acc[i][j] = v4i{0, 0, 0, 0};
    // (fragment: lane holds row ln, 16 bytes of k at chunk 4 h + lg)
    auto frag = [&](const int8_t* base, int r, int h) {
        return *reinterpret_cast<const v4i*>(base + r * BK + (((4 * h + lg) ^ ((r / RB) % C)) * 16));
    };
    auto stage = [&](int t, bool refill) {
        const int8_t* sa = ring + (t % NST) * STAGE;
        v4i fa[BK / 64][FM], fb[BK / 64][FN];
#pragma unroll
        for (int h = 0; h < BK / 64; ++h) {
#pragma unroll
            for (int i = 0; i < FM; ++i) fa[h][i] = frag(sa, 16 * i + ln, h);
#pragma unroll
            for (int j = 0; j < FN; ++j) fb[h][j] = frag(sa + BM * BK, 16 * j + ln, h);
        }
        // the fragments are in registers before the direct loads may overwrite where they were
        wave_lds_sync();
        __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
        wave_lds_sync();
        if (refill) load(t + NST);
#pragma unroll
        for (int h = 0; h < BK / 64; ++h)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int i = 0; i < FM; ++i) acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[h][j], fa[h][i], acc[i][j], 0, 0, 0);
    };
    int t = 0;
    for (; t + NST < n_st; ++t) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm((NST - 1) * (NA + NB)));
        wave_lds_sync();
        stage(t, true);
    }
    if (n_st > 0) {
        __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
        wave_lds_sync();
        for (; t < n_st; ++t) stage(t, false);
        // acc[i][j][q]: activation row 16 i + ln, column 16 j + 4 lg + q
        int* mine = reinterpret_cast<int*>(ring) + ln * LD + 4 * lg;
        wave_lds_sync();
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) *reinterpret_cast<v4i*>(mine + 16 * i * LD + 16 * j) = acc[i][j];
    }
    float S = 1.0f, Z = 0.0f;
    constexpr bool kRequant = MODE == OUT_REQUANT_I8 || MODE == OUT_REQUANT_JOIN || MODE == OUT_FAKEQUANT_F32;
    if (kRequant) S = g.out_scale[0], Z = g.out_zp[0];
    const QGrid G = make_qgrid(S, Z, float(g.out_qmin), float(g.out_qmax), kRequant, g.relu != 0, MODE == OUT_REQUANT_I8);
    JoinParams jp;
    if (MODE == OUT_REQUANT_JOIN) jp = load_join(g, G, true);
    const CodePack cpk = make_code_pack<MODE>(g, MODE == OUT_REQUANT_JOIN ? jp.out : G);
    lds_barrier();
    RangeKeep kept;
    if (finisher && nq < n_limit) {
#pragma unroll
        for (int i = 0; i < QPT; ++i) {
            const int row = row0 + i * ROWS, m = m0 + row;
            if (m >= g.M) break;
            const int* from = reinterpret_cast<const int*>(ks_smem) + row * LD + (tid % Cfg::QROW) * 4;
            v4i sum = *reinterpret_cast<const v4i*>(from);
#pragma unroll
            for (int p = 1; p < W; ++p)
                if (p < parts) sum += *reinterpret_cast<const v4i*>(from + p * (Cfg::RING / 4));
            uint4 v = epilogue_quad<MODE>(g, sum, as[i], cp, G);
            const size_t idx = size_t(m) * size_t(g.ldo) + size_t(nq);
            if (vec && (MODE != OUT_REQUANT_JOIN || jp.k2_exact)) {
                if (kFloatOut && g.residual != nullptr) {
                    v.x = __float_as_uint(__uint_as_float(v.x) + res[i].x), v.y = __float_as_uint(__uint_as_float(v.y) + res[i].y);
                    v.z = __float_as_uint(__uint_as_float(v.z) + res[i].z), v.w = __float_as_uint(__uint_as_float(v.w) + res[i].w);
                }
                if (MODE == OUT_REQUANT_JOIN) v = join_codes(jp, v, jv[i]);
                if (MODE == OUT_F32X)
                    kept.add(__uint_as_float(v.x)), kept.add(__uint_as_float(v.y)), kept.add(__uint_as_float(v.z)),
                        kept.add(__uint_as_float(v.w));
                store_vec4<MODE>(g, idx, v, cpk);
            } else {
                const uint32_t e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (nq + k < n_limit) {
                        const uint32_t y = finish_value<MODE>(g, e[k], m, nq + k, jp);
                        if (MODE == OUT_F32X) kept.add(__uint_as_float(y));
                        store_scalar<MODE>(g, idx + k, y, cpk);
                    }
            }
        }
    }
    if (MODE == OUT_F32X && g.range != nullptr) kept.store(g.range);
}

template <class Cfg, int BK, int MODE, int CONV>
int launch_ks_mode(const GemmArgs& g, int groups, hipStream_t st) {
    const void* fn = reinterpret_cast<const void*>(qgemm_ks_kernel<Cfg, BK, MODE, CONV>);
    static DeviceOnce attr_once;
    if (int rc = allow_dynamic_lds(attr_once, fn, Cfg::SMEM)) return rc;
    const long tiles = long((g.M + Cfg::BM - 1) / Cfg::BM) * ((g.N + Cfg::BN - 1) / Cfg::BN);
    LQ_REQUIRE(tiles <= 0x7fffffff, LQ_ERR_SHAPE, "K-split kernel: %ld tiles", tiles);
    LQ_REQUIRE(g.range == nullptr || tiles * groups <= kRangeSlots, LQ_ERR_SHAPE,
               "K-split kernel: %ld tiles are too many for a kept range", tiles * groups);
    GemmArgs copy = g;
    KsConv cv{FastDiv(unsigned(CONV ? g.cOH * g.cOW : 1)), FastDiv(unsigned(CONV ? g.cOW : 1))};
    void* kargs[] = {&copy, &cv};
    LQ_HIP(hipLaunchKernel(fn, dim3(unsigned(tiles), groups), dim3(Cfg::THREADS), kargs, Cfg::SMEM, st));
    return LQ_OK;
}

template <class Cfg, int BK, int CONV>
int launch_ks(const GemmArgs& g, int groups, hipStream_t st) {
    switch (g.out_mode) {
    case OUT_ACC_I32: return launch_ks_mode<Cfg, BK, OUT_ACC_I32, CONV>(g, groups, st);
    case OUT_F32:
        if (g.gelu || g.range != nullptr) {
            if (CONV) return fail(LQ_ERR_NOT_IMPLEMENTED, "K-split kernel: GELU / kept range are not built for convolutions");
            return launch_ks_mode<Cfg, BK, OUT_F32X, 0>(g, groups, st);
        }
        return launch_ks_mode<Cfg, BK, OUT_F32, CONV>(g, groups, st);
    case OUT_F16: return launch_ks_mode<Cfg, BK, OUT_F16, CONV>(g, groups, st);
    case OUT_REQUANT_I8:
        if (g.join_q != nullptr) return launch_ks_mode<Cfg, BK, OUT_REQUANT_JOIN, CONV>(g, groups, st);
        return launch_ks_mode<Cfg, BK, OUT_REQUANT_I8, CONV>(g, groups, st);
    default: return launch_ks_mode<Cfg, BK, OUT_FAKEQUANT_F32, CONV>(g, groups, st);
    }
}

template <class Cfg>
int launch_ks_shape(const GemmArgs& g, int conv, int groups, hipStream_t st) {
    if (!conv) return launch_ks<Cfg, 128, 0>(g, groups, st);
    return g.cCg % 128 == 0 ? launch_ks<Cfg, 128, 1>(g, groups, st) : launch_ks<Cfg, 64, 1>(g, groups, st);
}

}  // namespace
}  // namespace lq
