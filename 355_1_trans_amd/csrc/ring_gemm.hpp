// Ring GEMM for decode shapes (M <= 64) on gfx950: DMA waves stream B and A
// through a deep LDS ring, MFMA waves consume it.  MXFP8 / MXFP4 with
// row-major B, MXFP4 in aiter's formats (W16 B, e8m0_shuffle scales), and fp8
// with fp32 block scales (K-panel B' or fragment-order B'').
//
//  * a workgroup owns all rows (TM = 16 MB) of TN = 16 NB columns and a K
//    slice, in stages of 4 K-tiles: 512 bytes of each row, so a DMA of
//    row-major operands takes 2 rows x 512 contiguous bytes (copy-only
//    replays stream 16-row x 64-byte fragments at 3.7 TB/s, such runs at 5.1);
//  * four waves only issue DMAs: they keep NST - 1 stages (80-130 KB) in
//    flight whatever the MFMA waves do.  Waves that load, stage and multiply
//    by turns (row-run, slice, decode kernels) hold their next loads back
//    behind their own waits;
//  * MFMA wave w of four takes K-tile w of every stage (16x16x128, fp4 two per
//    K-tile) over the whole tile, so each operand byte is read from LDS
//    once; the four partial tiles meet in LDS at the end, in wave order;
//  * one barrier per stage: it says that stage s has been read (into
//    registers: the products follow it) and that stage s + 1 has landed;
//  * scales ride in the stage: PANEL, 16 (fp4: 32) bytes per row and DMA lane
//    where rows and K allow it, else a dword per row and K-tile; shuffled
//    scales as they lie (256 bytes per 32-row block and K-tile); B's fp32
//    scales one DMA (four DMAs instead cost 0.2-0.4 us of 6-12);
//  * every load's descriptor starts at its K offset and ends with the operand,
//    so the last, partial stage reads nothing past it, and its missing
//    K-tiles are not multiplied;
//  * K split over workgroups: fp32 partial planes, summed in slice order by
//    splitk_reduce_kernel, launched next (mid_gemm.hpp).
//
// Bound by the B stream (HBM) and, for 64 rows, by the CU's load path: A's
// rows come from L2 as often as there are column tiles.
// Graph-replayed over rotating weights, us, the kernel it replaced -> this one:
// MXFP8 M = 48, N = 5120, K = 8192 33.1 -> 17.9; M = 24, N = 14336, K = 8192
// 34.2 -> 24.7 (4.8 TB/s of B); M = 7, N = 6144, K = 3072 9.0 -> 6.9; MXFP4
// M = 64, N = 8000, K = 7168 15.5 -> 11.5; fp32 scales M = 48, N = 5120,
// K = 5120 30.5 -> 12.6; M = 32, N = 4096, K = 7168 13.9 -> 10.7; aiter's
// formats M = 57, N = 5120, K = 14336 21.6 -> 15.3.
#pragma once
#include "tile_args.hpp"

namespace qg {

struct RingArgs {
    TileArgs t;            // operands, shapes, strides (tiles_* / group_m unused)
    float* ws;             // fp32 partials [splitk][batch][M][N] (splitk > 1)
    int splitk, st_per_split, n_tiles;    // st_per_split: stages of 4 K-tiles
    int bf16;              // output type
    long long a_bytes, b_bytes, sfa_bytes, sfb_bytes;    // of one batch entry (the load ranges)
};

namespace ring {
constexpr int kLds = 159 * 1024;
// scale DMAs per stage of operand B (op_b) or A with `blocks` 16-row blocks,
// of 16 bytes per lane (wide) or 4
__host__ __device__ constexpr bool sc_wide(ScaleKind sk, bool panel, bool op_b) {
    return sk == ScaleKind::MXS || (panel && !(sk == ScaleKind::BSF32 && op_b));
}
__host__ __device__ constexpr int sc_dmas(ScaleKind sk, bool fp4, bool panel, int blocks, bool op_b) {
    if (sk == ScaleKind::BSF32 && op_b) return 1;    // one 128-column scale block: a float per K-tile
    if (sk == ScaleKind::MXS) return (blocks + 1) / 2;
    if (panel) return fp4 ? (blocks + 1) / 2 : 1;
    return fp4 ? 8 : 4;
}
__host__ __device__ constexpr int sc_bytes(ScaleKind sk, bool fp4, bool panel, int blocks, bool op_b) {
    return sc_dmas(sk, fp4, panel, blocks, op_b) * (sc_wide(sk, panel, op_b) ? 1024 : 256);
}
__host__ __device__ constexpr int stage_bytes(ScaleKind sk, bool fp4, bool panel, int mb, int nb) {
    return (mb + nb) * 16 * 512 + sc_bytes(sk, fp4, panel, mb, false) + sc_bytes(sk, fp4, panel, nb, true);
}
__host__ __device__ constexpr int stages(ScaleKind sk, bool fp4, bool panel, int mb, int nb) {
    const int n = kLds / stage_bytes(sk, fp4, panel, mb, nb);
    return n > 8 ? 8 : n;
}
}  // namespace ring

template <int FMT, ScaleKind SK, BLay BL, int MB, int NB, bool PANEL>
__global__ __launch_bounds__(512, 2) void ring_gemm_kernel(const RingArgs ra) {
    constexpr bool FP4 = FMT == kFmtFp4, MX = SK == ScaleKind::MX, MXS = SK == ScaleKind::MXS;
    constexpr bool BS = SK == ScaleKind::BSF32;
    static_assert(MX ? BL == BLay::RAW : MXS ? FP4 && BL == BLay::FRAG : BS && !FP4 && BL != BLay::RAW, "operands");
    constexpr bool LIN = BL == BLay::FRAG;        // 16-row blocks in operand order (B'', W16)
    constexpr int BKB = 128, RUN = 512, TM = 16 * MB, TN = 16 * NB;
    constexpr int KTB = FP4 ? 8 : 4;              // scale bytes per row and K-tile
    constexpr int PROW = 4 * KTB;                 // PANEL: scale bytes per row and stage
    constexpr int OFF_B = TM * RUN, OFF_SA = OFF_B + TN * RUN, OFF_SB = OFF_SA + ring::sc_bytes(SK, FP4, PANEL, MB, false);
    constexpr int STAGE = ring::stage_bytes(SK, FP4, PANEL, MB, NB), NST = ring::stages(SK, FP4, PANEL, MB, NB);
    static_assert(NST >= 3, "ring");
    constexpr int SA_N = ring::sc_dmas(SK, FP4, PANEL, MB, false), SB_N = ring::sc_dmas(SK, FP4, PANEL, NB, true);
    constexpr int UA = 2 * MB, UB = 2 * NB;       // operand DMAs per wave and stage
    constexpr int ND = UA + UB + (SA_N + SB_N) / 4;    // the fewest DMAs a wave issues per stage
    static_assert((NST - 2) * ND < 64, "vmcnt");
    constexpr int UNITS = MB * NB;
    static_assert(4 * UNITS * 1024 <= NST * STAGE, "the partial tiles reuse the ring");
    __shared__ __attribute__((aligned(1024))) uint8_t lds_mem[NST * STAGE];
    QG_LDS uint8_t* const lds = (QG_LDS uint8_t*)lds_mem;

    const TileArgs& p = ra.t;
    const int M = p.m, N = p.n, LDA = p.lda, LDB = p.ldb;
    const int nkt = p.kbytes / BKB;
    const int nt = blockIdx.x % ra.n_tiles, sk = blockIdx.x / ra.n_tiles, bz = blockIdx.y;
    const int n0 = nt * TN;
    const int st0 = sk * ra.st_per_split;
    const int ns = min((nkt + 3) / 4, st0 + ra.st_per_split) - st0;    // stages of this slice
    // wide tiles: step s of the slice is stage st0 + (s + nt) % ns, so that
    // workgroups in step, reading rows a power of two apart, do not meet in a
    // few memory channels (K = 16384: 18.4 -> 17.7 and 21.6 -> 20.3 us; one
    // 16-column block per workgroup lost, 11.9 -> 14.0, and keeps the order)
    const int rot = NB > 1 ? nt % ns : 0;
    auto stage_of = [&](int s) __attribute__((always_inline)) {
        const int x = s + rot;
        return st0 + (x >= ns ? x - ns : x);
    };
    const int tid = threadIdx.x, L = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
    const int q = L >> 4, l16 = L & 15;

    if (tid >= 256) {
        // ---- DMA waves ----
        auto rsrc = [](const uint8_t* base, long long off, long long bytes) __attribute__((always_inline)) {
            const long long left = bytes - off;
            return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base + off), 0,
                                                     (int)(left < 0 ? 0 : min(left, 0x7fffffffLL)), 0x00020000);
        };
        const uint8_t* A = p.a + bz * p.a_batch;
        const uint8_t* B = p.b + bz * p.b_batch;
        const uint8_t* SFA = p.sfa + (BS ? 4ll : 1ll) * bz * p.sfa_batch;
        const uint8_t* SFB = p.sfb + (BS ? 4ll : 1ll) * bz * p.sfb_batch;
        // operand DMA u of this wave is j = w + 4u of the stage's 8 MB (A)
        // and 8 NB (B).  Row-major: rows 2j, 2j + 1, lane L the 16-byte chunk
        // (L % 32) ^ (row % 16) of the row's 512 bytes.  B': 8 rows of one
        // K-tile, chunk (L % 8) ^ (row % 8).  B'' / W16: 1 KB of a block's 8.
        int a_off[UA], b_off[UB];
#pragma unroll
        for (int u = 0; u < UA; ++u) {
            const int row = 2 * (w + 4 * u) + (L >> 5);
            a_off[u] = min(row, M - 1) * LDA + (((L & 31) ^ (row & 15)) << 4);
        }
#pragma unroll
        for (int u = 0; u < UB; ++u) {
            const int j = w + 4 * u;
            if constexpr (LIN) {
                const int blk = min((n0 >> 4) + (j >> 3), ((N + 15) >> 4) - 1) - (n0 >> 4);
                b_off[u] = blk * nkt * 2048 + (j & 7) * 1024 + L * 16;
            } else if constexpr (BL == BLay::KPANEL) {
                const int row = (j % (2 * NB)) * 8 + (L >> 3);
                b_off[u] = (j / (2 * NB)) * N * BKB + (min(n0 + row, N - 1) - n0) * BKB + (((L & 7) ^ (row & 7)) << 4);
            } else {
                const int row = 2 * j + (L >> 5);
                b_off[u] = (min(n0 + row, N - 1) - n0) * LDB + (((L & 31) ^ (row & 15)) << 4);
            }
        }
        const long long b_base = LIN ? (long long)(n0 >> 4) * nkt * 2048
                                     : BL == BLay::KPANEL ? (long long)n0 * BKB : (long long)n0 * LDB;
        const long long b_step = LIN ? 8192 : BL == BLay::KPANEL ? 4ll * N * BKB : RUN;    // per stage
        // scale DMA x of operand op: lane -> byte offset, stage 0
        auto sc_off = [&](bool op_b, int x) __attribute__((always_inline)) {
            const int lim = op_b ? N - 1 - n0 : M - 1;
            const int sm = op_b ? p.sfb_sn : p.sfa_sm;
            if constexpr (MXS) {
                const int last = op_b ? ((N - 1) >> 5) - (n0 >> 5) : (M - 1) >> 5;
                return min(x, last) * sm + L * 16;
            } else if constexpr (BS) {
                if (op_b) return 4 * (L & 3);
                return 4 * (min(L, lim) * sm + (PANEL ? 0 : x * p.sfa_sk));
            } else if constexpr (PANEL) {
                return FP4 ? min(32 * x + (L >> 1), lim) * sm + (L & 1) * 16 : min(L, lim) * sm;
            } else {
                return min(L, lim) * sm + 4 * x;
            }
        };
        const long long sfa_step = MXS ? 1024 : BS ? 16ll * p.sfa_sk : PROW;
        const long long sfb_step = MXS ? 1024 : BS ? 16 : PROW;
        const long long sfb_base = MXS ? (long long)(n0 >> 5) * p.sfb_sn
                                       : BS ? 4ll * (n0 >> 7) * p.sfb_sn : (long long)n0 * p.sfb_sn;
        constexpr bool WA = ring::sc_wide(SK, PANEL, false), WB = ring::sc_wide(SK, PANEL, true);
        auto fill = [&](int s) __attribute__((always_inline)) {
            const int st = stage_of(s);
            QG_LDS uint8_t* dst = lds + (s % NST) * STAGE;
            const auto rsa = rsrc(SFA, st * sfa_step, ra.sfa_bytes);
            const auto rsb = rsrc(SFB, sfb_base + st * sfb_step, ra.sfb_bytes);
            // (the scales first: the waves' counts may differ by them, and an
            // early DMA waited for too much costs least)
#pragma unroll
            for (int x = 0; x < SA_N; ++x)
                if (x % 4 == w) {
                    if constexpr (WA) dma16_buf(rsa, dst + OFF_SA + x * 1024, sc_off(false, x), 0);
                    else dma4_buf(rsa, dst + OFF_SA + x * 256, sc_off(false, x), 0);
                }
#pragma unroll
            for (int x = 0; x < SB_N; ++x)
                if ((SA_N + x) % 4 == w) {
                    if constexpr (WB) dma16_buf(rsb, dst + OFF_SB + x * 1024, sc_off(true, x), 0);
                    else dma4_buf(rsb, dst + OFF_SB + x * 256, sc_off(true, x), 0);
                }
            const auto rb = rsrc(B, b_base + st * b_step, ra.b_bytes);
            const auto rA = rsrc(A, (long long)st * RUN, ra.a_bytes);
#pragma unroll
            for (int u = 0; u < UB; ++u) dma16_buf_nt(rb, dst + OFF_B + (w + 4 * u) * 1024, b_off[u], 0);
#pragma unroll
            for (int u = 0; u < UA; ++u) dma16_buf(rA, dst + (w + 4 * u) * 1024, a_off[u], 0);
        };
        // stage s is in LDS: all but the DMAs of the stages after it
        auto landed = [&](int s) __attribute__((always_inline)) {
            const int after = min(ns - 1 - s, NST - 2);
            if (after >= NST - 2) wait_vmcnt<(NST - 2) * ND>();
            else if (NST > 7 && after == 5) wait_vmcnt<5 * ND < 64 ? 5 * ND : 0>();
            else if (NST > 6 && after == 4) wait_vmcnt<4 * ND < 64 ? 4 * ND : 0>();
            else if (NST > 5 && after == 3) wait_vmcnt<3 * ND < 64 ? 3 * ND : 0>();
            else if (NST > 4 && after == 2) wait_vmcnt<2 * ND < 64 ? 2 * ND : 0>();
            else if (NST > 3 && after == 1) wait_vmcnt<ND>();
            else wait_vmcnt<0>();
            asm volatile("s_barrier" ::: "memory");
        };
        for (int s = 0; s < min(ns, NST - 1); ++s) fill(s);
        landed(0);
        if (ns > NST - 1) fill(NST - 1);
        for (int s = 0; s < ns; ++s) {
            landed(s + 1);
            if (s + NST < ns) fill(s + NST);
        }
        return;
    }

    // ---- MFMA waves: K-tile w of every stage ----
    f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    // 16-byte chunks of the lane's operand: q and q + 4 of the K-tile; row-
    // major fp4 2q and 2q + 1 (neighbours, so one u16 holds both scales)
    const int ca = FP4 && !MXS ? 2 * q : q, cb = FP4 && !MXS ? 2 * q + 1 : q + 4;
    const int run0 = l16 * RUN + (((8 * w + ca) ^ l16) << 4), run1 = l16 * RUN + (((8 * w + cb) ^ l16) << 4);
    const int kp0 = w * TN * BKB + l16 * BKB + ((ca ^ (l16 & 7)) << 4);
    const int kp1 = w * TN * BKB + l16 * BKB + ((cb ^ (l16 & 7)) << 4);
    const int b0 = LIN ? w * 2048 + L * 16 : BL == BLay::KPANEL ? kp0 : run0;
    const int b1 = LIN ? w * 2048 + 1024 + L * 16 : BL == BLay::KPANEL ? kp1 : run1;
    constexpr int B_BLK = BL == BLay::KPANEL ? 16 * BKB : 16 * RUN;
    // scale of block row x of an operand, as the lane's MFMA takes it
    auto sc_read = [&](const QG_LDS uint8_t* sc, int x) __attribute__((always_inline)) -> int {
        const int row = 16 * x + l16;
        if constexpr (MXS) return *(const QG_LDS int*)(sc + (x >> 1) * 1024 + w * 256 + q * 64 + l16 * 4);
        else if constexpr (FP4) {
            return PANEL ? *(const QG_LDS uint16_t*)(sc + row * PROW + w * 8 + 2 * q)
                         : *(const QG_LDS uint16_t*)(sc + (2 * w + (q >> 1)) * 256 + row * 4 + 2 * (q & 1));
        } else {
            return PANEL ? sc[row * PROW + w * 4 + q] : sc[w * 256 + row * 4 + q];
        }
    };
    auto cat8 = [](i32x4 lo, i32x4 hi) __attribute__((always_inline)) {
        return i32x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    };
    asm volatile("s_barrier" ::: "memory");    // stage 0 has landed
    for (int s = 0; s < ns; ++s) {
        const QG_LDS uint8_t* st = lds + (s % NST) * STAGE;
        i32x8 af[MB], bf[NB];
        int xa[MB], xb[NB];
        float fa[MB], fb = 0.f;
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            const QG_LDS uint8_t* blk = st + OFF_B + j * B_BLK;
            bf[j] = cat8(*(const QG_LDS i32x4*)(blk + b0), *(const QG_LDS i32x4*)(blk + b1));
        }
#pragma unroll
        for (int i = 0; i < MB; ++i) {
            const QG_LDS uint8_t* blk = st + i * 16 * RUN;
            af[i] = cat8(*(const QG_LDS i32x4*)(blk + run0), *(const QG_LDS i32x4*)(blk + run1));
        }
        if constexpr (BS) {
#pragma unroll
            for (int i = 0; i < MB; ++i) {
                const int row = 16 * i + l16;
                fa[i] = *(const QG_LDS float*)(st + OFF_SA + (PANEL ? row * PROW + w * 4 : w * 256 + row * 4));
            }
            fb = *(const QG_LDS float*)(st + OFF_SB + w * 4);
        } else {
#pragma unroll
            for (int j = 0; j < NB; ++j) xb[j] = sc_read(st + OFF_SB, j);
#pragma unroll
            for (int i = 0; i < MB; ++i) xa[i] = sc_read(st + OFF_SA, i);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (4 * stage_of(s) + w >= nkt) continue;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < NB; ++j) {
                if constexpr (BS) {
                    // zero scale operands select the unscaled fp8 MFMA (a plain product)
                    const f32x4 part = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(
                        bf[j], af[i], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0, 0, 0, 0);
                    const float f = fa[i] * fb;
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(part[e], f, acc[i][j][e]);
                } else if constexpr (FP4) {
                    const i32x8 bl = i32x8{bf[j][0], bf[j][1], bf[j][2], bf[j][3], 0, 0, 0, 0};
                    const i32x8 bh = i32x8{bf[j][4], bf[j][5], bf[j][6], bf[j][7], 0, 0, 0, 0};
                    const i32x8 al = i32x8{af[i][0], af[i][1], af[i][2], af[i][3], 0, 0, 0, 0};
                    const i32x8 ah = i32x8{af[i][4], af[i][5], af[i][6], af[i][7], 0, 0, 0, 0};
                    if constexpr (MXS) {
                        // byte (16-row half of the 32-row block) for group q, 2 + that for q + 4
                        const int hb = 8 * (((n0 >> 4) + j) & 1), ha = 8 * (i & 1);
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bl, al, acc[i][j], kFmtFp4, kFmtFp4, 0,
                                                                                     xb[j] >> hb, 0, xa[i] >> ha);
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bh, ah, acc[i][j], kFmtFp4, kFmtFp4, 0,
                                                                                     xb[j] >> (hb + 16), 0, xa[i] >> (ha + 16));
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bl, al, acc[i][j], kFmtFp4, kFmtFp4, 0,
                                                                                     xb[j], 0, xa[i]);
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bh, ah, acc[i][j], kFmtFp4, kFmtFp4, 1,
                                                                                     xb[j], 1, xa[i]);
                    }
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf[j], af[i], acc[i][j], kFmtFp8, kFmtFp8, 0,
                                                                                 xb[j], 0, xa[i]);
                }
            }
    }

    // ---- the waves' partial tiles, summed in wave order (the ring is free:
    // every stage has been read and no DMA is left) ----
    QG_LDS f32x4* red = (QG_LDS f32x4*)lds;
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) red[(w * UNITS + i * NB + j) * 64 + L] = acc[i][j];
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    const bool vec = ra.splitk > 1 ? (N & 3) == 0 : p.c_vec >= 4;    // aligned 4-element stores
    const long long plane = (long long)M * N;
    float* const part = ra.ws + ((long long)sk * gridDim.y + bz) * plane;
#pragma unroll
    for (int u0 = 0; u0 < UNITS; u0 += 4) {
        const int u = u0 + w;
        if (u >= UNITS) break;
        f32x4 v = red[u * 64 + L];
#pragma unroll
        for (int ww = 1; ww < 4; ++ww) {
            const f32x4 x = red[(ww * UNITS + u) * 64 + L];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += x[e];
        }
        const int m = 16 * (u / NB) + l16, n = n0 + 16 * (u % NB) + 4 * q;
        if (m >= M || n >= N) continue;
        const bool whole = vec && n + 3 < N;
        if (ra.splitk == 1 && ra.bf16) {
            uint16_t* c = (uint16_t*)p.c + bz * p.c_batch + (long long)m * p.ldc + n;
            if (whole) *(u32x2*)c = u32x2{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
            else
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) c[e] = bf16_bits(v[e]);
        } else {
            float* c = ra.splitk > 1 ? part + (long long)m * N + n : (float*)p.c + bz * p.c_batch + (long long)m * p.ldc + n;
            if (whole) *(f32x4*)c = v;
            else
                for (int e = 0; e < 4; ++e)
                    if (n + e < N) c[e] = v[e];
        }
    }
}

}  // namespace qg
