// Device-side quantizers and weight-layout transforms: the steps before the
// GEMM, on the GPU.
//
//   * fp32 / bf16 -> e4m3 with fp32 block scales amax / 448, per 1x128
//     activation block or 128x128 weight block (the block-scale recipe the
//     reference's fp32-scale kernels consume, BPS host.cc:66-90);
//   * the same with E8M0 block scales 2^ceil(log2(amax / 448)) (the SNAP
//     kernel's input, SNAP blockscale_bpreshuffle.py:3-4);
//   * MXFP8 (e4m3) and MXFP4 (e2m1, two per byte, even k in the low nibble)
//     with one E8M0 scale 2^ceil(log2(amax / qmax)) per 32 K elements, the
//     scales written row-major [rows][K/32] or in aiter's e8m0_shuffle order
//     (quant(..., shuffle=True), MX4 candidate_m9/README.md:6-12);
//   * the weight layouts: K-panel B' (BPS host.cc:92-111),
//     shuffle_weight(16,16) (SNAP host.cc:161-179, MX4 candidate_m10
//     host.cc:215-225), this library's B'' and e8m0_shuffle (MX4
//     candidate_m10 host.cc:194-206).
//
// All of it is HBM-bound byte work: one pass over the input with 16-byte
// loads, coalesced stores; only scales go through LDS.  The value codecs
// below are written from the format definitions (OCP E4M3 / E2M1, round to
// nearest even, saturating); groups of ordinary magnitudes use the hardware's
// conversions instead, which give the same codes, so all codes are
// bit-identical to the host quantizers the tests compare with.
#include <hip/hip_runtime.h>
#include <type_traits>

#include "common.hpp"
#include "launch.hpp"

namespace qg {

namespace {

// ---------------------------------------------------------------- codecs
// OCP E4M3FN, round to nearest even, saturating at 448 (0x7E); NaN -> 0x7F.
__device__ __forceinline__ uint32_t f32_to_e4m3(float x) {
    const uint32_t b = __float_as_uint(x);
    const uint32_t sign = (b >> 24) & 0x80u;
    const uint32_t a = b & 0x7fffffffu;
    if (a > 0x7f800000u) return sign | 0x7fu;             // NaN
    if (a >= 0x43e00000u) return sign | 0x7eu;            // |x| >= 448: saturate
    if (a < 0x3c800000u)                                  // |x| < 2^-6: subnormals, step 2^-9
        return sign | (uint32_t)__builtin_rintf(__uint_as_float(a) * 512.0f);   // 0..8 (8 = 2^-6)
    const uint32_t e = (a >> 23) - 120u;                  // biased e4m3 exponent 1..15
    uint32_t m = (a >> 20) & 7u;
    const uint32_t rem = a & 0xfffffu;
    if (rem > 0x80000u || (rem == 0x80000u && (m & 1u))) ++m;
    const uint32_t code = (e << 3) + m;                   // m == 8 carries into the exponent
    return sign | (code > 0x7eu ? 0x7eu : code);
}

// E2M1 {0, .5, 1, 1.5, 2, 3, 4, 6}, sign in bit 3, round to nearest even,
// saturating at 6; NaN -> 6 with its sign.
__device__ __forceinline__ uint32_t f32_to_e2m1(float x) {
    const uint32_t b = __float_as_uint(x);
    const uint32_t sign = (b >> 28) & 8u;
    const uint32_t a = b & 0x7fffffffu;
    if (a > 0x7f800000u) return sign | 7u;
    if (a < 0x3f800000u)                                  // |x| < 1: step 0.5
        return sign | (uint32_t)__builtin_rintf(__uint_as_float(a) * 2.0f);      // 0, 1, 2 (2 = 1.0)
    const int E = (int)(a >> 23) - 127;
    if (E > 2) return sign | 7u;
    uint32_t m = (a >> 22) & 1u;
    const uint32_t rem = a & 0x3fffffu;
    if (rem > 0x200000u || (rem == 0x200000u && (m & 1u))) ++m;
    const uint32_t code = ((uint32_t)(E + 1) << 1) + m;   // m == 2 carries
    return sign | (code > 7u ? 7u : code);
}

// ceil(log2(v)) of a positive float, subnormals included.
__device__ __forceinline__ int ceil_log2(float v) {
    const uint32_t b = __float_as_uint(v);
    const int e = (int)(b >> 23);
    const uint32_t m = b & 0x7fffffu;
    if (e == 0) return (31 - __clz((int)m)) - 149 + ((m & (m - 1u)) != 0u);
    return e - 127 + (m != 0u);
}

// Power-of-two scale exponent: the smallest E with amax / 2^E <= qmax,
// clamped to the E8M0 range; 0 (code 127) for an all-zero group.
__device__ __forceinline__ int mx_exp(float amax, float qmax) {
    if (!(amax > 0.0f)) return 0;
    const float v = amax / qmax;                          // IEEE division
    if (v == 0.0f) return -127;                           // the quotient underflows: the clamp
    const int e = ceil_log2(v);
    return e < -127 ? -127 : (e > 127 ? 127 : e);
}

// max over `width` consecutive lanes (width a power of two <= 64)
template <int WIDTH>
__device__ __forceinline__ float group_max(float v) {
#pragma unroll
    for (int d = 1; d < WIDTH; d <<= 1) v = fmaxf(v, __shfl_xor(v, d, 64));
    return v;
}

// The same over 4 or 16 lanes on bit patterns, by DPP (no LDS pipe): quad
// permutes, then row rotations, which leave every lane of a 16-lane row with
// the row's maximum.
template <int WIDTH>
__device__ __forceinline__ uint32_t group_max_bits(uint32_t v) {
    static_assert(WIDTH == 4 || WIDTH == 16, "one quad or one DPP row");
    auto step = [&](uint32_t o) { v = v > o ? v : o; };
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true));     // quad_perm [1,0,3,2]
    step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true));     // quad_perm [2,3,0,1]
    if constexpr (WIDTH == 16) {
        step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xF, 0xF, true));    // row_ror:4
        step((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, true));    // row_ror:8
    }
    return v;
}

// ---------------------------------------------------------------- fast codecs
// For a group whose |amax| is 0 or in [2^-80, inf) the codes come from the
// gfx950 conversion instructions, which round to nearest even exactly as the
// codecs above (all bf16 values x 207 scale exponents, all fp32 patterns up
// to 448 compared on the GPU: no difference); other groups (infinities,
// NaN, amax below 2^-80, where the quotient's remainder could underflow)
// take the codecs above.  Bit patterns of |x| order like the values, and NaN
// above infinity, so one integer maximum finds amax and both exceptions.
constexpr uint32_t kFastLo = (127u - 80u) << 23, kInfBits = 0x7f800000u;
__device__ __forceinline__ bool fast_group(uint32_t amax) { return amax == 0u || (amax >= kFastLo && amax < kInfBits); }

// mx_exp of a fast group from the bits of amax: the smallest E with
// amax <= qmax 2^E is amax's exponent less qmax's, one more when its
// mantissa is above qmax's (448 = 1.75 2^8, 6 = 1.5 2^2).  mx_exp's rounded
// quotient never crosses that line (every normal amax compared).
template <int FMT>
__device__ __forceinline__ int fast_exp(uint32_t amax) {
    if (amax == 0u) return 0;
    return FMT == 2 ? (int)((amax + 0x3fffffu) >> 23) - 129 : (int)((amax + 0x1fffffu) >> 23) - 135;
}

// x / s rounded to nearest, r = 1 / s rounded to nearest: one Newton step on
// the quotient, whose remainder is exact (P. Markstein, "Computation of
// elementary functions on the IBM RISC System/6000 processor", IBM J. Res.
// Dev. 34, 1990).  The remainder is taken with its sign turned so that x =
// -0 keeps its sign.
__device__ __forceinline__ float div_by(float x, float s, float r) {
    const float q = x * r;
    return fmaf(-fmaf(q, s, -x), r, q);
}

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8), aligned(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32_a2 __attribute__((aligned(2)));

// Eight consecutive input elements as loaded (16 or 32 bytes; the hardware
// takes vector loads and stores at dword, and for codes at byte, alignment).
template <bool BF16IN>
struct Unit;
template <>
struct Unit<true> {
    i32x4 w;
    __device__ __forceinline__ void load(const void* base, long long elem) {
        w = __builtin_bit_cast(i32x4, *(const bf16x8*)((const uint16_t*)base + elem));
    }
    __device__ __forceinline__ void zero() { w = i32x4{0, 0, 0, 0}; }
    __device__ __forceinline__ uint32_t amax_bits() const {
        u16x2 m = {0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(u16x2, w[i] & 0x7fff7fff));
        return (uint32_t)(m[0] > m[1] ? m[0] : m[1]) << 16;
    }
    __device__ __forceinline__ float f(int i) const {
        return __uint_as_float((i & 1) ? (uint32_t)w[i >> 1] & 0xffff0000u : (uint32_t)w[i >> 1] << 16);
    }
    __device__ __forceinline__ bf16x2 pair(int i) const {
        const int d = w[i];    // a value of its own: bit-casting the vector's element in place takes element 0
        return __builtin_bit_cast(bf16x2, d);
    }
    template <int I>
    __device__ __forceinline__ i16x2 cvt8(i16x2 old, float s) const {    // pair I of the unit into half I % 2
        return __builtin_amdgcn_cvt_scalef32_pk_fp8_bf16(old, pair(I), s, I & 1);
    }
    template <int I>
    __device__ __forceinline__ uint32_t cvt4(uint32_t old, float s) const {    // pair I into byte I
        return __builtin_amdgcn_cvt_scalef32_pk_fp4_bf16(old, pair(I), s, I);
    }
};
template <>
struct Unit<false> {
    f32x4 lo, hi;
    __device__ __forceinline__ void load(const void* base, long long elem) {
        lo = *(const f32x4*)((const float*)base + elem);
        hi = *(const f32x4*)((const float*)base + elem + 4);
    }
    __device__ __forceinline__ void zero() { lo = hi = f32x4{0.f, 0.f, 0.f, 0.f}; }
    __device__ __forceinline__ uint32_t amax_bits() const {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t b = __float_as_uint(f(i)) & 0x7fffffffu;
            m = m > b ? m : b;
        }
        return m;
    }
    __device__ __forceinline__ float f(int i) const { return i < 4 ? lo[i & 3] : hi[i & 3]; }
    template <int I>
    __device__ __forceinline__ i16x2 cvt8(i16x2 old, float s) const {
        return __builtin_amdgcn_cvt_scalef32_pk_fp8_f32(old, f(2 * I), f(2 * I + 1), s, I & 1);
    }
    template <int I>
    __device__ __forceinline__ uint32_t cvt4(uint32_t old, float s) const {
        return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(old, f(2 * I), f(2 * I + 1), s, I);
    }
};

// The codes of one unit of a fast group: FMT 0 e4m3 of x / sc (sc fp32),
// 1 e4m3 and 2 e2m1 of x 2^-E, sc = 2^E.  Two dwords (FMT 2: one).
template <int FMT, bool BF16IN>
__device__ __forceinline__ u32x2 fast_codes(const Unit<BF16IN>& v, float sc) {
    if constexpr (FMT == 0) {
        const float r = 1.0f / sc;
        float y[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) y[i] = div_by(v.f(i), sc, r);
        int a = __builtin_amdgcn_cvt_pk_fp8_f32(y[0], y[1], 0, false), b = __builtin_amdgcn_cvt_pk_fp8_f32(y[4], y[5], 0, false);
        a = __builtin_amdgcn_cvt_pk_fp8_f32(y[2], y[3], a, true);
        b = __builtin_amdgcn_cvt_pk_fp8_f32(y[6], y[7], b, true);
        return u32x2{(unsigned)a, (unsigned)b};
    } else if constexpr (FMT == 1) {
        i16x2 a = {0, 0}, b = {0, 0};
        a = v.template cvt8<0>(a, sc);
        a = v.template cvt8<1>(a, sc);
        b = v.template cvt8<2>(b, sc);
        b = v.template cvt8<3>(b, sc);
        return u32x2{__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b)};
    } else {
        uint32_t a = v.template cvt4<0>(0u, sc);
        a = v.template cvt4<1>(a, sc);
        a = v.template cvt4<2>(a, sc);
        a = v.template cvt4<3>(a, sc);
        return u32x2{a, 0u};
    }
}

// The same by the codecs above, for any group.
template <int FMT, bool BF16IN>
__device__ __forceinline__ u32x2 slow_codes(const Unit<BF16IN>& v, float sc, int E) {
    u32x2 w = {0, 0};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if constexpr (FMT == 0) w[i >> 2] |= f32_to_e4m3(v.f(i) / sc) << (8 * (i & 3));
        else if constexpr (FMT == 1) w[i >> 2] |= f32_to_e4m3(__builtin_ldexpf(v.f(i), -E)) << (8 * (i & 3));
        else w[0] |= f32_to_e2m1(__builtin_ldexpf(v.f(i), -E)) << (4 * i);
    }
    return w;
}

template <bool BF16IN>
__device__ __forceinline__ float amax8(const Unit<BF16IN>& v) {
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v.f(i)));
    return m;
}

// byte offset of (row, group) in aiter's e8m0_shuffle order (rows padded to
// 32, groups to 8; MX4 candidate_m10 host.cc:194-206)
__device__ __forceinline__ long long shuffled_scale_offset(int r, int g, int kg8) {
    return ((long long)(r >> 5) * (kg8 >> 3) + (g >> 3)) * 256 + (g & 3) * 64 + (r & 15) * 4 + ((g & 7) >> 2) * 2 +
           ((r & 31) >> 4);
}

struct QuantArgs {
    const void* x;
    uint8_t* q;
    void* s;                 // scales: fp32 or E8M0 bytes
    long long ldx, ldq;      // elements / bytes
    long long s_sm, s_sk;    // scale element strides along rows and K blocks (row-major / column-major)
    int rows, k;
    int kg8;                 // e8m0_shuffle: K/32 rounded up to 8
    int lc;                  // log2 of the tile's units of 8 columns
    int ctiles;              // tiles along K
};

// Row-wise group quantizer, GROUP elements per scale (32 for MX, 128 for
// the 1x128 activation blocks).
//   FMT  0: e4m3 with fp32 scale amax / 448 (x / scale, IEEE division)
//        1: e4m3 with E8M0 scale 2^ceil(log2(amax / 448))
//        2: e2m1 with E8M0 scale 2^ceil(log2(amax / 6))
// SHUF: E8M0 scales in e8m0_shuffle order instead of (s_sm, s_sk) strides.
//
// A workgroup takes a tile of 8 << lc columns and U (256 >> lc) rows, one
// unit of 8 elements per thread and row pass: a wave reads 1 KB (bf16) per
// load, all U loads first.  A group's amax is 4 or 16 neighbouring lanes'
// (one quad / DPP row).  The tile's scales meet in LDS and leave in the
// order of their layout: whole runs of a row, of a column, or (SHUF, tiles
// of 32 rows x 256 columns) the whole 256-byte shuffled block, whose padding
// rows and groups are written as 0x7F here rather than by a fill before.
//
// Bound by HBM.  One thread per 4 elements with the codecs in software (20
// instructions a code, 64-bit divisions for the row) was bound by its VALU
// work instead.  Time per launch in a graph, before -> after, bf16 in:
//   4096 x 7168   fp32 scales 37.9 -> 17.9 us (4.9 TB/s), E8M0 per 128
//                 35.4 -> 15.7 (5.6), MXFP8 33.7 -> 15.2 (5.8), MXFP4
//                 36.5 -> 13.7 (5.4), shuffled 39.2 -> 14.4 (5.1)
//   7168 x 16384  MXFP4 shuffled 150 -> 43.4 us (6.8 TB/s)
//   500 x 7168    MXFP8 6.7 -> 3.2 us
//   32 x 7168     fp32 scales 2.9 -> 2.3 us (an empty launch takes 1.8)
//   57 x 7168     MXFP4 shuffled, with the padding fill's launch 4.8 -> 2.4
// fp32 in: 1.2-2.9x, 5.2-7.2 TB/s from 4096 x 2048.
template <int FMT, int GROUP, bool BF16IN, bool SHUF, int U>
__global__ __launch_bounds__(256) void quant_rows_kernel(const QuantArgs p) {
    constexpr int UPG = GROUP / 8;                 // units (lanes) per group
    constexpr int LUPG = GROUP == 32 ? 2 : 4;
    constexpr int NSC = U * 256 / UPG;             // scales of a tile
    typedef typename std::conditional<FMT == 0, float, uint8_t>::type Scale;
    __shared__ Scale sc_tile[NSC];
    const int t = threadIdx.x, lc = p.lc;
    const int rt = (int)(blockIdx.x / (unsigned)p.ctiles), ct = (int)(blockIdx.x - (unsigned)rt * (unsigned)p.ctiles);
    const int rpp = 256 >> lc;                     // rows per pass
    const long long row0 = (long long)rt * (U * rpp);
    const int lr = t >> lc, lu = t & ((1 << lc) - 1), col = (ct << (lc + 3)) + 8 * lu;
    const bool col_ok = col < p.k;
    Unit<BF16IN> v[U];
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const long long r = row0 + i * rpp + lr;
        v[i].zero();
        if (col_ok && r < p.rows) v[i].load(p.x, r * p.ldx + col);
    }
#pragma unroll
    for (int i = 0; i < U; ++i) {
        const long long r = row0 + i * rpp + lr;
        const bool ok = col_ok && r < p.rows;
        const uint32_t amax = group_max_bits<UPG>(v[i].amax_bits());
        float sc = 1.0f;
        int E = 0;
        u32x2 w;
        if (fast_group(amax)) {
            if constexpr (FMT == 0) {
                sc = amax != 0u ? __uint_as_float(amax) / 448.0f : 1.0f;
            } else {
                E = fast_exp<FMT>(amax);
                sc = __uint_as_float((uint32_t)(E + 127) << 23);
            }
            w = fast_codes<FMT, BF16IN>(v[i], sc);
        } else {
            const float am = group_max<UPG>(amax8<BF16IN>(v[i]));
            if constexpr (FMT == 0) sc = am > 0.0f ? am / 448.0f : 1.0f;
            else E = mx_exp(am, FMT == 2 ? 6.0f : 448.0f);
            w = slow_codes<FMT, BF16IN>(v[i], sc, E);
        }
        if (ok) {
            uint8_t* q = p.q + r * p.ldq + (FMT == 2 ? col >> 1 : col);
            if constexpr (FMT == 2) *(u32_a2*)q = w[0];
            else *(u32x2_a4*)q = __builtin_bit_cast(u32x2_a4, w);
        }
        if ((lu & (UPG - 1)) == 0) {
            Scale o;
            if constexpr (FMT == 0) o = sc;
            else o = SHUF && !ok ? (uint8_t)0x7f : (uint8_t)(E + 127);
            sc_tile[((i * rpp + lr) << (lc - LUPG)) + (lu >> LUPG)] = o;
        }
    }
    __syncthreads();
    const int lg = lc - LUPG, g0 = ct << lg;       // log2 of the tile's groups per row; its first group
    if (t >= NSC) return;
    if constexpr (SHUF) {
        // padding included: rows to a multiple of 32, groups to one of 8
        int r, g;
        if constexpr (U == 4) {                    // e = byte of the tile's one shuffled block
            r = (t & 1) * 16 + ((t & 63) >> 2);
            g = ((t & 3) >> 1) * 4 + (t >> 6);
        } else {
            r = t >> lg;
            g = t & ((1 << lg) - 1);
        }
        if (row0 + r < (p.rows + 31LL) / 32 * 32 && g0 + g < p.kg8)
            ((uint8_t*)p.s)[shuffled_scale_offset((int)(row0 + r), g0 + g, p.kg8)] = sc_tile[(r << lg) + g];
    } else {
        const int lrows = 8 - lc + (U == 4 ? 2 : 0);
        int r, g;
        if (p.s_sk == 1) {                         // a row's groups are neighbours
            r = t >> lg;
            g = t & ((1 << lg) - 1);
        } else {                                   // a group's rows are neighbours
            g = t >> lrows;
            r = t & ((1 << lrows) - 1);
        }
        if (row0 + r < p.rows && g0 + g < p.k / GROUP)
            ((Scale*)p.s)[(row0 + r) * p.s_sm + (g0 + g) * p.s_sk] = sc_tile[(r << lg) + g];
    }
}

// 128 x 128 weight-block quantizer: one workgroup (4 waves) per block;
// thread t holds columns 8(t % 16) .. +7 of rows t/16 + 16i (i < 8) -- each
// load instruction covers four whole 256-byte (bf16) rows of the block -- and
// the block's amax meets in LDS.  Rows past N belong to no block element
// (masked).  Codes as in the row quantizers; the whole workgroup takes the
// software codecs when the block holds an infinity, NaN or a tiny amax.
//   FMT 0: fp32 scale amax / 448; 1: E8M0 2^ceil(log2(amax / 448)).
// HBM-bound.  Four columns per thread and the software codecs -> this, per
// launch in a graph, bf16 in, fp32 / E8M0 scales: 192 x 2048 14.9 / 13.2 ->
// 3.6 / 3.1 us, 4096 x 7168 39.8 / 35.8 -> 14.9 / 14.6 (5.9 TB/s),
// 7168 x 16384 143 / 132 -> 63 / 63; fp32 in 1.05-3.6x (5.3-6.8 TB/s).
template <int FMT, bool BF16IN>
__global__ __launch_bounds__(256) void quant_wgt_block_kernel(const QuantArgs p) {
    __shared__ uint32_t wmax[8];
    const int g = blockIdx.x, nb = blockIdx.y, t = threadIdx.x;
    const int col = g * 128 + 8 * (t & 15), r0 = t >> 4;
    const int rows = min(128, p.rows - nb * 128);
    Unit<BF16IN> v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = r0 + 16 * i;
        v[i].zero();
        if (r < rows) v[i].load(p.x, (long long)(nb * 128 + r) * p.ldx + col);
    }
    uint32_t bits = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t b = v[i].amax_bits();
        bits = bits > b ? bits : b;
    }
    bits = group_max_bits<16>(bits);
#pragma unroll
    for (int d = 16; d < 64; d <<= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)bits, d, 64);
        bits = bits > o ? bits : o;
    }
    if ((t & 63) == 0) wmax[t >> 6] = bits;
    __syncthreads();
    bits = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
    const bool fast = fast_group(bits);
    float amax = __uint_as_float(bits);
    if (!fast) {                                   // NaN does not count towards amax
        amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) amax = fmaxf(amax, amax8<BF16IN>(v[i]));
        amax = group_max<64>(amax);
        if ((t & 63) == 0) wmax[4 + (t >> 6)] = __float_as_uint(amax);
        __syncthreads();
        amax = fmaxf(fmaxf(__uint_as_float(wmax[4]), __uint_as_float(wmax[5])),
                     fmaxf(__uint_as_float(wmax[6]), __uint_as_float(wmax[7])));
    }
    float sc = 1.0f;
    int E = 0;
    if constexpr (FMT == 0) {
        sc = amax > 0.0f ? amax / 448.0f : 1.0f;
        if (t == 0) ((float*)p.s)[nb * p.s_sm + g] = sc;
    } else {
        E = mx_exp(amax, 448.0f);
        if (t == 0) ((uint8_t*)p.s)[nb * p.s_sm + g] = (uint8_t)(E + 127);
        if (fast) sc = __uint_as_float((uint32_t)(E + 127) << 23);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int r = r0 + 16 * i;
        if (r < rows) {
            const u32x2 w = fast ? fast_codes<FMT, BF16IN>(v[i], sc) : slow_codes<FMT, BF16IN>(v[i], sc, E);
            *(u32x2_a4*)(p.q + (long long)(nb * 128 + r) * p.ldq + col) = __builtin_bit_cast(u32x2_a4, w);
        }
    }
}

// ---------------------------------------------------------------- layouts
// K-panel [kt][n][128]; W16 [n/16][kbytes/16][16 rows][16] and FRAG, the same
// order with the rows padded by zeros to a multiple of 16 (per K-tile
// [h][q][row][16], chunk 4 h + q).
//
// A workgroup moves 16 rows x 2 U K-tiles, a thread U units of 16 bytes, all
// loads before the stores.  A wave's 64 units are 8 rows x one K-tile: whole
// 128-byte lines on both sides.  W16 / FRAG stores go through LDS, so that
// neighbouring lanes store neighbouring rows of a chunk (stored as loaded:
// 1.05-1.09x the time).  Every byte is touched once: nontemporal both ways
// (1.06-1.2x).  HBM-bound: walking the destination unit by unit, reading half
// lines -> this, us, N x K bytes: W16 and FRAG 7168 x 8192 23.8 -> 20.7, 4096 x
// 7168 14.5 -> 11.9, 2112 x 7168 9.0 -> 7.0, 16384 x 6144 40.2 -> 33.8 (6.0
// TB/s; a 1 GiB device copy 5.0); KPANEL 25.1 -> 22.7, 14.6 -> 10.9, 9.1 ->
// 6.5, 39.7 -> 35.3; 1536 x 2048 3.4 -> 3.1.
enum class Lay : int { KPANEL = 0, W16 = 1, FRAG = 2 };

template <Lay L, int U>
__global__ __launch_bounds__(256) void relayout_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                       int n, int kbytes, long long ld) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int r = (w & 1) * 8 + (lane >> 3), chunks = kbytes / 16;
    const int c0 = (blockIdx.x * 2 * U + (w >> 1)) * 8 + (lane & 7);    // chunk of unit 0; unit i: + 16 i
    __shared__ i32x4 turn[L == Lay::KPANEL ? 1 : 256];
    i32x4* const mine = turn + w * 64;
    const int blocks = n / 16 + (n % 16 != 0);
    for (int nb = blockIdx.y; nb < blocks; nb += gridDim.y) {
        const long long row = (long long)nb * 16 + r;
        if (L != Lay::FRAG && row >= n) continue;
        const uint8_t* const in = src + row * ld;
        i32x4 v[U];
#pragma unroll
        for (int i = 0; i < U; ++i) {
            v[i] = i32x4{0, 0, 0, 0};
            if (row < n && c0 + 16 * i < chunks) v[i] = __builtin_nontemporal_load((const i32x4*)(in + (c0 + 16 * i) * 16LL));
        }
#pragma unroll
        for (int i = 0; i < U; ++i) {
            if constexpr (L == Lay::KPANEL) {
                const int c = c0 + 16 * i;
                if (c < chunks) __builtin_nontemporal_store(v[i], (i32x4*)(dst + ((long long)(c >> 3) * n + row) * 128 + (c & 7) * 16));
            } else {    // through LDS, so that neighbouring lanes hold neighbouring rows of one chunk
                mine[lane ^ (lane >> 3)] = v[i];
                __builtin_amdgcn_wave_barrier();
                const i32x4 x = mine[((lane & 7) * 8 + (lane >> 3)) ^ (lane & 7)];
                __builtin_amdgcn_wave_barrier();
                const int c = c0 - (lane & 7) + (lane >> 3) + 16 * i;
                if (c < chunks) __builtin_nontemporal_store(x, (i32x4*)(dst + ((long long)nb * chunks + c) * 256 + ((w & 1) * 8 + (lane & 7)) * 16));
            }
        }
    }
}

// e8m0_shuffle: one thread per destination byte; padding bytes are 0x7F.
__global__ __launch_bounds__(256) void e8m0_shuffle_kernel(const uint8_t* __restrict__ src, uint8_t* __restrict__ dst,
                                                           int rows, int kg, long long ld, int kg8, long long bytes) {
    for (long long o = (long long)blockIdx.x * 256 + threadIdx.x; o < bytes; o += (long long)gridDim.x * 256) {
        const long long blk = o >> 8;
        const int w = (int)(o & 255);
        const long long rb = blk / (kg8 >> 3), gb = blk - rb * (kg8 >> 3);
        const long long r = rb * 32 + (w & 1) * 16 + ((w & 63) >> 2);
        const long long g = gb * 8 + ((w & 3) >> 1) * 4 + (w >> 6);
        dst[o] = (r < rows && g < kg) ? src[r * ld + g] : (uint8_t)0x7f;
    }
}

// e8m0_shuffle of one or two operands (all batch entries) in one launch: a
// workgroup turns one 32-row block x 16 K-tiles (128 groups) of row-major
// E8M0 into 16 contiguous 256-byte shuffled blocks.  Each row's 128-byte run
// is read with dword loads (8 threads per row) into LDS, and every thread
// then gathers and writes 16 contiguous destination bytes.  Rows past
// `rows` and groups past kg read as 0x7F.  Source rows and pitches are
// dword aligned, destinations 16-byte aligned.
__global__ __launch_bounds__(256) void e8m0_shuffle_blocks_kernel(const ShuffleArgs a) {
    __shared__ uint8_t run[32][132];    // 33 dwords per row: the gathers spread over the banks
    int u = blockIdx.x, op = 0;
    if (u >= a.units[0]) {
        u -= a.units[0];
        op = 1;
    }
    const int kg = a.kg, kt8 = (kg + 7) / 8, chunks = (kt8 + 15) / 16;
    const int rb = u / chunks, ch = u - rb * chunks;
    const int rows = a.rows[op];
    const uint8_t* src = a.src[op] + (long long)blockIdx.y * a.src_batch[op];
    uint8_t* dst = a.dst[op] + (long long)blockIdx.y * a.dst_batch[op];
    const int t = threadIdx.x, rl = t >> 3, seg = t & 7, row = rb * 32 + rl;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
        const int g = ch * 128 + seg * 16 + 4 * d;
        uint32_t v = 0x7F7F7F7Fu;
        if (row < rows) {
            const uint8_t* q = src + (long long)row * a.ld[op] + g;
            if (g + 3 < kg) {
                v = *(const uint32_t*)q;
            } else {
                v = 0;
                for (int e = 0; e < 4; ++e) v |= (uint32_t)(g + e < kg ? q[e] : 0x7Fu) << (8 * e);
            }
        }
        *(uint32_t*)&run[rl][seg * 16 + 4 * d] = v;
    }
    __syncthreads();
    const int j = t >> 4, kt = ch * 16 + j, w0 = (t & 15) * 16;
    if (kt >= kt8) return;
    uint32_t o[4] = {0, 0, 0, 0};
#pragma unroll
    for (int e = 0; e < 16; ++e) {
        const int w = w0 + e;
        const int r = (w & 1) * 16 + ((w & 63) >> 2), g = j * 8 + ((w & 3) >> 1) * 4 + (w >> 6);
        o[e >> 2] |= (uint32_t)run[r][g] << (8 * (e & 3));
    }
    *(i32x4*)(dst + (long long)rb * 32 * (kt8 * 8) + (long long)kt * 256 + w0) =
        i32x4{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
}

// Row passes of 256 threads up to which the row quantizer runs one per
// workgroup: 2048 workgroups are one round of the chip at eight per CU.
constexpr long long kQuantOnePass = 2048;
constexpr long long kGridMaxX = 0xffffffffLL / 256;    // workgroups of 256

unsigned grid_for(long long units) {
    const long long b = (units + 255) / 256;
    return (unsigned)(b < 8192 ? (b > 0 ? b : 1) : 8192);
}

}  // namespace

// ---------------------------------------------------------------- launchers
hipError_t launch_quant_rows(int fmt, int group, bool bf16in, bool shuffle, const void* x, long long ldx,
                             uint8_t* q, long long ldq, void* s, long long s_sm, long long s_sk, int rows, int k,
                             hipStream_t st) {
    QuantArgs p{};
    p.x = x;
    p.q = q;
    p.s = s;
    p.ldx = ldx;
    p.ldq = ldq;
    p.s_sm = s_sm;
    p.s_sk = s_sk;
    p.rows = rows;
    p.k = k;
    p.kg8 = (k / 32 + 7) / 8 * 8;
    // Tile: scales that run along K (row-major) take up to 1024 columns, so
    // a row's scales leave in runs of 8 floats or 32 bytes; column-major and
    // shuffled scales take 256 columns of 32 rows.  Narrow K takes a
    // narrower tile (no idle columns).  One row pass per workgroup while
    // that leaves the chip room (latency counts, not bytes per workgroup),
    // else four.
    const bool tall = shuffle || s_sk != 1;
    int lc = tall ? 5 : 7;
    while (!shuffle && lc > (group == 32 ? 2 : 4) && (4LL << lc) >= k) --lc;
    p.lc = lc;
    // (k rounded up to a tile passes INT_MAX; the last unit's column, 2^31 - 8, does not)
    p.ctiles = (int)((k + (8LL << lc) - 1) >> (lc + 3));
    const long long prow = shuffle ? (rows + 31LL) / 32 * 32 : rows;
    const long long passes = (prow + (256 >> lc) - 1) / (256 >> lc) * p.ctiles;
    const bool one = passes <= kQuantOnePass;
    const long long rpt = (256 >> lc) * (one ? 1 : 4);
    const long long blocks = (prow + rpt - 1) / rpt * p.ctiles;
    // A grid dimension holds 2^32 threads: more tiles go in several launches of
    // whole row tiles (a second dimension made calls of 500 - 4096 rows up to
    // 1.3% slower).
    if (blocks > kGridMaxX) {
        const long long part = kGridMaxX / p.ctiles * rpt;
        for (long long r = 0; r < rows; r += part) {
            const hipError_t e = launch_quant_rows(
                fmt, group, bf16in, shuffle, static_cast<const uint8_t*>(x) + r * ldx * (bf16in ? 2 : 4), ldx, q + r * ldq, ldq,
                static_cast<uint8_t*>(s) + r * (shuffle ? p.kg8 : s_sm * (fmt == 0 ? 4 : 1)), s_sm, s_sk,
                (int)(rows - r < part ? rows - r : part), k, st);
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }
    const unsigned grid = (unsigned)blocks;
#define QG_QUANT(F, G, B, S)                                                                            \
    if (fmt == F && group == G && bf16in == B && shuffle == S) {                                        \
        if (one) quant_rows_kernel<F, G, B, S, 1><<<grid, 256, 0, st>>>(p);                             \
        else quant_rows_kernel<F, G, B, S, 4><<<grid, 256, 0, st>>>(p);                                 \
        trace_launch("quant_rows<%s,g%d,%s%s>", F == 0 ? "e4m3,fp32" : F == 1 ? "e4m3,e8m0" : "e2m1,e8m0", G, \
                     B ? "bf16" : "fp32", S ? ",shuffled" : "");                                        \
        return hipGetLastError();                                                                       \
    }
    QG_QUANT(0, 128, false, false) QG_QUANT(0, 128, true, false)
    QG_QUANT(1, 128, false, false) QG_QUANT(1, 128, true, false)
    QG_QUANT(1, 32, false, false) QG_QUANT(1, 32, true, false) QG_QUANT(1, 32, false, true) QG_QUANT(1, 32, true, true)
    QG_QUANT(2, 32, false, false) QG_QUANT(2, 32, true, false) QG_QUANT(2, 32, false, true) QG_QUANT(2, 32, true, true)
#undef QG_QUANT
    return hipErrorInvalidValue;
}

hipError_t launch_quant_wgt_blocks(int fmt, bool bf16in, const void* w, long long ldw, uint8_t* q, long long ldq,
                                   void* s, long long ld_s, int n, int k, hipStream_t st) {
    QuantArgs p{};
    p.x = w;
    p.q = q;
    p.s = s;
    p.ldx = ldw;
    p.ldq = ldq;
    p.s_sm = ld_s;
    p.rows = n;
    p.k = k;
    const dim3 grid(k / 128, (n + 127) / 128);
#define QG_WQ(F, B)                                                                                      \
    if (fmt == F && bf16in == B) {                                                                       \
        quant_wgt_block_kernel<F, B><<<grid, 256, 0, st>>>(p);                                           \
        trace_launch("quant_wgt_block<%s,%s>", F == 0 ? "e4m3,fp32" : "e4m3,e8m0", B ? "bf16" : "fp32"); \
        return hipGetLastError();                                                                        \
    }
    QG_WQ(0, false) QG_WQ(0, true) QG_WQ(1, false) QG_WQ(1, true)
#undef QG_WQ
    return hipErrorInvalidValue;
}

template <Lay L>
static void relayout_go(const uint8_t* src, uint8_t* dst, int n, int kbytes, long long ld, hipStream_t st) {
    const int blocks = n / 16 + (n % 16 != 0), kt = kbytes / 128 + (kbytes % 128 != 0);
    const unsigned y = blocks < 65535 ? blocks : 65535;
    // four units per thread once 2048 workgroups of them remain, K-panel 512
    // (4096 x 7168 12.9 -> 10.9 us, 7168 x 2048 7.2 -> 6.3, 2112 x 7168 6.9 -> 6.5;
    // W16 / FRAG there 0.96-1.05x); else one
    if ((long long)blocks * kt >= (L == Lay::KPANEL ? 4096 : 16384)) relayout_kernel<L, 4><<<dim3((kt + 7) / 8, y), 256, 0, st>>>(src, dst, n, kbytes, ld);
    else relayout_kernel<L, 1><<<dim3((kt + 1) / 2, y), 256, 0, st>>>(src, dst, n, kbytes, ld);
}
hipError_t launch_relayout(int layout, const uint8_t* src, uint8_t* dst, int n, int kbytes, long long ld,
                           hipStream_t st) {
    switch (layout) {
        case 0: relayout_go<Lay::KPANEL>(src, dst, n, kbytes, ld, st); trace_launch("relayout<KPANEL>"); break;
        case 1: relayout_go<Lay::W16>(src, dst, n, kbytes, ld, st); trace_launch("relayout<W16>"); break;
        case 2: relayout_go<Lay::FRAG>(src, dst, n, kbytes, ld, st); trace_launch("relayout<FRAG>"); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_e8m0_shuffle_blocks(const ShuffleArgs& a, int batch, hipStream_t st) {
    const dim3 grid(a.units[0] + a.units[1], batch);
    e8m0_shuffle_blocks_kernel<<<grid, 256, 0, st>>>(a);
    trace_launch("e8m0_shuffle_blocks<%d>", a.units[1] ? 2 : 1);
    return hipGetLastError();
}

hipError_t launch_e8m0_shuffle(const uint8_t* src, uint8_t* dst, int rows, int kg, long long ld, hipStream_t st) {
    const int kg8 = (kg + 7) / 8 * 8;
    const long long bytes = (long long)(rows + 31) / 32 * 32 * kg8;
    e8m0_shuffle_kernel<<<grid_for(bytes), 256, 0, st>>>(src, dst, rows, kg, ld, kg8, bytes);
    trace_launch("e8m0_shuffle");
    return hipGetLastError();
}

}  // namespace qg
