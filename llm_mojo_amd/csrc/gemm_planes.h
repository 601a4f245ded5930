// Several-token matmul on the 16-bit matrix cores over activation planes: the
// kernel template behind gemm_planes_*.hip.
//
// One kernel covers every stored weight format whose codes, less their zero
// point (and times an integer sub-block scale), are exact in 16-bit floats.
//
// Float activations of every format but Q4_K (F32) are read as they are, and
// each workgroup splits its tokens' into three bf16 planes in LDS that sum to
// them exactly (float32's 24 bits are bf16's 8 three times, over the same
// exponents): v_mfma_f32_16x16x32_bf16 forms sum q (p0 + p1 + p2) with every
// product exact in its fp32 sums.  So a call needs no memory and no other
// kernel, an input (from 2^-110 on) keeps its last bit whatever its neighbours
// are, and what is left of the format is applied in fp32: the block's scale
// per chunk of 32 inputs (Q8_0, Q4_0, Q4_1, Q5_K's sub-blocks, groups of 32 to
// 128) or per superblock of 8 (Q6_K, one scale a row).  Q6_K's codes times
// their sub-block scale are 13 bits: two bf16 operands.  Q4_1 and Q5_K take
// their codes less 8 or 16 and the rest of the offset times the chunk's sum
// of x, both in fp32 (the sum on the fp32 matrix cores), which keeps the two
// large sums from cancelling.  Chunks of a token that bf16 could not hold
// (an infinity, a NaN, inputs from 2^100 on, or nothing above 2^-85) are left
// out of the planes and added to the outputs weight by weight at the end.
// Off the 64-bit result (476 x 768 x 2304, a residual stream; the fp32 matrix
// cores): Q8_0 1.0e-7 (2.9e-7), Q5_K 1.0e-7 (2.9e-7), Q6_K 1.2e-7 (2.9e-7),
// int8-ch 1.0e-7 (2.9e-7).  Two fp16 planes under an exponent a superblock
// (22 bits, Q4_K's record below) were as close there and took 2 products for
// 3, but lost a small input beside one 2^20 times as large, to all of it.
//
// Q4_K's activations come as the h16 record of gguf_gemm16.hip: per token and
// superblock of 256 inputs a power-of-two scale s and x s as two fp16
// planes, hi and lo (22 bits together).  v_mfma_f32_16x16x32_f16 forms sum q
// (hi + lo); the superblock's scale and 1 / s are applied in fp32, and the
// minima are one more product per superblock, of whole numbers (m_j) with
// the record's sums of each chunk.
//
// Mapping: a workgroup of WT x WR x WK waves owns WT TT token tiles and
// WR RT row tiles (16 each); a wave computes TT x RT of the 16 x 16 blocks,
// over the whole reduction axis (WK = 1) or every WK-th chunk of it (the
// waves' sums are then added in LDS, in wave order), so an output's bits do
// not depend on the other tokens of the call (but, through the tile, on how
// many they are).  The axis is walked in steps of S chunks: a step's codes
// and scales (and the record's planes) are copied into one of two LDS buffers
// (global-to-LDS loads) while the waves compute the other; the floats of the
// step after go through registers, which a step's splitting empties before
// its products.  A superblock's fields, sums and 1 / s go to a pair of
// buffers of their own.
//
// What bounds it: over floats, a block (16 x 16, one chunk) has 3 products of
// 16 cycles and ~15 vector instructions of 4 (7 decode its share of a row
// tile's codes, 4 scale it, 4 to 5 split its share of x), and each wave reads
// 3 KB of planes a token tile and chunk.  512 x 4096 x 11008 Q8_0 in the
// 256-row tile: matrix cores busy 34 % of the time, the vector units 53 %, LDS
// 35 % (counters), the rest waits at 4 waves a SIMD; 16 waves a CU did more
// than wider wave tiles at 8 (4 x 2: 218 us, 2 x 4: 223, 2 x 2: 166, 2 x 3 in
// 128 registers: 157).  Few workgroups are bound by a wave's own chain through
// a step (~1 us for 2 chunks): tiles whose waves share the chunks out (WK = 2,
// 4).  Over a record, the LDS reads take half of the products' time and the
// decode and scales come to their own time at TT = 2; three or four buffers
// in flight instead of two measured the same or slower at every size.
// 512 x 4096 x 11008, fp32 matrix cores and here: Q8_0 1059 us and 157, Q4_0
// 1134 and 161, Q4_1 1134 and 187, Q5_K 777 and 202, Q6_K 1168 and 274,
// int8-ch 1142 and 182, int4-g32 1148 and 165 (0.88 PFLOP/s of bf16 products
// at Q8_0); Q4_K 725 and 124 with its record.
//
// int16 activation codes (kA4, kA8) come as two exact planes of their own,
// 256 hi + lo: every partial sum of a segment (at most 256 inputs) is a whole
// number below 2^24, so hi + lo is the integer and one fma per output and
// segment, in the reference's order, gives the int8 matrix cores' bits
// (512 x 4096 x 4096 with the activations: int8-ch 109 -> 59 us, int4-ch
// 72 -> 57, int8-g32 88 -> 70).
#pragma once
#include <type_traits>

#include "common.h"

namespace planes {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));
typedef __bf16 v8b __attribute__((ext_vector_type(8)));
typedef float v4f_u __attribute__((ext_vector_type(4), aligned(4)));

enum Fmt { kQ8_0, kQ4_0, kQ4_1, kQ4_K, kQ5_K, kQ6_K, kQm4, kQm8, kA4, kA8 };

struct Args {
    const uint8_t *planes, *sums, *inv;        // the h16 record
    const float *x;                            // or the floats themselves
    int64_t ldx;
    const uint8_t *codes, *scales, *zps, *bits, *sb, *sbd;
    int T, n, ntiles, NC, NSB, NG, gshift, flags;  // NC chunks of 32 inputs, NSB superblocks, NG groups a row
    int rows_first;                                // workgroup order: row blocks fastest
    int64_t ldo;
    const float *bias, *sx;  // sx: the tokens' scales (A16)
    float *out;
};

// Bytes a format keeps per (16-row tile, chunk of 32 inputs) and superblock.
template <int F>
struct Tr {
    static constexpr bool KQ = F == kQ4_K || F == kQ5_K || F == kQ6_K;
    static constexpr bool A16 = F == kA4 || F == kA8;                       // int16 activation codes
    static constexpr bool QM = F == kQm4 || F == kQm8 || A16;
    static constexpr bool F32 = !A16 && F != kQ4_K;                         // float inputs, split here
    static constexpr int AB = F32 ? 3072 : 2048;                            // planes of a token tile
    static constexpr bool W8 = F == kQ8_0 || F == kQm8 || F == kA8;
    static constexpr int CB = W8 ? 512 : 256;                               // codes
    static constexpr int SCB = KQ ? 0 : F == kQ4_1 ? 64 : 32;               // scales
    static constexpr int ZB = QM ? 16 : 0;                                  // zero points
    static constexpr int HB = F == kQ5_K ? 64 : F == kQ6_K ? 128 : 0;       // high bits
    static constexpr int SBF = KQ ? 256 : 0, SBD = F == kQ6_K ? 32 : 0;     // superblock fields
    static constexpr bool SUMS = F == kQ4_K;                                // additive minima, over the record's sums
    static constexpr bool CENTER = F == kQ4_1 || F == kQ5_K;                // codes less 8 / 16, minima in fp32
};

// 1024 + the 8 bytes of (a, b) as fp16 pairs (a0, a1), (a2, a3), (b0, b1),
// (b2, b3): 0x6400 | n is 1024 + n in fp16 for n < 1024.
__device__ __forceinline__ void bytes_f16(uint32_t a, uint32_t b, v2h (&d)[4]) {
    d[0] = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, a, 0x04010400u));
    d[1] = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, a, 0x04030402u));
    d[2] = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, b, 0x04010400u));
    d[3] = __builtin_bit_cast(v2h, __builtin_amdgcn_perm(0x64646464u, b, 0x04030402u));
}
__device__ __forceinline__ float h2f(uint32_t bits) { return __half2float(__ushort_as_half((unsigned short)bits)); }
// A read at byte `at` of an LDS buffer, the whole offset as one index: the
// compiler keeps track of which buffer a read is from (and so does not make
// it wait for copies into the others) through a few address steps only.
template <class T>
__device__ __forceinline__ T lds(const uint8_t *buf, int at) {
    return *reinterpret_cast<const T *>(buf + at);
}
__device__ __forceinline__ v2h splat(float v) { return (v2h){(_Float16)v, (_Float16)v}; }
// The high halves of (a, b): two floats cut to bf16.
__device__ __forceinline__ uint32_t high2(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }
// fp16 halves to float, plus c or times s plus c, an instruction each.
#define LLMQ_MIX(f, h, s, c, sel) \
    asm("v_fma_mix_f32 %0, %1, " s ", %2 op_sel:[" sel ",0,0] op_sel_hi:[1,0,0]" : "=v"(f) : "v"(h), "v"(c))
__device__ __forceinline__ void halves_add(v2h h, float c, float &lo, float &hi) {
    LLMQ_MIX(lo, h, "1.0", c, "0");
    LLMQ_MIX(hi, h, "1.0", c, "1");
}
#undef LLMQ_MIX
// Signed byte B of c to float.
template <int B>
__device__ __forceinline__ float sbyte(uint32_t c) {
    float f;
    if constexpr (B == 0) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f) : "v"(c));
    if constexpr (B == 1) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f) : "v"(c));
    if constexpr (B == 2) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f) : "v"(c));
    if constexpr (B == 3) asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f) : "v"(c));
    return f;
}
// Whether the 32 inputs of a token and chunk go through the bf16 planes, m
// the bits of the largest |x| of them: not where one is infinite, NaN or so
// large that a sum of 256 products with codes could pass float32's range, nor
// where all are so small that bf16 could not hold their last bits.
__device__ __forceinline__ bool in_planes(int m) {
    constexpr uint32_t lo = (127 - 85) << 23, hi = (127 + 100) << 23;
    return m == 0 || (uint32_t)m - lo < hi - lo;
}

template <int F, int TT, int RT, int WT, int WR, int S>
struct Lay {
    using R = Tr<F>;
    static constexpr int NTT = WT * TT, NRT = WR * RT;
    static constexpr int A = NTT * S * R::AB, C = NRT * S * R::CB, SC = NRT * S * R::SCB, Z = NRT * S * R::ZB,
                         H = NRT * S * R::HB;
    static constexpr int oC = R::F32 ? 0 : A, oSC = oC + C, oZ = oSC + SC, oH = oZ + Z, STEP = oH + H;
    static constexpr int SBF = NRT * R::SBF, SBD = NRT * R::SBD, SU = R::SUMS ? NTT * 512 : 0, IV = R::SUMS ? NTT * 64 : 0;
    static constexpr int oSBD = SBF, oSU = oSBD + SBD, oIV = oSU + SU, SBUF = oIV + IV;
};

// Weight k of chunk c of row r of row tile rt, as the reference decoders
// compute it (decode_chunk of gguf_gemm.hip).
template <int F>
__device__ float weight(const Args &a, int rt, int r, int c, int k) {
    using R = Tr<F>;
    const int e = (rt * a.NC + c) * 16 + r, se = (rt * a.NSB + c / 8) * 16 + r;
    const int ge = (rt * a.NG + (c >> a.gshift)) * 16 + r;
    auto u16 = [](const uint8_t *p, int i) { return h2f(reinterpret_cast<const uint16_t *>(p)[i]); };
    int u;
    if constexpr (R::W8)
        u = a.codes[(rt * a.NC + c) * 512 + (k >> 4) * 256 + r * 16 + (k & 15)];
    else
        u = (a.codes[e * 16 + (k >> 1)] >> (4 * (k & 1))) & 15;
    if constexpr (R::QM) return ((float)u - (float)a.zps[ge]) * u16(a.scales, ge);
    if constexpr (F == kQ8_0) return u16(a.scales, e) * (float)(int8_t)u;
    if constexpr (F == kQ4_0) return ((float)u - 8.0f) * u16(a.scales, e);
    if constexpr (F == kQ4_1) return u16(a.scales, 2 * e) * (float)u + u16(a.scales, 2 * e + 1);
    const uint8_t *f = a.sb + (int64_t)se * 16;
    if constexpr (F == kQ5_K) {
        const int j = c & 7;
        const uint8_t *q = f + 4;
        const int sc = j < 4 ? q[j] & 63 : (q[j + 4] & 15) | (q[j - 4] >> 6 << 4);
        const int mn = j < 4 ? q[j + 4] & 63 : (q[j + 4] >> 4) | (q[j] >> 6 << 4);
        u |= ((a.bits[(int64_t)e * 4 + (k >> 3)] >> (k & 7)) & 1) << 4;
        return u16(f, 0) * (float)sc * (float)u - u16(f, 1) * (float)mn;
    }
    if constexpr (F == kQ6_K) {
        u |= ((a.bits[(int64_t)e * 8 + (k >> 2)] >> (2 * (k & 3))) & 3) << 4;
        return u16(a.sbd, se) * (float)(int8_t)f[2 * (c & 7) + (k >> 4)] * ((float)u - 32.0f);
    }
    return 0.0f;
}

// SEG0: chunks of 32 inputs that share a scale (1, 2, 4, or 8 for one scale a
// superblock or more; over floats 1 or 8).
template <int F, int SEG0, int TT, int RT, int WT, int WR, int WK, int S>
__global__ __launch_bounds__(WT * WR * WK * 64, Tr<F>::F32 ? 4 : 2) void gemm_planes_kernel(Args a) {
    using R = Tr<F>;
    using L = Lay<F, TT, RT, WT, WR, S>;
    constexpr int SPB = 8 / S;  // steps a superblock
    static_assert(8 % S == 0 && S % WK == 0 && 4 % WK == 0, "whole steps a superblock, chunks for every wave");
    constexpr int NW = WT * WR * WK, RB = NW * 1024;  // bytes a copy round: 16 a lane
    constexpr int SEG = R::F32 ? 1 : SEG0;  // (over floats every chunk's sums are scaled or added by themselves)
    // One scale a superblock: over a record the products of its chunks chain, over floats, with twice as many
    // and more of Q6_K, the chunks' sums are added (chained, Q6_K was 2.0e-7 off at 476 x 768 x 2304).
    constexpr bool CHAIN = F == kQ4_K, ONE = R::F32 && F != kQ5_K && (R::KQ || SEG0 == 8);
    // separate arrays, so that the compiler sees a copy into one cannot alias reads of another
    __shared__ __align__(16) uint8_t b0[L::STEP], b1[L::STEP], f0[L::SBUF ? L::SBUF : 16], f1[L::SBUF ? L::SBUF : 16];
    // F32: the step's planes, the superblock's sums of x a chunk, and which token tiles have inputs left out of the planes
    __shared__ __align__(16) uint8_t x0[R::F32 ? L::A : 16], x1[R::F32 ? L::A : 16], s0[R::CENTER ? L::NTT * 512 : 16], s1[R::CENTER ? L::NTT * 512 : 16];
    __shared__ int left[L::NTT];
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c16 = lane & 15, g = lane >> 4;
    const int wt = w / WR % WT, wr = w % WR, kk = w / (WT * WR);
    // Workgroups go to the 8 XCDs in turn (linear id mod 8); each XCD gets a
    // contiguous run of (token block, row block) pairs, the operand with
    // more bytes slowest, so that it is read by few XCDs.
    int bx, by;
    {
        const int gx = gridDim.x, gy = gridDim.y, nb = gx * gy, id = blockIdx.y * gx + blockIdx.x;
        const int x = id & 7, q = nb >> 3, rem = nb & 7, pos = x * q + min(x, rem) + (id >> 3);
        if (a.rows_first) {
            bx = pos % gx;
            by = pos / gx;
        } else {
            by = pos % gy;
            bx = pos / gy;
        }
    }
    const int rt0 = bx * L::NRT, tt0 = by * L::NTT, ttiles = (a.T + 15) >> 4;
    // A token tile past the record or a row tile past the matrix copies tile
    // 0 instead (its outputs are not stored).
    auto ttile = [&](int j) __attribute__((always_inline)) { return tt0 + j < ttiles ? tt0 + j : 0; };
    auto rtile = [&](int j) __attribute__((always_inline)) { return rt0 + j < a.ntiles ? rt0 + j : 0; };
    // One region's copy: the 16 bytes at region offset off(q) from voff[q] on
    // from src; a last partial round is shared out over all waves where it
    // divides.
    auto part = [](int N, int q) constexpr { return q < N / RB || N % RB % (16 * NW) ? 1024 : N % RB / NW; };
    auto off = [&](auto bytes, int q) __attribute__((always_inline)) {
        return q * RB + w * part(decltype(bytes)::value, q) + lane * 16;
    };
    auto copy = [&](const uint8_t *src, uint8_t *dst, auto bytes, const uint32_t *voff) __attribute__((always_inline)) {
        constexpr int N = decltype(bytes)::value;
#pragma unroll
        for (int q = 0; q < (N + RB - 1) / RB; q++) {
            const bool whole = (q + 1) * RB <= N;
            if (whole || (N % RB % (16 * NW) ? off(bytes, q) < N : lane * 16 < part(N, q)))
                __builtin_amdgcn_global_load_lds(src + voff[q],
                                                 (__attribute__((address_space(3))) void *)(dst + q * RB + w * part(N, q)), 16, 0, 0);
        }
    };
    constexpr int NA = (L::A + RB - 1) / RB, NCC = (L::C + RB - 1) / RB, NS = (L::SC + RB - 1) / RB,
                  NZ = (L::Z + RB - 1) / RB, NH = (L::H + RB - 1) / RB, NF = (L::SBF + RB - 1) / RB;
#define LLMQ_N(bytes) std::integral_constant<int, bytes>{}
    uint32_t vA[NA], vC[NCC], vS[NS ? NS : 1], vZ[NZ ? NZ : 1], vH[NH ? NH : 1], vF[NF ? NF : 1], vD[1], vU[1], vI[1];
    if constexpr (!R::F32) {
#pragma unroll
        for (int q = 0; q < NA; q++) {
            const int x = off(LLMQ_N(L::A), q);
            vA[q] = ttile(x / (S * 2048)) * a.NC * 2048 + x % (S * 2048);
        }
    }
#pragma unroll
    for (int q = 0; q < NCC; q++) {
        const int x = off(LLMQ_N(L::C), q);
        vC[q] = rtile(x / (S * R::CB)) * a.NC * R::CB + x % (S * R::CB);
    }
    if constexpr (R::SCB > 0 && !R::QM) {
#pragma unroll
        for (int q = 0; q < NS; q++) {
            const int x = off(LLMQ_N(L::SC), q);
            vS[q] = rtile(x / (S * R::SCB)) * a.NC * R::SCB + x % (S * R::SCB);
        }
    }
    if constexpr (R::HB > 0) {
#pragma unroll
        for (int q = 0; q < NH; q++) {
            const int x = off(LLMQ_N(L::H), q);
            vH[q] = rtile(x / (S * R::HB)) * a.NC * R::HB + x % (S * R::HB);
        }
    }
    if constexpr (R::SBF > 0) {
#pragma unroll
        for (int q = 0; q < NF; q++) {
            const int x = off(LLMQ_N(L::SBF), q);
            vF[q] = rtile(x / 256) * a.NSB * 256 + x % 256;
        }
    }
    static_assert(L::SBD <= RB && L::SU <= RB && L::IV <= RB, "one copy round each");
    if constexpr (R::SBD > 0) {
        const int x = off(LLMQ_N(L::SBD), 0);
        vD[0] = rtile(x / 32) * a.NSB * 32 + x % 32;
    }
    if constexpr (R::SUMS) {
        const int x = off(LLMQ_N(L::SU), 0);
        vU[0] = ttile(x / 512) * a.NSB * 512 + x % 512;
    }
    if constexpr (L::IV > 0) {
        const int x = off(LLMQ_N(L::IV), 0);
        vI[0] = ttile(x / 64) * a.NSB * 64 + x % 64;
    }
#define LLMQ_CP(base, dst, bytes, v, at) copy(base + (int64_t)(at), dst, LLMQ_N(bytes), v)
    auto stage = [&](int c0, uint8_t *buf) __attribute__((always_inline)) {  // chunks c0 .. c0 + S - 1
        if constexpr (!R::F32) LLMQ_CP(a.planes, buf, L::A, vA, c0 * 2048);
        LLMQ_CP(a.codes, buf + L::oC, L::C, vC, c0 * R::CB);
        if constexpr (R::QM) {  // the chunk's group
#pragma unroll
            for (int q = 0; q < NS; q++) {
                const int x = off(LLMQ_N(L::SC), q), u = x % (S * 32) / 32;
                vS[q] = (rtile(x / (S * 32)) * a.NG + ((c0 + u) >> a.gshift)) * 32 + x % 32;
            }
#pragma unroll
            for (int q = 0; q < NZ; q++) {
                const int x = off(LLMQ_N(L::Z), q), u = x % (S * 16) / 16;
                vZ[q] = (rtile(x / (S * 16)) * a.NG + ((c0 + u) >> a.gshift)) * 16;
            }
            LLMQ_CP(a.scales, buf + L::oSC, L::SC, vS, 0);
            LLMQ_CP(a.zps, buf + L::oZ, L::Z, vZ, 0);
        } else if constexpr (R::SCB > 0) {
            LLMQ_CP(a.scales, buf + L::oSC, L::SC, vS, c0 * R::SCB);
        }
        if constexpr (R::HB > 0) LLMQ_CP(a.bits, buf + L::oH, L::H, vH, c0 * R::HB);
    };
    auto stage_sb = [&](int sb, uint8_t *buf) __attribute__((always_inline)) {
        if constexpr (R::SBF > 0) LLMQ_CP(a.sb, buf, L::SBF, vF, sb * 256);
        if constexpr (R::SBD > 0) LLMQ_CP(a.sbd, buf + L::oSBD, L::SBD, vD, sb * 32);
        if constexpr (R::SUMS) LLMQ_CP(a.sums, buf + L::oSU, L::SU, vU, sb * 512);
        if constexpr (L::IV > 0) LLMQ_CP(a.inv, buf + L::oIV, L::IV, vI, sb * 64);
    };
#undef LLMQ_CP
    // F32: the floats of a (token tile, chunk) unit a wave, UW of them a step:
    // lane (token l % 16, inputs 8 (l / 16) ..) has 8 from fetch() on, and
    // split() leaves them in LDS as three bf16 planes, x = p0 + p1 + p2
    // exactly (the high 8 bits, the next 8, the rest), in the codes' order.
    constexpr int U = L::NTT * S, UW = (U + NW - 1) / NW;
    uint32_t vX[UW];
    v4f_u xr[UW][2];
    auto unit = [&](int q) __attribute__((always_inline)) { return U % NW == 0 || w + q * NW < U; };
    if constexpr (R::F32) {
#pragma unroll
        for (int q = 0; q < UW; q++) {
            const int id = w + q * NW, tok = (tt0 + id / S) * 16 + c16;
            vX[q] = (uint32_t)(tok < a.T ? tok : 0) * (uint32_t)a.ldx * 4u + id % S * 128 + g * 32;
        }
        if (tid < L::NTT) left[tid] = 0;
        __syncthreads();
    }
    auto fetch = [&](int c0) __attribute__((always_inline)) {
        const uint8_t *src = reinterpret_cast<const uint8_t *>(a.x) + (int64_t)c0 * 128;
#pragma unroll
        for (int q = 0; q < UW; q++) {
            if (!unit(q)) continue;
            xr[q][0] = *reinterpret_cast<const v4f_u *>(src + vX[q]);
            xr[q][1] = *reinterpret_cast<const v4f_u *>(src + vX[q] + 16);
        }
    };
    auto over_groups = [](auto v, auto op) __attribute__((always_inline)) {  // over the 4 lanes of a token
        using T = decltype(v);
        auto both = [&](uint32_t x, uint32_t y) { return op(__builtin_bit_cast(T, x), __builtin_bit_cast(T, y)); };
        const uint32_t b = __builtin_bit_cast(uint32_t, v);
        const auto r16 = __builtin_amdgcn_permlane16_swap(b, b, false, false);
        const uint32_t d = __builtin_bit_cast(uint32_t, both(r16[0], r16[1]));
        const auto r32 = __builtin_amdgcn_permlane32_swap(d, d, false, false);
        return both(r32[0], r32[1]);
    };
    auto split = [&](uint8_t *xb, uint8_t *sums, int j0) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < UW; q++) {
            if (!unit(q)) continue;
            const int id = w + q * NW;
            uint32_t b[8];
#pragma unroll
            for (int i = 0; i < 8; i++) b[i] = __float_as_uint(xr[q][i >> 2][i & 3]);
            // the largest |x|: of the negative ones the largest bits, of the others the largest integer
            uint32_t um = b[0];
            int sm = (int)b[0];
#pragma unroll
            for (int i = 1; i < 8; i++) {
                um = max(um, b[i]);
                sm = max(sm, (int)b[i]);
            }
            const int m = over_groups(max((int)(um & 0x7FFFFFFFu), sm), [](int x, int y) { return max(x, y); });
            if (__any(!in_planes(m))) {
                const bool ok = in_planes(m);
#pragma unroll
                for (int i = 0; i < 8; i++) b[i] = ok ? b[i] : 0u;
                if (!ok) left[id / S] = 1;
            }
            uint32_t p1[8], p2[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float r = __uint_as_float(b[i]) - __uint_as_float(b[i] & 0xFFFF0000u);
                p1[i] = __float_as_uint(r);
                p2[i] = __float_as_uint(r - __uint_as_float(p1[i] & 0xFFFF0000u));
            }
            uint8_t *o = xb + id * 3072 + lane * 16;
            auto put = [&](const uint32_t (&v)[8], int at) __attribute__((always_inline)) {
                if constexpr (R::W8)
                    *reinterpret_cast<uint4 *>(o + at) =
                        make_uint4(high2(v[0], v[1]), high2(v[2], v[3]), high2(v[4], v[5]), high2(v[6], v[7]));
                else
                    *reinterpret_cast<uint4 *>(o + at) =
                        make_uint4(high2(v[0], v[2]), high2(v[4], v[6]), high2(v[1], v[3]), high2(v[5], v[7]));
            };
            put(b, 0);
            put(p1, 1024);
            put(p2, 2048);
            if constexpr (R::CENTER) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; i++) x[i] = __uint_as_float(b[i]);
                float sx = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7]));
                sx = over_groups(sx, [](float x, float y) { return x + y; });
                if (g == 0) *reinterpret_cast<float *>(sums + id / S * 512 + c16 * 32 + (j0 + id % S) * 4) = sx;
            }
        }
    };
    const v4f zero = {0.0f, 0.0f, 0.0f, 0.0f};
    v4f acc[TT][RT], d[TT][RT];  // outputs; the superblock's sums in scale s
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int r = 0; r < RT; r++) acc[t][r] = zero;
    v4f seg[TT][RT], sel[TT][RT];   // A16, SEG > 1: the group's sums of the hi and the lo plane
    v2h sc[RT][4];                  // Q4_K: sub-block scales (sc_2i, sc_2i+1)
    uint32_t sl5[RT], sh5[RT];      // Q5_K: the same as bytes, 0-3 and 4-7
    uint32_t mp[RT][4];             // Q4_K: minima of the 8 chunks, fp16 pairs
    float cm[RT][2] = {};           // CENTER: the offsets of chunks g and 4 + g
    float rs[RT];                   // ONE: the row's scale

    // this lane's place in each region of a buffer (opaque, so that a read is one step from its buffer)
    auto place = [](int v) { asm("" : "+v"(v)); return v; };
    const int pA = place(wt * TT * S * R::AB + kk * R::AB + lane * 16);
    const int pC = place(L::oC + wr * RT * S * R::CB + kk * R::CB + (R::W8 ? (g >> 1) * 256 + c16 * 16 + (g & 1) * 8 : c16 * 16 + g * 4));
    const int pS = place(L::oSC + wr * RT * S * R::SCB + kk * R::SCB + c16 * (R::SCB / 16));
    const int pZ = place(L::oZ + wr * RT * S * 16 + kk * 16 + c16);
    const int pH = place(L::oH + wr * RT * S * R::HB + kk * R::HB + c16 * (R::HB / 16) + g * (R::HB / 64));
    const int pF = place(wr * RT * 256 + c16 * 16), pF6 = place(wr * RT * 256 + c16 * 16 + (g >> 1) + 2 * kk);
    const int pD = place(L::oSBD + wr * RT * 32 + c16 * 2);
    const int pU = place(R::CENTER ? wt * TT * 512 + c16 * 32 + g * 4 : L::oSU + wt * TT * 512 + (lane & 31) * 16);
    const int pI = place(L::oIV + wt * TT * 64 + g * 16);

    // F32: row tile r's sums x of chunk j, times the scale s unless that is the superblock's
    auto scale = [&](int j, int r, const v4f (&x)[TT], float s) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TT; t++) {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if constexpr (ONE)
                    d[t][r][i] = j == 0 ? x[t][i] : d[t][r][i] + x[t][i];
                else
                    d[t][r][i] = j == 0 ? s * x[t][i] : fmaf(s, x[t][i], d[t][r][i]);
            asm volatile("" : "+v"(d[t][r]));  // (formed here: sunk past a branch, its products' results would pile up)
        }
    };

    // chunks j0 .. j0 + S - 1 of a superblock from cur (F32: and xb), its fields in sbf, its sums in sums
    auto compute = [&](auto j0c, const uint8_t *cur, const uint8_t *xb, const uint8_t *sbf, const uint8_t *sums) __attribute__((always_inline)) {
        constexpr int j0 = decltype(j0c)::value;
        if constexpr ((F == kQ4_K || F == kQ5_K) && j0 == 0) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                // sc_j and m_j as bytes (k_scale_min, gguf.mojo:205-221, four at a time)
                const uint4 f = lds<uint4>(sbf, pF + r * 256);
                const uint32_t sl = f.y & 0x3F3F3F3Fu, ml = f.z & 0x3F3F3F3Fu;
                const uint32_t sh = (f.w & 0x0F0F0F0Fu) | ((f.y >> 2) & 0x30303030u);
                const uint32_t mh = ((f.w >> 4) & 0x0F0F0F0Fu) | ((f.z >> 2) & 0x30303030u);
                if constexpr (F == kQ5_K) {  // (WK > 1: this wave's chunks' bytes to each unit's first place)
                    sl5[r] = WK > 1 ? sl >> (8 * kk) : sl;
                    sh5[r] = WK > 1 ? sh >> (8 * kk) : sh;
                } else if constexpr (WK > 1) {
                    bytes_f16(sl >> (8 * kk), sh >> (8 * kk), sc[r]);
                } else {
                    bytes_f16(sl, sh, sc[r]);
                }
                if constexpr (F == kQ4_K) {
#pragma unroll
                    for (int i = 0; i < 4; i++) sc[r][i] = sc[r][i] - splat(1024.0f);
                    v2h m2[4];
                    bytes_f16(ml, mh, m2);
#pragma unroll
                    for (int i = 0; i < 4; i++) mp[r][i] = __builtin_bit_cast(uint32_t, m2[i] - splat(1024.0f));
                } else if (kk == 0) {  // 16 d sc - dmin m of chunks g and 4 + g
                    const float d16 = 16.0f * h2f(f.x & 0xFFFFu), dmin = h2f(f.x >> 16);
                    cm[r][0] = fmaf(d16, (float)((sl >> (8 * g)) & 255u), -dmin * (float)((ml >> (8 * g)) & 255u));
                    cm[r][1] = fmaf(d16, (float)((sh >> (8 * g)) & 255u), -dmin * (float)((mh >> (8 * g)) & 255u));
                }
            }
        }
#pragma unroll
        for (int u = 0; u < S; u += WK) {
            const int j = j0 + u;  // this wave's chunk is j + kk
            v4f px[TT];
            float ps = 0.0f;
            // (one array for either kind cost the record's kernels up to 20 more waits in the compiler's schedule)
            uint4 ap[TT][3], ah[TT], al[TT];
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const int p = pA + (t * S + u) * R::AB;
                if constexpr (R::F32) {
#pragma unroll
                    for (int q = 0; q < 3; q++) ap[t][q] = lds<uint4>(xb, p + q * 1024);
                } else {
                    ah[t] = lds<uint4>(cur, p);
                    al[t] = lds<uint4>(cur, p + 1024);
                }
            }
            // F32: with them the chunk's codes and scales, so that the wave waits once (512 x 4096 x 11008
            // Q8_0 in the 256-row tile: 175 us with the reads where they are used, 166 so; the widest has no
            // registers for it)
            uint2 cv[RT];
            uint32_t sv[RT], zv[RT];
            constexpr bool EARLY = R::F32 && RT < 3;
            if constexpr (EARLY) {
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    const int e = r * S + u;
                    if constexpr (R::W8)
                        cv[r] = lds<uint2>(cur, pC + e * 512);
                    else
                        cv[r].x = lds<uint32_t>(cur, pC + e * 256);
                    if constexpr (F == kQ4_1)
                        sv[r] = lds<uint32_t>(cur, pS + e * 64);
                    else if constexpr (!R::KQ)
                        sv[r] = lds<uint16_t>(cur, pS + e * 32);
                    if constexpr (R::QM) zv[r] = lds<uint8_t>(cur, pZ + e * 16);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const int e = r * S + u;  // (row tile, chunk) entry
                // the 8 codes of row c16, inputs 8 g .. 8 g + 7: F32 with 8 bits a code in that order, else 0 2 4 6 1 3 5 7
                uint32_t ev = 0, od = 0;
                uint2 cw = {};
                if constexpr (R::W8) {
                    cw = EARLY ? cv[r] : lds<uint2>(cur, pC + e * 512);
                    ev = __builtin_amdgcn_perm(cw.y, cw.x, 0x06040200u);
                    od = __builtin_amdgcn_perm(cw.y, cw.x, 0x07050301u);
                } else {
                    const uint32_t c4 = EARLY ? cv[r].x : lds<uint32_t>(cur, pC + e * 256);
                    ev = c4 & 0x0F0F0F0Fu;
                    od = (c4 >> 4) & 0x0F0F0F0Fu;
                }
                if constexpr (F == kQ5_K) {
                    // bits 0, 2, 4, 6 of the group's byte to bit 4 of four bytes (the product's other terms miss those)
                    const uint32_t hb = lds<uint8_t>(cur, pH + e * 64);
                    ev |= __umul24(hb & 0x55u, 0x00410410u) & 0x10101010u;
                    od |= __umul24((hb >> 1) & 0x55u, 0x00410410u) & 0x10101010u;
                }
                if constexpr (F == kQ6_K) {
                    // two bits a code: bytes 0 and 1 of the group's halfword apart, then to bits 4, 5 of each code's byte
                    const uint32_t h = lds<uint16_t>(cur, pH + e * 128);
                    const uint32_t y = (h | (h << 8)) & 0x00FF00FFu;
                    ev |= ((y << 4) & 0x00300030u) | ((y << 8) & 0x30003000u);
                    od |= ((y << 2) & 0x00300030u) | ((y << 6) & 0x30003000u);
                }
                v8h b;         // the weights in fp16
                uint4 bw, be;  // F32: in bf16; Q6_K: and what bf16 leaves of sc q
                if constexpr (R::F32) {
                    float f[8];
                    if constexpr (F == kQ8_0) {
                        f[0] = sbyte<0>(cw.x), f[1] = sbyte<1>(cw.x), f[2] = sbyte<2>(cw.x), f[3] = sbyte<3>(cw.x);
                        f[4] = sbyte<0>(cw.y), f[5] = sbyte<1>(cw.y), f[6] = sbyte<2>(cw.y), f[7] = sbyte<3>(cw.y);
                    } else {
                        v2h q[4];  // 1024 + code
                        if constexpr (R::W8)
                            bytes_f16(cw.x, cw.y, q);
                        else
                            bytes_f16(ev, od, q);
                        if constexpr (F == kQ6_K) {
                            // sub-block 2 j + g / 2's int8 scale: (u - 32) sc, 13 bits
                            const float s1 = (float)lds<int8_t>(sbf, pF6 + r * 256 + 2 * j), n1 = s1 * -1056.0f;
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                f[2 * i] = fmaf((float)q[i][0], s1, n1);
                                f[2 * i + 1] = fmaf((float)q[i][1], s1, n1);
                            }
                        } else {
                            float z = F == kQ5_K ? -1040.0f : -1032.0f;
                            if constexpr (R::QM) z = -1024.0f - (float)(EARLY ? zv[r] : lds<uint8_t>(cur, pZ + e * 16));
#pragma unroll
                            for (int i = 0; i < 4; i++) halves_add(q[i], z, f[2 * i], f[2 * i + 1]);
                        }
                    }
                    uint32_t fb[8];
#pragma unroll
                    for (int i = 0; i < 8; i++) fb[i] = __float_as_uint(f[i]);
                    bw = make_uint4(high2(fb[0], fb[1]), high2(fb[2], fb[3]), high2(fb[4], fb[5]), high2(fb[6], fb[7]));
                    if constexpr (F == kQ6_K) {
#pragma unroll
                        for (int i = 0; i < 8; i++) fb[i] = __float_as_uint(f[i] - __uint_as_float(fb[i] & 0xFFFF0000u));
                        be = make_uint4(high2(fb[0], fb[1]), high2(fb[2], fb[3]), high2(fb[4], fb[5]), high2(fb[6], fb[7]));
                    }
                } else {
                    v2h q[4];
                    bytes_f16(ev, od, q);
                    if constexpr (F == kQ4_K) {
                        // (1024 + u) sc - 1024 sc = u sc exactly (below 2048)
                        const _Float16 s1 = sc[r][j >> 1][j & 1], n1 = s1 * (_Float16)-1024.0f;
                        const v2h sv = {s1, s1}, nv = {n1, n1};
#pragma unroll
                        for (int i = 0; i < 4; i++) q[i] = __builtin_elementwise_fma(q[i], sv, nv);
                    } else {
                        const v2h z = __builtin_bit_cast(v2h, (uint32_t)lds<uint8_t>(cur, pZ + e * 16) * 0x10001u + 0x64006400u);
#pragma unroll
                        for (int i = 0; i < 4; i++) q[i] = q[i] - z;
                    }
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        b[2 * i] = q[i][0];
                        b[2 * i + 1] = q[i][1];
                    }
                }
                float s = 0.0f;
                if constexpr (F == kQ4_1) {
                    const uint32_t m = EARLY ? sv[r] : lds<uint32_t>(cur, pS + e * 64);
                    s = h2f(m & 0xFFFFu);
                    const float c = fmaf(8.0f, s, h2f(m >> 16));  // lane group j % 4 keeps chunk j's
                    cm[r][j >> 2] = (j & 3) + kk == g ? c : cm[r][j >> 2];
                } else if constexpr (F == kQ5_K) {
                    s = (float)(((j < 4 ? sl5[r] : sh5[r]) >> (8 * (j & 3))) & 255u);
                } else if constexpr (!R::KQ) {
                    if (R::F32 ? !ONE || j + WK == 8 : (j + 1) % SEG == 0) s = h2f(EARLY ? sv[r] : lds<uint16_t>(cur, pS + e * 32));
                    if (SEG0 == 8 && j + WK == 8) rs[r] = s;
                }
                if constexpr (R::A16) {
                    // sum 256 hi w and sum lo w over the group's chunks (256 inputs at most), each exact
                    // (multiples of 256 below 2^32, whole numbers below 2^24), and their one rounded sum
                    // float(G); int4 in groups of 32: |G| < 2^24, one exact chain
                    constexpr bool one = F == kA4 && SEG == 1;
                    v4f xh[TT], xl[TT];
#pragma unroll
                    for (int t = 0; t < TT; t++)
                        xh[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, ah[t]), b,
                                                                       j % SEG == 0 ? zero : seg[t][r], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < TT; t++)
                        xl[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            __builtin_bit_cast(v8h, al[t]), b, one ? xh[t] : j % SEG == 0 ? zero : sel[t][r], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < TT; t++) {
                        if ((j + 1) % SEG == 0) {  // tile_i16's flush
#pragma unroll
                            for (int i = 0; i < 4; i++)
                                acc[t][r][i] = fmaf(one ? xl[t][i] : xh[t][i] + xl[t][i], s, acc[t][r][i]);
                            asm volatile("" : "+v"(acc[t][r]));  // (formed here, as in scale())
                        } else {
                            seg[t][r] = xh[t];
                            sel[t][r] = xl[t];
                        }
                    }
                    continue;
                }
                v4f x[TT];
#pragma unroll
                for (int t = 0; t < TT; t++)
                    x[t] = CHAIN && j > 0 ? d[t][r] : zero;
                if constexpr (R::F32) {
                    // Largest first: what a product is added to, the matrix cores round to nearest where it is
                    // the larger, but cut downwards where it is the smaller (smallest first left a mean error of
                    // -0.9e-7 of the results' size at 301 x 4096 x 1000; so -1e-9).
                    auto product = [&](int q, const uint4 &wb) __attribute__((always_inline)) {
#pragma unroll
                        for (int t = 0; t < TT; t++)
                            x[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8b, ap[t][q]),
                                                                           __builtin_bit_cast(v8b, wb), x[t], 0, 0, 0);
                    };
                    product(0, bw);
                    product(1, bw);
                    if constexpr (F == kQ6_K) product(0, be);
                    product(2, bw);
                    if constexpr (F == kQ6_K) {
                        product(1, be);
                        product(2, be);
                    }
                } else {
#pragma unroll
                    for (int t = 0; t < TT; t++)
                        x[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, ah[t]), b, x[t], 0, 0, 0);
#pragma unroll
                    for (int t = 0; t < TT; t++)
                        x[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, al[t]), b, x[t], 0, 0, 0);
                }
                if constexpr (CHAIN) {
#pragma unroll
                    for (int t = 0; t < TT; t++) d[t][r] = x[t];
                } else {
                    // the scale of the block before this one (its products are done by now), and no
                    // product ahead of it: more results in flight would not fit the registers
                    if (r > 0) scale(j, r - 1, px, ps);
#pragma unroll
                    for (int t = 0; t < TT; t++) px[t] = x[t];
                    ps = s;
                    __builtin_amdgcn_sched_barrier(0x104);  // (LDS reads and scalar work may cross)
                    if (r + 1 == RT) scale(j, r, px, ps);
                }
            }
        }
        if constexpr (j0 + S == 8 && !R::A16) {  // the superblock's minima, scale and 1 / s
            float dd[RT], dmin[RT];
            v8h bm[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) {
                if constexpr (F == kQ5_K) {
                    dd[r] = h2f(lds<uint16_t>(sbf, pF + r * 256));
                } else if constexpr (F == kQ4_K) {
                    const uint32_t f = lds<uint32_t>(sbf, pF + r * 256);
                    dd[r] = h2f(f & 0xFFFFu);
                    dmin[r] = -h2f(f >> 16);
                } else if constexpr (F == kQ6_K) {
                    rs[r] = h2f(lds<uint16_t>(sbf, pD + r * 32));
                }
                if constexpr (F == kQ4_K) {  // the minima in groups 0 and 1, against the sums' hi and lo planes
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        const v2h m2 = __builtin_bit_cast(v2h, g < 2 && kk == 0 ? mp[r][i] : 0u);
                        bm[r][2 * i] = m2[0];
                        bm[r][2 * i + 1] = m2[1];
                    }
                }
            }
#pragma unroll
            for (int t = 0; t < TT; t++) {
                v4f iv = zero;
                if constexpr (!R::F32) iv = lds<v4f>(sbf, pI + t * 64);
                uint4 sq = make_uint4(0u, 0u, 0u, 0u);
                float xs[2] = {0.0f, 0.0f};
                if constexpr (R::CENTER) {  // token c16's sums of chunks g and 4 + g
                    xs[0] = lds<float>(sums, pU + t * 512);
                    xs[1] = lds<float>(sums, pU + t * 512 + 16);
                } else if constexpr (R::SUMS) {
                    sq = lds<uint4>(sbf, pU + t * 512);
                    if (g >= 2) sq = make_uint4(0u, 0u, 0u, 0u);
                }
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    v4f dm = zero;
                    if constexpr (R::CENTER) {
                        dm = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[0], cm[r][0], zero, 0, 0, 0);
                        dm = __builtin_amdgcn_mfma_f32_16x16x4f32(xs[1], cm[r][1], dm, 0, 0, 0);
                    } else if constexpr (R::SUMS)
                        dm = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, sq), bm[r], zero, 0, 0, 0);
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        float v = d[t][r][i];
                        if constexpr (F == kQ4_K)
                            v = fmaf(dmin[r], dm[i], dd[r] * v);
                        else if constexpr (F == kQ5_K)
                            v = fmaf(dd[r], v, dm[i]);
                        else if constexpr (F == kQ4_1)
                            v += dm[i];
                        acc[t][r][i] = ONE ? fmaf(rs[r], v, acc[t][r][i])
                                           : R::F32 ? acc[t][r][i] + v : fmaf(iv[i], v, acc[t][r][i]);
                    }
                }
            }
        }
    };
    // One step: wait for its copies, start those of the next step into the
    // buffer that the step before has left, compute.
    auto step = [&](int sb, auto odd, auto j0c) __attribute__((always_inline)) {
        constexpr int j0 = decltype(j0c)::value, P = decltype(odd)::value;
        constexpr bool even = (P * SPB + j0 / S) % 2 == 0;
        __builtin_amdgcn_s_waitcnt(0x0070);  // vmcnt(0), lgkmcnt(0): this wave's copies are in, its reads done
        llmq_lds_barrier();
        const bool more = sb * 8 + j0 + S < a.NC;
        if (more) {
            stage(sb * 8 + j0 + S, even ? b1 : b0);
            if constexpr (j0 + S == 8) stage_sb(sb + 1, P ? f0 : f1);
        }
        if constexpr (R::F32) {
            if (more) split(even ? x1 : x0, (j0 + S == 8) != (P == 1) ? s1 : s0, (j0 + S) % 8);
            if (sb * 8 + j0 + 2 * S < a.NC) fetch(sb * 8 + j0 + 2 * S);
        }
        compute(j0c, even ? b0 : b1, even ? x0 : x1, P ? f1 : f0, P ? s1 : s0);
    };
    auto superblock = [&](int sb, auto odd) __attribute__((always_inline)) {
        step(sb, odd, LLMQ_N(0));
        if constexpr (S == 2) step(sb, odd, LLMQ_N(2));
        if constexpr (S <= 4) step(sb, odd, LLMQ_N(4));
        if constexpr (S == 2) step(sb, odd, LLMQ_N(6));
    };
    if constexpr (R::F32) fetch(0);
    stage(0, b0);
    stage_sb(0, f0);
    if constexpr (R::F32) {
        split(x0, s0, 0);
        if (S < a.NC) fetch(S);
    }
    for (int sb = 0; sb < a.NSB; sb += 2) {
        superblock(sb, LLMQ_N(0));
        if (sb + 1 < a.NSB) superblock(sb + 1, LLMQ_N(1));
    }
#undef LLMQ_N
    if constexpr (WK > 1) {  // the waves' sums over their chunks, in wave order
        static_assert((WK - 1) * WT * WR * TT * RT * 1024 <= (R::F32 ? L::A : L::STEP), "the sums fit a step's buffer");
        __syncthreads();
        v4f *const p = reinterpret_cast<v4f *>(R::F32 ? x0 : b0) + (w % (WT * WR)) * TT * RT * 64 + lane;
        constexpr int KS = WT * WR * TT * RT * 64;
        if (kk > 0) {
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int r = 0; r < RT; r++) p[(kk - 1) * KS + (t * RT + r) * 64] = acc[t][r];
        }
        __syncthreads();
        if (kk > 0) return;
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int q = 0; q < WK - 1; q++) acc[t][r] += p[q * KS + (t * RT + r) * 64];
    }
    if constexpr (R::F32) {
        // the inputs left out of the planes: their float32 products, a token's in turn (i of tile t)
#pragma unroll 1
        for (int e = 0; e < TT * 4; e++) {
            if (!__builtin_amdgcn_readfirstlane(left[wt * TT + e / 4])) continue;
            const int tok = (tt0 + wt * TT + e / 4) * 16 + 4 * g + e % 4;
            float v[RT] = {};
            if (tok < a.T) {
#pragma unroll 1
                for (int c = 0; c < a.NC; c++) {
                    const float *x = a.x + (int64_t)tok * a.ldx + c * 32;
                    int m = 0;
                    for (int k = 0; k < 32; k++) m = max(m, (int)(__float_as_uint(x[k]) & 0x7FFFFFFFu));
                    if (in_planes(m)) continue;
#pragma unroll 1
                    for (int k = 0; k < 32; k++)
#pragma unroll
                        for (int r = 0; r < RT; r++)
                            v[r] = fmaf(x[k], weight<F>(a, rtile(wr * RT + r), c16, c, k), v[r]);
                }
            }
#pragma unroll
            for (int t = 0; t < TT; t++)
#pragma unroll
                for (int i = 0; i < 4; i++)
#pragma unroll
                    for (int r = 0; r < RT; r++) acc[t][r][i] = 4 * t + i == e ? acc[t][r][i] + v[r] : acc[t][r][i];
        }
    }
    // store_out: bias, GELU, residual
#pragma unroll
    for (int r = 0; r < RT; r++) {
        const int o = (rt0 + wr * RT + r) * 16 + c16;
        const bool rok = o < a.n && rt0 + wr * RT + r < a.ntiles;
        const float bo = rok && (a.flags & LLMQ_BIAS) ? a.bias[o] : 0.0f;
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int tok = (tt0 + wt * TT + t) * 16 + 4 * g + i;
                if (!rok || tok >= a.T) continue;
                float v = acc[t][r][i];
                if constexpr (R::A16) v *= a.sx[tok];
                if (a.flags & LLMQ_BIAS) v += bo;
                if (a.flags & LLMQ_GELU) v = gelu_ref(v);
                float *dst = a.out + (int64_t)tok * a.ldo + o;
                if (a.flags & LLMQ_RESID) v += *dst;
                *dst = v;
            }
    }
}

// The tiles, as TT, RT, WT, WR, WK, S (gemm_planes.hip has what each costs).
template <int F, int SEG>
int launch_tile(hipStream_t st, int tile, const Args &a) {
    const int tt = (a.T + 15) / 16, rt = a.ntiles;
#define LLMQ_PK(TT, RT, WT, WR, WK, S)                                                                              \
    hipLaunchKernelGGL((gemm_planes_kernel<F, SEG, TT, RT, WT, WR, WK, S>),                                     \
                       dim3((unsigned)((rt + WR * RT - 1) / (WR * RT)), (unsigned)((tt + WT * TT - 1) / (WT * TT))), \
                       dim3(WT *WR * WK * 64), 0, st, a)
    if constexpr (Tr<F>::A16) {  // the segments' fma order is the reference's: no tiles that split the axis
        switch (tile) {
        case 1: LLMQ_PK(2, 4, 2, 2, 1, 2); break;
        case 2: LLMQ_PK(2, 2, 2, 2, 1, 2); break;
        case 3: LLMQ_PK(2, 1, 1, 4, 1, 4); break;
        default: LLMQ_PK(1, 1, 1, 4, 1, 4); break;
        }
        LLMQ_HIP(hipGetLastError());
        return LLMQ_OK;
    } else if constexpr (Tr<F>::F32) {
        switch (tile) {
        case 0:  // (only where 128 registers hold it)
            if constexpr (Tr<F>::KQ || Tr<F>::CENTER || SEG == 8)
                LLMQ_PK(2, 2, 1, 8, 1, 2);
            else
                LLMQ_PK(2, 3, 1, 8, 1, 2);
            break;
        case 1: LLMQ_PK(2, 2, 1, 8, 1, 2); break;
        case 2: LLMQ_PK(2, 1, 1, 8, 2, 4); break;
        case 3: LLMQ_PK(1, 2, 1, 4, 4, 8); break;
        case 4: LLMQ_PK(1, 1, 1, 4, 4, 8); break;
        default: LLMQ_PK(1, 1, 1, 2, 4, 8); break;
        }
    } else {
        switch (tile) {
        case 0: LLMQ_PK(4, 4, 1, 4, 1, 2); break;
        case 1: LLMQ_PK(2, 4, 2, 2, 1, 2); break;
        case 2: LLMQ_PK(2, 2, 2, 2, 1, 2); break;
        case 3: LLMQ_PK(2, 1, 1, 4, 1, 4); break;
        case 4: LLMQ_PK(1, 1, 1, 4, 1, 4); break;
        case 5: LLMQ_PK(1, 1, 1, 4, 4, 8); break;
        default: LLMQ_PK(1, 1, 1, 2, 4, 8); break;
        }
    }
#undef LLMQ_PK
    LLMQ_HIP(hipGetLastError());
    return LLMQ_OK;
}

}  // namespace planes
