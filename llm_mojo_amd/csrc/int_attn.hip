// IntAttnKV (int_attention.mojo:62-269): an int8 key / value cache with
// per-(position, head) scales held as integers (scale * 2^24), and attention
// computed in integers with intmath.masked_exp (intmath.mojo:48-123).
//
// Layout in HBM: the int8 cache's [layer, pos, head, head_dim] codes and
// [layer, pos, head] int32 scales (the reference's VNNI blocking is a CPU
// layout for VPDPWSSD; the arithmetic does not depend on it).
//
// Every step is integer arithmetic except the final float multiply, which
// follows the reference: per 256-position segment the exact int32 value sums
// become float and add in segment order, then out = sums * f32(vmax 2^15 /
// (2^24 total)).  The integer sums are exact in any order, so the kernels
// reproduce the reference's results bit for bit.
#include "common.h"

namespace {

constexpr int kKS = 24;  // fraction bits of the key / value scales (int_attention.mojo:54)
constexpr int kSF = 16;  // fraction bits of the fixed-point scores (:55)
constexpr int kFB = 16;  // fraction bits of the base-2 exponent (intmath.mojo:31)
constexpr int kMB = 24;  // extra fraction bits of the multiplier (:32)
constexpr int kThreads = 256;
constexpr int kRun = 64;           // prompt kernel: positions a wave takes at a time,
constexpr int kPromptWaves = 8;    // waves a workgroup (16 tokens of a head)

// A native vector (not HIP's int4 struct, whose copies kept the value rows
// in scratch memory).
typedef int v4i __attribute__((ext_vector_type(4)));

// maxima over the wave (order-free), without LDS
__device__ __forceinline__ float wave_max_f(float v) { return llmq_wave_max_all(v); }
__device__ __forceinline__ int wave_max_i(int v) { return llmq_wave_max_all(v); }
__device__ __forceinline__ int64_t wave_sum_l(int64_t v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

__device__ __forceinline__ void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// exp2_neg (intmath.mojo:53-65): 2^(-d scale log2 e) in Q30 for d >= 0, the
// integer part of the exponent as a shift and the fraction by a degree-3
// polynomial; exponents >= 31 give 0.  The reference's 64-bit steps on 32-bit
// multiplies' high halves: with the scores' multiplier (kMult) every d from
// 1408218 on gives 0 (so the cap at 2^31 is never reached), and below 2^21
// (d mult) >> 24 = (2^8 d mult) >> 32 and (p r) >> 16 = (2 p 2^15 r) >> 32,
// with 2 p and 2^15 r within 31 bits and a sign (checked for every d).
constexpr uint32_t kMult = 24204406;  // exp_multiplier(1 / 2^16) (intmath.mojo:48-50, int_attention.mojo:174)
__device__ __forceinline__ uint32_t exp2_neg(uint32_t d) {
    constexpr int C0 = 1073741824, C1 = -742598100, C2 = 248207216, C3 = -42480028;  // :40-43
    const uint32_t y = __umulhi(d << (32 - kMB), kMult);
    const uint32_t q = y >> kFB;
    const int r = (int)((y & ((1u << kFB) - 1)) << 15);
    int p = __mulhi(2 * C3, r) + C2;
    p = __mulhi(2 * p, r) + C1;
    p = __mulhi(2 * p, r) + C0;
    return d >= (1u << 21) || q >= 31 ? 0u : (uint32_t)p >> q;
}

// IntAttnKV.quantize_head (int_attention.mojo:140-168) with one wave:
// s = max|x| / 127 (1 if zero), codes round(x * (1 / s)); returns s * 2^24
// rounded, as int32.  Codes go to dst (global) and, when given, lds_copy.
template <int HD>
__device__ __forceinline__ int32_t quantize_head(const float *__restrict__ src, int8_t *__restrict__ dst,
                                                 int8_t *lds_copy, int lane) {
    float xs[HD / 64];
    float m = 0.0f;
#pragma unroll
    for (int e = 0; e < HD / 64; e++) {
        xs[e] = src[lane + 64 * e];
        m = fmaxf(m, fabsf(xs[e]));
    }
    m = wave_max_f(m);
    float s = m / 127.0f;
    if (s == 0.0f) s = 1.0f;
    const float inv = 1.0f / s;
#pragma unroll
    for (int e = 0; e < HD / 64; e++) {
        const int8_t c = (int8_t)llmq_to_int(roundf(xs[e] * inv));
        dst[lane + 64 * e] = c;
        if (lds_copy) lds_copy[lane + 64 * e] = c;
    }
    return (int32_t)(int64_t)round((double)s * (double)(1 << kKS));
}

// IntAttnKV.store (int_attention.mojo:132-138) for token t = blockIdx.y at
// position pos0 + t, head h = blockIdx.x; keys and values are columns C..
// and 2C.. of qkv row t.
template <int HD>
__global__ __launch_bounds__(64) void ikv_store_kernel(const float *__restrict__ qkv, int64_t ld, int C, int pos0,
                                                       const int *__restrict__ pos_dev, int layer, int max_t,
                                                       int n_head, int8_t *__restrict__ K8, int8_t *__restrict__ V8,
                                                       int32_t *__restrict__ KQ, int32_t *__restrict__ VQ) {
    const int h = blockIdx.x, t = blockIdx.y, lane = threadIdx.x;
    const int pos = (pos_dev ? *pos_dev : pos0) + t;
    const int64_t sl = ((int64_t)layer * max_t + pos) * n_head + h;
    const float *row = qkv + (int64_t)t * ld + (int64_t)h * HD;
    const int32_t kq = quantize_head<HD>(row + C, K8 + sl * HD, nullptr, lane);
    const int32_t vq = quantize_head<HD>(row + 2 * C, V8 + sl * HD, nullptr, lane);
    if (lane == 0) {
        KQ[sl] = kq;
        VQ[sl] = vq;
    }
}

// IntAttnKV.attend_one (int_attention.mojo:170-269) for token t = blockIdx.y
// (position pos0 + t, or state[0] + t on the device-driven decode path) and
// head h = blockIdx.x, 256 threads:
//   1. query -> int16 (wave 0) and the score multiplier qm = sq / sqrt(HD) 2^40;
//   2-3. thread i scores positions i, i + 256, ...: the int32 dot product of
//      the int16 query with the int8 key, rescaled to 16 fraction bits
//      ((dot kq + 2^23) >> 24, then (. qm + 2^23) >> 24);
//   4. masked_exp over the scores (maximum, exp2_neg, int64 total);
//   5. int16 weights w = min((e r16 + 2^30) >> 31, 32767) with r16 the value
//      scale relative to the largest, Q16; per 256-position segment the
//      int32 sums of w v (exact) become float and add in segment order;
//   6. out = sums * f32(vmax 2^15 / (2^24 total)).
// STAGE copies each position's value row into LDS while scoring, so the
// value pass reads no global memory.  STORE (one token: decode) quantizes the
// head's new key and value first (IntAttnKV.store) and uses them from LDS.
template <int HD, bool STAGE, bool STORE>
__global__ __launch_bounds__(kThreads) void ikv_attend_kernel(const float *__restrict__ qkv, int64_t ld, int C,
                                                              int pos0, const int *__restrict__ pos_dev, int layer,
                                                              int max_t, int n_head, int8_t *__restrict__ K8,
                                                              int8_t *__restrict__ V8, int32_t *__restrict__ KQ,
                                                              int32_t *__restrict__ VQ, float *__restrict__ out,
                                                              int64_t ldo, double sqrt_hd) {
    constexpr int NV = HD / 16;         // 16-byte pieces of a row
    constexpr int DG = HD / 4;          // value pass: dimension groups of 4
    constexpr int SLICES = kThreads / DG;  // and position slices
    extern __shared__ __align__(16) int32_t ism[];
    int32_t *scores = ism;             // [max_t]
    int32_t *vqs = scores + max_t;     // [max_t] value scales
    int16_t *w = reinterpret_cast<int16_t *>(vqs + max_t);  // [max_t] weights
    int8_t *vrow = reinterpret_cast<int8_t *>(w + ((max_t + 7) & ~7));  // [max_t][HD] (STAGE)
    __shared__ __align__(16) int16_t qi[HD];
    __shared__ __align__(16) int8_t knew[HD], vnew[HD];
    __shared__ __align__(16) int32_t part[SLICES * HD];
    __shared__ int64_t qm_s, red64[4];
    __shared__ int32_t red_m[4], red_v[4], kq_new;
    const int h = blockIdx.x, t = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int npos = (pos_dev ? *pos_dev : pos0) + t + 1;
    const int cur = npos - 1;
    const int64_t base = (int64_t)layer * max_t * n_head + h;  // slot of position 0
    const float *qrow = qkv + (int64_t)t * ld + (int64_t)h * HD;

    // This thread's first rows, requested before anything else (positions
    // past the end re-read the last one and are not used).
    v4i kr[NV], vr[NV];
    int32_t kqr, vqr;
    auto load_row = [&](int s) {
        const int64_t sl = base + (int64_t)s * n_head;
        const v4i *kp = reinterpret_cast<const v4i *>(K8 + sl * HD);
        const v4i *vp = reinterpret_cast<const v4i *>(V8 + sl * HD);
#pragma unroll
        for (int i = 0; i < NV; i++) {
            kr[i] = kp[i];
            if (STAGE) vr[i] = vp[i];
        }
        kqr = KQ[sl];
        vqr = VQ[sl];
    };
    load_row(tid < npos ? tid : cur);
    __builtin_amdgcn_sched_barrier(0);

    if (wid == 0) {
        // 1. Query -> int16, symmetric (int_attention.mojo:183-197).
        float qv[HD / 64];
        float m = 0.0f;
#pragma unroll
        for (int e = 0; e < HD / 64; e++) {
            qv[e] = qrow[lane + 64 * e];
            m = fmaxf(m, fabsf(qv[e]));
        }
        m = wave_max_f(m);
        float sq = m / 32767.0f;
        if (sq == 0.0f) sq = 1.0f;
        const float invq = 1.0f / sq;
#pragma unroll
        for (int e = 0; e < HD / 64; e++) qi[lane + 64 * e] = (int16_t)llmq_to_int(roundf(qv[e] * invq));
        if (lane == 0) qm_s = (int64_t)round((double)sq / sqrt_hd * (double)((int64_t)1 << (kSF + kKS)));
    } else if (STORE && (wid == 1 || wid == 2)) {
        // IntAttnKV.store for this head's new key (wave 1) and value (wave 2).
        const int kv = wid - 1;
        const int64_t sl = base + (int64_t)cur * n_head;
        // LDS copies: the workgroup reads the new rows from there, not back
        // from global memory.
        int8_t *copy = kv == 0 ? knew : (STAGE ? vrow + (int64_t)cur * HD : vnew);
        const int32_t q = quantize_head<HD>(qrow + (int64_t)(1 + kv) * C, (kv ? V8 : K8) + sl * HD, copy, lane);
        if (lane == 0) {
            (kv ? VQ : KQ)[sl] = q;
            if (kv == 0)
                kq_new = q;
            else
                vqs[cur] = q;
        }
    }
    lds_barrier();

    // 2-3. Scores in 16 fraction bits; the maxima of the scores and scales.
    uint32_t qpair[HD / 2];  // the int16 query, two dimensions a word
#pragma unroll
    for (int i = 0; i < HD / 8; i++) {
        const int4 q4 = reinterpret_cast<const int4 *>(qi)[i];
        qpair[4 * i] = (uint32_t)q4.x;
        qpair[4 * i + 1] = (uint32_t)q4.y;
        qpair[4 * i + 2] = (uint32_t)q4.z;
        qpair[4 * i + 3] = (uint32_t)q4.w;
    }
    const int64_t qm = qm_s;
    int smax = INT32_MIN, vmax = 0;
    for (int s = tid; s < npos; s += kThreads) {
        if (s != tid) load_row(s);  // only past 256 positions
        const bool fresh = STORE && s == cur;
        if (fresh) {
#pragma unroll
            for (int i = 0; i < NV; i++) kr[i] = reinterpret_cast<const v4i *>(knew)[i];
            kqr = kq_new;
            vqr = vqs[cur];
        }
        // int32 dot product (at most HD 32767 127: no overflow for HD <= 512)
        int32_t acc = 0;
#pragma unroll
        for (int i = 0; i < NV; i++) {
            const uint32_t kw[4] = {(uint32_t)kr[i].x, (uint32_t)kr[i].y, (uint32_t)kr[i].z, (uint32_t)kr[i].w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t q01 = qpair[8 * i + 2 * j], q23 = qpair[8 * i + 2 * j + 1];
                acc += (int32_t)(int16_t)q01 * (int32_t)(int8_t)kw[j];
                acc += (int32_t)(int16_t)(q01 >> 16) * (int32_t)(int8_t)(kw[j] >> 8);
                acc += (int32_t)(int16_t)q23 * (int32_t)(int8_t)(kw[j] >> 16);
                acc += (int32_t)(int16_t)(q23 >> 16) * (int32_t)(int8_t)(kw[j] >> 24);
            }
        }
        const int64_t t1 = ((int64_t)acc * kqr + ((int64_t)1 << (kKS - 1))) >> kKS;
        const int32_t sc = (int32_t)((t1 * qm + ((int64_t)1 << (kKS - 1))) >> kKS);
        scores[s] = sc;
        smax = max(smax, sc);
        vmax = max(vmax, vqr);
        if (!fresh) {
            vqs[s] = vqr;
            if (STAGE) {
#pragma unroll
                for (int i = 0; i < NV; i++) *reinterpret_cast<v4i *>(vrow + (int64_t)s * HD + 16 * i) = vr[i];
            }
        }
    }
    smax = wave_max_i(smax);
    vmax = wave_max_i(vmax);
    if (lane == 0) {
        red_m[wid] = smax;
        red_v[wid] = vmax;
    }
    lds_barrier();
    const int64_t m = max(max(red_m[0], red_m[1]), max(red_m[2], red_m[3]));
    vmax = max(max(red_v[0], red_v[1]), max(red_v[2], red_v[3]));

    // 4-5. e = exp2_neg(m - score) in Q30, the total, the int16 weights.
    const int64_t inv47 = vmax > 0 ? ((int64_t)1 << 47) / vmax : 0;
    int64_t tot = 0;
    for (int s = tid; s < npos; s += kThreads) {
        const int64_t e = exp2_neg((uint32_t)(m - scores[s]));
        tot += e;
        const int64_t r16 = ((int64_t)vqs[s] * inv47) >> 31;
        const int64_t ww = min((e * r16 + ((int64_t)1 << 30)) >> 31, (int64_t)32767);
        w[s] = e == 0 ? 0 : (int16_t)ww;
    }
    tot = wave_sum_l(tot);
    if (lane == 0) red64[wid] = tot;
    lds_barrier();
    const int64_t total = red64[0] + red64[1] + red64[2] + red64[3];
    float *o = out + (int64_t)t * ldo + (int64_t)h * HD;
    if (vmax == 0 || total == 0) {
        for (int i = tid; i < HD; i += kThreads) o[i] = 0.0f;
        return;
    }

    // Weighted value sums: thread (dg, slice) takes dimensions 4dg..4dg+3 of
    // positions slice, slice + SLICES, ... of each 256-position segment.
    const int dg = tid % DG, slice = tid / DG;
    float accf = 0.0f;  // dimension tid (tid < HD)
    for (int seg = 0; seg < npos; seg += 256) {
        const int end = min(seg + 256, npos);
        int32_t a0 = 0, a1 = 0, a2 = 0, a3 = 0;
        for (int s = seg + slice; s < end; s += SLICES) {
            const int32_t ws = w[s];
            uint32_t vw;
            if (STAGE)
                vw = *reinterpret_cast<const uint32_t *>(vrow + (int64_t)s * HD + 4 * dg);
            else if (STORE && s == cur)
                vw = *reinterpret_cast<const uint32_t *>(vnew + 4 * dg);
            else
                vw = *reinterpret_cast<const uint32_t *>(V8 + (base + (int64_t)s * n_head) * HD + 4 * dg);
            a0 += ws * (int32_t)(int8_t)(vw);
            a1 += ws * (int32_t)(int8_t)(vw >> 8);
            a2 += ws * (int32_t)(int8_t)(vw >> 16);
            a3 += ws * (int32_t)(int8_t)(vw >> 24);
        }
        *reinterpret_cast<int4 *>(part + slice * HD + 4 * dg) = make_int4(a0, a1, a2, a3);
        lds_barrier();
        if (tid < HD) {
            int32_t v = 0;
#pragma unroll
            for (int p = 0; p < SLICES; p++) v += part[p * HD + tid];
            accf += (float)v;
        }
        lds_barrier();
    }
    // 6. Back to float: * (vmax / 2^24) * 2^15 / total.
    const float fs = (float)((double)vmax * (double)(1 << 15) / ((double)(1 << kKS) * (double)total));
    if (tid < HD) o[tid] = accf * fs;
}

// Attention of 16 tokens of one head (workgroup (head, tile), 8 waves) on the
// int8 matrix cores: the same integers as ikv_attend_kernel, hence the same
// bits.  A wave takes runs of 64 positions (run, run + 8, ...; RPW of them at
// most), whose scores stay in its registers between the passes.
//   scores: mfma(keys, query bytes).  The int16 query is 256 qh + (ql + 128)
//     with both bytes signed; the 128 sum(k) comes from a product with ones.
//     A lane ends with positions 16 b + 4 g + r (b, r = 0..3) of one token.
//   values: mfma(values transposed, weight bytes), split the same way.  The
//     reduction's order is free, so a lane's own 16 weights are its operand
//     as they lie; the other operand is 16 dwords of value rows (4 dimensions
//     of positions 16 b + 4 g + r), 4 x 4 bytes transposed by v_perm, whose
//     row i of tile c is dimension 4 i + c.  No exchange through LDS but the
//     tokens' maxima and totals and the segments' sums (LDS atomics on whole
//     numbers: any order gives the same sum).
// What bounds it: the ~60 32- and 64-bit integer instructions a score (rescale,
// exp2_neg, weight), which a workgroup per token and head spent beside ~250
// for its two scalar dot products and its own reads of every cached row.
// 476 tokens of 12 heads of 64: 65.4 -> 16.9 us with the store (4.9 of it).
template <int HD, int RPW>
__global__ __launch_bounds__(64 * kPromptWaves) void ikv_prompt_kernel(
    const float *__restrict__ qkv, int64_t ld, int pos0, int T, int layer, int max_t, int n_head,
    const int8_t *__restrict__ K8, const int8_t *__restrict__ V8, const int32_t *__restrict__ KQ,
    const int32_t *__restrict__ VQ, float *__restrict__ out, int64_t ldo, double sqrt_hd) {
    constexpr int NT = 64 * kPromptWaves;
    constexpr int KS = HD / 64;    // reduction steps of a score, halves of a value row
    constexpr int PS = HD + 1;     // padded row of the segments' sums: tokens on different banks
    extern __shared__ __align__(16) int32_t ism[];
    __shared__ __align__(16) int8_t qh[16 * HD], ql[16 * HD];
    __shared__ int64_t qm_s[16];
    __shared__ unsigned long long tot_s[16];
    __shared__ int32_t max_s[16], vmax_s[16];
    const int h = blockIdx.x, t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * 16;  // longest contexts first
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int tn = lane & 15, g = lane >> 4;
    const int last = pos0 + min(t0 + 15, T - 1);  // the tile's last position
    const int runs = last / kRun + 1, segs = last / 256 + 1;
    const int64_t base = (int64_t)layer * max_t * n_head + h;
    int32_t *kqs = ism, *vqs = kqs + runs * kRun, *part = vqs + runs * kRun;  // part[segs][16][PS]

    // The first run's rows (positions past the tile's last re-read it; their
    // scores are masked and their weights 0).
    v4i kr[4][KS];
    uint32_t vr[16 * KS];
    auto load_keys = [&](int p0) {
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int i = 0; i < KS; i++)
                kr[b][i] = *reinterpret_cast<const v4i *>(
                    K8 + (base + (int64_t)min(p0 + 16 * b + tn, last) * n_head) * HD + 64 * i + 16 * g);
    };
    auto load_values = [&](int p0) {
#pragma unroll
        for (int j = 0; j < 16; j++) {
            const int8_t *v = V8 + (base + (int64_t)min(p0 + 16 * (j >> 2) + 4 * g + (j & 3), last) * n_head) * HD;
#pragma unroll
            for (int i = 0; i < KS; i++) vr[16 * i + j] = *reinterpret_cast<const uint32_t *>(v + 64 * i + 4 * tn);
        }
    };
    if (wid < runs) {
        load_keys(wid * kRun);
        load_values(wid * kRun);
    }
    for (int p = tid; p < runs * kRun; p += NT) {
        const int64_t sl = base + (int64_t)min(p, last) * n_head;
        kqs[p] = KQ[sl];
        vqs[p] = VQ[sl];
    }
    for (int i = tid; i < segs * 16 * PS; i += NT) part[i] = 0;
    if (tid < 16) {
        tot_s[tid] = 0;
        max_s[tid] = INT32_MIN;
        vmax_s[tid] = 0;
    }
    // Queries -> int16 (int_attention.mojo:183-197), two tokens a wave.
#pragma unroll
    for (int u = 0; u < 16 / kPromptWaves; u++) {
        const int tk = wid * (16 / kPromptWaves) + u;
        const float *qrow = qkv + (int64_t)min(t0 + tk, T - 1) * ld + (int64_t)h * HD;
        float qv[KS];
        float m = 0.0f;
#pragma unroll
        for (int e = 0; e < KS; e++) {
            qv[e] = qrow[lane + 64 * e];
            m = fmaxf(m, fabsf(qv[e]));
        }
        m = wave_max_f(m);
        float sq = m / 32767.0f;
        if (sq == 0.0f) sq = 1.0f;
        const float invq = 1.0f / sq;
#pragma unroll
        for (int e = 0; e < KS; e++) {
            const int c = (int16_t)llmq_to_int(roundf(qv[e] * invq));
            qh[tk * HD + lane + 64 * e] = (int8_t)(c >> 8);
            ql[tk * HD + lane + 64 * e] = (int8_t)((c & 255) - 128);
        }
        if (lane == 0) qm_s[tk] = (int64_t)round((double)sq / sqrt_hd * (double)((int64_t)1 << (kSF + kKS)));
    }
    __syncthreads();

    // Scores in 16 fraction bits; the maxima of the scores and value scales.
    const int cur = min(pos0 + t0 + tn, last);  // this lane's token's position
    const int64_t qm = qm_s[tn];
    const v4i ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
    int32_t sc[RPW][16];
    int smax = INT32_MIN, vmax = 0;
#pragma unroll
    for (int rr = 0; rr < RPW; rr++) {
        const int p0 = (wid + rr * kPromptWaves) * kRun;
        if (p0 > last) break;
        if (rr) load_keys(p0);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            v4i dh = {0, 0, 0, 0}, dl = {0, 0, 0, 0}, ks = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < KS; i++) {
                const v4i qhv = *reinterpret_cast<const v4i *>(qh + tn * HD + 64 * i + 16 * g);
                const v4i qlv = *reinterpret_cast<const v4i *>(ql + tn * HD + 64 * i + 16 * g);
                dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(kr[b][i], qhv, dh, 0, 0, 0);
                dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(kr[b][i], qlv, dl, 0, 0, 0);
                ks = __builtin_amdgcn_mfma_i32_16x16x64_i8(kr[b][i], ones, ks, 0, 0, 0);
            }
            const int p = p0 + 16 * b + 4 * g;
            const v4i kq = *reinterpret_cast<const v4i *>(kqs + p);
            const v4i vq = *reinterpret_cast<const v4i *>(vqs + p);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int32_t acc = (int32_t)(((uint32_t)dh[r] << 8) + (uint32_t)dl[r] + ((uint32_t)ks[r] << 7));
                const int64_t t1 = ((int64_t)acc * kq[r] + ((int64_t)1 << (kKS - 1))) >> kKS;
                const int32_t s = (int32_t)((t1 * qm + ((int64_t)1 << (kKS - 1))) >> kKS);
                sc[rr][4 * b + r] = s;
                if (p + r <= cur) {
                    smax = max(smax, s);
                    vmax = max(vmax, vq[r]);
                }
            }
        }
    }
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) {
        smax = max(smax, __shfl_xor(smax, o));
        vmax = max(vmax, __shfl_xor(vmax, o));
    }
    if (g == 0) {
        atomicMax(&max_s[tn], smax);
        atomicMax(&vmax_s[tn], vmax);
    }
    __syncthreads();

    // e in Q30, the totals, the int16 weights and the value sums.
    const uint32_t m = (uint32_t)max_s[tn];
    vmax = vmax_s[tn];
    const int64_t inv47 = vmax > 0 ? ((int64_t)1 << 47) / vmax : 0;
    uint64_t tot = 0;
#pragma unroll
    for (int rr = 0; rr < RPW; rr++) {
        const int p0 = (wid + rr * kPromptWaves) * kRun;
        if (p0 > last) break;
        if (rr) load_values(p0);
        v4i wh, wl;
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int p = p0 + 16 * b + 4 * g;
            const v4i vq = *reinterpret_cast<const v4i *>(vqs + p);
            uint32_t hw = 0, lw = 0;
            // A scale that overflowed int32 (a head's values past 16256) is
            // negative: then the 64-bit form; else r16 <= 2^16 and 32 x 32 bits do.
            const bool wide = __any((vq[0] | vq[1] | vq[2] | vq[3]) < 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const uint32_t e = p + r <= cur ? exp2_neg(m - (uint32_t)sc[rr][4 * b + r]) : 0u;
                tot += e;
                int w;
                if (wide) {
                    const int64_t r16 = ((int64_t)vq[r] * inv47) >> 31;
                    const int64_t ww = ((int64_t)e * r16 + ((int64_t)1 << 30)) >> 31;
                    w = (int16_t)(ww < 32767 ? ww : 32767);
                } else {
                    const uint64_t lo = (uint64_t)(uint32_t)vq[r] * (uint32_t)inv47;
                    const uint32_t hi = (uint32_t)vq[r] * (uint32_t)(inv47 >> 32) + (uint32_t)(lo >> 32);
                    const uint32_t r16 = (hi << 1) | ((uint32_t)lo >> 31);
                    const uint64_t ww = (uint64_t)e * r16 + (1u << 30);
                    w = min((int)(ww >> 31), 32767);
                }
                if (e == 0) w = 0;
                hw |= (uint32_t)((w >> 8) & 255) << (8 * r);
                lw |= (uint32_t)(w & 255) << (8 * r);
            }
            wh[b] = (int)hw;
            wl[b] = (int)(lw ^ 0x80808080u);  // less 128
        }
        int32_t *pp = part + ((p0 >> 8) * 16 + tn) * PS;
#pragma unroll
        for (int i = 0; i < KS; i++) {
            v4i vt[4];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const uint32_t *x = vr + 16 * i + 4 * b;
                const uint32_t a0 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u);
                const uint32_t a1 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u);
                const uint32_t a2 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u);
                const uint32_t a3 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
                vt[0][b] = (int)__builtin_amdgcn_perm(a1, a0, 0x05040100u);
                vt[1][b] = (int)__builtin_amdgcn_perm(a1, a0, 0x07060302u);
                vt[2][b] = (int)__builtin_amdgcn_perm(a3, a2, 0x05040100u);
                vt[3][b] = (int)__builtin_amdgcn_perm(a3, a2, 0x07060302u);
            }
#pragma unroll
            for (int c = 0; c < 4; c++) {
                const v4i z = {0, 0, 0, 0};
                const v4i dh = __builtin_amdgcn_mfma_i32_16x16x64_i8(vt[c], wh, z, 0, 0, 0);
                const v4i dl = __builtin_amdgcn_mfma_i32_16x16x64_i8(vt[c], wl, z, 0, 0, 0);
                const v4i vs = __builtin_amdgcn_mfma_i32_16x16x64_i8(vt[c], ones, z, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++)
                    atomicAdd(pp + 64 * i + 4 * (4 * g + r) + c,
                              (int32_t)(((uint32_t)dh[r] << 8) + (uint32_t)dl[r] + ((uint32_t)vs[r] << 7)));
            }
        }
    }
    tot += __shfl_xor(tot, 16);
    tot += __shfl_xor(tot, 32);
    if (g == 0 && wid < runs) atomicAdd(&tot_s[tn], (unsigned long long)tot);
    __syncthreads();

    // The segments' sums become float and add in segment order; the scale.
    const int tk = tid / (NT / 16), d0 = tid % (NT / 16);
    if (t0 + tk >= T) return;
    const int64_t total = (int64_t)tot_s[tk];
    const int tv = vmax_s[tk], tsegs = (pos0 + t0 + tk) / 256 + 1;
    const float fs = (float)((double)tv * (double)(1 << 15) / ((double)(1 << kKS) * (double)total));
    float *o = out + (int64_t)(t0 + tk) * ldo + (int64_t)h * HD;
    for (int d = d0; d < HD; d += NT / 16) {
        float a = 0.0f;
        for (int sg = 0; sg < tsegs; sg++) a += (float)part[(sg * 16 + tk) * PS + d];
        o[d] = tv == 0 || total == 0 ? 0.0f : a * fs;
    }
}

template <int HD, int RPW>
int prompt_launch(llmq_ctx *ctx, const llmq_kv *kv, float *out, const float *qkv, int layer, int T, int pos0,
                  int64_t ld) {
    const int C = kv->n_head * kv->head_dim, n = pos0 + T;
    // at most 49 KB for HD 64 and 81 KB for HD 128, at 2048 positions: 16 of scales, 33 or 65 of sums
    const size_t lds = ((size_t)(n + kRun - 1) / kRun * kRun * 2 + (size_t)(n + 255) / 256 * 16 * (HD + 1)) * 4;
    static size_t granted = 64 * 1024;
    if (lds > granted) {
        LLMQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ikv_prompt_kernel<HD, RPW>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        granted = lds;
    }
    hipLaunchKernelGGL((ikv_prompt_kernel<HD, RPW>), dim3(kv->n_head, (T + 15) / 16), dim3(64 * kPromptWaves), lds,
                       ctx->stream, qkv, ld ? ld : 3 * C, pos0, T, layer, kv->max_t, kv->n_head, kv->k, kv->v, kv->kq,
                       kv->vq, out, (int64_t)C, sqrt((double)HD));
    LLMQ_HIP(hipGetLastError());
    return LLMQ_OK;
}

template <int HD, bool STAGE, bool STORE>
int attend_launch(llmq_ctx *ctx, const llmq_kv *kv, float *out, const float *qkv, int layer, int T, int pos0,
                  const int *pos_dev, int64_t ld, size_t lds) {
    static size_t granted = 64 * 1024;
    if (lds > granted) {
        LLMQ_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(&ikv_attend_kernel<HD, STAGE, STORE>),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        granted = lds;
    }
    const int C = kv->n_head * kv->head_dim;
    hipLaunchKernelGGL((ikv_attend_kernel<HD, STAGE, STORE>), dim3(kv->n_head, T), dim3(kThreads), lds, ctx->stream,
                       qkv, ld ? ld : 3 * C, C, pos0, pos_dev, layer, kv->max_t, kv->n_head, kv->k, kv->v, kv->kq,
                       kv->vq, out, (int64_t)C, sqrt((double)HD));
    LLMQ_HIP(hipGetLastError());
    return LLMQ_OK;
}

template <int HD>
int attend_hd(llmq_ctx *ctx, const llmq_kv *kv, float *out, const float *qkv, int layer, int T, int pos0,
              const int *pos_dev, int64_t ld, bool store) {
    const size_t base = (size_t)kv->max_t * 8 + (size_t)((kv->max_t + 7) & ~7) * 2;
    const size_t staged = base + (size_t)kv->max_t * HD;
    // The prompt kernel from where a workgroup per token and head no longer
    // runs in one round: its LDS lets one or two share a CU (more of the
    // unstaged ones, 5 KB each, do not run faster), 256 CUs.  12 heads of 64,
    // max_t 1024, 40 tokens (480 workgroups) after 100 and 850: 5.7 and 15.3
    // us against 7.3 and 15.0 here; 44 (528): 8.0 and 23.2 against 7.3 and
    // 15.0; 140: 16.7 and 48.4 against 7.5 and 15.2.  8 heads of 128, max_t
    // 1024 (one a CU), after 100: 32 tokens 6.5 against 8.6, 40 11.2 against
    // 8.7.  Positions the host does not know, one token's fused store and
    // contexts past a wave's four runs stay on the other.
    const size_t lds = (staged <= 150 * 1024 ? staged : base) + 5 * 1024;
    const int64_t round = 256 * (2 * lds <= 160 * 1024 ? 2 : 1);
    if (T > 1 && !pos_dev && !store && (int64_t)T * kv->n_head > round && pos0 + T <= 4 * kRun * kPromptWaves) {
        const int runs = (pos0 + T + kRun - 1) / kRun;
        if (runs <= kPromptWaves) return prompt_launch<HD, 1>(ctx, kv, out, qkv, layer, T, pos0, ld);
        if (runs <= 2 * kPromptWaves) return prompt_launch<HD, 2>(ctx, kv, out, qkv, layer, T, pos0, ld);
        return prompt_launch<HD, 4>(ctx, kv, out, qkv, layer, T, pos0, ld);
    }
    // Staged values fit the 160 KB of LDS up to max_t = 1920 at HD 64.
    if (staged <= 150 * 1024)
        return store ? attend_launch<HD, true, true>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, staged)
                     : attend_launch<HD, true, false>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, staged);
    LLMQ_REQUIRE(base <= 150 * 1024, "int attention: max_t %d needs more LDS than a workgroup has", kv->max_t);
    return store ? attend_launch<HD, false, true>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, base)
                 : attend_launch<HD, false, false>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, base);
}

}  // namespace

int launch_ikv_store(llmq_ctx *ctx, llmq_kv *kv, int layer, int pos0, const int *pos_dev, const float *qkv, int T,
                     int64_t ld) {
    const int C = kv->n_head * kv->head_dim;
    if (kv->head_dim == 64)
        hipLaunchKernelGGL(ikv_store_kernel<64>, dim3(kv->n_head, T), dim3(64), 0, ctx->stream, qkv, ld ? ld : 3 * C,
                           C, pos0, pos_dev, layer, kv->max_t, kv->n_head, kv->k, kv->v, kv->kq, kv->vq);
    else if (kv->head_dim == 128)
        hipLaunchKernelGGL(ikv_store_kernel<128>, dim3(kv->n_head, T), dim3(64), 0, ctx->stream, qkv, ld ? ld : 3 * C,
                           C, pos0, pos_dev, layer, kv->max_t, kv->n_head, kv->k, kv->v, kv->kq, kv->vq);
    else
        return llmq_set_error(LLMQ_EUNSUPPORTED, "int attention: head_dim %d (64 or 128)", kv->head_dim);
    LLMQ_HIP(hipGetLastError());
    return LLMQ_OK;
}

int launch_ikv_attend(llmq_ctx *ctx, const llmq_kv *kv, float *out, const float *qkv, int layer, int T, int pos0,
                      const int *pos_dev, int64_t ld, bool store) {
    if (kv->head_dim == 64) return attend_hd<64>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, store);
    if (kv->head_dim == 128) return attend_hd<128>(ctx, kv, out, qkv, layer, T, pos0, pos_dev, ld, store);
    return llmq_set_error(LLMQ_EUNSUPPORTED, "int attention: head_dim %d (64 or 128)", kv->head_dim);
}
