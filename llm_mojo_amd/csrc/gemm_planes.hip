// The activation-plane matmul (gemm_planes.h): which matrices it takes, the
// tile of a call, and the operands.  The kernels are in gemm_planes_*.hip.
#include "gemm_planes.h"

namespace planes {

#define LLMQ_PX(F, SEG) extern template int launch_tile<F, SEG>(hipStream_t, int, const Args &);
LLMQ_PX(kQ8_0, 1) LLMQ_PX(kQ4_0, 1) LLMQ_PX(kQ4_1, 1) LLMQ_PX(kQ4_K, 8) LLMQ_PX(kQ5_K, 1) LLMQ_PX(kQ6_K, 8)
LLMQ_PX(kQm4, 1) LLMQ_PX(kQm4, 8) LLMQ_PX(kQm8, 1) LLMQ_PX(kQm8, 8)
LLMQ_PX(kA4, 1) LLMQ_PX(kA4, 2) LLMQ_PX(kA4, 4) LLMQ_PX(kA4, 8)
LLMQ_PX(kA8, 1) LLMQ_PX(kA8, 2) LLMQ_PX(kA8, 4) LLMQ_PX(kA8, 8)
#undef LLMQ_PX

namespace {

// Chunks of 32 inputs that share one of a QuantMatrix's scales, as the
// kernel's SEG (8: one scale a superblock or more) and the shift from a
// chunk to its group; false for groups the kernel does not take.
bool qm_groups(const llmq_mat *w, int *seg, int *shift) {
    if (w->NG == 1) {
        *seg = 8;
        *shift = 31;
        return true;
    }
    const int64_t cpg = w->group / 32;
    if (cpg < 1 || (cpg & (cpg - 1))) return false;
    *shift = __builtin_ctzll((unsigned long long)cpg);
    *seg = cpg < 8 ? (int)cpg : 8;
    return true;
}

// The tiles over a record: their size in 16-token and 16-row tiles, and what
// they took with one scale a superblock at 4096 x 4096 and 4096 x 11008: the
// time of a superblock in microseconds with few workgroups, how many of them
// run before that time grows, and the time before the first superblock.  The
// choice over 89 calls of Q4_K (48 to 1024 tokens, 768 to 8192 inputs, 768
// to 12000 rows) is 4 % off the best tile's time in the mean and 23 % at
// worst, over 355 calls of int4-g32, int4-g128, int8-g32 and int8-ch with
// int16 activations (16 to 1024 tokens) 1.1 and 23 %.
struct Tile {
    int tt, rt;
    float us, full, start;
};
constexpr Tile kTiles[] = {{4, 16, 5.2f, 280.0f, 4.0f}, {4, 8, 3.6f, 328.0f, 3.0f}, {4, 4, 2.4f, 386.0f, 2.0f},
                           {2, 4, 1.5f, 440.0f, 1.0f},  {1, 4, 1.2f, 510.0f, 0.6f}, {1, 4, 0.7f, 275.0f, 0.6f},
                           {1, 2, 0.6f, 292.0f, 0.6f}};

float tile_us(const Tile &k, int64_t token_tiles, int64_t row_tiles, int64_t inputs) {
    const float wgs = (float)((token_tiles + k.tt - 1) / k.tt * ((row_tiles + k.rt - 1) / k.rt));
    return k.start + (float)(inputs / 256) * k.us * (wgs > k.full ? wgs / k.full : 1.0f);
}

}  // namespace
}  // namespace planes

bool gemm_planes_ok(const llmq_mat *w) {
    if (!w || !is_float_act(w) || w->k % 256 != 0) return false;
    int seg, shift;
    return w->kind == MAT_GGUF || planes::qm_groups(w, &seg, &shift);
}

// LLMQ_PLANES_TILE, or -1.
static int forced_tile() {
    const char *e = getenv("LLMQ_PLANES_TILE");
    if (!e) return -1;
    const int t = atoi(e);
    return t < 0 ? 0 : t > 6 ? 6 : t;
}

// The tile from `first` on with the least time by kTiles' figures, and that time.
static int least_tile(const llmq_mat *w, int64_t T, int first, float *us) {
    using namespace planes;
    int best = first;
    *us = tile_us(kTiles[first], (T + 15) / 16, w->ntiles, w->k);
    for (int i = first + 1; i < (int)(sizeof(kTiles) / sizeof(kTiles[0])); i++) {
        const float t = tile_us(kTiles[i], (T + 15) / 16, w->ntiles, w->k);
        if (t < *us) {
            best = i;
            *us = t;
        }
    }
    return best;
}

// Q4_K's tile (few tokens have a kernel of their own).
static int q4k_tile(const llmq_mat *w, int64_t T) {
    const int forced = forced_tile();
    float us;
    return forced >= 0 ? forced : least_tile(w, T, 0, &us);
}

// The tiles over floats (the widest only where the kernel has it): what a
// superblock costs in microseconds with one workgroup on the fullest of the
// 256 CUs, and each further one there.  Fitted to 237 calls of Q8_0, int4-g32
// and int8-ch (16 to 1024 tokens, 768 to 8192 inputs, 768 to 12000 rows), 6
// to 12 % off a tile's times and within 1 % of the best of them by the choice;
// within 10 % on 79 of Q6_K, whose products are twice as many.
//
// The fp32 kernel (22 MAC a picosecond) is further off the 64-bit result, so
// it has only what it is the clearly faster one for: the line lies at 4 us
// and the least of kTiles' times, a little above the times here (10 x 1280 x
// 7224 Q4_1, near it: 7.3 us and 3.6e-7 off there, 8.2 and 1.0e-7 here; 16
// tokens of 4096 x 4096 Q8_0 12.2 us there and 16.8 here, 64 tokens 50 and
// 18.5).
int gemm_floats_tile(const llmq_mat *w, int64_t T) {
    using namespace planes;
    struct FloatTile {
        int tt, rt;
        float us, more;
    };
    static constexpr FloatTile tiles[] = {{2, 24, 5.88f, 4.66f}, {2, 16, 4.09f, 3.31f}, {2, 8, 2.53f, 3.17f},
                                          {1, 8, 1.60f, 2.06f},  {1, 4, 1.02f, 1.27f},  {1, 2, 0.74f, 0.70f}};
    int best = forced_tile();
    if (best >= 0) return best;
    int seg = 1, shift;
    if (w->kind == MAT_QUANT) qm_groups(w, &seg, &shift);
    const int ty = float_act_type(w);
    const bool wide = w->kind == MAT_QUANT ? seg < 8 : ty == LLMQ_GGML_Q8_0 || ty == LLMQ_GGML_Q4_0;
    float least;
    least_tile(w, T, wide || ty == LLMQ_GGML_Q4_1 ? 1 : 0, &least);
    if (3.5f + (float)T * (float)w->k * (float)w->n / 22e6f < 4.0f + least) return -1;
    for (int i = wide ? 0 : 1; i < (int)(sizeof(tiles) / sizeof(tiles[0])); i++) {
        const FloatTile &k = tiles[i];
        const int64_t wgs = ((T + 15) / 16 + k.tt - 1) / k.tt * ((w->ntiles + k.rt - 1) / k.rt);
        const float us = k.us + k.more * (float)((wgs + 255) / 256 - 1);
        if (best < 0 || us < least) {
            best = i;
            least = us;
        }
    }
    return best;
}

namespace planes {
namespace {

// The weights' and the outputs' side of a call (seg: chunks that share a scale).
int args(const llmq_mat *w, int64_t T, float *out, int64_t ldo, const float *bias, int flags, Args *a, int *seg) {
    LLMQ_REQUIRE(gemm_planes_ok(w), "gemm_planes: not a matrix of this kernel");
    LLMQ_REQUIRE(out && T > 0, "gemm_planes: bad arguments");
    LLMQ_REQUIRE(!(flags & LLMQ_BIAS) || bias, "gemm_planes: LLMQ_BIAS without a bias");
    const int64_t T16 = (T + 15) / 16 * 16;
    const int64_t ntc = (w->ntiles * w->CK + LLMQ_PAD_CHUNKS) * 16;
    LLMQ_REQUIRE(ntc * 16 < (int64_t)kLlmqOOB, "gemm_planes: operands too large");
    *a = Args{};
    a->codes = w->codes;
    *seg = 8;
    if (w->kind == MAT_QUANT) {
        qm_groups(w, seg, &a->gshift);
        a->scales = reinterpret_cast<const uint8_t *>(w->scales);
        a->zps = w->zps;
        a->NG = (int)w->NG;
    } else if (w->ggml_type == LLMQ_GGML_Q4_1) {
        a->scales = reinterpret_cast<const uint8_t *>(w->g_meta32);
    } else if (w->ggml_type == LLMQ_GGML_Q8_0 || w->ggml_type == LLMQ_GGML_Q4_0) {
        a->scales = reinterpret_cast<const uint8_t *>(w->g_meta16);
    } else {
        a->sb = reinterpret_cast<const uint8_t *>(w->g_sb16);
        if (w->ggml_type == LLMQ_GGML_Q5_K) {
            a->bits = reinterpret_cast<const uint8_t *>(w->g_bits32);
        } else if (w->ggml_type == LLMQ_GGML_Q6_K) {
            a->bits = reinterpret_cast<const uint8_t *>(w->g_bits64);
            a->sbd = reinterpret_cast<const uint8_t *>(w->g_meta16);
        }
    }
    a->T = (int)T;
    a->n = (int)w->n;
    a->ntiles = (int)w->ntiles;
    a->NC = (int)(w->k / 32);
    a->NSB = (int)(w->k / 256);
    a->flags = flags;
    a->rows_first = T16 * w->k * 4 > ntc * 16;
    a->ldo = ldo;
    a->bias = bias ? bias : out;
    a->out = out;
    return LLMQ_OK;
}

}  // namespace
}  // namespace planes

int launch_gemm_planes(llmq_ctx *ctx, const llmq_mat *w, const void *rec, int64_t T, float *out, int64_t ldo,
                       const float *bias, int flags) {
    using namespace planes;
    Args a;
    int seg;
    RC(args(w, T, out, ldo, bias, flags, &a, &seg));
    LLMQ_REQUIRE(gguf_gemm_h16_ok(w) && rec && h16_rec_bytes(T, w->k) < (int64_t)kLlmqOOB,
                 "gemm_planes: not a record of this kernel");
    uint8_t *pl;
    _Float16 *su;
    float *iv;
    h16_rec_parts(const_cast<void *>(rec), T, w->k, &pl, &su, &iv);
    a.planes = pl;
    a.sums = reinterpret_cast<const uint8_t *>(su);
    a.inv = reinterpret_cast<const uint8_t *>(iv);
    return launch_tile<kQ4_K, 8>(ctx->stream, q4k_tile(w, T), a);
}

int launch_gemm_floats(llmq_ctx *ctx, const llmq_mat *w, const float *x, int64_t ldx, int64_t T, float *out,
                       int64_t ldo, const float *bias, int flags, int tile) {
    using namespace planes;
    Args a;
    int seg;
    RC(args(w, T, out, ldo, bias, flags, &a, &seg));
    LLMQ_REQUIRE(tile >= 0 && x && ldx >= w->k && T * ldx * 4 < (int64_t)kLlmqOOB, "gemm_floats: bad arguments");
    a.x = x;
    a.ldx = ldx;
    hipStream_t st = ctx->stream;
    switch (float_act_type(w)) {  // (groups of 64 and 128 take their scale a chunk at a time)
    case kQmFloat4: return seg == 8 ? launch_tile<kQm4, 8>(st, tile, a) : launch_tile<kQm4, 1>(st, tile, a);
    case kQmFloat8: return seg == 8 ? launch_tile<kQm8, 8>(st, tile, a) : launch_tile<kQm8, 1>(st, tile, a);
    case LLMQ_GGML_Q8_0: return launch_tile<kQ8_0, 1>(st, tile, a);
    case LLMQ_GGML_Q4_0: return launch_tile<kQ4_0, 1>(st, tile, a);
    case LLMQ_GGML_Q4_1: return launch_tile<kQ4_1, 1>(st, tile, a);
    case LLMQ_GGML_Q5_K: return launch_tile<kQ5_K, 1>(st, tile, a);
    case LLMQ_GGML_Q6_K: return launch_tile<kQ6_K, 8>(st, tile, a);
    default: return llmq_set_error(LLMQ_EUNSUPPORTED, "gemm_floats: type %d", float_act_type(w));
    }
}

bool gemm_planes_a16_ok(const llmq_mat *w) {
    int seg, shift;
    return w && w->kind == MAT_QUANT && w->k % 256 == 0 && planes::qm_groups(w, &seg, &shift);
}

int launch_gemm_planes_a16(llmq_ctx *ctx, const llmq_mat *w, const uint8_t *pl, const float *sx, int64_t T, int64_t n,
                           float *out, int64_t ldo, const float *bias, int flags) {
    using namespace planes;
    LLMQ_REQUIRE(gemm_planes_a16_ok(w) && n <= w->n, "gemm_planes_a16: not a matrix of this kernel");
    Args a{};
    a.planes = pl;
    a.sx = sx;
    a.codes = w->codes;
    a.scales = reinterpret_cast<const uint8_t *>(w->scales);
    a.zps = w->zps;
    a.NG = (int)w->NG;
    int seg = 8;
    qm_groups(w, &seg, &a.gshift);
    a.T = (int)T;
    a.n = (int)n;
    a.ntiles = (int)(n / 16);
    a.NC = (int)(w->k / 32);
    a.NSB = (int)(w->k / 256);
    a.flags = flags;
    a.rows_first = (T + 15) / 16 * 16 * w->k * 4 > w->ntiles * w->CK * 256;
    a.ldo = ldo;
    a.bias = bias ? bias : out;
    a.out = out;
    int tile = 1;
    if (const char *e = getenv("LLMQ_PLANES_TILE")) {
        tile = atoi(e) < 1 ? 1 : atoi(e) > 4 ? 4 : atoi(e);
    } else {
        float least = 0.0f;
        for (int i = 1; i <= 4; i++) {
            const float us = tile_us(kTiles[i], (T + 15) / 16, a.ntiles, w->k);
            if (i == 1 || us < least) {
                tile = i;
                least = us;
            }
        }
    }
    hipStream_t st = ctx->stream;
#define LLMQ_PS(F)                                             \
    switch (seg) {                                             \
    case 1: return launch_tile<F, 1>(st, tile, a);             \
    case 2: return launch_tile<F, 2>(st, tile, a);             \
    case 4: return launch_tile<F, 4>(st, tile, a);             \
    default: return launch_tile<F, 8>(st, tile, a);            \
    }
    if (w->bits == 4) {
        LLMQ_PS(kA4)
    }
    LLMQ_PS(kA8)
#undef LLMQ_PS
}
