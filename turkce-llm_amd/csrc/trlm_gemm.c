/* trlm_gemm.c -- host dispatch of the fp32 GEMM kernels (gemm.hip, gemm_split.hip,
 * gemm_small.hip).
 *
 * Plays the role of the reference's gemm()/gemm1()/bf16_gemm*() launch
 * helpers (model/gpu_train.c:42-118): same operand conventions (NN, NT, TN;
 * batched with element strides; alpha/beta; bias and residual epilogue),
 * with the tile shape and split-K chosen per problem for 256 CUs:
 *   - (tile, split-K) minimise a load-balance cost model (select_plan): the
 *     busiest CU's share of workgroups, the variant's residency and
 *     efficiency, and the split partials' HBM round trip.  The plan depends
 *     on (M, N, K, batch) only, so reruns are bit-identical;
 *   - split-K (single GEMMs: weight gradients with K = B*T, dX with
 *     K = vocab, short-M shapes): splits write raw partials to a workspace
 *     that k_gemm_splitk_reduce sums in split order, so the result stays
 *     deterministic (no atomics);
 *   - operands whose rows are not 16-byte aligned go to the _u variants,
 *     which load value by value.
 */
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>

#include "gpu_internal.h"

#include "kernel_params.h"   /* GemmParams: the argument block the kernels read */

enum { L_NN = 0, L_NT = 1, L_TN = 2 };
static const char* LAYOUT_NAME[4] = { "nn", "nt", "tn", "tt" };

/* Aligned tile variants: name suffix, tile rows/cols, k step of the fp32
 * kernels (gemm.hip, k_gemm_*).  128x128, 64x128_k32 and 64x64_k32 also come
 * from exact three-way bf16 splits (gemm_split.hip, k_xgemm_*, k step 32),
 * which an engine takes for them unless it keeps to fp32. */
typedef struct TileDef { const char* name; int bm, bn, bk; } TileDef;
enum { T_256x128, T_128x256, T_128x128, T_128x128_K32, T_64x128, T_64x128_K32, T_64x64, T_64x64_K32, T_COUNT };
static const TileDef TILES[T_COUNT] = {
    { "256x128", 256, 128, 16 }, { "128x256", 128, 256, 16 }, { "128x128", 128, 128, 16 },
    { "128x128_k32", 128, 128, 32 }, { "64x128", 64, 128, 16 }, { "64x128_k32", 64, 128, 32 },
    { "64x64", 64, 64, 16 }, { "64x64_k32", 64, 64, 32 },
};

static int has_split(int t) { return t == T_128x128 || t == T_64x128_K32 || t == T_64x64_K32; }

#define CUS 256
#define KCHUNK_ALIGN 32  /* split-K chunks are multiples of every variant's k step */

struct TrlmGemm {
    HipCtx* ctx;
    hipFunction_t k[3][T_COUNT];   /* fp32 tiles (gemm.hip) */
    hipFunction_t x[3][T_COUNT];   /* split products (gemm_split.hip), for the tiles that have them */
    int fp32;                      /* keep to the fp32 tiles */
    hipFunction_t ku[4];           /* unaligned operands: fp32 64x64_u */
    hipFunction_t xu[4], xu128[3]; /* the same from split products, 64x64_u and 128x128_u */
    hipFunction_t reduce;
    hipFunction_t reduce4;   /* four columns per thread, for 16-byte aligned operands */
    hipFunction_t small[2][3];   /* k_smallgemm_<layout>[_u]: 32x32 tiles, k shared out over a workgroup's waves */
    hipFunction_t small_glu;
    hipFunction_t glu;             /* SwiGLU epilogue: fp32 64x64_k32 */
    hipFunction_t xglu, xglu128;   /* split products, 64x64_k32 and 128x128 */
    hipDeviceptr_t ws;
    u64 ws_floats;
    char last[48];
    i32 last_splits;
    i32 force_tile;    /* -1: automatic selection */
    i32 force_splits;  /* 0: automatic split-K */
};

static TrlmGemm* create(HipCtx* ctx, int fp32) {
    TrlmGemm* e = (TrlmGemm*)calloc(1, sizeof(TrlmGemm));
    e->ctx = ctx;
    e->force_tile = -1;
    e->fp32 = fp32;
    char name[64];
    for (int l = 0; l < 3; l++)
        for (int t = 0; t < T_COUNT; t++) {
            snprintf(name, sizeof(name), "k_gemm_%s_%s", LAYOUT_NAME[l], TILES[t].name);
            e->k[l][t] = hip_get_kernel(ctx, name);
            if (fp32 || !has_split(t)) continue;
            snprintf(name, sizeof(name), "k_xgemm_%s_%s", LAYOUT_NAME[l], TILES[t].name);
            e->x[l][t] = hip_get_kernel(ctx, name);
        }
    for (int l = 0; l < 4; l++) {
        snprintf(name, sizeof(name), "k_gemm_%s_64x64_u", LAYOUT_NAME[l]);
        e->ku[l] = hip_get_kernel(ctx, name);
        if (fp32) continue;
        snprintf(name, sizeof(name), "k_xgemm_%s_64x64_u", LAYOUT_NAME[l]);
        e->xu[l] = hip_get_kernel(ctx, name);
        if (l == 3) break;
        snprintf(name, sizeof(name), "k_xgemm_%s_128x128_u", LAYOUT_NAME[l]);
        e->xu128[l] = hip_get_kernel(ctx, name);
    }
    for (int l = 0; l < 3; l++)
        for (int u = 0; u < 2; u++) {
            snprintf(name, sizeof(name), "k_smallgemm_%s%s", LAYOUT_NAME[l], u ? "_u" : "");
            e->small[u][l] = hip_get_kernel(ctx, name);
        }
    snprintf(name, sizeof(name), "k_smallgemm_%s_glu", LAYOUT_NAME[L_NN]);
    e->small_glu = hip_get_kernel(ctx, name);
    e->reduce = hip_get_kernel(ctx, "k_gemm_splitk_reduce");
    e->reduce4 = hip_get_kernel(ctx, "k_gemm_splitk_reduce4");
    e->glu = hip_get_kernel(ctx, "k_gemm_nn_64x64_k32_glu");
    if (!fp32) {
        e->xglu = hip_get_kernel(ctx, "k_xgemm_nn_64x64_k32_glu");
        e->xglu128 = hip_get_kernel(ctx, "k_xgemm_nn_128x128_glu");
    }
    trlm_noalloc_setup(ctx->device);
    return e;
}

TrlmGemm* trlm_gemm_create(HipCtx* ctx) { return create(ctx, 0); }

TrlmGemm* trlm_gemm_create_fp32(HipCtx* ctx) { return create(ctx, 1); }

/* The engine's products keep to the fp32 matrix cores, with the tiles and
 * split-K of the fp32 plan (products of few tiles take k_smallgemm_*, which is
 * fp32 too).  The trainer's engines do: an optimizer's first steps magnify any
 * other rounding, however small (AdamW divides by the gradient's size: after
 * one step of the 12-layer model two correct roundings of it, each 1.7e-6 or
 * less from 64 bits, have gradients 7e-6 to 2e-5 apart), and the evaluation's
 * loss is bit for bit the training step's, so its products go with them. */
void trlm_gemm_keep_fp32(TrlmGemm* e) { e->fp32 = 1; }

void trlm_gemm_destroy(TrlmGemm* e) {
    if (!e) return;
    if (e->ws) hip_free(e->ws);
    free(e);
}

i32 trlm_gemm_device(const TrlmGemm* e) { return e->ctx->device; }

const char* trlm_gemm_last_variant(TrlmGemm* e, i32* splits) {
    if (splits) *splits = e->last_splits;
    return e->last;
}

i32 trlm_gemm_force(TrlmGemm* e, const char* tile, i32 splits) {
    e->force_tile = -1;
    e->force_splits = splits > 0 ? splits : 0;
    if (!tile || !tile[0]) return 0;
    for (int t = 0; t < T_COUNT; t++)
        if (strcmp(tile, TILES[t].name) == 0) {
            e->force_tile = t;
            return 0;
        }
    return -1;
}

static int cdiv(long long a, long long b) { return (int)((a + b - 1) / b); }

static int aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

/* Row statistics: 2 entries per tile column (one per wave column half);
 * the caller's buffer holds stats_cap entries per row. */
static void set_stats(GemmParams* p, hipDeviceptr_t stats, i32 stats_cap, int bn) {
    int n = 2 * cdiv(p->N, bn);
    if (n > stats_cap) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: row statistics need %d entries per row, buffer has %d\n", n, stats_cap);
        _exit(1);
    }
    p->stats = (float*)stats;
    p->stats_ld = n;
}

static void launch(hipFunction_t f, GemmParams* p, u32 gz) {
    void* args[] = { p };
    hip_launch(f, (u32)(p->tiles_m * p->tiles_n), 1, gz, 256, 1, 1, 0, args);
}

static long long tiles_of(int t, int M, int N, u32 batch) {
    return (long long)cdiv(M, TILES[t].bm) * cdiv(N, TILES[t].bn) * batch;
}

/* Split-K factor for a single GEMM with few output tiles and a long K:
 * enough splits for ~2 workgroups per CU, each split >= 256 deep.  Used
 * when a tile is forced without a split factor. */
static int auto_splits(long long tiles, int K) {
    if (K < 512 || tiles >= CUS) return 1;
    int s = cdiv(2 * CUS, tiles);
    if (s > K / 256) s = K / 256;
    if (s > 32) s = 32;
    return s < 1 ? 1 : s;
}

/* Plan model: the tiles' workgroups are spread evenly over the 256 CUs, so
 * the busiest CU runs n = ceil(workgroups / 256) of them, `occ` at a time
 * (the variant's resident workgroups per CU).  A CU with c resident
 * workgroups runs at cu_rate of the variant's steady-state rate (a lone
 * workgroup's split and LDS phases leave its matrix cores idle, several
 * workgroups' phases overlap).  The last resident batch adds an imbalance
 * term proportional to a workgroup's duration, and no plan is faster than
 * the chip's sustained rate (the matrix cores' clock falls under load).
 * Split-K adds the partials' round trip through HBM plus the reduction
 * launch.  Constants fitted to MI355X timings of the three split-product
 * variants and every split on the model's GEMMs at 300-8192 rows and five
 * others (within 0.8 % of the per-shape best over those 80 shapes). */
typedef struct PlanTile { int tile; int occ; double rate, lone, start; } PlanTile;
static const PlanTile PLAN_TILES[] = {
    { T_128x128, 3, 0.820e12, 0.781, 2e-6 },
    { T_64x128_K32, 4, 0.627e12, 0.450, 0 },
    { T_64x64_K32, 5, 0.644e12, 0.662, 0 },
};
static const int PLAN_SPLITS[] = { 1, 2, 3, 4, 6, 7, 8, 12, 16, 24, 32 };
#define PLAN_CAP_FLOPS 227e12    /* the chip's sustained rate, FLOP/s */
#define PLAN_SPLIT_BW 3.06e12    /* effective bytes/s of the partials' round trip */
#define PLAN_SPLIT_FIXED 1.91e-6 /* reduction launch, s */
#define PLAN_TAIL 0.123          /* last-round imbalance, in resident-batch durations */

static double cu_rate(const PlanTile* pt, long long c) {
    return pt->lone + (1.0 - pt->lone) * (double)(c - 1) / (pt->occ - 1);
}

static double plan_cost(const PlanTile* pt, int M, int N, int K, u32 batch, int splits) {
    const TileDef* td = &TILES[pt->tile];
    double wg = (double)cdiv(M, td->bm) * cdiv(N, td->bn) * batch * splits;
    int kch = splits > 1 ? cdiv(cdiv(K, splits), KCHUNK_ALIGN) * KCHUNK_ALIGN : K;
    long long n = (long long)((wg + CUS - 1) / CUS);
    double flops = 2.0 * td->bm * td->bn * (double)kch;
    double w = flops / pt->rate;
    long long full = n / pt->occ, rest = n % pt->occ, last = n < pt->occ ? n : pt->occ;
    double t = (double)full * pt->occ * w;
    if (rest) t += (double)rest * w / cu_rate(pt, rest);
    /* workgroups of one resident batch finish unevenly: long workgroups
     * leave CUs idle at the end, which more, shorter ones even out */
    t += PLAN_TAIL * (double)last * w / cu_rate(pt, last);
    if (t < wg * flops / PLAN_CAP_FLOPS) t = wg * flops / PLAN_CAP_FLOPS;
    t += pt->start;   /* first loads and last stores of a workgroup, over the smallest tile's */
    if (splits > 1) t += (splits + 1) * (double)M * N * 4.0 / PLAN_SPLIT_BW + PLAN_SPLIT_FIXED;
    return t;
}

static void select_plan(int M, int N, int K, u32 batch, int* tile, int* splits) {
    double best = 0.0;
    *tile = T_128x128;
    *splits = 1;
    /* Products of few tiles with one side of at most 128: each workgroup's k
     * loop is latency-bound (0.75 us per 32-deep step alone on its CU), so
     * split K down to 64-deep chunks over up to 8 partitions, 128-deep up to
     * 16 and 256-deep beyond, two workgroups per CU at most.  Measured on
     * MI355X against at most 8: 17x1374x7742 35.3 -> 27.2 us (16).  One
     * workgroup per CU where that leaves chunks of at most 512: the fp32
     * tile's case (see trlm_gemm_ws), 36x3795x1091 16.2 (7 splits) -> 14.3 us
     * (4), 3644x63x1428 19.2 (8) -> 16.7 (4). */
    if ((M <= 128 || N <= 128) && batch == 1) {
        long long tiles = (long long)cdiv(M, 64) * cdiv(N, 64);
        if (tiles < 128) {
            long long smax = K / 64;
            if (smax > 8) smax = 8;
            if (smax < K / 128) smax = K / 128 < 16 ? K / 128 : 16;
            if (smax < K / 256) smax = K / 256;
            const long long per_cu = (long long)K * tiles <= 512ll * CUS ? 1 : 2;
            if (smax > per_cu * CUS / tiles) smax = per_cu * CUS / tiles;
            *tile = T_64x64_K32;
            for (size_t j = 0; j < sizeof(PLAN_SPLITS) / sizeof(PLAN_SPLITS[0]); j++)
                if (PLAN_SPLITS[j] <= smax) *splits = PLAN_SPLITS[j];
            return;
        }
    }
    for (size_t i = 0; i < sizeof(PLAN_TILES) / sizeof(PLAN_TILES[0]); i++)
        for (size_t j = 0; j < sizeof(PLAN_SPLITS) / sizeof(PLAN_SPLITS[0]); j++) {
            int sp = PLAN_SPLITS[j];
            if (sp > 1 && (batch != 1 || K / sp < 256)) continue;
            double c = plan_cost(&PLAN_TILES[i], M, N, K, batch, sp);
            if ((i == 0 && j == 0) || c < best) {
                best = c;
                *tile = PLAN_TILES[i].tile;
                *splits = sp;
            }
        }
}

/* Plan model of the fp32 tiles (an engine that keeps them, see
 * trlm_gemm_keep_fp32): the tiles' workgroups are spread evenly over the 256 CUs, so
 * the busiest CU runs n = ceil(workgroups / 256) of them, `occ` at a time
 * (the variant's resident workgroups per CU).  A CU with c resident
 * workgroups runs at fp32_cu_rate(c) of its steady-state rate (one resident
 * 4-wave workgroup cannot hide its own load latency), and each variant has
 * its own steady-state efficiency.  The last resident batch adds an
 * imbalance term proportional to a workgroup's duration.  Split-K adds the
 * partials' round trip through HBM plus the reduction launch.  Constants
 * fitted to MI355X timings of every variant/split on the model's GEMMs at
 * 512-8192 rows (within 0.6 % of the per-shape best over those 45 shapes). */
typedef struct Fp32Tile { int tile; int occ; double eff; } Fp32Tile;
static const Fp32Tile FP32_TILES[] = {
    { T_128x128, 3, 1.047 }, { T_128x256, 2, 0.977 }, { T_256x128, 2, 1.008 },
    { T_64x128_K32, 2, 0.955 }, { T_64x64_K32, 4, 0.992 },
};
#define FP32_CU_FLOPS 0.6e12     /* per-CU steady-state fp32 MFMA rate, FLOP/s */
#define FP32_SPLIT_BW 1.63e12    /* effective bytes/s of the partials' round trip */
#define FP32_SPLIT_FIXED 1.25e-6 /* reduction launch, s */
#define FP32_TAIL 0.075          /* last-round imbalance, in resident-batch durations */

static double fp32_cu_rate(int c) { return c <= 1 ? 0.916 : 1.0; }

static double fp32_cost(const Fp32Tile* pt, int M, int N, int K, u32 batch, int splits) {
    const TileDef* td = &TILES[pt->tile];
    double wg = (double)cdiv(M, td->bm) * cdiv(N, td->bn) * batch * splits;
    int kch = splits > 1 ? cdiv(cdiv(K, splits), KCHUNK_ALIGN) * KCHUNK_ALIGN : K;
    long long n = (long long)((wg + CUS - 1) / CUS);
    double w = 2.0 * td->bm * td->bn * (double)kch / (pt->eff * FP32_CU_FLOPS);
    long long full = n / pt->occ, rest = n % pt->occ;
    double t = (double)full * pt->occ * w / fp32_cu_rate(pt->occ);
    if (rest) t += (double)rest * w / fp32_cu_rate((int)rest);
    /* workgroups of one resident batch finish unevenly: long workgroups
     * leave CUs idle at the end, which more, shorter ones even out */
    t += FP32_TAIL * pt->occ * w / fp32_cu_rate((int)(n < pt->occ ? n : pt->occ));
    if (splits > 1) t += (splits + 1) * (double)M * N * 4.0 / FP32_SPLIT_BW + FP32_SPLIT_FIXED;
    return t;
}

static void select_fp32(int M, int N, int K, u32 batch, int* tile, int* splits) {
    double best = 0.0;
    *tile = T_128x128;
    *splits = 1;
    /* Decode-sized products (M <= 128 rows, few tiles): each workgroup's
     * k loop is latency-bound (~1 us per 32-deep step), so split K down to
     * 64-deep chunks over up to 8 partitions, one workgroup per CU at most.
     * Measured on MI355X at M = 64: QKV 12.8 -> 9.0 us, attention-out 11.8
     * -> 8.6, gate_up 12.4 -> 8.2, down (K = 1024) 12.6 -> 10.4, reduction
     * included. */
    if (M <= 128 && batch == 1) {
        long long tiles = (long long)cdiv(M, 64) * cdiv(N, 64);
        if (tiles < 128) {
            long long smax = K / 64;
            if (smax > 8) smax = 8;
            if (smax > CUS / tiles) smax = CUS / tiles;
            *tile = T_64x64_K32;
            for (size_t j = 0; j < sizeof(PLAN_SPLITS) / sizeof(PLAN_SPLITS[0]); j++)
                if (PLAN_SPLITS[j] <= smax) *splits = PLAN_SPLITS[j];
            return;
        }
    }
    for (size_t i = 0; i < sizeof(FP32_TILES) / sizeof(FP32_TILES[0]); i++)
        for (size_t j = 0; j < sizeof(PLAN_SPLITS) / sizeof(PLAN_SPLITS[0]); j++) {
            int sp = PLAN_SPLITS[j];
            if (sp > 1 && (batch != 1 || K / sp < 256)) continue;
            double c = fp32_cost(&FP32_TILES[i], M, N, K, batch, sp);
            if ((i == 0 && j == 0) || c < best) {
                best = c;
                *tile = FP32_TILES[i].tile;
                *splits = sp;
            }
        }
}

/* Products of few tiles (gemm_small.hip, k_smallgemm_*): one 32x32 tile per
 * workgroup, k shared out over its waves.  Up to two tiles per
 * CU, measured on MI355X against the planned tile (us): 64x1152x384 5.8 / 8.0,
 * 128x2048x384 (256 tiles) 6.1 / 9.9, 512x384x384 (192) 6.0 / 11.9,
 * 512x1024x384 (512) 9.9 / 10.8, but 512x1152x384 (576) 12.4 / 12.2; with less
 * than 96 k up to one tile per CU (384x1152x64, 432 tiles: 5.2 / 4.9).  Up to
 * 768 k, 1152 where neither side is at most 128 (512x384x1024 11.0 / 13.4,
 * 358x137x1099 12.9 / 14.6, but 64x384x1024, which select_plan splits into
 * more partitions, 10.8 / 9.4).  Unaligned operands, which this kernel loads
 * with the fewer idle lanes, up to three tiles per CU where k is short (704
 * tiles: 701x1001x101 7.3 / 9.2, but 1000x701x333 17.2 / 14.9). */
static int small_gemm(int M, int N, int K, u32 batch, int aligned) {
    const long long tiles = (long long)cdiv(M, 32) * cdiv(N, 32);
    const int most = !aligned && K <= 192 ? 3 * CUS : K >= 96 ? 2 * CUS : CUS;
    return batch == 1 && K <= (M > 128 && N > 128 ? 1152 : 768) && tiles <= most;
}

#define ANY_ROOM (~0ull)   /* a workspace that grows */

/* What runs a product: the kernel's family and tile, the split-K factor and
 * each split's share of k. */
enum { FP32, SPLIT, SMALL };
typedef struct Plan { int family, tile, splits, kchunk; } Plan;

/* What a product asks of its plan beside its shape. */
typedef struct PlanOpts {
    int aligned;                /* 16-byte rows */
    int fp32;                   /* keeps to the fp32 tiles */
    int stats, whole;           /* row statistics; an epilogue that needs whole sums (stats, RoPE) */
    int force_tile, force_splits;
    u64 slab, ws_floats;        /* floats of one split's partials, and that there is room for */
} PlanOpts;

/* Shares k out over `splits`, each a multiple of KCHUNK_ALIGN. */
static void set_splits(Plan* p, int K, int splits) {
    p->splits = splits;
    p->kchunk = K;
    if (splits > 1) {
        p->kchunk = cdiv(cdiv(K, splits), KCHUNK_ALIGN) * KCHUNK_ALIGN;
        p->splits = cdiv(K, p->kchunk);
    }
}

static Plan make_plan(int layout, int M, int N, int K, u32 batch, const PlanOpts* o) {
    Plan p = { FP32, T_64x64_K32, 1, K };
    if (layout != 3 && !o->stats && o->force_tile < 0 && o->force_splits == 0 &&
        small_gemm(M, N, K, batch, o->aligned)) {
        p.family = SMALL;
        return p;
    }
    int splits;
    if (o->fp32) select_fp32(M, N, K, batch, &p.tile, &splits);
    else select_plan(M, N, K, batch, &p.tile, &splits);
    if (!o->aligned) {
        /* the unaligned kernels: one fp32 tile without split-K, two of the
         * split products' tiles */
        if (o->fp32 || p.tile != T_128x128 || layout == 3 || o->stats) p.tile = T_64x64_K32;
        if (o->fp32 || layout == 3) splits = 1;
    } else if (o->force_tile >= 0) {
        p.tile = o->force_tile;
        splits = batch == 1 ? auto_splits(tiles_of(p.tile, M, N, 1), K) : 1;
    }
    if (o->force_splits > 0 && batch == 1 && (o->aligned || (!o->fp32 && layout != 3))) splits = o->force_splits;
    if (o->whole || K < 2 * KCHUNK_ALIGN) splits = 1;
    set_splits(&p, K, splits);
    if (p.splits > 1 && (u64)p.splits * o->slab > o->ws_floats) {
        /* A fixed workspace that cannot hold the plan's partials: run the
         * most splits whose partials fit (one split needs none).  The k
         * chunks are formed as for a forced split count, so the result
         * equals this engine's trlm_gemm forced to that many splits. */
        u64 fit = o->ws_floats / o->slab;
        set_splits(&p, K, fit < 2 ? 1 : (int)fit);
    }
    if (!o->fp32 && (!o->aligned || has_split(p.tile))) p.family = SPLIT;
    /* At most one 64x64 workgroup per CU: nothing hides a lone workgroup's
     * splitting, and the fp32 tile of the same plan is the faster.  MI355X,
     * split products / fp32 tiles (us): 43x8816x710 TN (138 workgroups) 22.4 /
     * 17.8, 173x28x7365 TN (24 splits, 72) 16.5 / 13.5, 11x15x1051 NT (7) 10.7
     * / 9.6; over 46 drawn shapes up to 256 workgroups 0.79 to 1.02 of the
     * time, 257 to 320 0.95 to 1.08, beyond them 1.00 to 1.29. */
    if (o->aligned && p.tile == T_64x64_K32 && o->force_tile < 0 &&
        tiles_of(p.tile, M, N, p.splits > 1 ? (u32)p.splits : batch) <= CUS)
        p.family = FP32;
    return p;
}

/* The plan of the gate/up product [M, 2F] with the SwiGLU epilogue.  MI355X,
 * small / fp32 64x64 / split 64x64 / split 128x128 (us), K = 384, F = 1024:
 * 100 rows (256 small tiles) 6.4 / 11.1 / 13.6 / 29, 256 rows (512) 10.1 / 11.4 / 13.8,
 * 320 rows 14.4 / 11.7 / 13.9; K = 768, F = 2048: 64 rows (256) 12.3 / 18.3,
 * 100 rows (512) 21.8 / 18.4 -- so one small tile per CU beyond 384 k.  At most one 64x64
 * workgroup per CU takes the fp32 tile as in make_plan: 512 rows (256)
 * 12.1 / 14.3, 768 rows (384) 18.6 / 16.9.  Beyond, the 128-wide tile where F
 * holds whole half tiles and the plan model finds it the faster of the two. */
static Plan make_glu_plan(int M, int F, int K, int fp32) {
    Plan p = { fp32 ? FP32 : SPLIT, T_64x64_K32, 1, K };
    if (small_gemm(M, 2 * F, K, 1, 1) && (K <= 384 || (long long)cdiv(M, 32) * cdiv(2 * F, 32) <= CUS))
        p.family = SMALL;
    else if (tiles_of(p.tile, M, 2 * F, 1) <= CUS)
        p.family = FP32;
    else if (!fp32 && F % 64 == 0 &&
             plan_cost(&PLAN_TILES[0], M, 2 * F, K, 1, 1) < plan_cost(&PLAN_TILES[2], M, 2 * F, K, 1, 1))
        p.tile = T_128x128;
    return p;
}

/* The kernel's name in the code object. */
static void plan_name(char* out, size_t size, const Plan* p, int layout, int aligned, int glu) {
    const char* l = LAYOUT_NAME[layout];
    const char* end = glu ? "_glu" : aligned ? "" : "_u";
    if (p->family == SMALL) snprintf(out, size, "k_smallgemm_%s%s", l, end);
    else
        snprintf(out, size, "k_%sgemm_%s_%s%s", p->family == SPLIT ? "x" : "", l,
                 aligned ? TILES[p->tile].name : p->tile == T_128x128 ? "128x128" : "64x64", end);
}

const char* trlm_gemm_plan_ex(i32 trans_a, i32 trans_b, i32 M, i32 N, i32 K, u32 batch, i32 fp32, i32 glu_F,
                              i32* splits) {
    static __thread char name[48];
    const int layout = trans_a ? (trans_b ? 3 : L_TN) : (trans_b ? L_NT : L_NN);
    const PlanOpts o = { .aligned = layout != 3, .fp32 = fp32, .force_tile = -1, .ws_floats = ANY_ROOM };
    const Plan p = glu_F > 0 ? make_glu_plan(M, glu_F, K, fp32) : make_plan(layout, M, N, K, batch ? batch : 1, &o);
    plan_name(name, sizeof(name), &p, layout, o.aligned, glu_F > 0);
    if (splits) *splits = p.splits;
    return name;
}

const char* trlm_gemm_plan(i32 trans_a, i32 trans_b, i32 M, i32 N, i32 K, u32 batch, i32* splits) {
    return trlm_gemm_plan_ex(trans_a, trans_b, M, N, K, batch, 0, 0, splits);
}

void trlm_gemm(TrlmGemm* e, i32 trans_a, i32 trans_b, hipDeviceptr_t A, hipDeviceptr_t B, hipDeviceptr_t C,
               i32 M, i32 N, i32 K, i32 lda, i32 ldb, i32 ldc, u32 batch, i64 sA, i64 sB, i64 sC,
               f32 alpha, f32 beta, hipDeviceptr_t bias, hipDeviceptr_t resid, i32 ldr) {
    trlm_gemm_ex(e, trans_a, trans_b, A, B, C, M, N, K, lda, ldb, ldc, batch, sA, sB, sC, alpha, beta, bias, resid,
                 ldr, NULL);
}

i32 trlm_gemm_ex(TrlmGemm* e, i32 trans_a, i32 trans_b, hipDeviceptr_t A, hipDeviceptr_t B, hipDeviceptr_t C,
                 i32 M, i32 N, i32 K, i32 lda, i32 ldb, i32 ldc, u32 batch, i64 sA, i64 sB, i64 sC,
                 f32 alpha, f32 beta, hipDeviceptr_t bias, hipDeviceptr_t resid, i32 ldr, const TrlmGemmExtra* x) {
    return trlm_gemm_ws(e, trans_a, trans_b, A, B, C, M, N, K, lda, ldb, ldc, batch, sA, sB, sC, alpha, beta, bias,
                        resid, ldr, x, NULL, 0);
}

i32 trlm_gemm_ws(TrlmGemm* e, i32 trans_a, i32 trans_b, hipDeviceptr_t A, hipDeviceptr_t B, hipDeviceptr_t C,
                 i32 M, i32 N, i32 K, i32 lda, i32 ldb, i32 ldc, u32 batch, i64 sA, i64 sB, i64 sC,
                 f32 alpha, f32 beta, hipDeviceptr_t bias, hipDeviceptr_t resid, i32 ldr, const TrlmGemmExtra* x,
                 hipDeviceptr_t fixed_ws, u64 fixed_floats) {
    hipDeviceptr_t stats = x ? x->stats : NULL, csum = x ? x->csum : NULL;
    i32 stats_cap = x ? x->stats_cap : 0;
    int rope = x && x->rope_cos;
    if (M <= 0 || N <= 0 || batch == 0) return 0;
    if (rope && (batch != 1 || x->rope_T <= 0 || x->rope_hd <= 0 || x->rope_hd % 4 || x->rope_cols % 4)) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: RoPE epilogue needs a single GEMM and head width a multiple of 4\n");
        _exit(1);
    }
    if (stats && (batch != 1 || beta != 0.0f || bias || resid || trans_a || !trans_b)) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: row statistics need a single NT GEMM (the LM head's) with no beta, "
                        "bias or residual\n");
        _exit(1);
    }
    if (x && (x->tgt || x->tgt_val || x->no_store) && (!stats || (x->tgt == NULL) != (x->tgt_val == NULL))) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: target values and no_store need row statistics (and both target buffers)\n");
        _exit(1);
    }
    if (x && x->glu_h) {
        /* the SwiGLU epilogue: one fixed kernel, so only the shapes it tiles exactly */
        if (trans_a || trans_b || batch != 1 || beta != 0.0f || resid || stats || csum || rope || fixed_ws ||
            x->glu_F <= 0 || x->glu_F % 32 || N != 2 * x->glu_F || K <= 0 || K % 32 || !aligned16(A) ||
            !aligned16(B) || !aligned16(C) || !aligned16(x->glu_h) || lda % 4 || ldb % 4 || ldc % 4 ||
            (bias && !aligned16(bias))) {
            fprintf(stderr, "[HIP ERROR] trlm_gemm: the SwiGLU epilogue needs a single aligned NN GEMM, N = 2F with "
                            "F %% 32 == 0, K %% 32 == 0, no beta, residual or other epilogue\n");
            _exit(1);
        }
        GemmParams p;
        memset(&p, 0, sizeof(p));
        p.A = (const float*)A; p.B = (const float*)B; p.C = (float*)C; p.bias = (const float*)bias;
        p.M = M; p.N = N; p.K = K; p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.ldr = ldr;
        p.splits = 1; p.kchunk = K; p.alpha = alpha; p.beta = 0.0f;
        const Plan pl = make_glu_plan(M, x->glu_F, K, e->fp32);
        const int tile = pl.family == SMALL ? 32 : TILES[pl.tile].bm;
        p.tiles_m = cdiv(M, tile); p.tiles_n = cdiv(N, tile);
        p.glu_h = (float*)x->glu_h; p.glu_F = x->glu_F;
        plan_name(e->last, sizeof(e->last), &pl, L_NN, 1, 1);
        e->last_splits = 1;
        launch(pl.family == SMALL ? e->small_glu : pl.family == FP32 ? e->glu : pl.tile == T_128x128 ? e->xglu128
                                                                                                     : e->xglu, &p, 1);
        return 0;
    }
    if (csum && (batch != 1 || trans_b)) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: column sums need a single GEMM with B stored [K,N]\n");
        _exit(1);
    }
    if (M > (1 << 30) || N > (1 << 30) || K < 0) {
        fprintf(stderr, "[HIP ERROR] trlm_gemm: bad shape M=%d N=%d K=%d\n", M, N, K);
        _exit(1);
    }
    GemmParams p;
    memset(&p, 0, sizeof(p));
    p.A = (const float*)A; p.B = (const float*)B; p.C = (float*)C;
    p.bias = (const float*)bias; p.resid = (const float*)resid;
    p.sA = sA; p.sB = sB; p.sC = sC; p.sW = 0;
    p.M = M; p.N = N; p.K = K;
    p.lda = lda; p.ldb = ldb; p.ldc = ldc; p.ldr = ldr;
    p.splits = 1; p.kchunk = K > 0 ? K : 1;
    p.alpha = alpha; p.beta = beta;
    p.csum = (float*)csum;
    if (stats) {
        p.tgt = (const u32*)x->tgt;
        p.tgt_val = (float*)x->tgt_val;
        p.no_store = x->no_store != 0;
    }
    if (rope) {
        p.rope_cos = x->rope_cos; p.rope_sin = x->rope_sin;
        p.rope_T = x->rope_T; p.rope_hd = x->rope_hd; p.rope_cols = x->rope_cols;
    }

    int layout = trans_a ? (trans_b ? 3 : L_TN) : (trans_b ? L_NT : L_NN);
    int aligned = layout != 3 && aligned16(A) && aligned16(B) && (lda % 4 == 0) && (ldb % 4 == 0) &&
                  (batch == 1 || ((sA % 4 == 0) && (sB % 4 == 0)));
    /* split-K: raw partials into the workspace, then an ordered reduction;
     * with column sums each split's slab has one more row, M, for them */
    const u64 slab = ((u64)M + (csum ? 1u : 0u)) * (u64)N;
    /* row statistics and column sums are the fp32 kernels' */
    const PlanOpts o = { aligned, e->fp32 || stats || csum, stats != NULL, stats || rope, e->force_tile, e->force_splits, slab,
                         fixed_ws ? fixed_floats : ANY_ROOM };
    const Plan pl = make_plan(layout, M, N, K, batch, &o);
    const int tile = pl.tile, splits = pl.splits;
    plan_name(e->last, sizeof(e->last), &pl, layout, aligned, 0);
    e->last_splits = splits;
    if (pl.family == SMALL) {
        p.tiles_m = cdiv(M, 32); p.tiles_n = cdiv(N, 32);
        launch(e->small[!aligned][layout], &p, 1);
        return 0;
    }
    hipFunction_t kernel;
    if (!aligned) kernel = pl.family == FP32 ? e->ku[layout] : tile == T_128x128 ? e->xu128[layout] : e->xu[layout];
    else kernel = (pl.family == SPLIT ? e->x : e->k)[layout][tile];
    p.tiles_m = cdiv(M, TILES[tile].bm);
    p.tiles_n = cdiv(N, TILES[tile].bn);
    if (stats) set_stats(&p, stats, stats_cap, TILES[tile].bn);
    if (splits <= 1) {
        launch(kernel, &p, batch);
        return p.stats ? 2 * p.tiles_n : 0;
    }
    u64 need = (u64)splits * slab;
    hipDeviceptr_t W = fixed_ws;
    if (!fixed_ws) {
        if (need > e->ws_floats) {
            if (e->ws) hip_free(e->ws);
            e->ws = hip_alloc(need * sizeof(f32));
            e->ws_floats = need;
        }
        W = e->ws;
    }
    GemmParams q = p;
    q.C = (float*)W;
    q.ldc = N;
    q.sW = (long long)slab;
    q.kchunk = pl.kchunk;
    q.splits = splits;
    q.alpha = 1.0f; q.beta = 0.0f; q.bias = NULL; q.resid = NULL;
    launch(kernel, &q, (u32)splits);
    long long total = (long long)slab;
    i32 sp = splits;
    i64 sW = (i64)slab;
    void* args[] = { &W, &sp, &sW, &C, &M, &N, &ldc, &alpha, &beta, &bias, &resid, &ldr, &csum };
    /* four columns per thread when every row segment of four is 16-byte
     * aligned in each operand: same per-element order, same bits */
    const int vec4 = (N % 4) == 0 && (ldc % 4) == 0 && (!resid || (ldr % 4) == 0) &&
                     (((uintptr_t)W | (uintptr_t)C | (uintptr_t)bias | (uintptr_t)resid | (uintptr_t)csum) & 15u) == 0;
    if (vec4)
        hip_launch(e->reduce4, (u32)((total / 4 + 255) / 256), 1, 1, 256, 1, 1, 0, args);
    else
        hip_launch(e->reduce, (u32)((total + 255) / 256), 1, 1, 256, 1, 1, 0, args);
    return 0;
}

void trlm_timer_create(TrlmTimer* t) {
    hipEventCreate(&t->start);
    hipEventCreate(&t->stop);
}

void trlm_timer_destroy(TrlmTimer* t) {
    hipEventDestroy(t->start);
    hipEventDestroy(t->stop);
}

void trlm_timer_start(TrlmTimer* t) { hipEventRecord(t->start, hip_current_stream()); }

f32 trlm_timer_stop_ms(TrlmTimer* t) {
    float ms = 0.f;
    hipEventRecord(t->stop, hip_current_stream());
    hipEventSynchronize(t->stop);
    hipEventElapsedTime(&ms, t->start, t->stop);
    return ms;
}

const char* trlm_version(void) { return "trlm-mi355x 0.1 (gfx950, fp32 and split bf16 MFMA)"; }

u64 trlm_sizeof_gpu_trainer(void) { return (u64)sizeof(GpuTrainer); }
u64 trlm_sizeof_hip_ctx(void) { return (u64)sizeof(HipCtx); }
