// MoE layer of libw4a16hip.so: expert arenas, routing, slot alignment and the routed-expert FFN; and the launch of dense
// linears at a few dozen rows.
// Stands in for build_marlin_moe_arenas (w4a16_dec/upload.rs:1116-1235), moe_topk (w4a16_dec/mod.rs:168-185),
// moe_align_launch (moe/moe_align.rs:4-22) and marlin_moe_ffn_dev (kernels/marlin_moe.rs:290-422).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>

#include "w4a16_internal.h"

static inline unsigned ceil_div(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

// ------------------------------------------------------------------------------------------------ arenas
static void free_experts(w4a16_ctx* ctx, W4Experts& E) {
    (void)w4a16_free(ctx, E.q13);
    (void)w4a16_free(ctx, E.s13);
    (void)w4a16_free(ctx, E.q2);
    (void)w4a16_free(ctx, E.s2);
    E = W4Experts();
}

// Tile one projection of every expert: raw [n_exp][n][k/8] + [n_exp][n][k/group] on the host -> arena on the device.
static int tile_arena(w4a16_ctx* ctx, const void* q, const void* s, size_t n_exp, size_t n, size_t k, size_t group,
                      bool to_f16, uint64_t* q_arena, uint64_t* s_arena, size_t* q_stride, size_t* s_stride) {
    const size_t row_blocks = (n + 15) / 16, kt_n = k / 128, kg_n = k / group;
    const size_t q_raw_e = n * (k / 2), s_raw_e = n * kg_n * 2;
    *q_stride = row_blocks * kt_n * 1024;
    *s_stride = row_blocks * kg_n * 32;
    W4_TRY(w4a16_alloc(ctx, *q_stride * n_exp, q_arena));
    W4_TRY(w4a16_alloc(ctx, *s_stride * n_exp, s_arena));
    // stage the operands through a bounded device buffer, a few experts at a time
    const size_t per = std::max<size_t>(1, std::min<size_t>(n_exp, (size_t)(256u << 20) / (q_raw_e + s_raw_e)));
    uint64_t dq = 0, ds = 0;
    int rc = w4a16_alloc(ctx, per * q_raw_e, &dq);
    if (!rc) rc = w4a16_alloc(ctx, per * s_raw_e, &ds);
    for (size_t e0 = 0; e0 < n_exp && !rc; e0 += per) {
        const size_t cnt = std::min(per, n_exp - e0);
        rc = w4a16_h2d(ctx, dq, static_cast<const char*>(q) + e0 * q_raw_e, cnt * q_raw_e);
        if (!rc) rc = w4a16_h2d(ctx, ds, static_cast<const char*>(s) + e0 * s_raw_e, cnt * s_raw_e);
        for (size_t i = 0; i < cnt && !rc; i++) {
            uint64_t qr = dq + i * q_raw_e, sr = ds + i * s_raw_e;
            uint64_t qt = *q_arena + (e0 + i) * *q_stride, st = *s_arena + (e0 + i) * *s_stride;
            int ni = (int)n, ki = (int)k, rbi = (int)row_blocks, kgi = (int)kg_n;
            void* pq[] = {&qr, &qt, &ni, &ki, &rbi};
            rc = w4_launch(ctx, "w4a16_tile_q", ceil_div(*q_stride / 4, 256), 1, 256, 0, pq);
            void* ps[] = {&sr, &st, &ni, &kgi, &rbi};
            if (!rc) rc = w4_launch(ctx, to_f16 ? "w4a16_tile_s_f16" : "w4a16_tile_s", ceil_div(*s_stride / 2, 256), 1, 256, 0, ps);
        }
        if (!rc) rc = w4a16_sync(ctx);  // the staging buffer is reused by the next batch
    }
    const std::string keep = w4_err_save();
    (void)w4a16_free(ctx, dq);
    (void)w4a16_free(ctx, ds);
    if (rc) w4_err_restore(keep);
    return rc;
}

extern "C" int w4a16_upload_experts(w4a16_ctx* ctx, const char* name, size_t n_experts, const void* q13,
                                    size_t q13_bytes, const void* s13, size_t s13_bytes, const void* q2,
                                    size_t q2_bytes, const void* s2, size_t s2_bytes, size_t h, size_t n_ff,
                                    size_t group, int scale_bf16) {
    if (!ctx || !name || !q13 || !s13 || !q2 || !s2) return w4_fail(W4A16_ERR_ARG, "upload_experts: null argument");
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    if (group != 128 && group != 32)
        return w4_fail(W4A16_ERR_UNSUPPORTED, "upload_experts %s: unsupported group=%zu", name, group);
    if (n_experts == 0 || n_experts > 1024 || h == 0 || n_ff == 0 || h % 128 != 0 || n_ff % 128 != 0)
        return w4_fail(W4A16_ERR_SHAPE, "upload_experts %s: experts=%zu h=%zu n_ff=%zu (1..1024 experts, h and n_ff multiples of 128)",
                       name, n_experts, h, n_ff);
    if (q13_bytes != n_experts * 2 * n_ff * (h / 2) || s13_bytes != n_experts * 2 * n_ff * (h / group) * 2 ||
        q2_bytes != n_experts * h * (n_ff / 2) || s2_bytes != n_experts * h * (n_ff / group) * 2)
        return w4_fail(W4A16_ERR_SHAPE, "upload_experts %s: q13=%zu s13=%zu q2=%zu s2=%zu != experts%zu h%zu n_ff%zu g%zu contract",
                       name, q13_bytes, s13_bytes, q2_bytes, s2_bytes, n_experts, h, n_ff, group);
    if (2 * n_ff * (h / 2) >= 0x80000000ull || h * (n_ff / 2) >= 0x80000000ull)
        return w4_fail(W4A16_ERR_SHAPE, "upload_experts %s: one expert reaches 2 GiB", name);
    W4Experts E;
    E.n_exp = n_experts;
    E.h = h;
    E.n_ff = n_ff;
    E.group = group;
    E.scale_bf16 = scale_bf16 ? 1 : 0;
    auto all = [&](bool (*test)(const uint16_t*, size_t)) {
        return test(static_cast<const uint16_t*>(s13), s13_bytes / 2) && test(static_cast<const uint16_t*>(s2), s2_bytes / 2);
    };
    E.fold = scale_bf16 && group == 32 && all(w4_bf16_folds);  // the narrowest range: no further scan
    // the MFMA-tiled grouped kernels carry the running unit of the prefill kernel: they are taken only for arenas
    // whose every scale that kernel can divide by (the streaming kernels only multiply by scales and take any)
    E.scales_regular = E.fold || (w4_scales_regular(static_cast<const uint16_t*>(s13), s13_bytes / 2, scale_bf16) &&
                                  w4_scales_regular(static_cast<const uint16_t*>(s2), s2_bytes / 2, scale_bf16));
    // bf16 scales that f16 holds exactly are stored as f16: the f16 kernels read the same values without a conversion per scale
    const bool to_f16 = E.fold || (scale_bf16 && all(w4_bf16_fits_f16));
    E.tiled_bf16 = scale_bf16 && !to_f16;
    int rc = tile_arena(ctx, q13, s13, n_experts, 2 * n_ff, h, group, to_f16, &E.q13, &E.s13, &E.q13_stride, &E.s13_stride);
    if (!rc) rc = tile_arena(ctx, q2, s2, n_experts, h, n_ff, group, to_f16, &E.q2, &E.s2, &E.q2_stride, &E.s2_stride);
    if (rc) {
        const std::string keep = w4_err_save();
        free_experts(ctx, E);
        w4_err_restore(keep);
        return rc;
    }
    auto it = ctx->experts.find(name);
    if (it != ctx->experts.end()) free_experts(ctx, it->second);
    ctx->experts[name] = E;
    return 0;
}

static int find_experts(w4a16_ctx* ctx, const char* name, W4Experts** out) {
    if (!ctx || !name) return w4_fail(W4A16_ERR_ARG, "experts: null argument");
    auto it = ctx->experts.find(name);
    if (it == ctx->experts.end()) return w4_fail(W4A16_ERR_NOT_FOUND, "experts %s: not registered", name);
    *out = &it->second;
    return 0;
}

extern "C" int w4a16_experts_info(w4a16_ctx* ctx, const char* name, size_t* n_experts, size_t* h, size_t* n_ff,
                                  size_t* group, int* scale_bf16) {
    W4Experts* E = nullptr;
    W4_TRY(find_experts(ctx, name, &E));
    if (n_experts) *n_experts = E->n_exp;
    if (h) *h = E->h;
    if (n_ff) *n_ff = E->n_ff;
    if (group) *group = E->group;
    if (scale_bf16) *scale_bf16 = E->scale_bf16;
    return 0;
}

extern "C" int w4a16_experts_dequant_dump(w4a16_ctx* ctx, const char* name, int which, size_t expert,
                                          uint64_t out_f32_dev) {
    W4Experts* E = nullptr;
    W4_TRY(find_experts(ctx, name, &E));
    if (!out_f32_dev || (which != 0 && which != 1) || expert >= E->n_exp)
        return w4_fail(W4A16_ERR_ARG, "experts_dequant_dump %s: which=%d expert=%zu", name, which, expert);
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    const size_t n = which == 0 ? 2 * E->n_ff : E->h, k = which == 0 ? E->h : E->n_ff;
    uint64_t qt = (which == 0 ? E->q13 + expert * E->q13_stride : E->q2 + expert * E->q2_stride);
    uint64_t st = (which == 0 ? E->s13 + expert * E->s13_stride : E->s2 + expert * E->s2_stride);
    int ni = (int)n, ki = (int)k, gi = (int)E->group, rbi = (int)((n + 15) / 16);
    void* p[] = {&qt, &st, &out_f32_dev, &ni, &ki, &gi, &rbi};
    return w4_launch(ctx, E->tiled_bf16 ? "w4a16_dump_tiled_bf16" : "w4a16_dump_tiled_f16",
                     ceil_div((size_t)rbi * (k / 128) * 256, 256), 1, 256, 0, p);
}

// ------------------------------------------------------------------------------------------------ routing
extern "C" int w4a16_moe_topk_host(const float* logits, size_t t, size_t n_exp, size_t top_k, int32_t* idx, float* w) {
    if (!logits || !idx || !w) return w4_fail(W4A16_ERR_ARG, "moe_topk: null argument");
    if (n_exp == 0 || top_k == 0 || top_k > n_exp)
        return w4_fail(W4A16_ERR_SHAPE, "moe_topk: n_exp=%zu top_k=%zu", n_exp, top_k);
    std::vector<float> p(n_exp);
    std::vector<char> taken(n_exp);
    for (size_t ti = 0; ti < t; ti++) {
        const float* l = logits + ti * n_exp;
        float mx = -INFINITY;
        for (size_t i = 0; i < n_exp; i++) mx = std::fmax(mx, l[i]);
        float sum = 0.0f;
        for (size_t i = 0; i < n_exp; i++) {
            p[i] = std::exp(l[i] - mx);
            sum += p[i];
        }
        for (size_t i = 0; i < n_exp; i++) p[i] /= sum;
        std::fill(taken.begin(), taken.end(), 0);
        float wsum = 0.0f;
        for (size_t r = 0; r < top_k; r++) {  // descending probability, ties to the lower index
            size_t best = n_exp;
            for (size_t i = 0; i < n_exp; i++)
                if (!taken[i] && (best == n_exp || p[i] > p[best])) best = i;
            taken[best] = 1;
            idx[ti * top_k + r] = (int32_t)best;
            wsum += p[best];
        }
        for (size_t r = 0; r < top_k; r++) w[ti * top_k + r] = p[(size_t)idx[ti * top_k + r]] / wsum;
    }
    return 0;
}

extern "C" int w4a16_moe_route(w4a16_ctx* ctx, uint64_t logits_dev, size_t t, size_t n_exp, size_t top_k,
                               uint64_t idx_dev, uint64_t wt_dev) {
    if (!ctx || !logits_dev || !idx_dev || !wt_dev) return w4_fail(W4A16_ERR_ARG, "moe_route: null argument");
    if (t == 0 || n_exp == 0 || n_exp > 1024 || top_k == 0 || top_k > 64 || top_k > n_exp || t > 0x7fffffffu / n_exp)
        return w4_fail(W4A16_ERR_SHAPE, "moe_route: t=%zu n_exp=%zu top_k=%zu (n_exp <= 1024, top_k <= min(64, n_exp))", t,
                       n_exp, top_k);
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    int ti = (int)t, ni = (int)n_exp, ki = (int)top_k;
    void* p[] = {&logits_dev, &idx_dev, &wt_dev, &ti, &ni, &ki};
    return w4_launch(ctx, "w4a16_moe_topk_t", ceil_div(t, 4), 1, 256, 0, p);
}

extern "C" int w4a16_moe_align(w4a16_ctx* ctx, uint64_t idx_dev, size_t ns, size_t n_exp, size_t block,
                               uint64_t sorted_dev, uint64_t expert_ids_dev, uint64_t num_post_dev) {
    if (!ctx || !idx_dev || !sorted_dev || !expert_ids_dev || !num_post_dev)
        return w4_fail(W4A16_ERR_ARG, "moe_align: null argument");
    if (ns == 0 || ns > 0x3fffffffu || n_exp == 0 || n_exp > 1024 || block == 0 || block > 1024)
        return w4_fail(W4A16_ERR_SHAPE, "moe_align: ns=%zu n_exp=%zu block=%zu", ns, n_exp, block);
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    int nsi = (int)ns, ni = (int)n_exp, bi = (int)block;
    // one workgroup per 2048 slots, at most 16 (each counts all slots; kernels/moe.hip).  LDS: 16 per-wave count rows,
    // totals, offsets and (several workgroups) slots ahead, one entry per expert each
    int wgs = (int)std::min<size_t>(16, (ns + 2047) / 2048);
    void* p[] = {&idx_dev, &nsi, &ni, &bi, &sorted_dev, &expert_ids_dev, &num_post_dev, &wgs};
    return w4_launch(ctx, wgs > 1 ? "w4a16_moe_align_wide" : "w4a16_moe_align", (unsigned)wgs, 1, 64 * kW4MoeAlignWaves,
                     (unsigned)((kW4MoeAlignWaves + (wgs > 1 ? 3 : 2)) * n_exp * 4), p);
}

// ------------------------------------------------------------------------------------------------ FFN
int w4_ensure(w4a16_ctx* ctx, uint64_t* buf, size_t* cap, size_t bytes) {
    if (bytes <= *cap) return 0;
    if (ctx->capturing)
        return w4_fail(W4A16_ERR_ARG, "a scratch buffer would grow to %zu bytes while the launch stream is capturing: run the sequence once before the capture", bytes);
    if (*buf) {
        W4_TRY(w4a16_sync(ctx));  // earlier launches may still read the old buffer
        ctx->scratch_gen++;       // graphs captured so far hold its address: w4a16_graph_launch refuses them from now on
    }
    (void)w4a16_free(ctx, *buf);
    *buf = 0;
    *cap = 0;
    W4_TRY(w4a16_alloc(ctx, bytes, buf));
    *cap = bytes;
    return 0;
}

// Segment size (slots of one expert per workgroup).  Up to 15 tokens (top_k <= 8) skip the alignment; otherwise up to 8
// tokens run the streaming kernel on 16-slot segments; beyond that the LDS-staged kernel, whose segment size follows
// the mean run per expert: 32 slots below a mean of 24, 48 below 40, else 64.  The reference picks the smallest of
// 16/32/48/64 that the mean run fills to under 90 % (kernels/marlin_moe.rs:309-315); measured here (128 experts,
// top-8, T = 16..1024) 32-slot segments beat 16-slot ones at every T, and the larger sizes win once most experts would
// need a second segment.
static size_t pick_block(size_t t, size_t ns, size_t n_exp, size_t top_k) {
    // direct mode (no alignment, two launches, see w4a16_moe_ffn): streams an expert once per token that chose it,
    // which still beats the two extra launches up to fifteen tokens (128 experts, top-8: 35.6 vs 52.9 us at t = 8,
    // 49.3 vs 61.3 us at t = 12, 62.9 vs 64.7 us at t = 15, level at t = 16, 79.3 vs 65.4 us at t = 20)
    if (t <= 15 && top_k <= 8) return 1;
    if (t <= 4) return 4;
    if (t <= 8) return 16;
    const double mean = (double)ns / (double)n_exp;
    return mean < 24.0 ? 32 : mean < 40.0 ? 48 : 64;
}

// What an expert launch makes of its scales: f16 (or bf16 kept as f16), bf16, folded (W4Experts::fold).
enum MoeScales { kMoeF16 = 0, kMoeBf16 = 1, kMoeFold = 2 };
static MoeScales moe_scales(const W4Experts& E) { return E.fold ? kMoeFold : E.tiled_bf16 ? kMoeBf16 : kMoeF16; }

// Every expert's run is padded to a multiple of block: at most ns / block full segments plus one partial per expert.
static size_t moe_max_segs(size_t ns, size_t block, size_t n_exp) { return std::min(ns, ns / block + n_exp); }

// Segment size of an expert FFN (1: the direct mode, no alignment), and whether its GEMMs are the MFMA-tiled kernels.
struct MoeRoute {
    size_t block;
    bool tiled;
};

static MoeRoute plan_moe_route(size_t t, size_t top_k, size_t n_exp, bool scales_regular, int block_pin, int tiled_pin) {
    const size_t ns = t * top_k;
    // Where 64-slot segments are mostly full the MFMA-tiled grouped kernel (one segment x 256 columns per workgroup, x through
    // LDS, 32x32x16 tiles) takes over from the streaming kernels.  Mean run per expert from which it wins: 68 slots (us per FFN,
    // streaming / tiled: group 32, 128 experts top-8 h 2048 n_ff 768, T = 850 163 / 160, T = 1024 201 / 184; 32 experts top-4
    // n_ff 1024 T = 512 80 / 83, T = 600 96 / 88; group 128, 64 experts top-6 n_ff 1408 T = 600 133 / 134, T = 700 155 / 152).
    // Folded scales gain there too, and earlier (128 experts, T = 768 129 / 124, T = 1024 174 / 156), but the tiled kernels' sums, one
    // chain of MFMAs over all of k, lie about twice as far from 64-bit sums as the streaming ones (k = 2048 2.2e-7 and 1.0e-7 of
    // their rms): the line stays.
    const bool tiled = tiled_pin > 0 || (tiled_pin == 0 && block_pin == 0 && scales_regular && ns >= 68 * n_exp);
    return {tiled ? 64 : block_pin ? (size_t)block_pin : pick_block(t, ns, n_exp, top_k), tiled};
}

// The build of one aligned expert GEMM: gate|up (glu) or down.
struct MoeBuild {
    char sym[80];
    int waves;  // per workgroup
    bool two;   // two k tiles per stage
};

static MoeBuild plan_moe_build(bool glu, size_t n_exp, size_t h, size_t n_ff, size_t group, MoeScales scales, size_t ns, size_t block, bool tiled,
                               int waves_pin, size_t cus) {
    const size_t n = glu ? 2 * n_ff : h, kt_n = (glu ? h : n_ff) / 128;
    const char *kind = glu ? "glu" : "lin", *fam = scales == kMoeBf16 ? "bf16" : "f16";
    MoeBuild P{{0}, waves_pin ? waves_pin : 4, false};
    if (tiled) {
        snprintf(P.sym, sizeof P.sym, "w4a16_moe_g%zu_%s_pf_%s", group, scales == kMoeFold ? "f16x" : fam, kind);
        return P;
    }
    if (block <= 16) {
        // in-block split-K: each wave needs at least one k tile
        P.waves = std::max(1, std::min(std::min(P.waves, 8), (int)kt_n));
        snprintf(P.sym, sizeof P.sym, "w4a16_moe_g%zu_%s_dec_%s_x%d", group, fam, kind, block <= 4 ? 1 : 4);
        return P;
    }
    P.waves = P.waves >= 8 ? 8 : 4;  // the x staging needs at least 4 waves
    const int tt = (int)(block / 16);
    const size_t row_blocks = (n + 15) / 16, units = glu ? row_blocks / 2 : (row_blocks + 1) / 2, waves = (size_t)P.waves;
    const size_t max_segs = moe_max_segs(ns, block, n_exp), wide = (units + waves - 1) / waves * waves;  // waves of a segment's workgroups
    // Two k tiles per stage (kernels/moe.hip) for runs of up to 32 slots, at group 128 where the launch has at most three workgroups
    // per CU: 8 experts T = 100 62.5 -> 54.6 us per FFN, 32 experts top-4 n_ff 1024 T = 40 33.3 -> 30.8; beyond, the LDS they
    // take costs more than the wait they hide (8 experts T = 256 91 / 101, 64 experts top-6 n_ff 1408 T = 24 57.4 / 59.9).  At group
    // 32 (f16 scales or bf16 kept as f16), whose tiles take longer to multiply, where one segment per expert gives at most one
    // workgroup per CU (folded / f16 scales, 128 or 256 of them: 4 experts h 4096 n_ff 3584 T = 16 51.6 -> 40.8 / 54.5 -> 43.4, 8 experts
    // n_ff 2048 T = 24 45.5 -> 39.1 / 45.9 -> 38.8, T = 100 47.9 -> 45.3 / 56.8 -> 57.2; 384: 12 experts T = 24 50.6 / 51.2, T = 100
    // 56.2 / 58.5 / 61.5 / 64.2).
    const size_t few = group == 128 ? max_segs * wide : scales == kMoeBf16 ? ~(size_t)0 : 3 * n_exp * wide;
    P.two = tt <= 3 && ns < 32 * n_exp && few <= 12 * cus;
    // Folded scales (compute_fold, kernels/moe.hip) from eight k tiles, below which folded sums are the less exact, and eight slots per
    // expert; in segments of two 16-slot blocks only where one segment per expert gives at most 20 waves per CU: the folded build
    // has registers for five waves per SIMD, the other for six (128 experts top-8 n_ff 768 T = 200 scaled / folded 77.2 / 83.4 us,
    // 64 experts top-6 n_ff 1408 T = 100 67.4 / 71.9; 32 experts top-4 n_ff 1024 T = 100 38.3 / 37.2, 8 experts n_ff 3584 T = 100 65.5 / 57.6).
    const bool fold = scales == kMoeFold && kt_n >= 8 && ns >= 8 * n_exp &&
                      (tt > 2 || n_exp * wide <= 20 * cus);
    snprintf(P.sym, sizeof P.sym, "w4a16_moe_g%zu_%s_mm_%s_t%d%s", group, fold ? "f16x" : fam, kind, tt, P.two ? "_k2" : "");
    return P;
}

static int launch_moe_gemm(w4a16_ctx* ctx, const W4Experts& E, bool glu, uint64_t x, size_t x_rows, size_t x_div,
                           uint64_t y, int y_f16, uint64_t topw, size_t ns, size_t block, size_t max_segs,
                           uint64_t sorted, uint64_t eids, uint64_t npost, bool tiled = false) {
    const size_t n = glu ? 2 * E.n_ff : E.h, k = glu ? E.h : E.n_ff;
    const size_t row_blocks = (n + 15) / 16;
    const size_t units = glu ? row_blocks / 2 : (row_blocks + 1) / 2;
    if (x_rows * k * 2 >= 0x80000000ull)
        return w4_fail(W4A16_ERR_SHAPE, "moe: activations reach 2 GiB, beyond the buffer-descriptor range");
    uint64_t qa = glu ? E.q13 : E.q2, sa = glu ? E.s13 : E.s2;
    unsigned long long qs = glu ? E.q13_stride : E.q2_stride, ss = glu ? E.s13_stride : E.s2_stride;
    int xr = (int)x_rows, xd = (int)x_div, yf = y_f16, blk = (int)block, nsi = (int)ns, rbi = (int)row_blocks,
        ki = (int)k, ni = (int)n, nei = (int)E.n_exp;
    const MoeBuild P = plan_moe_build(glu, E.n_exp, E.h, E.n_ff, E.group, moe_scales(E), ns, block, tiled, ctx->moe_waves, (size_t)std::max(ctx->cu_count, 1));
    int waves = P.waves;
    int act_kind = ctx->moe_act_kind;  // read by the gate|up kernels only
    void* p[] = {&qa, &sa, &qs, &ss, &x, &xr, &xd, &y, &yf, &topw, &sorted, &eids, &npost, &blk, &nsi, &rbi, &ki, &ni, &nei,
                 &waves, &act_kind};
    if (tiled) {
        // MFMA-tiled grouped kernel (kernels/prefill.hip, MODE 1 / 2): block tile = one 64-slot segment x 256 columns
        // (gate|up: 128 gate + the 128 matching up columns); LDS = two x stages of 64 rows x 128 k, overlaid at the end by the
        // waves' padded f16 tiles, then slot ids and routing weights; rows always leave as f16
        if (block != 64) return w4_fail(W4A16_ERR_ARG, "moe: the tiled grouped kernel needs 64-slot segments (got %zu)", block);
        if (!y_f16) return w4_fail(W4A16_ERR_UNSUPPORTED, "moe: the tiled grouped kernel writes f16 rows only");
        const size_t cols = glu ? E.n_ff : n, per_tile = glu ? 128 : 256;
        const size_t blocks = (max_segs * ((cols + per_tile - 1) / per_tile) + 7) / 8 * 8;
        if (blocks > 0x7fffffffu) return w4_fail(W4A16_ERR_SHAPE, "moe: %zu segments exceed the grid", max_segs);
        return w4_launch(ctx, P.sym, (unsigned)blocks, 1, 256, kW4PfMoeIdsAt + 64 * 8, p);
    }
    if (block <= 16) {
        const unsigned shmem = waves > 1 ? (unsigned)(waves * 2 * 64 * 16) : 0;
        return w4_launch(ctx, P.sym, (unsigned)(max_segs * units), 1, (unsigned)(waves * 64), shmem, p);
    }
    const size_t blocks = max_segs * ((units + (size_t)waves - 1) / (size_t)waves);
    const unsigned shmem = (unsigned)((P.two ? 4 : 2) * block * 256);  // two stages of one or two x tiles of 128 k
    return w4_launch(ctx, P.sym, (unsigned)blocks, 1, (unsigned)(waves * 64), shmem, p);
}

// Launch plan of the 17..64-row kernel (kernels/mid.hip): waves along n and k of a workgroup, k slices across workgroups.
// Every shape gives the same bits for a given number of slices.  Units are pairs of row blocks, those of all segments of a launch
// beyond 64 rows.  Fitted to sweeps of every shape with cold weights (28 widths 512..28672, 20 k 2048..20480, t = 20..64, both
// groups: 1632 points, over which it loses 0.6 % to the best shape, 20 % at worst; 424 at 72..1024 rows, 1.1 %).  Against the
// kernel before this one it is slower by more than 2 % at 32 of 2944 shapes, 8 % at worst, and 32 % faster on average.  Figures:
// us, group 128, what it takes / the other.
//   * up to one unit per CU (n = 8192): a wave per unit and four along k, every unit's workgroup on a CU of its own
//     (5120 x 5120 t = 64 15.3, two units per workgroup 18.8);
//   * k slices of those where the CUs are many times the units, whose hand-over costs about 3 us: up to 64 units four, from a k
//     on that falls with the token blocks (1280 x 3584 t = 20 7.0 / 7.5 whole, 704 x 2560 t = 56 9.1 / 9.8), up to 32 with a
//     long k eight (512 x 17408 t = 40 11.2); up to 128 two, where the launch still is one workgroup per CU (2560 x 9216 t = 24
//     11.8 / 15.4 in eight slices of four units, 4096 x 17408 t = 24 19.7 / 22.0);
//   * else the lower price, in k tiles of a unit on the fullest CU.  k whole: a workgroup's start counts as 1.2 units (34816 x
//     5120 gated t = 64: five waves along n 34.5, four 49.2; 28672 x 4096: four 24.7, five 26.4).  Workgroups of four units
//     that walk k alone, where many of them share a CU (32 KiB of LDS at two token blocks, 48 at three, 64 at four: five, three,
//     two per CU, at least two to hide each other's latency): 7168 x 5120 t = 1024 93 / 110.  Those in k slices, all resident at once,
//     if the chip is not full without; their hand-over counts 55 and 4 for every unit and slice per CU.  13824 x 17408 t = 40
//     47.3 in four slices / 56.7 whole (eight are not resident: 58.8), t = 64 53.8 / 63.1; 9216 x 13312 t = 24 26.4 in eight /
//     33.9; 28672 x 20480 t = 56 97.7 in two / 110.  Between 129 and 256 units and 66..94 k tiles slices come up to 18 % too
//     early at two token blocks (4104 x 8448 t = 20 15.8 / 13.4 whole).
struct MidPlan {
    int wn = 1, wk = kW4MidParts;
    size_t nks = 1;
};

static MidPlan plan_mid(size_t units, size_t segs, size_t kt_n, size_t t, size_t cus, int ksplit, bool may_split) {
    const size_t u = units * segs * 256 / cus, tt = t <= 32 ? 2 : t <= 48 ? 3 : 4;  // units per 256 CUs; token blocks
    MidPlan P;
    if (may_split && ksplit > 0) {
        P.nks = std::max<size_t>(1, std::min(std::min<size_t>((size_t)ksplit, kW4MoeMaxKsplit), kt_n / 2));
        if (P.nks > 1 && u > 96) P.wn = 4, P.wk = 1;
        if (P.nks > 1) return P;
    }
    const bool slices = may_split && ksplit == 0;
    if (u <= 64) {
        if (slices && kt_n >= 18 && kt_n * tt >= 56) P.nks = u <= 32 && kt_n * tt >= 120 ? 8 : 4;
        return P;
    }
    if (u <= 128) {
        if (slices && u > 96 && tt == 4 && kt_n >= 80) return MidPlan{4, 1, 8};
        if (slices && kt_n * tt >= u + 4) P.nks = 2;
        return P;
    }
    double best = 1e30;
    auto take = [&](const MidPlan& c, double per_k_tile, double once) {
        const double cost = (double)kt_n * per_k_tile + once;
        if (cost < best) best = cost, P = c;
    };
    if (u <= 256) take(MidPlan{}, 2.1, 0.0);
    else
        for (const MidPlan& c : {MidPlan{2, 4, 1}, MidPlan{3, 4, 1}, MidPlan{4, 2, 1}, MidPlan{5, 2, 1}}) {
            const size_t wgs = (units + (size_t)c.wn - 1) / (size_t)c.wn * segs;
            take(c, (double)((wgs + cus - 1) / cus) * (c.wn + 1.2), 0.0);
        }
    for (size_t nks : {1, 2, 4, 8}) {
        if (nks > 1 && (!slices || kt_n < 2 * nks)) continue;
        const size_t per_cu = ((units + 3) / 4 * segs * nks + cus - 1) / cus, room = 10 / tt, gens = (per_cu + room - 1) / room;
        if (nks > 1 && gens > 1) continue;
        take(MidPlan{4, 1, nks}, (double)(gens * std::max<size_t>(2, std::min(per_cu, room))) * (nks > 1 ? 4.0 / (double)nks : 4.25),
             nks > 1 ? 55.0 + 4.0 * (double)(nks * u) / 256.0 : 0.0);
    }
    return P;
}

extern "C" int w4a16_plan_stream(size_t n, size_t k, size_t t, int cu_count, int glu, int* waves_n, int* waves_k, int* k_slices) {
    if (n == 0 || k == 0 || k % 128 != 0 || t == 0 || cu_count <= 0 || (glu && n % 32 != 0))
        return w4_fail(W4A16_ERR_ARG, "plan_stream: n=%zu k=%zu t=%zu cus=%d glu=%d", n, k, t, cu_count, glu);
    const size_t row_blocks = (n + 15) / 16, rows = t <= 32 ? 32 : t <= 48 ? 48 : 64;
    const MidPlan P = plan_mid(glu ? row_blocks / 2 : (row_blocks + 1) / 2, (t + rows - 1) / rows, k / 128, t, (size_t)cu_count, 0, !glu);
    if (waves_n) *waves_n = P.wn;
    if (waves_k) *waves_k = P.wk;
    if (k_slices) *k_slices = (int)P.nks;
    return 0;
}

// glu_act >= 0: the linear is a fused gate|up projection and y receives f16 [t][n/2] = act(gate) * up on the f32 sums; the
// gated launch never splits over k.
int w4_dense_mid(w4a16_ctx* ctx, const W4Lin& L, uint64_t x, uint64_t y, size_t t, int out_f16, int glu_act) {
    const bool glu = glu_act >= 0;
    if (!L.q_tiled) return w4_fail(W4A16_ERR_UNSUPPORTED, "stream: linear has no tiled copy (needs k %% 128 == 0)");
    if (t > 0x7fffffffu / 2) return w4_fail(W4A16_ERR_SHAPE, "stream: t=%zu too large", t);
    if (glu && L.n % 32 != 0) return w4_fail(W4A16_ERR_SHAPE, "stream glu: n=%zu must be a multiple of 32", L.n);
    // x is switched off row by row with an offset of 2 GiB; weights only by an empty descriptor, so they may fill all of its range
    if (t * L.k * 2 >= 0x80000000ull) return w4_fail(W4A16_ERR_SHAPE, "stream: x reaches 2 GiB, beyond the buffer-descriptor range");
    if (L.row_blocks * (L.k / 128) * 1024 > 0xffffffffull)
        return w4_fail(W4A16_ERR_SHAPE, "stream: tiled weights of 4 GiB or more exceed the buffer-descriptor range");
    const size_t units = glu ? L.row_blocks / 2 : (L.row_blocks + 1) / 2, cus = (size_t)std::max(ctx->cu_count, 1);
    const size_t tt = t <= 32 ? 2 : t <= 48 ? 3 : 4, segs = (t + 16 * tt - 1) / (16 * tt);
    const MidPlan P = plan_mid(units, segs, L.k / 128, t, cus, ctx->decode_ksplit, !glu);
    const size_t wn = (size_t)P.wn, wk = (size_t)P.wk, groups = (units + wn - 1) / wn, blocks = groups * segs;
    uint64_t ws = 0, tk = 0;
    if (P.nks > 1) {  // partial tiles and per-wave tickets, shared with the decode kernel
        const size_t ws_need = blocks * wn * 2 * tt * 1024 * P.nks, tk_need = blocks * wn * wk * 4;
        if (ws_need > 0xffffffffull) return w4_fail(W4A16_ERR_SHAPE, "stream: %zu bytes of partial tiles", ws_need);
        W4_TRY(w4_ensure(ctx, &ctx->decode_ws, &ctx->decode_ws_cap, ws_need));
        if (tk_need > ctx->decode_tickets_cap) {
            W4_TRY(w4_ensure(ctx, &ctx->decode_tickets, &ctx->decode_tickets_cap, std::max<size_t>(tk_need, 16384)));
            W4_TRY(w4a16_memset0(ctx, ctx->decode_tickets, ctx->decode_tickets_cap));
        }
        ws = ctx->decode_ws;
        tk = ctx->decode_tickets;
    }
    // At group 32 bf16 scales that fold (w4_bf16_folds) are multiplied into the weights (bf16x) where a slice has 24 k tiles or more,
    // else group sums are scaled.  Folded sums round once per k tile instead of once per group but inside the MFMAs as well, which
    // exact integer products do not: against 64-bit sums, folded / scaled, k = 2048 9.3e-8 / 8.5e-8, 3072 9.7e-8 / 9.9e-8, 5120
    // 1.05e-7 / 1.22e-7, 17408 in eight slices 1.10e-7 / 1.22e-7 but 8192 in four 1.04e-7 / 8.8e-8: below 24 k tiles the folded ones
    // are the less exact.
    const bool fold = L.fold && L.k / 128 >= 24 * P.nks;
    const char* fam = !L.scale_bf16 ? "f16" : fold ? "bf16x" : "bf16";
    char sym[64];
    snprintf(sym, sizeof sym, "w4a16_mid_g%zu_%s_t%zu_n%dk%d%s", L.group, fam, tt, P.wn, P.wk, glu ? "_glu" : "");
    // staged x (two buffers of unpadded rows; a lone wave along n: one of padded rows), overlaid by the groups' results; then,
    // where a wave sums several parts, its slot for the finished ones (kernels/mid.hip: XB, OB)
    const size_t xb = wk * 16 * tt * (wn > 1 ? 2 * 256 : 2 * (size_t)kW4MoeLdx), tiles = wk * wn * 2 * tt * 1024;
    const size_t shmem = std::max(xb, wk > 1 ? tiles : 0) + (P.wk < kW4MidParts ? tiles : 0);
    uint64_t qt = L.q_tiled, st = L.s_tiled;
    int row_blocks = (int)L.row_blocks, ki = (int)L.k, ni = (int)L.n, ti = (int)t, of = out_f16 ? 1 : 0, act = glu ? glu_act : 0,
        nksi = (int)P.nks, gp = (int)groups;
    void* params[] = {&qt, &st, &x, &y, &row_blocks, &ki, &ni, &ti, &of, &act, &ws, &tk, &nksi, &gp};
    return w4_launch(ctx, sym, (unsigned)blocks, (unsigned)P.nks, (unsigned)(wn * wk * 64), (unsigned)shmem, params);
}

// Direct mode for decode steps: no alignment pass.  The gate|up GEMM runs one segment per slot — the segment table is
// the identity, the expert table is idx itself, the "padded total" a constant no slot index reaches — and
// w4a16_moe_*_down_sum folds the down projection of a token's experts, the routing-weight multiply, the f16 rounding
// of c2 and the slot-order sum into one launch of top_k waves per block.  Experts chosen by several tokens are
// streamed once per token, which is cheaper than the two extra launches for a handful of tokens.
static int moe_ffn_direct(w4a16_ctx* ctx, const char* name, const W4Experts& E, uint64_t x_dev, uint64_t idx_dev,
                          uint64_t wt_dev, size_t t, size_t top_k, uint64_t y_dev) {
    if (top_k > 8) return w4_fail(W4A16_ERR_UNSUPPORTED, "moe_ffn %s: direct mode needs top_k <= 8 (got %zu)", name, top_k);
    const size_t ns = t * top_k;
    W4MoeScratch& S = ctx->moe;
    S.block = 1;
    S.sorted_len = S.expert_len = S.c2_len = 0;
    S.act_len = ns * E.n_ff * 2;
    W4_TRY(w4_ensure(ctx, &S.act, &S.act_cap, S.act_len));
    if (S.iota_cap < ns) {
        const size_t cap = std::max<size_t>(ns, 256);
        std::vector<int32_t> host(cap);
        for (size_t i = 0; i < cap; i++) host[i] = (int32_t)i;
        size_t bytes_cap = S.iota_cap * 4;
        W4_TRY(w4_ensure(ctx, &S.iota, &bytes_cap, cap * 4));
        W4_TRY(w4a16_h2d(ctx, S.iota, host.data(), cap * 4));
        S.iota_cap = cap;
    }
    if (!S.always) {
        const int32_t big[2] = {0x7fffffff, 0};
        W4_TRY(w4a16_alloc(ctx, 8, &S.always));
        W4_TRY(w4a16_h2d(ctx, S.always, big, 8));
    }
    // gate|up with the SiLU*up epilogue, one slot per segment
    W4_TRY(launch_moe_gemm(ctx, E, true, x_dev, t, top_k, S.act, 1, 0, ns, 1, ns, S.iota, idx_dev, S.always));
    // down + routing weight + f16 rounding + slot-order sum
    // units of one row block while units of two would leave CUs without a workgroup
    const size_t row_blocks = (E.h + 15) / 16;
    const size_t rbu = (ctx->moe_waves == 2 || (ctx->moe_waves == 0 && t * ((row_blocks + 1) / 2) < (size_t)std::max(ctx->cu_count, 1))) ? 1 : 2;
    const size_t units = (row_blocks + rbu - 1) / rbu;
    uint64_t qa = E.q2, sa = E.s2;
    unsigned long long qs = E.q2_stride, ss = E.s2_stride;
    int tk = (int)top_k, nsi = (int)ns, rbi = (int)row_blocks, ki = (int)E.n_ff, ni = (int)E.h, nei = (int)E.n_exp;
    void* p[] = {&qa, &sa, &qs, &ss, &S.act, &idx_dev, &wt_dev, &y_dev, &tk, &nsi, &rbi, &ki, &ni, &nei};
    char sym[80];
    snprintf(sym, sizeof sym, "w4a16_moe_g%zu_%s_down_sum%s", E.group, E.tiled_bf16 ? "bf16" : "f16", rbu == 1 ? "1" : "");
    return w4_launch(ctx, sym, (unsigned)(t * units), 1, (unsigned)(top_k * 64), (unsigned)(top_k * rbu * 64 * 16), p);
}

extern "C" int w4a16_plan_moe(size_t t, size_t top_k, size_t n_exp, size_t h, size_t n_ff, size_t group, int scales, int cu_count,
                              size_t* segment, char* gate_up, char* down, size_t cap) {
    if (t == 0 || top_k == 0 || top_k > n_exp || t > 0x3fffffffu / top_k || h == 0 || n_ff == 0 || h % 128 != 0 || n_ff % 128 != 0 ||
        (group != 128 && group != 32) || scales < kMoeF16 || scales > kMoeFold || (scales == kMoeFold && group != 32) || cu_count <= 0 ||
        !segment || !gate_up || !down || cap < sizeof(MoeBuild::sym))
        return w4_fail(W4A16_ERR_ARG, "plan_moe: t=%zu top_k=%zu experts=%zu h=%zu n_ff=%zu group=%zu scales=%d cus=%d", t, top_k, n_exp, h, n_ff, group,
                       scales, cu_count);
    const MoeRoute R = plan_moe_route(t, top_k, n_exp, true, 0, 0);
    *segment = R.block;
    gate_up[0] = down[0] = 0;
    if (R.block == 1) return 0;
    for (bool glu : {true, false}) {
        const MoeBuild P = plan_moe_build(glu, n_exp, h, n_ff, group, (MoeScales)scales, t * top_k, R.block, R.tiled, 0, (size_t)cu_count);
        std::memcpy(glu ? gate_up : down, P.sym, sizeof P.sym);
    }
    return 0;
}

extern "C" int w4a16_moe_ffn(w4a16_ctx* ctx, const char* name, uint64_t x_dev, uint64_t idx_dev, uint64_t wt_dev,
                             size_t t, size_t top_k, uint64_t y_dev) {
    return w4a16_moe_ffn_act(ctx, name, x_dev, idx_dev, wt_dev, t, top_k, y_dev, W4A16_ACT_SILU);
}

extern "C" int w4a16_moe_ffn_act(w4a16_ctx* ctx, const char* name, uint64_t x_dev, uint64_t idx_dev, uint64_t wt_dev,
                                 size_t t, size_t top_k, uint64_t y_dev, int act) {
    W4Experts* E = nullptr;
    W4_TRY(find_experts(ctx, name, &E));
    if (!x_dev || !idx_dev || !wt_dev || !y_dev) return w4_fail(W4A16_ERR_ARG, "moe_ffn %s: null operand", name);
    if (act != W4A16_ACT_SILU && act != W4A16_ACT_GELU_TANH)
        return w4_fail(W4A16_ERR_ARG, "moe_ffn %s: activation %d (0 = silu, 1 = gelu, tanh form)", name, act);
    ctx->moe_act_kind = act;  // read by the gate|up launches of this call
    if (t == 0 || top_k == 0 || top_k > E->n_exp || t > 0x3fffffffu / top_k)
        return w4_fail(W4A16_ERR_SHAPE, "moe_ffn %s: t=%zu top_k=%zu experts=%zu", name, t, top_k, E->n_exp);
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    const size_t ns = t * top_k;
    if (ctx->moe_tiled > 0 && !E->scales_regular)
        return w4_fail(W4A16_ERR_UNSUPPORTED, "moe_ffn %s: the MFMA-tiled grouped kernels were requested (set_moe_tiled 1) but the experts hold a zero, non-finite or out-of-range scale; the streaming kernels serve them", name);
    const MoeRoute R = plan_moe_route(t, top_k, E->n_exp, E->scales_regular, ctx->moe_block, ctx->moe_tiled);
    const bool tiled = R.tiled;
    const size_t block = R.block;
    if (block != 1 && block != 4 && block != 16 && block != 32 && block != 48 && block != 64)
        return w4_fail(W4A16_ERR_ARG, "moe_ffn %s: segment size %zu not in {1,4,16,32,48,64}", name, block);
    if (block == 1) return moe_ffn_direct(ctx, name, *E, x_dev, idx_dev, wt_dev, t, top_k, y_dev);
    const size_t max_segs = moe_max_segs(ns, block, E->n_exp);
    W4MoeScratch& S = ctx->moe;
    S.block = block;
    S.sorted_len = (ns + E->n_exp * block) * 4;
    S.expert_len = (ns / block + E->n_exp + 1) * 4;
    S.act_len = ns * E->n_ff * 2;
    S.c2_len = ns * E->h * 2;
    W4_TRY(w4_ensure(ctx, &S.sorted, &S.sorted_cap, S.sorted_len));
    W4_TRY(w4_ensure(ctx, &S.expert_ids, &S.expert_cap, S.expert_len));
    size_t np_cap = S.num_post ? 8 : 0;
    W4_TRY(w4_ensure(ctx, &S.num_post, &np_cap, 8));
    W4_TRY(w4_ensure(ctx, &S.act, &S.act_cap, S.act_len));
    W4_TRY(w4_ensure(ctx, &S.c2, &S.c2_cap, S.c2_len));
    W4_TRY(w4a16_moe_align(ctx, idx_dev, ns, E->n_exp, block, S.sorted, S.expert_ids, S.num_post));
    // gate|up with the SiLU*up epilogue: slot j reads token j / top_k
    W4_TRY(launch_moe_gemm(ctx, *E, true, x_dev, t, top_k, S.act, 1, 0, ns, block, max_segs, S.sorted, S.expert_ids,
                           S.num_post, tiled));
    // down, multiplied by the routing weight: slot j reads act row j
    W4_TRY(launch_moe_gemm(ctx, *E, false, S.act, ns, 1, S.c2, 1, wt_dev, ns, block, max_segs, S.sorted, S.expert_ids,
                           S.num_post, tiled));
    int ti = (int)t, hi = (int)E->h, ki = (int)top_k;
    void* p[] = {&S.c2, &y_dev, &ti, &hi, &ki};
    return w4_launch(ctx, "w4a16_moe_topk_sum_f16", std::min<unsigned>(ceil_div(t * E->h / (E->h % 8 == 0 ? 8 : 1), 256), 4096), 1, 256, 0, p);
}

extern "C" int w4a16_moe_scratch(w4a16_ctx* ctx, int which, uint64_t* dptr, size_t* bytes, size_t* block) {
    if (!ctx || !dptr || !bytes) return w4_fail(W4A16_ERR_ARG, "moe_scratch: null argument");
    const W4MoeScratch& S = ctx->moe;
    switch (which) {
        case 0: *dptr = S.sorted; *bytes = S.sorted_len; break;
        case 1: *dptr = S.expert_ids; *bytes = S.expert_len; break;
        case 2: *dptr = S.num_post; *bytes = S.num_post ? 8 : 0; break;
        case 3: *dptr = S.act; *bytes = S.act_len; break;
        case 4: *dptr = S.c2; *bytes = S.c2_len; break;
        default: return w4_fail(W4A16_ERR_ARG, "moe_scratch: which=%d outside 0..4", which);
    }
    if (!*dptr) return w4_fail(W4A16_ERR_NOT_FOUND, "moe_scratch: no MoE call has run on this context");
    if (block) *block = S.block;
    return 0;
}

extern "C" int w4a16_set_moe_shape(w4a16_ctx* ctx, int block, int waves) {
    if (!ctx) return w4_fail(W4A16_ERR_ARG, "set_moe_shape: null context");
    if ((block != 0 && block != 1 && block != 4 && block != 16 && block != 32 && block != 48 && block != 64) || waves < 0 ||
        waves > 8)
        return w4_fail(W4A16_ERR_ARG, "set_moe_shape: block in {0,1,4,16,32,48,64}, waves in 0..8");
    ctx->moe_block = block;
    ctx->moe_waves = waves;
    return 0;
}

extern "C" int w4a16_set_moe_tiled(w4a16_ctx* ctx, int mode) {
    if (!ctx) return w4_fail(W4A16_ERR_ARG, "set_moe_tiled: null context");
    if (mode < -1 || mode > 1) return w4_fail(W4A16_ERR_ARG, "set_moe_tiled: -1 = never, 0 = automatic, 1 = always");
    ctx->moe_tiled = mode;
    return 0;
}

extern "C" int w4a16_bench_moe(w4a16_ctx* ctx, const char* const* names, size_t n_names, uint64_t x_dev,
                               uint64_t idx_dev, uint64_t wt_dev, size_t t, size_t top_k, uint64_t y_dev, size_t warmup,
                               size_t reps, float* ms_events, double* ms_wall) {
    if (!ctx || !names || n_names == 0 || reps == 0) return w4_fail(W4A16_ERR_ARG, "bench_moe: null argument");
    W4_TRY(w4_hip(hipSetDevice(ctx->device), "hipSetDevice"));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    W4_TRY(w4_hip(hipEventCreate(&e0), "hipEventCreate"));
    int rc = w4_hip(hipEventCreate(&e1), "hipEventCreate");
    for (size_t i = 0; i < warmup && !rc; i++)
        rc = w4a16_moe_ffn(ctx, names[i % n_names], x_dev, idx_dev, wt_dev, t, top_k, y_dev);
    if (!rc) rc = w4_hip(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    auto w0 = std::chrono::steady_clock::now();
    if (!rc) rc = w4_hip(hipEventRecord(e0, ctx->stream), "hipEventRecord");
    for (size_t i = 0; i < reps && !rc; i++)
        rc = w4a16_moe_ffn(ctx, names[(warmup + i) % n_names], x_dev, idx_dev, wt_dev, t, top_k, y_dev);
    if (!rc) rc = w4_hip(hipEventRecord(e1, ctx->stream), "hipEventRecord");
    if (!rc) rc = w4_hip(hipStreamSynchronize(ctx->stream), "hipStreamSynchronize");
    auto w1 = std::chrono::steady_clock::now();
    float ms = 0.f;
    if (!rc) rc = w4_hip(hipEventElapsedTime(&ms, e0, e1), "hipEventElapsedTime");
    if (ms_events) *ms_events = ms;
    if (ms_wall) *ms_wall = std::chrono::duration<double, std::milli>(w1 - w0).count();
    const std::string keep = w4_err_save();
    (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (rc) w4_err_restore(keep);
    return rc;
}
