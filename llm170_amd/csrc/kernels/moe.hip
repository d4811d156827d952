// MoE expert FFN on W4A16 experts: routing, slot alignment, grouped/ragged expert GEMMs, top-k reduction.
// Role of the reference's route -> align -> grouped gate+up -> SiLU*up -> grouped down (x top-k weight) -> sum
// sequence (w4a16_dec/kernels/marlin_moe.rs:290-422 over assets/moe.cu:686-759, 860-908, 1599-1674 and the vendored
// grouped Marlin kernels), designed for CDNA4:
//   * a "slot" is one (token, chosen expert) pair, slot j = token * top_k + choice.  The align kernel sorts slots by
//     expert (stable) and pads every expert's run to a multiple of the segment size; a segment = up to BLK slots of
//     one expert.  Workgroups are numbered (segment, output-row group); segments past the padded total exit at once.
//   * expert weights live in one arena in the tiled layout of w4a16_common.hpp, experts at a fixed stride; the
//     gate and up projections are one fused matrix (rows 0..n_ff gate, n_ff..2 n_ff up; upload.rs:1116-1235).
//   * both regimes multiply on v_mfma_f32_16x16x32_f16 with weights as exact integers (A operand = one dword of the
//     64 lanes of a tile) and apply the group scale to the f32 group sum, like the dense decode kernel.
//       - moe_dec (segments of <= 4 or <= 16 slots, decode steps): HBM streaming, in-block split-K over the waves,
//         x gathered straight from global memory (one load + DPP row shifts for <= 4 slots);
//       - moe_mm (segments of 16..64 slots, prefill chunks): the waves of a block take different output rows of the
//         same segment and share the gathered x rows through LDS (LDS DMA, double buffered, one k tile per stage), so x
//         is fetched once per block instead of once per wave.
//   * decode steps of at most four tokens skip the alignment: the gate|up GEMM runs one segment per slot (segment table
//     = identity, expert table = idx itself) and moe_down_sum does the down projection of a token's experts, the
//     routing-weight multiply, the f16 rounding and the slot-order sum in one launch — two launches per FFN;
//   * GLU epilogue: a wave owns gate row block u and up row block u + n_ff/16, rounds both sums to f16 (the reference
//     materialises them as f16, moe.cu:1649-1660) and writes silu(g)*u as f16 — the intermediate never reaches
//     memory.  LIN epilogue: optional multiply by the slot's routing weight, f16 or f32 rows scattered by slot id.
//   * for group size 32 the four scale groups of a k tile come with ONE load per row block: lane c of each quad
//     fetches group c % 4 and v_mov_b32_dpp quad_perm broadcasts group w when MFMA w needs it.
#include <type_traits>

#include "w4a16_common.hpp"

template <int W>
__device__ __forceinline__ unsigned w4_quad_bcast(unsigned v) {
    return __builtin_amdgcn_update_dpp(0u, v, W * 0x55, 0xF, 0xF, true);
}

template <int SH>
__device__ __forceinline__ u4_t moe_row_shl(u4_t v) {
    u4_t r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = __builtin_amdgcn_update_dpp(0u, v[i], 0x100 + SH, 0xF, 0xF, true);
    return r;
}

// The four scales (rows 4q..4q+3 of the row block) of scale group W of the current k tile, as f32.
// s = the lane's b64 scale load: for G = 128 the tile's only group, for G = 32 group (lane % 4).
template <int G, bool SBF, int W>
__device__ __forceinline__ f4_t moe_scale4(u2_t s) {
    unsigned d0 = s[0], d1 = s[1];
    if (G == 32) {
        d0 = w4_quad_bcast<W>(d0);
        d1 = w4_quad_bcast<W>(d1);
    }
    f4_t r;
    r[0] = w4_scale_fast<SBF>(d0 & 0xFFFFu);
    r[1] = w4_scale_fast<SBF>(d0 >> 16);
    r[2] = w4_scale_fast<SBF>(d1 & 0xFFFFu);
    r[3] = w4_scale_fast<SBF>(d1 >> 16);
    return r;
}

__device__ __forceinline__ float moe_round_f16(float v) { return (float)(_Float16)v; }

// Epilogue of one 16 x 16 result tile pair for one token column.  a0/a1: the lane's four rows of row blocks 0/1 of
// the unit.  GLU: a0 = gate, a1 = up -> act[slot][u*16 + 4q + i] = f16(silu(f16(g)) * f16(u)).
// LIN: rows of row blocks rbA / rbB, scaled by wgt, as f16 or f32.
template <bool GLU>
__device__ __forceinline__ void moe_store(f4_t a0, f4_t a1, int slot, int q, int u, int rbA, int rbB, bool haveB,
                                          void* __restrict__ y, int y_f16, float wgt, int n, int act_kind) {
    if (GLU) {
        const int n_ff = n >> 1;
        h4_t o;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // gate and up are f16 tensors in the reference and are rounded first
            float v = w4_act_mul(moe_round_f16(a0[i]), moe_round_f16(a1[i]), act_kind);
            asm volatile("" : "+v"(v));  // the product is rounded to f32 before the f16 conversion
            o[i] = (_Float16)v;
        }
        *reinterpret_cast<h4_t*>(reinterpret_cast<_Float16*>(y) + (size_t)slot * n_ff + u * 16 + 4 * q) = o;
    } else {
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            if (rb == 1 && !haveB) break;
            const f4_t a = (rb == 0 ? a0 : a1) * wgt;
            const int row = (rb == 0 ? rbA : rbB) * 16 + 4 * q;
            if (y_f16) {
                _Float16* yo = reinterpret_cast<_Float16*>(y) + (size_t)slot * n + row;
                if (row + 3 < n) {
                    h4_t v = {(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3]};
                    *reinterpret_cast<h4_t*>(yo) = v;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (row + i < n) yo[i] = (_Float16)a[i];
                }
            } else {
                float* yo = reinterpret_cast<float*>(y) + (size_t)slot * n + row;
                if (row + 3 < n) {
                    *reinterpret_cast<f4_t*>(yo) = a;
                } else {
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (row + i < n) yo[i] = a[i];
                }
            }
        }
    }
}

// Arguments shared by the two grouped kernels.
//   qa/sa: arena bases, expert e at qa + e*q_stride / sa + e*s_stride (bytes); each expert is row_blocks x k/128
//          tiles and [row_blocks][k/G][16] scales.  x: f16 [x_rows][k]; slot j reads row j / x_div.
//   y: GLU -> f16 [ns][n/2]; LIN -> f16 or f32 [ns][n].  topw: null or f32 [ns] (LIN only).
//   sorted_ids[seg*blk + i]: slot id or the sentinel ns; expert_ids[seg]; num_post[0] = padded slot total.
//   A segment whose expert id is outside 0..n_exp-1 is skipped (its slots stay unwritten).
//   act_kind (GLU only): 0 = silu(gate) * up (w4a16_moe_act_silu_f16), 1 = the tanh form of gelu on the gate
//   (w4a16_moe_act_gelu_f16, assets/moe.cu:1635-1647).
//   wpb: waves per block (the block size, as an argument: read from the dispatch packet it costs one more dependent
//   scalar-cache miss before the first weight load).
#define MOE_PARAMS                                                                                                  \
    const char *__restrict__ qa, const char *__restrict__ sa, unsigned long long q_stride,                          \
        unsigned long long s_stride, const uint16_t *__restrict__ x, int x_rows, int x_div, void *__restrict__ y,   \
        int y_f16, const float *__restrict__ topw, const int *__restrict__ sorted_ids,                              \
        const int *__restrict__ expert_ids, const int *__restrict__ num_post, int blk, int ns, int row_blocks, int k, \
        int n, int n_exp, int wpb, int act_kind
#define MOE_ARGS \
    qa, sa, q_stride, s_stride, x, x_rows, x_div, y, y_f16, topw, sorted_ids, expert_ids, num_post, blk, ns, row_blocks, k, n, n_exp, wpb, act_kind

// ---------------------------------------------------------------------------------------------------- moe_dec
template <int RB, int XL>
struct MoeDecStage {
    u4_t q[RB];
    u2_t s[RB];
    u4_t x[XL];
};

// One block = (segment, unit of two row blocks); its W waves split k.  XL = 1: blk <= 4; XL = 4: blk <= 16.
template <int G, bool SBF, bool GLU, int XL, int DEPTH>
__device__ __forceinline__ void moe_dec_body(MOE_PARAMS) {
    extern __shared__ f4_t red[];  // [W][2][64]
    constexpr int GPT = W4_TILE_K / G;
    constexpr int C = 4 / XL, TPL = 16 / C;
    const int lane = threadIdx.x & 63, W = wpb;
    // every kernel argument is fetched here, in one batch: left to the compiler they arrive in three dependent
    // scalar-cache misses spread over the prologue, each ahead of the first weight load
    asm volatile("" ::"s"(qa), "s"(sa), "s"(q_stride), "s"(s_stride), "s"(x), "s"(x_rows), "s"(x_div), "s"(y), "s"(topw),
                 "s"(sorted_ids), "s"(blk), "s"(ns), "s"(row_blocks), "s"(k), "s"(n),
                 "s"(n_exp), "s"(wpb));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int units = GLU ? row_blocks >> 1 : (row_blocks + 1) >> 1;
    const int seg = blockIdx.x / units, u = blockIdx.x % units;
    const int m = lane & 15, g = lane >> 4;
    const int xtok = m % TPL, xchunk = m / TPL;
    // The three table reads (padded total, the segment's expert, the lane's slot id) are issued together, ahead of
    // the tests that use them: one memory round trip before the first weight load instead of three.  The tables hold
    // an entry for every segment the grid was sized for.
    int np = num_post[0], e = expert_ids[seg], xslot = sorted_ids[seg * blk + min(xtok, blk - 1)];
    asm volatile("" : "+s"(np), "+s"(e), "+v"(xslot));
    if (seg * blk >= np) return;
    if ((unsigned)e >= (unsigned)n_exp) return;  // uniform for the block
    if (xtok >= blk) xslot = ns;
    const int kt_n = k / W4_TILE_K, kg_n = kt_n * GPT;
    const int kt0 = (kt_n * wave) / W, kt1 = (kt_n * (wave + 1)) / W;
    const int rbA = GLU ? u : 2 * u, rbB = GLU ? u + units : min(2 * u + 1, row_blocks - 1);
    const bool haveB = GLU || 2 * u + 1 < row_blocks;

    const __amdgpu_buffer_rsrc_t qr =
        w4_make_rsrc(qa + (unsigned long long)e * q_stride, (unsigned)row_blocks * (unsigned)kt_n * 1024u);
    const __amdgpu_buffer_rsrc_t sr =
        w4_make_rsrc(sa + (unsigned long long)e * s_stride, (unsigned)row_blocks * (unsigned)kg_n * 32u);
    const __amdgpu_buffer_rsrc_t xr = w4_make_rsrc(x, (unsigned)x_rows * (unsigned)k * 2u);

    const unsigned xoff =
        xslot < ns ? ((unsigned)(xslot / x_div) * (unsigned)k + (unsigned)(xchunk * 32 + g * 8)) * 2u : W4_OOB;
    const unsigned qoff[2] = {(unsigned)rbA * (unsigned)kt_n * 1024u + (unsigned)lane * 16u,
                              (unsigned)rbB * (unsigned)kt_n * 1024u + (unsigned)lane * 16u};
    // scale load: G = 128 -> the tile's group; G = 32 -> group (lane % 4) of the tile's four
    const unsigned sg = G == 32 ? (unsigned)(lane & 3) * 32u : 0u;
    const unsigned soff[2] = {(unsigned)rbA * (unsigned)kg_n * 32u + sg + (unsigned)g * 8u,
                              (unsigned)rbB * (unsigned)kg_n * 32u + sg + (unsigned)g * 8u};
    f4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};

    MoeDecStage<2, XL> stage[DEPTH];
    auto load = [&](MoeDecStage<2, XL>& s_, int kt) {
        const bool live = kt < kt1;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
            s_.q[rb] = __builtin_amdgcn_raw_buffer_load_b128(qr, live ? qoff[rb] + (unsigned)kt * 1024u : W4_OOB, 0, 2);
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
            s_.s[rb] = __builtin_amdgcn_raw_buffer_load_b64(sr, live ? soff[rb] + (unsigned)kt * (GPT * 32u) : W4_OOB, 0, 0);
#pragma unroll
        for (int l = 0; l < XL; l++)
            s_.x[l] = __builtin_amdgcn_raw_buffer_load_b128(
                xr, live ? xoff + (unsigned)(kt * W4_TILE_K + l * C * 32) * 2u : W4_OOB, 0, 0);
    };
    auto compute = [&](const MoeDecStage<2, XL>& s_) {
        u4_t xb[4];
#pragma unroll
        for (int l = 0; l < XL; l++) {
            xb[l * C] = s_.x[l];
            if (C == 4) {
                xb[1] = moe_row_shl<TPL>(s_.x[l]);
                xb[2] = moe_row_shl<2 * TPL>(s_.x[l]);
                xb[3] = moe_row_shl<3 * TPL>(s_.x[l]);
            }
        }
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            const f4_t zero = {0.f, 0.f, 0.f, 0.f};
            if (G == 128) {
                f4_t part = zero;
#pragma unroll
                for (int w = 0; w < 4; w++)
                    part = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][w]),
                                                                  __builtin_bit_cast(h8_t, xb[w]), part, 0, 0, 0);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 0>(s_.s[rb]), part, acc[rb]);
            } else {
                f4_t p0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][0]), __builtin_bit_cast(h8_t, xb[0]), zero, 0, 0, 0);
                f4_t p1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][1]), __builtin_bit_cast(h8_t, xb[1]), zero, 0, 0, 0);
                f4_t p2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][2]), __builtin_bit_cast(h8_t, xb[2]), zero, 0, 0, 0);
                f4_t p3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][3]), __builtin_bit_cast(h8_t, xb[3]), zero, 0, 0, 0);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 0>(s_.s[rb]), p0, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 1>(s_.s[rb]), p1, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 2>(s_.s[rb]), p2, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 3>(s_.s[rb]), p3, acc[rb]);
            }
        }
    };

    // counted loop: round -1 fills the ring with compute skipped, so the loads outstanding at every stage's wait are
    // in ring order (see the dense decode kernel)
    const int tiles = kt1 - kt0;
    const int rounds = tiles / DEPTH;
    for (int r = -1; r < rounds; r++) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            __builtin_amdgcn_s_setprio(1);  // compute ahead of the waves that are queueing loads (1-2 % at T <= 4)
            if (r >= 0) compute(stage[d]);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            load(stage[d], kt0 + (r + 1) * DEPTH + d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        if (rounds * DEPTH + d < tiles) compute(stage[d]);

    if (W > 1) {
        if (wave != 0) {
            red[(wave * 2 + 0) * 64 + lane] = acc[0];
            red[(wave * 2 + 1) * 64 + lane] = acc[1];
        }
        __syncthreads();
        if (wave != 0) return;
        for (int w = 1; w < W; w++) {
            acc[0] += red[(w * 2 + 0) * 64 + lane];
            acc[1] += red[(w * 2 + 1) * 64 + lane];
        }
    }
    const int slot = m < blk ? sorted_ids[seg * blk + m] : ns;
    if (slot >= ns) return;
    const float wgt = (!GLU && topw) ? topw[slot] : 1.0f;
    moe_store<GLU>(acc[0], acc[1], slot, g, u, rbA, rbB, haveB, y, y_f16, wgt, n, act_kind);
}

// ---------------------------------------------------------------------------------------------------- moe_down_sum
// Decode steps (a handful of tokens): the down projection of all of a token's experts and the slot-order sum in one
// launch.  One block = (token, unit of two row blocks); wave w < top_k owns slot token*top_k + w: it streams that
// expert's rows over the whole k range with the slot's activation row as x, multiplies by the routing weight and
// rounds to f16 exactly as the staged path materialises c2; wave 0 then adds the waves' values in slot order in f32
// (the same order as the separate sum kernel) and writes y f32 [t][n].  No alignment pass is needed: the expert of
// a slot is read straight from idx.
// RB: row blocks of a workgroup's unit — 2, or 1 for a handful of tokens, when units of two leave most CUs without work.
template <int G, bool SBF, int DEPTH, int RB>
__device__ __forceinline__ void moe_down_sum_body(const char* __restrict__ qa, const char* __restrict__ sa,
                                                  unsigned long long q_stride, unsigned long long s_stride,
                                                  const uint16_t* __restrict__ act, const int* __restrict__ idx,
                                                  const float* __restrict__ topw, float* __restrict__ y, int top_k,
                                                  int ns, int row_blocks, int k, int n, int n_exp) {
    extern __shared__ f4_t red[];  // [top_k][RB][64]
    constexpr int GPT = W4_TILE_K / G;
    const int lane = threadIdx.x & 63;
    // every kernel argument is fetched here, in one batch (see moe_dec_body)
    asm volatile("" ::"s"(qa), "s"(sa), "s"(q_stride), "s"(s_stride), "s"(act), "s"(idx), "s"(topw), "s"(y), "s"(top_k),
                 "s"(ns), "s"(row_blocks), "s"(k), "s"(n), "s"(n_exp));
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int units = (row_blocks + RB - 1) / RB;
    const int token = blockIdx.x / units, u = blockIdx.x % units;
    const int slot = token * top_k + wave;
    const int e_raw = __builtin_amdgcn_readfirstlane(idx[slot]);
    const bool valid = (unsigned)e_raw < (unsigned)n_exp;  // an out-of-range expert id contributes zero
    const int e = valid ? e_raw : 0;
    const int kt_n = k / W4_TILE_K, kg_n = kt_n * GPT;
    const int m = lane & 15, g = lane >> 4;
    const int rbA = RB * u, rbB = min(RB * u + 1, row_blocks - 1);
    const bool haveB = RB == 2 && 2 * u + 1 < row_blocks;

    const __amdgpu_buffer_rsrc_t qr = w4_make_rsrc(qa + (unsigned long long)e * q_stride,
                                                   valid ? (unsigned)row_blocks * (unsigned)kt_n * 1024u : 0u);
    const __amdgpu_buffer_rsrc_t sr = w4_make_rsrc(sa + (unsigned long long)e * s_stride,
                                                   valid ? (unsigned)row_blocks * (unsigned)kg_n * 32u : 0u);
    const __amdgpu_buffer_rsrc_t xr = w4_make_rsrc(act, (unsigned)ns * (unsigned)k * 2u);
    // one x load per k tile: lane m = 4c fetches chunk c of the slot's row; DPP row shifts bring chunk c to column 0
    const unsigned xoff = (m & 3) == 0 ? ((unsigned)slot * (unsigned)k + (unsigned)((m >> 2) * 32 + g * 8)) * 2u : W4_OOB;
    const unsigned qoff[2] = {(unsigned)rbA * (unsigned)kt_n * 1024u + (unsigned)lane * 16u,
                              (unsigned)rbB * (unsigned)kt_n * 1024u + (unsigned)lane * 16u};
    const unsigned sg = G == 32 ? (unsigned)(lane & 3) * 32u : 0u;
    const unsigned soff[2] = {(unsigned)rbA * (unsigned)kg_n * 32u + sg + (unsigned)g * 8u,
                              (unsigned)rbB * (unsigned)kg_n * 32u + sg + (unsigned)g * 8u};
    f4_t acc[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) acc[rb] = (f4_t){0.f, 0.f, 0.f, 0.f};

    MoeDecStage<RB, 1> stage[DEPTH];
    auto load = [&](MoeDecStage<RB, 1>& s_, int kt) {
        const bool live = kt < kt_n;
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
            s_.q[rb] = __builtin_amdgcn_raw_buffer_load_b128(qr, live ? qoff[rb] + (unsigned)kt * 1024u : W4_OOB, 0, 2);
#pragma unroll
        for (int rb = 0; rb < RB; rb++)
            s_.s[rb] = __builtin_amdgcn_raw_buffer_load_b64(sr, live ? soff[rb] + (unsigned)kt * (GPT * 32u) : W4_OOB, 0, 0);
        s_.x[0] = __builtin_amdgcn_raw_buffer_load_b128(xr, live ? xoff + (unsigned)(kt * W4_TILE_K) * 2u : W4_OOB, 0, 0);
    };
    auto compute = [&](const MoeDecStage<RB, 1>& s_) {
        u4_t xb[4];
        xb[0] = s_.x[0];
        xb[1] = moe_row_shl<4>(s_.x[0]);
        xb[2] = moe_row_shl<8>(s_.x[0]);
        xb[3] = moe_row_shl<12>(s_.x[0]);
#pragma unroll
        for (int rb = 0; rb < RB; rb++) {
            const f4_t zero = {0.f, 0.f, 0.f, 0.f};
            if (G == 128) {
                f4_t part = zero;
#pragma unroll
                for (int w = 0; w < 4; w++)
                    part = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][w]),
                                                                  __builtin_bit_cast(h8_t, xb[w]), part, 0, 0, 0);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 0>(s_.s[rb]), part, acc[rb]);
            } else {
                f4_t p0 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][0]), __builtin_bit_cast(h8_t, xb[0]), zero, 0, 0, 0);
                f4_t p1 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][1]), __builtin_bit_cast(h8_t, xb[1]), zero, 0, 0, 0);
                f4_t p2 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][2]), __builtin_bit_cast(h8_t, xb[2]), zero, 0, 0, 0);
                f4_t p3 = __builtin_amdgcn_mfma_f32_16x16x32_f16(w4_deq8(s_.q[rb][3]), __builtin_bit_cast(h8_t, xb[3]), zero, 0, 0, 0);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 0>(s_.s[rb]), p0, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 1>(s_.s[rb]), p1, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 2>(s_.s[rb]), p2, acc[rb]);
                acc[rb] = w4_fma4(moe_scale4<G, SBF, 3>(s_.s[rb]), p3, acc[rb]);
            }
        }
    };
    const int rounds = kt_n / DEPTH;
    for (int r = -1; r < rounds; r++) {
#pragma unroll
        for (int d = 0; d < DEPTH; d++) {
            __builtin_amdgcn_s_setprio(1);  // compute ahead of the waves that are queueing loads (1-2 % at T <= 4)
            if (r >= 0) compute(stage[d]);
            __builtin_amdgcn_s_setprio(0);
            __builtin_amdgcn_sched_barrier(0);
            load(stage[d], (r + 1) * DEPTH + d);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH - 1; d++)
        if (rounds * DEPTH + d < kt_n) compute(stage[d]);

    // c2 of this slot: routing weight, one rounding to f16 (the value the staged path stores), back to f32
    const float wgt = topw[slot];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
#pragma unroll
        for (int i = 0; i < 4; i++) {
            // the product is rounded to f32 first, as where c2 is materialised (the compiler would otherwise fold the
            // multiply into the conversion, v_fma_mixlo_f16: one rounding of the exact product instead of two)
            float p = acc[rb][i] * wgt;
            asm volatile("" : "+v"(p));
            acc[rb][i] = moe_round_f16(p);
        }
        red[(wave * RB + rb) * 64 + lane] = acc[rb];
    }
    __syncthreads();
    if (wave != 0 || m != 0) return;
    f4_t sum[RB];
#pragma unroll
    for (int rb = 0; rb < RB; rb++) sum[rb] = (f4_t){0.f, 0.f, 0.f, 0.f};
    for (int w = 0; w < top_k; w++) {
#pragma unroll
        for (int rb = 0; rb < RB; rb++) sum[rb] += red[(w * RB + rb) * 64 + lane];
    }
#pragma unroll
    for (int rb = 0; rb < RB; rb++) {
        if (rb == 1 && !haveB) break;
        const int row = (rb == 0 ? rbA : rbB) * 16 + 4 * g;
        float* yo = y + (size_t)token * n + row;
        if (row + 3 < n) {
            *reinterpret_cast<f4_t*>(yo) = sum[rb];
        } else {
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (row + i < n) yo[i] = sum[rb][i];
        }
    }
}

#define MOE_DOWN_SUM_KERNEL(NAME, G, SBF, RB)                                                                     \
    extern "C" __global__ __launch_bounds__(512) void NAME(                                                       \
        const char* qa, const char* sa, unsigned long long q_stride, unsigned long long s_stride,                 \
        const uint16_t* act, const int* idx, const float* topw, float* y, int top_k, int ns, int row_blocks, int k, \
        int n, int n_exp) {                                                                                       \
        moe_down_sum_body<G, SBF, 3, RB>(qa, sa, q_stride, s_stride, act, idx, topw, y, top_k, ns, row_blocks, k, \
                                         n, n_exp);                                                               \
    }
MOE_DOWN_SUM_KERNEL(w4a16_moe_g32_f16_down_sum, 32, false, 2)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g32_bf16_down_sum, 32, true, 2)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g128_f16_down_sum, 128, false, 2)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g128_bf16_down_sum, 128, true, 2)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g32_f16_down_sum1, 32, false, 1)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g32_bf16_down_sum1, 32, true, 1)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g128_f16_down_sum1, 128, false, 1)
MOE_DOWN_SUM_KERNEL(w4a16_moe_g128_bf16_down_sum1, 128, true, 1)

// ---------------------------------------------------------------------------------------------------- moe_mm
template <int RB, bool FOLD>
struct MoeMmStage {
    u4_t q[RB];
    typename std::conditional<FOLD, unsigned, u2_t>::type s[RB];
};

// One block = (segment of blk = 16*TT slots, group of W units); wave w owns unit group*W + w over the whole k range.
// TT: the 16-slot blocks of the segment this workgroup multiplies (those that hold a slot).  KT: k tiles per stage.
template <int G, bool SBF, bool GLU, int TT, int KT, bool FOLD>
__device__ __forceinline__ void moe_mm_body(MOE_PARAMS) {
    extern __shared__ _Float16 xs[];  // [2][KT][16*TT][128]
    constexpr int GPT = W4_TILE_K / G;
    constexpr int ROWS = 16 * TT;
    const int tid = threadIdx.x, lane = tid & 63, W = wpb;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int units = GLU ? row_blocks >> 1 : (row_blocks + 1) >> 1;
    const int groups = (units + W - 1) / W;
    const int seg = blockIdx.x / groups, grp = blockIdx.x % groups;
    // the table reads (padded total, the segment's expert, this lane's slot ids) are issued together, ahead of the tests that
    // use them (see moe_dec_body); x load p of wave w brings rows 4 * (w + p * W) ..+3 of the segment, 16 lanes to a row
    int np = num_post[0], e = expert_ids[seg];
    int slot_of[TT];
#pragma unroll
    for (int p = 0; p < TT; p++) slot_of[p] = sorted_ids[seg * blk + min(4 * (wave + p * W) + (lane >> 4), ROWS - 1)];
    asm volatile("" : "+s"(np), "+s"(e));
#pragma unroll
    for (int p = 0; p < TT; p++) asm volatile("" : "+v"(slot_of[p]));
    if (seg * blk >= np) return;  // uniform for the block, before any barrier
    const int u_raw = grp * W + wave;
    const bool active = u_raw < units;  // a surplus wave repeats the last unit and stores nothing
    const int u = min(u_raw, units - 1);
    if ((unsigned)e >= (unsigned)n_exp) return;  // uniform for the block, before any barrier
    const int kt_n = k / W4_TILE_K, kg_n = kt_n * GPT;
    const int c = lane & 15, q = lane >> 4;
    const int rbA = GLU ? u : 2 * u, rbB = GLU ? u + units : min(2 * u + 1, row_blocks - 1);
    const bool haveB = GLU || 2 * u + 1 < row_blocks;

    const char* const qe = qa + (unsigned long long)e * q_stride;
    const char* const se = sa + (unsigned long long)e * s_stride;
    const unsigned q_bytes = (unsigned)row_blocks * (unsigned)kt_n * 1024u, s_bytes = (unsigned)row_blocks * (unsigned)kg_n * 32u;

    // x staging: one k tile of the segment's rows, gathered straight into LDS by DMA (no registers held), rows of 256 B whose
    // 16-byte chunks are swizzled, chunk p of row r at position p ^ (r & 15), so that the 16 rows of a B operand's read fall
    // into distinct banks.  W >= 4: at most TT loads per wave.
    unsigned xg_off[TT];
#pragma unroll
    for (int p = 0; p < TT; p++) {
        const int row = 4 * (wave + p * W) + q, slot = row < ROWS ? slot_of[p] : ns;
        xg_off[p] = slot < ns ? ((unsigned)(slot / x_div) * (unsigned)k + (unsigned)((c ^ (row & 15)) * 8)) * 2u : W4_OOB;
    }
    typedef __attribute__((address_space(3))) char lds_char_t;
    auto load_x = [&](int kt, int buf) {
        const __amdgpu_buffer_rsrc_t xr = w4_make_rsrc(x, kt < kt_n ? (unsigned)x_rows * (unsigned)k * 2u : 0u);
#pragma unroll
        for (int p = 0; p < TT; p++)
            if (wave + p * W < 4 * TT)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    xr, (__attribute__((address_space(3))) void*)((lds_char_t*)xs + (buf * ROWS + 4 * (wave + p * W)) * 256), 16, xg_off[p],
                    kt * (W4_TILE_K * 2), 0, 0);
    };
    unsigned x_get[4];  // halves: operand of MFMA w, row c of a 16-row block
#pragma unroll
    for (int w = 0; w < 4; w++) x_get[w] = (unsigned)(c * 128 + ((w * 4 + q) ^ c) * 8);

    const unsigned qoff[2] = {(unsigned)rbA * (unsigned)kt_n * 1024u + (unsigned)lane * 16u,
                              (unsigned)rbB * (unsigned)kt_n * 1024u + (unsigned)lane * 16u};
    // scales: the four rows of the lane's results (group 32: of group lane % 4); FOLD: one of the k tile's 64 per lane
    const unsigned sg = G == 32 ? (unsigned)(lane & 3) * 32u : 0u;
    const unsigned soff[2] = {FOLD ? (unsigned)rbA * (unsigned)kg_n * 32u + (unsigned)lane * 2u : (unsigned)rbA * (unsigned)kg_n * 32u + sg + (unsigned)q * 8u,
                              FOLD ? (unsigned)rbB * (unsigned)kg_n * 32u + (unsigned)lane * 2u : (unsigned)rbB * (unsigned)kg_n * 32u + sg + (unsigned)q * 8u};
    typedef MoeMmStage<2, FOLD> Stage;
    Stage stage[2][KT];
    auto load_w = [&](Stage& s_, int kt) {
        const bool live = kt < kt_n;
        const __amdgpu_buffer_rsrc_t qr = w4_make_rsrc(qe, live ? q_bytes : 0u), sr = w4_make_rsrc(se, live ? s_bytes : 0u);
#pragma unroll
        for (int rb = 0; rb < 2; rb++) s_.q[rb] = __builtin_amdgcn_raw_buffer_load_b128(qr, qoff[rb], kt * 1024, 2);
#pragma unroll
        for (int rb = 0; rb < 2; rb++) {
            if constexpr (FOLD) s_.s[rb] = __builtin_amdgcn_raw_buffer_load_b16(sr, soff[rb], kt * (GPT * 32), 0);
            else s_.s[rb] = __builtin_amdgcn_raw_buffer_load_b64(sr, soff[rb], kt * (GPT * 32), 0);
        }
    };

    f4_t acc[2][TT];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) acc[rb][tt] = (f4_t){0.f, 0.f, 0.f, 0.f};

    auto compute = [&](const auto& s_, int buf) {
        const _Float16* xb = xs + buf * (ROWS * 128);
        const f4_t zero = {0.f, 0.f, 0.f, 0.f};
        f4_t part[2][TT];
        auto step = [&](auto wc) {
            constexpr int w = decltype(wc)::value;
            h8_t b[TT];
#pragma unroll
            for (int tt = 0; tt < TT; tt++) b[tt] = *reinterpret_cast<const h8_t*>(xb + x_get[w] + tt * 16 * 128);
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                // G = 32 (segments of 64 slots only; smaller ones run compute32 below): every 32-k group's products are
                // scaled on their own, and left alone the compiler issues all 8 * TT MFMAs of a k tile into separate
                // result registers before the first scaled sum.  The empty asm statements pin the order group by group:
                // this group's unpack starts after the previous group's sums, so one group's results are live at a time.
                unsigned qw = s_.q[rb][w];
                if (G == 32) asm volatile("" : "+v"(qw));
                const h8_t a = w4_deq8(qw);
                if (G == 32) {
                    const f4_t sc = moe_scale4<G, SBF, w>(s_.s[rb]);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        acc[rb][tt] = w4_fma4(sc, __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[tt], zero, 0, 0, 0), acc[rb][tt]);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) asm volatile("" : "+v"(acc[rb][tt]));
                } else {
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        part[rb][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[tt], w == 0 ? zero : part[rb][tt], 0, 0, 0);
                }
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        if (G == 128) {
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                const f4_t sc = moe_scale4<G, SBF, 0>(s_.s[rb]);
#pragma unroll
                for (int tt = 0; tt < TT; tt++) acc[rb][tt] = w4_fma4(sc, part[rb][tt], acc[rb][tt]);
            }
        }
    };

    // Group size 32, up to three 16-slot blocks, software-pipelined by hand: a k tile is eight groups (32 k x one row
    // block), each TT MFMAs into fresh results, the scale conversion and 4 * TT scaled sums.  Issue order per group: its
    // MFMAs; then the NEXT group's unpack (and, when the 32-k chunk changes, the next B operands from LDS) while the
    // matrix pipe works; then this group's scaled sums; then the next group's MFMAs, whose operands are ready.  A wave
    // does not wait for its own MFMAs (the order "unpack, MFMAs, sums" group by group left 5-8 idle cycles after every
    // MFMA for the other waves to fill).  Scheduling barriers hold the phases in this order; one group's results are
    // live at a time.  128 experts, top-8: T = 64 77.6 -> 76.1 us, T = 512 117.9 -> 115.6 us; with four blocks the
    // extra registers cost a wave per SIMD (T = 1024 +2 %), so 64-slot segments keep the plain order.
    auto compute32 = [&](const auto& s_, int buf) {
        const _Float16* xb = xs + buf * (ROWS * 128);
        const f4_t zero = {0.f, 0.f, 0.f, 0.f};
        h8_t b[TT];
#pragma unroll
        for (int tt = 0; tt < TT; tt++) b[tt] = *reinterpret_cast<const h8_t*>(xb + x_get[0] + tt * 16 * 128);
        h8_t a = w4_deq8(s_.q[0][0]);
        auto group = [&](auto gc) {
            constexpr int g = decltype(gc)::value, w = g >> 1, rb = g & 1;
            f4_t p[TT];
#pragma unroll
            for (int tt = 0; tt < TT; tt++) p[tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[tt], zero, 0, 0, 0);
            if constexpr (TT == 1) asm volatile("" : "+v"(p[0]));
            if constexpr (TT == 2) asm volatile("" : "+v"(p[0]), "+v"(p[1]));
            if constexpr (TT == 3) asm volatile("" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]));
            if constexpr (TT == 4) asm volatile("" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (g < 7) {
                constexpr int w2 = (g + 1) >> 1, rb2 = (g + 1) & 1;
                if constexpr (w2 != w) {
#pragma unroll
                    for (int tt = 0; tt < TT; tt++) b[tt] = *reinterpret_cast<const h8_t*>(xb + x_get[w2] + tt * 16 * 128);
                }
                a = w4_deq8(s_.q[rb2][w2]);
                asm volatile("" : "+v"(a));
            }
            __builtin_amdgcn_sched_barrier(0);
            const f4_t sc = moe_scale4<G, SBF, w>(s_.s[rb]);
#pragma unroll
            for (int tt = 0; tt < TT; tt++) acc[rb][tt] = w4_fma4(sc, p[tt], acc[rb][tt]);
#pragma unroll
            for (int tt = 0; tt < TT; tt++) asm volatile("" : "+v"(acc[rb][tt]));
            __builtin_amdgcn_sched_barrier(0);
        };
        group(std::integral_constant<int, 0>{});
        group(std::integral_constant<int, 1>{});
        group(std::integral_constant<int, 2>{});
        group(std::integral_constant<int, 3>{});
        group(std::integral_constant<int, 4>{});
        group(std::integral_constant<int, 5>{});
        group(std::integral_constant<int, 6>{});
        group(std::integral_constant<int, 7>{});
    };

    // FOLD: scaled weights (w4_deq8_scaled); a k tile's four MFMAs are summed from zero and added once, so an accumulator rounds as often
    // as there are k tiles and not at every MFMA: at three 16-slot blocks a quarter of the vector ALU work of scaled group sums is gone.
    // A k tile is eight groups (32 k x one row block), issued like those of compute32: a group's MFMAs, then the next group's unpack,
    // the B operands of the next 32 k one group early (in the order the compiler finds by itself 128 experts top-8 take 74.2 instead
    // of 71.7 us per FFN at T = 64).  Mean distance from 64-bit sums over their rms, scaled group sums / MFMAs chained straight into the
    // accumulators / this: k = 512 0.67e-7 / - / 0.73e-7, 768 0.76e-7 / 1.32e-7 / 0.83e-7, 1024 0.90e-7 / 1.65e-7 / 0.80e-7, 2048
    // 1.09e-7 / 2.1e-7 / 0.93e-7, 3584 1.40e-7 / 2.7e-7 / 1.0e-7: below eight k tiles the launch keeps scaled sums.  us per FFN,
    // scaled / this (gate and up; down where it has eight k tiles): 128 experts top-8 n_ff 768 T = 517 114.4 / 109.2, T = 640 125.8 / 118.5;
    // 8 experts top-2 n_ff 3584 T = 64 62.1 / 56.4, T = 250 108.1 / 93.2; runs below eight slots per expert gain nothing (T = 64 71.4 / 71.7).
    auto compute_fold = [&](const auto& s_, int buf) {
        const _Float16* xb = xs + buf * (ROWS * 128);
        const f4_t zero = {0.f, 0.f, 0.f, 0.f};
        f4_t part[2][TT];
        unsigned sc[2][4];
        h8_t b[2][TT];
#pragma unroll
        for (int tt = 0; tt < TT; tt++) b[0][tt] = *reinterpret_cast<const h8_t*>(xb + x_get[0] + tt * 16 * 128);
#pragma unroll
        for (int rb = 0; rb < 2; rb++) w4_spread_groups(s_.s[rb], sc[rb]);
        h8_t a = w4_deq8_scaled(s_.q[0][0], sc[0][0]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 8; g++) {
            const int w = g >> 1, rb = g & 1;
            if (rb == 0 && w < 3) {
#pragma unroll
                for (int tt = 0; tt < TT; tt++) b[(w + 1) & 1][tt] = *reinterpret_cast<const h8_t*>(xb + x_get[w + 1] + tt * 16 * 128);
            }
#pragma unroll
            for (int tt = 0; tt < TT; tt++) part[rb][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[w & 1][tt], w == 0 ? zero : part[rb][tt], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if (g < 7) a = w4_deq8_scaled(s_.q[(g + 1) & 1][(g + 1) >> 1], sc[(g + 1) & 1][(g + 1) >> 1]);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) acc[rb][tt] += part[rb][tt];
    };

    // one stage ahead: its DMA and weights are issued ahead of this stage's MFMAs and waited for (vmcnt 0) at the barrier
    // that ends them.  Few registers, many waves: x in flight in registers and weights two (group 32) or four (group 128) tiles
    // ahead, the wait for x behind the youngest weights, were slower throughout (128 experts, us per FFN: group 32 f16 T = 64
    // 75.6 -> 70.7, T = 517 117 -> 113; group 128 T = 64 74.9 -> 67.4, T = 517 111.5 -> 98.5).
    auto load_stage = [&](int kt, int d) {  // out of range past the last tile: zeros, no traffic
#pragma unroll
        for (int j = 0; j < KT; j++) {
            load_x(kt + j, d * KT + j);
            load_w(stage[d][j], kt + j);
        }
    };
    load_stage(0, 0);
    w4_dma_barrier();
    for (int kt0 = 0; kt0 < kt_n; kt0 += 2 * KT) {
#pragma unroll
        for (int d = 0; d < 2; d++) {
            const int kt = kt0 + d * KT;
            load_stage(kt + KT, d ^ 1);
            __builtin_amdgcn_sched_barrier(0);
            // a wave that holds a landed tile issues ahead of the waves that are queueing loads (about 1 % at every T)
            __builtin_amdgcn_s_setprio(1);
#pragma unroll
            for (int j = 0; j < KT; j++)
                if (kt + j < kt_n) {
                    if constexpr (FOLD) compute_fold(stage[d][j], d * KT + j);
                    else if constexpr (G == 32 && TT <= 3) compute32(stage[d][j], d * KT + j);
                    else compute(stage[d][j], d * KT + j);
                }
            __builtin_amdgcn_s_setprio(0);
            w4_dma_barrier();
        }
    }

    if (!active) return;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        const int slot = sorted_ids[seg * blk + tt * 16 + c];
        if (slot >= ns) continue;
        const float wgt = (!GLU && topw) ? topw[slot] : 1.0f;
        moe_store<GLU>(acc[0][tt], acc[1][tt], slot, q, u, rbA, rbB, haveB, y, y_f16, wgt, n, act_kind);
    }
}

// A segment's slots are a prefix of it (the alignment pads an expert's run at its end), so the first slot of each
// 16-slot block tells whether the block holds any: the workgroup runs the body built for the blocks that do, and the
// MFMAs, scaled sums and x rows of all-padding blocks are never issued (128 experts, top-8, T = 512: runs of 32 +- 6
// slots in 48-slot segments, every other expert fills two blocks of three).
template <int G, bool SBF, bool GLU, int TT, int KT, bool FOLD>
__device__ __forceinline__ void moe_mm_entry(MOE_PARAMS) {
    const int units = GLU ? row_blocks >> 1 : (row_blocks + 1) >> 1;
    const int seg = blockIdx.x / ((units + wpb - 1) / wpb);
    int live = 1;
#pragma unroll
    for (int p = 1; p < TT; p++) live += sorted_ids[seg * blk + 16 * p] < ns ? 1 : 0;
    if (live == 1) moe_mm_body<G, SBF, GLU, 1, KT, FOLD>(MOE_ARGS);
    else if (TT == 2 || live == 2) moe_mm_body<G, SBF, GLU, 2, KT, FOLD>(MOE_ARGS);
    else if (TT == 3 || live == 3) moe_mm_body<G, SBF, GLU, TT >= 3 ? 3 : 2, KT, FOLD>(MOE_ARGS);
    else moe_mm_body<G, SBF, GLU, TT, KT, FOLD>(MOE_ARGS);
}

#define MOE_DEC_KERNEL(NAME, G, SBF, GLU, XL, DEPTH)                                  \
    extern "C" __global__ __launch_bounds__(512) void NAME(MOE_PARAMS) {              \
        moe_dec_body<G, SBF, GLU, XL, DEPTH>(MOE_ARGS);                               \
    }
#define MOE_MM_BUILD(NAME, G, SBF, GLU, TT, KT, FOLD)                                 \
    extern "C" __global__ __launch_bounds__(512) void NAME(MOE_PARAMS) {              \
        moe_mm_entry<G, SBF, GLU, TT, KT, FOLD>(MOE_ARGS);                            \
    }
#define MOE_MM_KERNEL(NAME, G, SBF, GLU, TT, KT) MOE_MM_BUILD(NAME, G, SBF, GLU, TT, KT, false)
// Ring depths of the streaming kernels, from sweeps on the 128-expert shape: the one-slot segments of the direct mode run
// best with two k tiles in flight per wave (T = 4..12: 9-11 % faster than four: fewer registers, more waves resident at
// once); so do the segments of up to 16 slots (5 % faster than three).
#define MOE_FAMILY(PFX, G, SBF)                             \
    MOE_DEC_KERNEL(PFX##_dec_glu_x1, G, SBF, true, 1, 2)     \
    MOE_DEC_KERNEL(PFX##_dec_glu_x4, G, SBF, true, 4, 2)     \
    MOE_DEC_KERNEL(PFX##_dec_lin_x1, G, SBF, false, 1, 2)    \
    MOE_DEC_KERNEL(PFX##_dec_lin_x4, G, SBF, false, 4, 2)    \
    MOE_MM_KERNEL(PFX##_mm_glu_t2, G, SBF, true, 2, 1)    \
    MOE_MM_KERNEL(PFX##_mm_glu_t3, G, SBF, true, 3, 1)    \
    MOE_MM_KERNEL(PFX##_mm_glu_t4, G, SBF, true, 4, 1)    \
    MOE_MM_KERNEL(PFX##_mm_lin_t2, G, SBF, false, 2, 1)   \
    MOE_MM_KERNEL(PFX##_mm_lin_t3, G, SBF, false, 3, 1)   \
    MOE_MM_KERNEL(PFX##_mm_lin_t4, G, SBF, false, 4, 1)

MOE_FAMILY(w4a16_moe_g32_f16, 32, false)
MOE_FAMILY(w4a16_moe_g32_bf16, 32, true)
MOE_FAMILY(w4a16_moe_g128_f16, 128, false)
MOE_FAMILY(w4a16_moe_g128_bf16, 128, true)

// Folded scales (f16x: arenas of bf16 scales kept as f16, W4Experts::fold)
#define MOE_MM_FOLD(PFX)                                    \
    MOE_MM_BUILD(PFX##_mm_glu_t2, 32, false, true, 2, 1, true)   \
    MOE_MM_BUILD(PFX##_mm_glu_t3, 32, false, true, 3, 1, true)   \
    MOE_MM_BUILD(PFX##_mm_glu_t4, 32, false, true, 4, 1, true)   \
    MOE_MM_BUILD(PFX##_mm_lin_t2, 32, false, false, 2, 1, true)  \
    MOE_MM_BUILD(PFX##_mm_lin_t3, 32, false, false, 3, 1, true)  \
    MOE_MM_BUILD(PFX##_mm_lin_t4, 32, false, false, 4, 1, true)
MOE_MM_FOLD(w4a16_moe_g32_f16x)

// Two k tiles per stage, for launches of few workgroups (the rule is at the launch, w4a16_moe.cc): one tile in flight per wave
// does not cover the trip to memory there.  Same sums in the same order.  Group 128, 8 experts top-2, h 4096, n_ff
// 3584, us per FFN, x and weights four tiles ahead in registers / one tile per stage / two: T = 16 52.5 / 57.8 / 49.2, T = 40
// 50.3 / 57.3 / 45.7, T = 100 57.8 / 62.5 / 54.6; four tiles per stage lose (51.1, 49.4, 71.3).  Group
// 32, folded bf16 / f16 scales, one tile / two: same shape T = 16 58.3 / 52.4 and 57.9 / 52.3, T = 100 66.0 / 63.4 and 69.3 / 67.6.
#define MOE_MM_KT2(PFX, G, SBF, FOLD)                              \
    MOE_MM_BUILD(PFX##_mm_glu_t2_k2, G, SBF, true, 2, 2, FOLD)     \
    MOE_MM_BUILD(PFX##_mm_glu_t3_k2, G, SBF, true, 3, 2, FOLD)     \
    MOE_MM_BUILD(PFX##_mm_lin_t2_k2, G, SBF, false, 2, 2, FOLD)    \
    MOE_MM_BUILD(PFX##_mm_lin_t3_k2, G, SBF, false, 3, 2, FOLD)
MOE_MM_KT2(w4a16_moe_g128_f16, 128, false, false)
MOE_MM_KT2(w4a16_moe_g128_bf16, 128, true, false)
MOE_MM_KT2(w4a16_moe_g32_f16, 32, false, false)
MOE_MM_KT2(w4a16_moe_g32_f16x, 32, false, true)

// ---------------------------------------------------------------------------------------------------- routing
// Routing rule of the reference (w4a16_dec/mod.rs:168-185, device counterpart assets/moe.cu:686-759): softmax over all
// experts, the k largest probabilities with ties to the lower index, weights renormalised by the selected sum.
// One wave per token, n <= 1024; the body is built for 2, 4 and 16 experts per lane (n <= 128, 256, 1024).  The kernel is
// a chain of dependent wave-wide steps and nothing else, so a selection round is kept short: the probability's bit
// pattern (monotone for non-negative floats; NaN of all ones held one lower) plus one is a 32-bit key, 0 for an absent or
// taken expert; a lane's largest key, six v_max_u32 with DPP operands and one lane read give the round's probability, and
// one ballot per expert of a lane, in index order, names the lowest index that holds it.  (Rounds on a 64-bit key with the index in its low half
// and shuffles through LDS, always 16 experts per lane: 6.9 us at one token and 8.9 at 2048, 128 experts, top-8; this form
// 2.8 and 3.4.)
template <int CTRL>
__device__ __forceinline__ unsigned topk_dpp_max(unsigned v) {
    const unsigned o = __builtin_amdgcn_update_dpp(0u, v, CTRL, 0xF, 0xF, true);  // lanes without a source read 0
    return o > v ? o : v;
}

template <int PER_LANE>
__device__ __forceinline__ void moe_topk_body(const float* __restrict__ logits, int* __restrict__ idx,
                                              float* __restrict__ wt, int n, int k) {
    const int lane = threadIdx.x & 63;
    float e[PER_LANE];
    float top = -INFINITY;
#pragma unroll
    for (int j = 0; j < PER_LANE; j++) {
        const int i = lane + 64 * j;
        e[j] = i < n ? logits[i] : -INFINITY;
    }
#pragma unroll
    for (int j = 0; j < PER_LANE; j++) top = fmaxf(top, e[j]);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off));
    float total = 0.f;
#pragma unroll
    for (int j = 0; j < PER_LANE; j++) {
        e[j] = lane + 64 * j < n ? expf(e[j] - top) : 0.f;
        total += e[j];  // lane-local sum in index order, then the butterfly (the host statement adds all in index order)
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) total += __shfl_xor(total, off);
    unsigned key[PER_LANE];
#pragma unroll
    for (int j = 0; j < PER_LANE; j++)
        key[j] = lane + 64 * j < n ? min(__builtin_bit_cast(unsigned, e[j] / total), 0xfffffffeu) + 1u : 0u;
    float chosen_sum = 0.f, kept = 0.f;  // lane r keeps the r-th chosen probability and expert (k <= 64)
    int kept_i = 0;
    for (int r = 0; r < k; r++) {
        unsigned best = key[0];
#pragma unroll
        for (int j = 1; j < PER_LANE; j++) best = key[j] > best ? key[j] : best;
        best = topk_dpp_max<0x111>(best);  // row_shr 1, 2, 4, 8: lane 15 of a row holds the row's maximum
        best = topk_dpp_max<0x112>(best);
        best = topk_dpp_max<0x114>(best);
        best = topk_dpp_max<0x118>(best);
        best = topk_dpp_max<0x142>(best);  // row_bcast 15, 31: lane 63 holds the wave's
        best = topk_dpp_max<0x143>(best);
        best = (unsigned)__builtin_amdgcn_readlane((int)best, 63);
        int at = 0;
#pragma unroll
        for (int j = PER_LANE - 1; j >= 0; j--) {  // the last that matches is the lowest j
            const unsigned long long hit = __ballot(key[j] == best);
            if (hit) at = 64 * j + __builtin_ctzll(hit);
        }
#pragma unroll
        for (int j = 0; j < PER_LANE; j++) key[j] = lane + 64 * j == at ? 0u : key[j];
        const float p = __builtin_bit_cast(float, best - 1u);
        kept = lane == r ? p : kept;
        kept_i = lane == r ? at : kept_i;
        chosen_sum += p;
    }
    if (lane < k) {
        idx[lane] = kept_i;
        wt[lane] = kept / chosen_sum;
    }
}

extern "C" __global__ __launch_bounds__(256) void w4a16_moe_topk_t(const float* __restrict__ lg, int* __restrict__ idx,
                                                                   float* __restrict__ wt, int t, int n, int k) {
    const int token = blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (token >= t) return;
    const float* const logits = lg + (size_t)token * n;
    int* const oi = idx + (size_t)token * k;
    float* const ow = wt + (size_t)token * k;
    if (n <= 128) moe_topk_body<2>(logits, oi, ow, n, k);
    else if (n <= 256) moe_topk_body<4>(logits, oi, ow, n, k);
    else moe_topk_body<16>(logits, oi, ow, n, k);
}

// Stable counting sort of slots by expert with every expert's run padded to a multiple of `block`
// (assets/moe.cu:860-908 + 1599-1633 in one launch).  Workgroups of 1024 threads, n_exp <= 1024.
//   sorted_ids: slot ids in expert order, padding = sentinel ns; expert_ids[b]: expert of segment b;
//   num_post[0] = padded total, num_post[1] = number of distinct experts hit.
// A workgroup owns a contiguous range of slots, its wave w the w-th chunk of it: per-wave counts, an exclusive prefix
// over the waves per expert, a two-level scan over the experts' padded counts, then every wave places its slots in
// order.  An out-of-range expert id is dropped (its slot is never placed).
// The placement (a ballot per bit of the expert id for every 64 slots) is what a launch spends its time on, so beyond
// 2048 slots it is spread over workgroups, about two steps of 64 slots per wave; each of them counts ALL slots (LDS atomics,
// a fraction of the placement's cost), which gives it the number of slots ahead of its range per expert and the totals
// without a second launch (128 experts: 4136 slots 7.4 -> 6.0 us, 16384 18.1 -> 7.6, 32768 32.7 -> 9.6).
#define MOE_ALIGN_WAVES 16
#define MOE_ALIGN_THREADS (64 * MOE_ALIGN_WAVES)
#define MOE_ALIGN_KEEP 4  // 64-slot steps of a wave whose expert ids stay in registers between the two passes
template <bool WIDE>
__device__ __forceinline__ void moe_align_body(const int* __restrict__ idx, int ns, int n_exp, int block,
                                               int* __restrict__ sorted_ids, int* __restrict__ expert_ids,
                                               int* __restrict__ num_post, int wgs) {
    extern __shared__ unsigned align_lds[];  // cnt[WAVES][n_exp] (per wave count, then the slots of the expert ahead
                                             // of the wave's), tot[n_exp], poff[n_exp], WIDE: pre[n_exp] (slots ahead of the range)
    unsigned* const cnt = align_lds;
    unsigned* const tot = cnt + MOE_ALIGN_WAVES * n_exp;
    unsigned* const poff = tot + n_exp;
    unsigned* const pre = poff + n_exp;
    __shared__ unsigned wsum[MOE_ALIGN_WAVES], whit[MOE_ALIGN_WAVES];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int i = tid; i < (MOE_ALIGN_WAVES + (WIDE ? 3 : 0)) * n_exp; i += MOE_ALIGN_THREADS) cnt[i] = 0;
    const int wg = WIDE ? (int)blockIdx.x : 0;
    if (!WIDE) wgs = 1;
    const int chunk = ((ns + wgs * MOE_ALIGN_WAVES * 64 - 1) / (wgs * MOE_ALIGN_WAVES * 64)) * 64;  // slots per wave, multiple of 64
    const int lo = wg * MOE_ALIGN_WAVES * chunk, hi = min(ns, lo + MOE_ALIGN_WAVES * chunk);  // this workgroup's slots
    const int j0 = lo + wave * chunk, steps = chunk / 64;
    int keep[MOE_ALIGN_KEEP];
#pragma unroll
    for (int s = 0; s < MOE_ALIGN_KEEP; s++) {
        const int j = j0 + s * 64 + lane;
        int e = (s < steps && j < ns) ? idx[j] : -1;
        keep[s] = (unsigned)e < (unsigned)n_exp ? e : -1;
    }
    auto expert_of = [&](int s) -> int {
        int e = -1;
#pragma unroll
        for (int i = 0; i < MOE_ALIGN_KEEP; i++)
            if (i == s) e = keep[i];
        if (s >= MOE_ALIGN_KEEP) {
            const int j = j0 + s * 64 + lane;
            e = j < ns ? idx[j] : -1;
            if ((unsigned)e >= (unsigned)n_exp) e = -1;
        }
        return e;
    };
    __syncthreads();
    for (int s = 0; s < steps; s++) {
        const int e = expert_of(s);
        if (e >= 0) atomicAdd(&cnt[wave * n_exp + e], 1u);
    }
    if (WIDE) {  // the other workgroups' slots, four loads in flight per thread
        for (int j = tid; j < ns; j += 4 * MOE_ALIGN_THREADS) {
            int e[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int ju = j + u * MOE_ALIGN_THREADS;
                e[u] = ju < ns && (ju < lo || ju >= hi) ? idx[ju] : -1;
            }
#pragma unroll
            for (int u = 0; u < 4; u++)
                if ((unsigned)e[u] < (unsigned)n_exp) atomicAdd(j + u * MOE_ALIGN_THREADS < lo ? &pre[e[u]] : &tot[e[u]], 1u);
        }
    }
    __syncthreads();
    // thread i owns expert i: total over the waves, then a scan of the padded totals over all threads
    unsigned padded = 0, hits = 0;
    {
        const int e = tid;
        unsigned run = 0;
        if (e < n_exp) {
            if (WIDE) run = pre[e];
            for (int w = 0; w < MOE_ALIGN_WAVES; w++) {
                const unsigned c = cnt[w * n_exp + e];
                cnt[w * n_exp + e] = run;
                run += c;
            }
            if (WIDE) run += tot[e];
            tot[e] = run;
        }
        padded = ((run + block - 1) / block) * block;
        hits = run != 0;
    }
    unsigned incl = padded, hincl = hits;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned v = __shfl_up(incl, off), hv = __shfl_up(hincl, off);
        if (lane >= off) {
            incl += v;
            hincl += hv;
        }
    }
    if (lane == 63) {
        wsum[wave] = incl;
        whit[wave] = hincl;
    }
    __syncthreads();
    unsigned base = 0, all = 0, allhit = 0;
#pragma unroll
    for (int w = 0; w < MOE_ALIGN_WAVES; w++) {
        if (w < wave) base += wsum[w];
        all += wsum[w];
        allhit += whit[w];
    }
    const unsigned pos0 = base + incl - padded;
    if (tid < n_exp) poff[tid] = pos0;
    // Padding sentinels.  A workgroup alone writes one to every position, coalesced, and places the slots over them after
    // the barrier (which waits for the stores issued before it, so the order of the two writes to a position is fixed);
    // several write the padding behind every expert's run only, after the barrier.
    if (!WIDE)
        for (unsigned p = tid; p < all; p += MOE_ALIGN_THREADS) sorted_ids[p] = ns;
    if (wg == 0) {
        if (tid < n_exp)
            for (unsigned b = 0; b < padded / block; b++) expert_ids[pos0 / block + b] = tid;
        if (tid == 0) {
            num_post[0] = (int)all;
            num_post[1] = (int)allhit;
        }
    }
    __syncthreads();
    // padding sentinels of several workgroups: eight threads to an expert, experts dealt to the workgroups
    for (int i = wg * MOE_ALIGN_THREADS + tid; WIDE && i < n_exp * 8; i += wgs * MOE_ALIGN_THREADS) {
        const unsigned n_e = tot[i >> 3], end = ((n_e + block - 1) / block) * block;
        for (unsigned p = n_e + (i & 7); p < end; p += 8) sorted_ids[poff[i >> 3] + p] = ns;
    }
    // placement in slot order: every wave walks its range 64 slots at a time; rank among equal experts in the step.
    // The wave's row of cnt is private to it and LDS operations of one wave execute in order, so the loop needs no
    // workgroup barrier; the wave-scope fences keep the compiler from reordering the LDS accesses.
    int nbits = 1;  // bits that tell experts 0..n_exp-1 apart; the bit above them tells a dropped slot (-1) from all
    while ((1 << nbits) < n_exp) nbits++;
    for (int s = 0; s < steps; s++) {
        const int e = expert_of(s);
        // lanes of the step with this lane's expert: one ballot per bit of the expert id, each lane keeps the side
        // of the ballot its own bit is on (a dropped slot, e = -1, matches only other dropped slots and is not placed)
        unsigned long long peers = ~0ull;
        for (int bit = 0; bit <= nbits; bit++) {
            const bool on = (e >> bit) & 1;
            const unsigned long long bal = __ballot(on);
            peers &= on ? bal : ~bal;
        }
        const unsigned same = (unsigned)__popcll(peers);
        const unsigned rank = __builtin_amdgcn_mbcnt_hi((unsigned)(peers >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)peers, 0u));
        unsigned before = 0;
        if (e >= 0) before = cnt[wave * n_exp + e];
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if (e >= 0) {
            sorted_ids[poff[e] + before + rank] = j0 + s * 64 + lane;
            if (rank + 1 == same) cnt[wave * n_exp + e] = before + same;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

// (Two kernels: the few instructions more cost the one-workgroup launch 0.35 of its 3.8 us.)
extern "C" __global__ __launch_bounds__(MOE_ALIGN_THREADS) void w4a16_moe_align(const int* idx, int ns, int n_exp, int block,
                                                                               int* sorted_ids, int* expert_ids,
                                                                               int* num_post) {
    moe_align_body<false>(idx, ns, n_exp, block, sorted_ids, expert_ids, num_post, 1);
}
extern "C" __global__ __launch_bounds__(MOE_ALIGN_THREADS) void w4a16_moe_align_wide(const int* idx, int ns, int n_exp,
                                                                                    int block, int* sorted_ids,
                                                                                    int* expert_ids, int* num_post, int wgs) {
    moe_align_body<true>(idx, ns, n_exp, block, sorted_ids, expert_ids, num_post, wgs);
}

// out[t][c] = sum over the token's k slots of f16 c2[slot][c], added in slot order in f32 (assets/moe.cu:1662-1674).
// Eight columns per thread when h % 8 == 0 (16-byte loads), one otherwise.
extern "C" __global__ __launch_bounds__(256) void w4a16_moe_topk_sum_f16(const uint16_t* __restrict__ c2,
                                                                         float* __restrict__ out, int t, int h, int top_k) {
    if ((h & 7) == 0) {
        const size_t total = (size_t)t * h / 8;
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
            const size_t r = (i * 8) / h, c = (i * 8) % h;
            float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            for (int kk = 0; kk < top_k; kk++) {
                const h8_t v = *reinterpret_cast<const h8_t*>(c2 + (r * top_k + kk) * h + c);
#pragma unroll
                for (int j = 0; j < 8; j++) acc[j] += (float)v[j];
            }
            f4_t* o = reinterpret_cast<f4_t*>(out + i * 8);
            o[0] = (f4_t){acc[0], acc[1], acc[2], acc[3]};
            o[1] = (f4_t){acc[4], acc[5], acc[6], acc[7]};
        }
        return;
    }
    const size_t total = (size_t)t * h;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
        const size_t r = i / h, c = i % h;
        float acc = 0.f;
        for (int kk = 0; kk < top_k; kk++)
            acc += (float)__builtin_bit_cast(_Float16, c2[(r * top_k + kk) * h + c]);
        out[i] = acc;
    }
}
