// Prefill regime (t > 16 activation rows): tiled GEMM  y[t][n] = x[t][k] * W^T  on v_mfma_f32_32x32x16_f16.
// Role of the reference's prefill path gemm_launch -> marlin_gemm_try / w4a16_gemm_g128_mma
// (w4a16_dec/kernels/gemm.rs:4-51, kernels/marlin.rs:94-213, assets/gptq4.cu:984-1147), designed for CDNA4:
//   * workgroup = 4 waves along n, block tile 128 (m) x 256 (n), wave tile 128 x 64 = 4 x 2 MFMA tiles of 32 x 32 with
//     f32 accumulators in arch VGPRs (128 registers); two workgroups per CU, so one block's barriers and LDS writes
//     overlap the other's MFMAs;
//   * x (the A operand) is staged through LDS a k tile at a time (in the 96-row tile, whose registers leave no room for the
//     addresses, half of one), double buffered, by LDS DMA (buffer_load ... lds: no staging registers, no ds_write), one
//     barrier per stage; against stages of 64 k (us): 5120 x 34816 gated t = 300 114.8 -> 112.3; t = 4096, seven boxes, 1187 -> 1179,
//     1166 -> 1157, 1187 -> 1178, 1204 -> 1200, 1251 -> 1253, 1219 -> 1210, 1172 -> 1161; group 32 1649 -> 1470 (its 256-register
//     build spilled); 17408 x 5120 t = 4096 614 -> 608; but 17408 x 2560 t = 400 in eight slices 57.5 -> 61.7; rows are unpadded and their 16-byte chunks swizzled by row so the ds_read_b128 fragment reads are
//     bank-conflict free; rows >= t come from out-of-range loads (zeros);
//   * the weights (B operand) never touch LDS: the tiled layout of w4a16_common.hpp already is the MFMA B layout —
//     lane (n = l % 32, khalf = l / 32) reads 16 B of tile lane g = 2h + khalf, r = n % 16 of its row block, dword w of
//     which is the k16 block (w, h) of the k tile — so each wave fetches its 64 x 128 weights with four coalesced
//     dwordx4 loads per k tile (one k tile ahead) and unpacks them in registers (9 VALU ops per MFMA operand);
//   * weights enter the MFMA as exact integers.  The per-group scale is carried as a running unit: the accumulator
//     holds sum / s_g; at each group boundary it is multiplied by s_prev / s_cur and the new group's integer products
//     are added by the MFMA itself; the epilogue multiplies by the last scale.  No weight is rounded to f16 and no
//     second accumulator set is needed.  (Linears with a zero or non-finite scale are not routed here.)
//   * the live block tiles are numbered without gaps and every XCD takes an eighth of them, neighbours in super-tiles (8 x 8 block
//     tiles on large grids: each x slab and each weight panel is fetched into that L2 once per eight uses).
#include "w4a16_common.hpp"

// s_prev / s_cur of a group boundary: the hardware reciprocal (1 ulp) and one Newton step on the quotient (the residual
// s_prev - q * s_cur is exact in a fused multiply-add), which leaves the quotient within about half an ulp.  The
// accumulators are re-expressed with this factor once per scale group, so its error enters every output once per
// group: with the bare reciprocal the kernel's distance from the exact dot product was several times that of the f32
// lane order at k = 17408 (136 groups); with the corrected quotient it is of the same size.  Three instructions per scale
// instead of the ten of an IEEE division (+2 % at group 128, +4.5 % at group 32 at M = 4096 for the division).
__device__ __forceinline__ float pf_ratio(float s_prev, float s_cur) {
    const float r = __builtin_amdgcn_rcpf(s_cur);
    const float q = s_prev * r;
    return __builtin_fmaf(__builtin_fmaf(-q, s_cur, s_prev), r, q);
}

#define PF_BN 256
#define PF_KS 128         // k per LDS stage, half of that in the 96-row tile
#define PF_THREADS 256
#define PF_MOE_IDS_AT 36864  // grouped: LDS bytes ahead of the slot ids, the larger of the two stages and four padded f16 tiles

// MI = 32-row MFMA tiles along m per wave: 4 (block tile 128 x 256, 128 accumulator registers, two workgroups per CU) or
// 2 (64 x 256, 64 registers, three workgroups per CU) for a few dozen to a couple of hundred rows, where 128-row tiles
// would spend half their MFMAs on padding and leave too few workgroups.
//
// Grouped form for the expert FFN (MODE 1, 2): the role of the reference's grouped Marlin GEMM at prefill sizes
// (assets/moe.cu:686-759 via kernels/marlin_moe.rs:290-422).  The rows of a block tile are one 64-slot segment of the
// alignment pass (sorted_ids, padded with the sentinel ns; expert_ids per segment; num_post = padded slot total), the
// weights are those of the segment's expert in its arena, x rows are gathered by slot id (slot j reads row j / x_div)
// straight into the LDS stage by the same DMA, and the epilogue scatters by slot id:
//   MODE 1 (gate|up, n = 2 n_ff): a wave's two 32-column sub-tiles are gate columns c.. and up columns n_ff + c.., so
//     the lane that holds a gate sum holds the matching up sum; both are rounded to f16 (the reference materialises
//     them as f16) and act[slot][c] = f16(act(gate) * up) is written, f16 [ns][n_ff];
//   MODE 2 (down, n = hidden): y[slot][c] = f16(sum * topw[slot]), f16 [ns][n].
//
// Dense gated form (MODE 3): a fused gate|up linear (rows 0..n/2 gate, n/2..n up) with the element-wise kernel that
// follows it in the reference's prefill chain (lin_forward + ew, w4a16_dec/prefill.rs:148-207, assets/ew.cu:9-57)
// folded into the epilogue: column pairing as in MODE 1, tile numbering and split-K as in MODE 0, and
// y[m][c] = f16(act(g) * u) on the f32 sums g, u (f16 [t][n/2]) — the bits of the MODE 0 launch with f32 output
// followed by w4a16_act_mul_f16, without the [t][n] f32 round trip (285 of the 419 MB a 4096-row launch moves on the
// 27B gate|up shape).  A split launch writes f32 partials of all n columns and w4a16_prefill_splitk_sum applies the
// activation after adding them.
template <int MODE>
struct PfGroup {
    const int* sorted_ids;
    const int* expert_ids;
    const int* num_post;
    const float* topw;
    unsigned long long q_stride, s_stride;  // bytes per expert
    int ns, x_rows, x_div, n_exp, act_kind;
    int m0, n0, expert;  // the block tile: first position in sorted_ids, first column, expert
};

// Epilogue options of the dense kernels (MODE 0 and 3), the prefill-regime form of what the decode kernel does for a
// normalisation deferred across linears (the element-wise parts of the reference's norm_resid, assets/norm.cu:4-48,
// moved into the linears either side of it).  Every part is optional (a null pointer / 0 / 1.0 switches it off):
//   consumer side: stats_in [n_stats_in][ld_stats] are partial sums of squares of the INPUT rows left by the launch
//     that produced x; the output row m is multiplied by 1/sqrt(sum_e stats_in[e][m] * inv_cols_in + 1e-6) * in_scale
//     (in_scale = 2^e undoes the power-of-two factor x was handed over with); ldx = halves between x rows (0 = k);
//   producer side: resid f32 [t][n] takes the output (v = resid + y, written back); stats_out[c / 64][m] receives
//     the partial sum of v^2 over the 64 columns from c that a wave holds, those below stat_cols (no atomics); nw f32 [n] multiplies what y receives; out_scale = 2^-e is applied last.
struct PfEpi {
    const float* stats_in;
    float* stats_out;
    float* resid;
    const float* nw;
    int n_stats_in, ld_stats, stat_cols, ldx;
    float inv_cols_in, in_scale, out_scale;
};

// FOLD (grouped form, group 32): scales multiplied into the weights (w4_deq8_scaled), no running unit: 7 instead of 18 vector ALU
// instructions per MFMA.  128 experts top-8 n_ff 768, us per FFN: T = 2048 265 -> 232, T = 1152 188 -> 168.  Dense linears keep the
// unit: their f32 results would lie 15 % further from 64-bit sums (5120 x 5120 t = 1024 2.6e-7 instead of 2.3e-7), which the f16
// rows of the expert FFN do not show (4.0e-4 either way).  us they would save: 34816 x 5120 t = 2048 773 -> 657.
template <int G, bool SBF, int MI, int MODE = 0, int WNW = 4, int KG = 1, bool FOLD = false>
__device__ __forceinline__ void prefill_body(const u4_t* __restrict__ qt, const uint16_t* __restrict__ st,
                                             const uint16_t* __restrict__ x, void* __restrict__ y, int row_blocks,
                                             int k, int n, int t, int out_f16, int walk, int nks,
                                             const PfGroup<MODE> gp = PfGroup<MODE>(), const PfEpi epi = PfEpi()) {
    extern __shared__ _Float16 lds[];  // 2 stages x [PF_BM][KS]; then row factors, a word per thread (dense) / slot ids, weights (grouped)
    constexpr int GPT = W4_TILE_K / G;
    constexpr int BN = 64 * WNW, GT = 64 * WNW;  // block tile columns, threads of a k group
    constexpr int PF_BM = 32 * MI, KS = MI == 3 ? PF_KS / 2 : PF_KS;
    constexpr int PF_STAGE_BYTES = PF_BM * KS * 2, CPR = KS / 8;  // 16-byte chunks per staged x row
    constexpr int NA = (PF_BM * CPR + GT - 1) / GT, SPT = W4_TILE_K / KS;  // x loads per thread and stage, stages per k tile
    // LDS: per k group two stages of x, overlaid by what the groups hand over at the end; then a word per thread
    constexpr int HAND = KG > 1 ? KG * (KG - 1) * WNW * MI * 2 * 1024 : 0, XB = KG * 2 * PF_STAGE_BYTES, LDS_ROWS_AT = XB > HAND ? XB : HAND;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = KG > 1 ? wave % WNW : wave, kg = KG > 1 ? wave / WNW : 0;
    const int kt_n = k / W4_TILE_K, kg_n = kt_n * GPT;

    // XCD-aware tile numbering.  Block b runs on XCD b % 8 and is the (b / 8)-th block of that XCD.  walk: sup_m in the low 16 bits, sup_n,
    // signed, in the high ones (one word, so that a launch's arguments fill two lines of 64 bytes and not a little of a third, which
    // is fetched cold in every launch: gated 2688 x 1152 group 32 t = 171 12.25 us, 12.5 with the third).  The live block tiles are numbered
    // without gaps: panels of sup_n tile columns, in a panel super-tiles of sup_m tile rows, in a super-tile m fastest (sup_n < 0:
    // bands of sup_m tile rows, in a band super-tiles of -sup_n columns), and a tile's k slices one after the other.  Every XCD
    // takes an eighth of the numbers, one run, so the blocks resident on it at a time share x slabs and weight panels through its L2,
    // and no XCD and no CU has more block tiles than an even share.  (Whole super-tiles dealt round-robin, those at the edges
    // partly empty, left some CUs with a block more: 5120 x 5120 t = 1568 99 us, now 80; 14336 x 5248 t = 1041 203 / 144; over 256
    // shapes of 65..4096 rows 5 % on average.  Slices as the outermost dimension cost launches of one block per CU two us: 2448 x 8064
    // t = 177 in eight slices 27.3 / 24.6.)
    int m0, n0, slice = 0;
    constexpr bool DENSE = MODE == 0 || MODE == 3, PAIRED = MODE == 1 || MODE == 3;  // PAIRED: gate and up columns per wave
    if (DENSE) {
        const int tiles_m = (t + PF_BM - 1) / PF_BM,
                  tiles_n = MODE == 3 ? ((n >> 1) + BN / 2 - 1) / (BN / 2) : (n + BN - 1) / BN;
        const unsigned work = (unsigned)(tiles_m * tiles_n) * (unsigned)nks, xcd = blockIdx.x & 7;
        const unsigned at = (unsigned)((unsigned long long)work * xcd / 8) + (blockIdx.x >> 3);
        if (at >= (unsigned)((unsigned long long)work * (xcd + 1) / 8)) return;  // uniform for the whole block
        const int r = (int)(at / (unsigned)nks);
        slice = (int)(at - (unsigned)(r * nks));
        // outer: the dimension cut into panels or bands, inner: the one walked within
        const int sup_m = walk & 0xffff, sup_n = walk >> 16;
        const bool bands = sup_n < 0;
        const int so = bands ? sup_m : sup_n, si = bands ? -sup_n : sup_m, to = bands ? tiles_m : tiles_n, ti = bands ? tiles_n : tiles_m;
        const int o = r / (ti * so), in_o = r - o * (ti * so), wide = min(so, to - o * so);
        const int super = in_o / (si * wide), in_super = in_o - super * (si * wide), deep = min(si, ti - super * si);
        // m fastest inside a super-tile
        const int rows = bands ? wide : deep, i_n = in_super / rows, i_m = in_super - i_n * rows;
        const int tm = (bands ? o * so : super * si) + i_m, tn = (bands ? super * si : o * so) + i_n;
        m0 = tm * PF_BM;
        n0 = tn * (MODE == 3 ? BN / 2 : BN);
    } else {
        m0 = gp.m0;
        n0 = gp.n0;
        qt = reinterpret_cast<const u4_t*>(reinterpret_cast<const char*>(qt) + (size_t)gp.expert * gp.q_stride);
        st = reinterpret_cast<const uint16_t*>(reinterpret_cast<const char*>(st) + (size_t)gp.expert * gp.s_stride);
    }

    const unsigned ldx = DENSE && epi.ldx ? (unsigned)epi.ldx : (unsigned)k;  // halves between x rows
    const __amdgpu_buffer_rsrc_t xr = w4_make_rsrc(x, DENSE ? ((unsigned)(t - 1) * ldx + (unsigned)k) * 2u : (unsigned)gp.x_rows * (unsigned)k * 2u);
    const __amdgpu_buffer_rsrc_t qr = w4_make_rsrc(qt, (unsigned)row_blocks * (unsigned)kt_n * 1024u);
    const __amdgpu_buffer_rsrc_t sr = w4_make_rsrc(st, (unsigned)row_blocks * (unsigned)kg_n * 32u);

    // ---- x staging by LDS DMA (buffer_load ... lds: global -> LDS without passing through registers).  A stage is
    // PF_BM rows x KS k = PF_BM * CPR chunks of 16 B; one instruction of a wave fills 1 KiB of LDS, lane i at byte 16*i,
    // so rows are 2 KS bytes apart without padding.  To keep the fragment reads conflict free the chunks of a
    // row are stored swizzled: chunk position p of row r holds k chunk p ^ (r % CPR) — the lane that fills position p
    // simply fetches that k chunk.  Rows >= t fetch out of range: zeros.
    typedef __attribute__((address_space(3))) char lds_char_t;
    lds_char_t* const lds_base = (lds_char_t*)lds;
    unsigned xa_off[NA];
#pragma unroll
    for (int i = 0; i < NA; i++) {
        const int c = wn * 64 + lane + i * GT, row = c / CPR, kc = (c % CPR) ^ (row % CPR);
        if (DENSE) {
            xa_off[i] = (m0 + row < t) ? ((unsigned)(m0 + row) * ldx + (unsigned)kc * 8u) * 2u : W4_OOB;
        } else {
            const int id = gp.sorted_ids[m0 + row];  // padding rows carry the sentinel ns: zeros, never stored
            xa_off[i] = id < gp.ns ? ((unsigned)(id / gp.x_div) * (unsigned)k + (unsigned)kc * 8u) * 2u : W4_OOB;
        }
    }
    int* const seg_ids = reinterpret_cast<int*>(lds_base + (DENSE ? LDS_ROWS_AT : PF_MOE_IDS_AT));
    float* const seg_w = reinterpret_cast<float*>(seg_ids + PF_BM);
    if (!DENSE && tid < PF_BM) {  // visible after the first barrier
        const int id = gp.sorted_ids[m0 + tid];
        seg_ids[tid] = id;
        if (MODE == 2) seg_w[tid] = gp.topw != nullptr && id < gp.ns ? gp.topw[id] : 1.0f;
    }
    // Dense, input statistics given: the row factors of this block's PF_BM input rows, through a word per thread behind the
    // stages.  The entries of a row are dealt to RP threads, eight loads in flight each, while the first stage of x and weights
    // is on its way (one thread per row ahead of those loads: a chain of up to n / 512 loads in which nothing else runs); the
    // thread of part 0 adds the parts after the first barrier and leaves the factor for the epilogue in its own word.  The
    // order of the additions is fixed: the same bits on every run.
    constexpr int RP = GT * KG / PF_BM;
    float* const row_fac = reinterpret_cast<float*>(lds_base + LDS_ROWS_AT);
    const bool has_stats = DENSE && epi.stats_in != nullptr;
    auto sum_stats = [&]() {
        const int row = tid % PF_BM, part = tid / PF_BM;
        if (part >= RP) return;
        const float* const sp = epi.stats_in + min(m0 + row, t - 1);
        float sum = 0.f;
        for (int e = part; e < epi.n_stats_in; e += 8 * RP) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; j++) v[j] = sp[(size_t)min(e + j * RP, epi.n_stats_in - 1) * epi.ld_stats];
#pragma unroll
            for (int j = 0; j < 8; j++) sum += e + j * RP < epi.n_stats_in ? v[j] : 0.f;
        }
        row_fac[tid] = sum;
    };
    auto make_factor = [&]() {
        float sum = row_fac[tid];
#pragma unroll
        for (int p = 1; p < RP; p++) sum += row_fac[p * PF_BM + tid];
        row_fac[tid] = (float)(1.0 / sqrt((double)sum * (double)epi.inv_cols_in + 1e-6)) * epi.in_scale;
    };
    auto load_a = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < NA; i++)
            if (PF_BM * CPR % GT == 0 || i * GT + wn * 64 < PF_BM * CPR)  // uniform for the wave
                __builtin_amdgcn_raw_ptr_buffer_load_lds(
                    xr, (__attribute__((address_space(3))) void*)(lds_base + (kg * 2 + buf) * PF_STAGE_BYTES + (i * GT + wn * 64) * 16),
                    16, xa_off[i], s * (KS * 2), 0, 0);
    };

    // ---- weights: lane (nl = l % 32, khalf = l / 32); per n sub-tile ni and half h one dwordx4 per k tile
    const int nl = lane & 31, khalf = lane >> 5;
    unsigned q_off[2][2], s_off[2];
#pragma unroll
    for (int ni = 0; ni < 2; ni++) {
        const int nrow = PAIRED ? ni * (n >> 1) + n0 + wn * 32 + nl : n0 + wn * 64 + ni * 32 + nl;
        const unsigned rb = (unsigned)min(nrow >> 4, row_blocks - 1);  // rows past n re-read the last block, never stored
        const unsigned r = (unsigned)(nrow & 15);
#pragma unroll
        for (int h = 0; h < 2; h++) q_off[ni][h] = (rb * (unsigned)kt_n * 64u + (unsigned)(2 * h + khalf) * 16u + r) * 16u;
        s_off[ni] = (rb * (unsigned)kg_n * 16u + r) * 2u;
    }
    u4_t bq[2][2], bqn[2][2];
    unsigned sc[2][GPT], scn[2][GPT];
    auto load_b = [&](u4_t (&dst)[2][2], unsigned (&sdst)[2][GPT], int kt) {
#pragma unroll
        for (int ni = 0; ni < 2; ni++) {
#pragma unroll
            for (int h = 0; h < 2; h++)
                dst[ni][h] = __builtin_amdgcn_raw_buffer_load_b128(qr, q_off[ni][h], kt * 1024, 0);  // k tile in the scalar offset
#pragma unroll
            for (int gi = 0; gi < GPT; gi++)
                sdst[ni][gi] = __builtin_amdgcn_raw_buffer_load_b16(sr, s_off[ni], (kt * GPT + gi) * 32, 0);
        }
    };

    f16_t acc[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; mi++)
#pragma unroll
        for (int ni = 0; ni < 2; ni++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[mi][ni][e] = 0.f;
    float unit[2] = {1.f, 1.f};  // scale the accumulator of sub-tile ni is currently expressed in

    const int a_row = nl;  // + mi * 32
    // split-K over nks slices (narrow outputs at moderate t, where the tile grid alone cannot fill the chip): this
    // block covers k tiles [kt_lo, kt_hi) and writes an f32 partial; a second launch adds the partials in order
    // KG > 1: the k range is dealt to the groups of the workgroup's waves instead, contiguous runs of equal length (the last
    // shorter or empty); every group runs as many iterations, for the barriers, and skips those past its run
    const int kt_a = DENSE && KG == 1 ? (kt_n * slice) / nks : 0,
              kt_b = DENSE && KG == 1 ? (kt_n * (slice + 1)) / nks : kt_n;
    const int per = (kt_b - kt_a + KG - 1) / KG;
    const int kt_lo = kt_a + kg * per, kt_hi = KG > 1 ? min(kt_b, kt_lo + per) : kt_b;
    const int stages = SPT * kt_hi;
    constexpr bool PF_WAVE_PRIO = G == 128;  // wave priority over a stage's MFMAs (see the k loop)

    if (KG == 1 || kt_lo < kt_hi) {
        load_a(SPT * kt_lo, 0);
        load_b(bq, sc, kt_lo);
    }
    if (has_stats) sum_stats();
    w4_dma_barrier();
    if (has_stats && tid < PF_BM) make_factor();  // read after the barriers of the k loop
    if (KG > 1) {
        // The first weights are waited for here: pending at the loop's head they make its first use wait, in every iteration,
        // for as many loads as were just issued.
#pragma unroll
        for (int ni = 0; ni < 2; ni++) {
#pragma unroll
            for (int h = 0; h < 2; h++) asm volatile("" : "+v"(bq[ni][h]));
#pragma unroll
            for (int gi = 0; gi < GPT; gi++) asm volatile("" : "+v"(sc[ni][gi]));
        }
    }

    for (int kt = kt_lo; kt < kt_lo + per; kt++) {
#pragma unroll
        for (int half = 0; half < SPT; half++) {
            const int s = kt * SPT + half;
            // stage s+1 goes into the buffer that stage s-1 was read from: every wave is past the barrier that ended it
            if (s + 1 < stages) load_a(s + 1, (s + 1 - SPT * kt_lo) & 1);
            if (half == 0 && kt + 1 < kt_hi) load_b(bqn, scn, kt + 1);
            const _Float16* abuf = lds + (kg * 2 + ((s - SPT * kt_lo) & 1)) * (PF_BM * KS) + a_row * KS;
            if (KG == 1 || kt < kt_hi)  // uniform for the wave
#pragma unroll
            for (int kbl = 0; kbl < KS / 16; kbl++) {
                const int kb = half * (KS / 16) + kbl, w = kb >> 1, h = kb & 1;
                // Group boundary: re-express the accumulators in the next group's scale.
                //   group 128: the multiply is done at the END of a k tile, tile by tile right after each tile's last
                //   MFMA of the group, with the scale of the next k tile (already loaded), so the VALU work of tile j
                //   runs in the shadow of the MFMAs of tiles j+1.. instead of stalling the next stage's first MFMAs;
                //   group 32: at the first k16 of each 32-k group, before the tile's first MFMA.
                // Wave priority: raised while a stage's MFMAs issue, dropped for the accumulator rescale at the end of a
                // k tile, so that a wave in that VALU-only stretch yields the issue port to the waves that feed the
                // matrix pipe.  64- and 96-row tiles (three waves per SIMD): M = 512 186 -> 180 us, M = 1024 328 -> 317 us
                // on 5120 x 34816; 17408 x 5120 at M = 4096 630 -> 620 us.  128-row tile (two waves per SIMD), built with
                // the max-ILP scheduler: 5120 x 34816 at M = 4096 -0.5...-1.5 % on five boxes (with the default
                // scheduler the same lost 0.4-0.9 % on the faster boxes).  Group 32 rescales inside the stage and has no
                // such stretch.
                if (PF_WAVE_PRIO && kbl == 0) __builtin_amdgcn_s_setprio(1);
                const bool boundary32 = G == 32 && h == 0 && !FOLD;
                float ratio[2] = {1.f, 1.f};
                if (boundary32) {
#pragma unroll
                    for (int ni = 0; ni < 2; ni++) {
                        const float s_cur = w4_scale_fast<SBF>(sc[ni][w]);
                        ratio[ni] = pf_ratio(unit[ni], s_cur);
                        unit[ni] = s_cur;
                    }
                }
                if (G == 128 && kb == 0 && kt == kt_lo) {  // the very first group: unit = its scale, accumulators are zero
#pragma unroll
                    for (int ni = 0; ni < 2; ni++) unit[ni] = w4_scale_fast<SBF>(sc[ni][0]);
                }
                h8_t a[MI];
#pragma unroll
                for (int mi = 0; mi < MI; mi++)
                    a[mi] = *reinterpret_cast<const h8_t*>(abuf + mi * 32 * KS + (((kbl * 2 + khalf) ^ (nl % CPR)) * 8));
                const bool last128 = G == 128 && kb == 7;  // branch free: the last k tile multiplies by 1
                // The next scales' arithmetic stays here: moved up by the scheduler it waits for loads just issued (the 64-row
                // f16 build did so after the second MFMA: 2048 x 11008 t = 256 28.2 us instead of 26.2).
                if (MI == 2 && last128) __builtin_amdgcn_sched_barrier(0x9c);  // SALU, MFMA and memory may cross, VALU may not
                float next_ratio[2] = {1.f, 1.f};
                if (last128) {
                    const bool more = kt + 1 < kt_hi;
#pragma unroll
                    for (int ni = 0; ni < 2; ni++) {
                        const float s_next = more ? w4_scale_fast<SBF>(scn[ni][0]) : unit[ni];
                        next_ratio[ni] = pf_ratio(unit[ni], s_next);
                        unit[ni] = s_next;
                    }
                }
#pragma unroll
                for (int ni = 0; ni < 2; ni++) {
                    h8_t b;
                    if constexpr (FOLD) b = w4_deq8_scaled(bq[ni][h][w], sc[ni][w]);
                    else b = w4_deq8(bq[ni][h][w]);
#pragma unroll
                    for (int mi = 0; mi < MI; mi++) {
                        if (boundary32) acc[mi][ni] *= ratio[ni];
                        acc[mi][ni] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[mi], b, acc[mi][ni], 0, 0, 0);
                    }
                }
                if (last128) {
                    if (PF_WAVE_PRIO) __builtin_amdgcn_s_setprio(0);
#pragma unroll
                    for (int ni = 0; ni < 2; ni++)
#pragma unroll
                        for (int mi = 0; mi < MI; mi++) acc[mi][ni] *= next_ratio[ni];
                }
            }
            w4_dma_barrier();
        }
#pragma unroll
        for (int ni = 0; ni < 2; ni++) {
#pragma unroll
            for (int h = 0; h < 2; h++) bq[ni][h] = bqn[ni][h];
#pragma unroll
            for (int gi = 0; gi < GPT; gi++) sc[ni][gi] = scn[ni][gi];
        }
    }

    f4_t own[MI][2];  // KG > 1: the finished sums of this group's rows
    if constexpr (KG > 1) {
        // Add the groups' sums, in group order: group g takes rows 8g + 4 khalf ..+3 of every 32 (accumulator registers 4g..4g+3),
        // gets them from the other groups through LDS and runs the epilogue for them.
        static_assert(KG == 4, "a group's share is four accumulator registers");
        f4_t* const hand = reinterpret_cast<f4_t*>(lds_base);  // [share][other group][wave along n][tile][lane]
        auto at = [&](int share, int from) { return ((share * (KG - 1) + (from < share ? from : from - 1)) * WNW + wn) * (MI * 2 * 64) + lane; };
#pragma unroll
        for (int g = 0; g < KG; g++) {
            if (g == kg) continue;
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int ni = 0; ni < 2; ni++) {
                    const f4_t v = {acc[mi][ni][4 * g] * unit[ni], acc[mi][ni][4 * g + 1] * unit[ni], acc[mi][ni][4 * g + 2] * unit[ni],
                                    acc[mi][ni][4 * g + 3] * unit[ni]};
                    hand[at(g, kg) + (mi * 2 + ni) * 64] = v;
                }
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < KG; g++) {
            if (g != kg) continue;
#pragma unroll
            for (int mi = 0; mi < MI; mi++)
#pragma unroll
                for (int ni = 0; ni < 2; ni++) {
                    const f4_t mine = {acc[mi][ni][4 * g] * unit[ni], acc[mi][ni][4 * g + 1] * unit[ni], acc[mi][ni][4 * g + 2] * unit[ni],
                                acc[mi][ni][4 * g + 3] * unit[ni]};
                    f4_t sum;
#pragma unroll
                    for (int from = 0; from < KG; from++) {
                        const f4_t v = from == g ? mine : hand[at(g, from) + (mi * 2 + ni) * 64];
                        sum = from == 0 ? v : sum + v;
                    }
                    own[mi][ni] = sum;
                }
        }
    }

    // ---- epilogue: y[m][n] = acc * unit; D register e of lane (nl, khalf) is row 8*(e/4) + 4*khalf + e%4, column nl
    constexpr int NE = KG > 1 ? 4 : 16;  // registers of a 32-row tile that this wave finishes
    auto value = [&](int mi, int ni, int e) { return KG > 1 ? own[mi][ni][e] : acc[mi][ni][e] * unit[ni]; };
    auto row_of = [&](int mi, int e) { return m0 + mi * 32 + 8 * (KG > 1 ? kg : e >> 2) + 4 * khalf + (e & 3); };
    if (!DENSE) {
        // Grouped: the wave's f16 tile goes through its own part of the stages' LDS (free after the last barrier, a wave's LDS
        // operations run in order) and out in 16-byte pieces of whole row segments: one store per 1 KiB instead of 2 bytes per
        // lane; the routing weights were fetched once per row, not once per element.  128 experts top-8 h 2048 n_ff 768,
        // T = 2048: down projection 126 -> 85 us, gate|up level (its stores cost 17 us, the activation keeps them busy).
        constexpr int COLS = MODE == 1 ? 32 : 64, LD = COLS + 8, PER_ROW = COLS / 8;
        const int n_out = MODE == 1 ? n >> 1 : n, col = n0 + wn * COLS;
        if (col >= n_out) return;  // uniform for the wave (n_out % 64 == 0)
        _Float16* const tile = lds + wave * (PF_BM * LD);
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
#pragma unroll
            for (int e = 0; e < 16; e++) {
                const int r = mi * 32 + 8 * (e >> 2) + 4 * khalf + (e & 3);
                if (MODE == 1) {
                    const float gt = (float)(_Float16)(acc[mi][0][e] * unit[0]), up = (float)(_Float16)(acc[mi][1][e] * unit[1]);
                    tile[r * LD + nl] = (_Float16)w4_act_mul(gt, up, gp.act_kind);
                } else {
                    const float w = seg_w[r];
#pragma unroll
                    for (int ni = 0; ni < 2; ni++) {
                        float v = acc[mi][ni][e] * unit[ni] * w;
                        asm volatile("" : "+v"(v));  // the product is rounded to f32 before the f16 conversion
                        tile[r * LD + ni * 32 + nl] = (_Float16)v;
                    }
                }
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
#pragma unroll
        for (int i = 0; i < PF_BM * PER_ROW / 64; i++) {
            const int r = i * (64 / PER_ROW) + lane / PER_ROW, piece = lane % PER_ROW, slot = seg_ids[r];
            const u4_t v = *reinterpret_cast<const u4_t*>(tile + r * LD + piece * 8);
            if (slot < gp.ns) *reinterpret_cast<u4_t*>(reinterpret_cast<_Float16*>(y) + (size_t)slot * n_out + col + piece * 8) = v;
        }
        return;
    }
    // x arrived as its true value times 1/in_scale and (with input statistics) un-normalised: one factor per row
    const bool use_fac = DENSE && (has_stats || (epi.in_scale != 1.0f && epi.in_scale != 0.0f));
    if (MODE == 3 && (KG > 1 || nks == 1)) {
        const int n_ff = n >> 1, col = n0 + wn * 32 + nl;
        if (col >= n_ff) return;
#pragma unroll
        for (int mi = 0; mi < MI; mi++) {
#pragma unroll
            for (int e = 0; e < NE; e++) {
                const int row = row_of(mi, e);
                if (row < t) {
                    float gt = value(mi, 0, e), up = value(mi, 1, e);
                    asm volatile("" : "+v"(gt), "+v"(up));  // the sums are rounded to f32 as the separate launch stores them
                    if (use_fac) {
                        const float f = has_stats ? row_fac[row - m0] : epi.in_scale;
                        gt *= f;
                        up *= f;
                    }
                    float v = w4_act_mul(gt, up, gp.act_kind);
                    asm volatile("" : "+v"(v));  // and the product before the f16 conversion, as in the separate kernel
                    if (epi.out_scale != 1.0f && epi.out_scale != 0.0f) {
                        v *= epi.out_scale;
                        asm volatile("" : "+v"(v));
                    }
                    reinterpret_cast<_Float16*>(y)[(size_t)row * n_ff + col] = (_Float16)v;
                }
            }
        }
        return;
    }
    // a partial (f32) of a split launch: w4a16_prefill_splitk_sum finishes (activation, epilogue options).  Gated launches end here or
    // above; said without nks, or the compiler keeps the plain epilogue for them too, which doubles their code (55 KB instead of 30 at
    // 64 rows) and what a launch fetches of it.
    if (KG == 1 && (MODE == 3 || nks > 1)) {
        y = reinterpret_cast<float*>(y) + (size_t)slice * (size_t)t * (size_t)n;
#pragma unroll
        for (int ni = 0; ni < 2; ni++) {
            const int col = MODE == 3 ? ni * (n >> 1) + n0 + wn * 32 + nl : n0 + wn * 64 + ni * 32 + nl;
            if (MODE == 3 ? n0 + wn * 32 + nl >= (n >> 1) : col >= n) continue;
#pragma unroll
            for (int mi = 0; mi < MI; mi++) {
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    const int row = m0 + mi * 32 + 8 * (e >> 2) + 4 * khalf + (e & 3);
                    if (row < t) reinterpret_cast<float*>(y)[(size_t)row * n + col] = acc[mi][ni][e] * unit[ni];
                }
            }
        }
        return;
    }
    // MODE 0, whole k range: y = acc * unit, then the optional parts in the order of the decode kernel's epilogue — row
    // factor, residual stream, statistics of what continues, norm weight, power-of-two hand-over factor
    const bool plain = !use_fac && epi.resid == nullptr && epi.stats_out == nullptr && epi.nw == nullptr && (epi.out_scale == 1.0f || epi.out_scale == 0.0f);
    // The residual stream's values and norm weights are fetched ahead of the stores that the compiler may not move them across:
    // a wait per four rows (k groups: one in all) instead of one per element.
    int col[2];
    float nwv[2] = {1.f, 1.f};
#pragma unroll
    for (int ni = 0; ni < 2; ni++) {
        col[ni] = n0 + wn * 64 + ni * 32 + nl;
        if (epi.nw != nullptr) nwv[ni] = epi.nw[min(col[ni], n - 1)];
    }
    constexpr int MB = KG > 1 ? MI : 1;  // tiles per batch of four rows
#pragma unroll
    for (int mb = 0; mb < MI * NE; mb += 4 * MB) {
        const int m_at = mb / NE, e_at = mb % NE;
        float rv[MB][4][2];
        if (epi.resid != nullptr) {
#pragma unroll
            for (int i = 0; i < MB; i++)
#pragma unroll
                for (int e = 0; e < 4; e++)
#pragma unroll
                    for (int ni = 0; ni < 2; ni++)
                        rv[i][e][ni] = epi.resid[(size_t)min(row_of(m_at + i, e_at + e), t - 1) * n + min(col[ni], n - 1)];
        }
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const int mi = m_at + i;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = row_of(mi, e_at + e);
                float p = 0.f;  // this lane's share of the row's sum of squares
                if (row < t) {
                    const float f = !use_fac ? 1.0f : has_stats ? row_fac[row - m0] : epi.in_scale;
#pragma unroll
                    for (int ni = 0; ni < 2; ni++) {
                        if (col[ni] >= n) continue;
                        const size_t at = (size_t)row * n + col[ni];
                        float v = value(mi, ni, e_at + e);
                        if (!plain) {
                            asm volatile("" : "+v"(v));
                            if (use_fac) v *= f;
                            if (epi.resid != nullptr) {
                                v += rv[i][e][ni];
                                epi.resid[at] = v;
                            }
                            if (col[ni] < epi.stat_cols) p = __builtin_fmaf(v, v, p);
                            if (epi.nw != nullptr) v *= nwv[ni];
                            if (epi.out_scale != 1.0f && epi.out_scale != 0.0f) {
                                v *= epi.out_scale;
                                asm volatile("" : "+v"(v));  // rounded to f32 on its own, not fused into the f16 conversion
                            }
                        }
                        if (out_f16)
                            reinterpret_cast<_Float16*>(y)[at] = (_Float16)v;
                        else
                            reinterpret_cast<float*>(y)[at] = v;
                    }
                }
                if (epi.stats_out != nullptr) {  // uniform: the 32 lanes of a row (same khalf) add up in a fixed order
#pragma unroll
                    for (int off = 16; off > 0; off >>= 1) p += __shfl_xor(p, off);
                    if (nl == 0 && row < t && n0 + wn * 64 < epi.stat_cols)
                        epi.stats_out[(size_t)((n0 + wn * 64) >> 6) * epi.ld_stats + row] = p;
                }
            }
        }
    }
}

#define PREFILL_KERNEL(NAME, G, SBF, MI, WPE)                                                                      \
    extern "C" __global__ __launch_bounds__(PF_THREADS) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void NAME(      \
        const u4_t* qt, const uint16_t* st, const uint16_t* x, void* y, int row_blocks, int k, int n, int t,          \
        int out_f16, int walk, int nks, int act_kind, PfEpi epi) {                                                  \
        (void)act_kind;                                                                                                \
        prefill_body<G, SBF, MI>(qt, st, x, y, row_blocks, k, n, t, out_f16, walk, nks, PfGroup<0>(), epi);         \
    }

// Dense gated kernels: same arguments (the plain kernels ignore act_kind, W4A16_ACT_*); y is f16 [t][n/2], or the f32
// partials [slices][t][n] of a split launch.
#define PREFILL_GLU_KERNEL(NAME, G, SBF, MI, WPE)                                                                  \
    extern "C" __global__ __launch_bounds__(PF_THREADS) __attribute__((amdgpu_waves_per_eu(WPE, WPE))) void NAME(      \
        const u4_t* qt, const uint16_t* st, const uint16_t* x, void* y, int row_blocks, int k, int n, int t,          \
        int out_f16, int walk, int nks, int act_kind, PfEpi epi) {                                                  \
        PfGroup<3> gp;                                                                                                 \
        gp.act_kind = act_kind;                                                                                        \
        prefill_body<G, SBF, MI, 3>(qt, st, x, y, row_blocks, k, n, t, out_f16, walk, nks, gp, epi);                \
    }

// Block tile of a grouped workgroup.  Every XCD (block b runs on XCD b % 8) takes an eighth of the live block tiles, segments in
// order and column tiles fastest, so that the segments of one expert's run fetch its weights, and the column tiles of a segment
// its x rows, into one L2 at about the same time (128 experts, T = 2048: -3 %).  Dealt by whole segments, a count just over a
// multiple of eight leaves most XCDs waiting for one (8 experts top-2, h 4096, n_ff 3584, us per FFN, by segments / by tiles:
// group 32 T = 1024 298 / 272, group 128 T = 700 182 / 155; level elsewhere).  Gate|up tiles span 128 gate and the 128
// matching up columns.  A segment whose second half is padding (its slots are a prefix of it) runs the 32-row body: an expert's
// last segment is partly filled (T = 1536 246 -> 225 us per FFN, T = 2048 284 -> 264).
template <int MODE>
__device__ __forceinline__ bool pf_moe_tile(PfGroup<MODE>& gp, const int* num_post, int n, int* rows) {
    const int tiles = MODE == 1 ? ((n >> 1) + PF_BN / 2 - 1) / (PF_BN / 2) : (n + PF_BN - 1) / PF_BN;
    const unsigned work = (unsigned)(num_post[0] / 64) * (unsigned)tiles, xcd = blockIdx.x & 7;
    const unsigned at = (unsigned)((unsigned long long)work * xcd / 8) + (blockIdx.x >> 3);
    if (at >= (unsigned)((unsigned long long)work * (xcd + 1) / 8)) return false;
    const int seg = (int)(at / (unsigned)tiles);
    gp.m0 = seg * 64;
    gp.n0 = (int)(at % (unsigned)tiles) * (MODE == 1 ? PF_BN / 2 : PF_BN);
    gp.expert = gp.expert_ids[seg];
    *rows = gp.sorted_ids[gp.m0 + 32] < gp.ns ? 64 : 32;
    return (unsigned)gp.expert < (unsigned)gp.n_exp;
}

// k-group kernels, for outputs too narrow to fill the chip with 256-column tiles: 64 rows x 64 WNW columns, WNW waves along n times
// four k groups in one workgroup (8 or 12 waves, 128 or 144 KiB of LDS: one workgroup per CU).  What bounds these launches is
// not the matrix pipe but a chain per k tile (x by DMA, barrier, 32 MFMAs a wave) too few waves are there to hide, plus, when
// k slices filled the chip instead, writing the slices' f32 sums to memory and a second launch that adds them.  Here each group
// walks a quarter of k with x stages of its own, the groups' sums meet in LDS in group order (same bits on every run), and each
// group runs the epilogue, options included, for a quarter of the rows.  5120 x 5120 t = 300 32.0 -> 27.4 us (200
// workgroups instead of 400 and a second launch), 4096 x 2048 t = 300 26.3 -> 12.9, group 32 5120 x 2048 t = 300 32.1 -> 16.1.
// One wave along n (64 columns) needs twice the waves for the same x traffic and won 0.3 % over the range: not built.
#define PREFILL_KG_KERNEL(NAME, G, SBF, WNW, MODE)                                                                    \
    extern "C" __global__ __launch_bounds__(64 * WNW * 4) __attribute__((amdgpu_waves_per_eu(WNW, WNW))) void NAME(       \
        const u4_t* qt, const uint16_t* st, const uint16_t* x, void* y, int row_blocks, int k, int n, int t,          \
        int out_f16, int walk, int nks, int act_kind, PfEpi epi) {                                                  \
        PfGroup<MODE> gp;                                                                                              \
        gp.act_kind = act_kind;                                                                                        \
        prefill_body<G, SBF, 2, MODE, WNW, 4>(qt, st, x, y, row_blocks, k, n, t, out_f16, walk, nks, gp, epi);      \
    }
#define PREFILL_KG_FAMILY(PFX, G, SBF)                    \
    PREFILL_KG_KERNEL(PFX##_m64_n2k4, G, SBF, 2, 0)       \
    PREFILL_KG_KERNEL(PFX##_m64_n3k4, G, SBF, 3, 0)       \
    PREFILL_KG_KERNEL(PFX##_m64_n2k4_glu, G, SBF, 2, 3)   \
    PREFILL_KG_KERNEL(PFX##_m64_n3k4_glu, G, SBF, 3, 3)

// Grouped kernels for the expert FFN: same arguments as the streaming grouped kernels of moe.hip (blk must be 64, the
// rows of a block tile, and y_f16 1: the host refuses others; wpb is unused).
#define PREFILL_MOE_BUILD(NAME, G, SBF, MODE, FOLD)                                                                   \
    extern "C" __global__ __launch_bounds__(PF_THREADS) __attribute__((amdgpu_waves_per_eu(3, 3))) void NAME(            \
        const char* qa, const char* sa, unsigned long long q_stride, unsigned long long s_stride, const uint16_t* x,      \
        int x_rows, int x_div, void* y, int y_f16, const float* topw, const int* sorted_ids, const int* expert_ids,      \
        const int* num_post, int blk, int ns, int row_blocks, int k, int n, int n_exp, int wpb, int act_kind) {                                                                                                  \
        PfGroup<MODE> gp;                                                                                                \
        gp.sorted_ids = sorted_ids;                                                                                      \
        gp.expert_ids = expert_ids;                                                                                      \
        gp.num_post = num_post;                                                                                          \
        gp.topw = topw;                                                                                                  \
        gp.q_stride = q_stride;                                                                                          \
        gp.s_stride = s_stride;                                                                                          \
        gp.ns = ns;                                                                                                      \
        gp.x_rows = x_rows;                                                                                              \
        gp.x_div = x_div;                                                                                                \
        gp.n_exp = n_exp;                                                                                                \
        gp.act_kind = act_kind;                                                                                          \
        (void)blk, (void)wpb;                                                                   \
        int rows;                                                                                                        \
        if (!pf_moe_tile<MODE>(gp, num_post, n, &rows)) return;                                                          \
        const u4_t* qt = reinterpret_cast<const u4_t*>(qa);                                                              \
        const uint16_t* st = reinterpret_cast<const uint16_t*>(sa);                                                      \
        if (rows <= 32) prefill_body<G, SBF, 1, MODE, 4, 1, FOLD>(qt, st, x, y, row_blocks, k, n, 0, y_f16, 0, 1, gp);         \
        else prefill_body<G, SBF, 2, MODE, 4, 1, FOLD>(qt, st, x, y, row_blocks, k, n, 0, y_f16, 0, 1, gp);                    \
    }

#define PREFILL_MOE_KERNEL(NAME, G, SBF, MODE) PREFILL_MOE_BUILD(NAME, G, SBF, MODE, false)

// This file builds two code objects.  Compiled on its own it holds everything but the dense group-128 kernels;
// prefill_g128.hip includes it with PF_DENSE_G128 defined and holds those (the k-group ones as well), built with the backend's max-ILP
// instruction scheduler (5120 x 34816 at M = 4096: 1.204 -> 1.193 ms, the other layer shapes -0.2...-0.6 %; the
// group-32 builds spill registers under that scheduler and keep the default).
#ifdef PF_DENSE_G128
PREFILL_KERNEL(w4a16_prefill_g128_f16, 128, false, 4, 2)
PREFILL_KERNEL(w4a16_prefill_g128_bf16, 128, true, 4, 2)
PREFILL_KERNEL(w4a16_prefill_g128_f16_m64, 128, false, 2, 3)
PREFILL_KERNEL(w4a16_prefill_g128_bf16_m64, 128, true, 2, 3)
PREFILL_KERNEL(w4a16_prefill_g128_f16_m96, 128, false, 3, 3)
PREFILL_KERNEL(w4a16_prefill_g128_bf16_m96, 128, true, 3, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_f16_glu, 128, false, 4, 2)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_bf16_glu, 128, true, 4, 2)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_f16_m64_glu, 128, false, 2, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_bf16_m64_glu, 128, true, 2, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_f16_m96_glu, 128, false, 3, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g128_bf16_m96_glu, 128, true, 3, 3)
PREFILL_KG_FAMILY(w4a16_prefill_g128_f16, 128, false)
PREFILL_KG_FAMILY(w4a16_prefill_g128_bf16, 128, true)
#else
// y[i] = sum over the nks partials of a split-K launch, added in split order in f32; f32 or f16 out.
// glu != 0: the partials are those of a fused gate|up linear, [slices][t][n]; y is f16 [t][n/2] = act(g) * u on the
// summed gate and up columns (act_kind as in w4_act_mul), the same arithmetic as the unsplit gated epilogue.
extern "C" __global__ __launch_bounds__(256) void w4a16_prefill_splitk_sum(const float* __restrict__ part, void* __restrict__ y,
                                                                           int nks, size_t count, int out_f16, int glu,
                                                                           int n, int act_kind) {
    if (glu) {
        const size_t n_ff = (size_t)(n >> 1), q_ff = n_ff / 4, total = (count / (size_t)n) * q_ff;  // n_ff % 4 == 0 (host)
        for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (size_t)gridDim.x * blockDim.x) {
            const size_t row = i / q_ff, c4 = i - row * q_ff;
            const float* pg = part + row * (size_t)n + c4 * 4;
            f4_t g = *reinterpret_cast<const f4_t*>(pg), u = *reinterpret_cast<const f4_t*>(pg + n_ff);
            for (int ks = 1; ks < nks; ks++) {
                g += *reinterpret_cast<const f4_t*>(pg + (size_t)ks * count);
                u += *reinterpret_cast<const f4_t*>(pg + (size_t)ks * count + n_ff);
            }
            h4_t o;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                float v = w4_act_mul(g[j], u[j], act_kind);
                asm volatile("" : "+v"(v));
                o[j] = (_Float16)v;
            }
            reinterpret_cast<h4_t*>(y)[row * q_ff + c4] = o;
        }
        return;
    }
    const size_t n4 = count / 4;  // count = t*n with n % 4 == 0 is guaranteed by the host
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (size_t)gridDim.x * blockDim.x) {
        f4_t a = reinterpret_cast<const f4_t*>(part)[i];
        for (int ks = 1; ks < nks; ks++) a += reinterpret_cast<const f4_t*>(part + (size_t)ks * count)[i];
        if (out_f16) {
            h4_t v = {(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3]};
            reinterpret_cast<h4_t*>(y)[i] = v;
        } else {
            reinterpret_cast<f4_t*>(y)[i] = a;
        }
    }
}

// Finish of a split launch that carries epilogue options (MODE 0 only; n % 1024 == 0): one workgroup per (row,
// 1024-column chunk) adds the slices in order and applies the options of PfEpi in the order of the unsplit epilogue.
// Statistics: one entry per chunk, stats_out[chunk][row] (the four waves' sums folded in wave order).
extern "C" __global__ __launch_bounds__(256) void w4a16_prefill_splitk_finish(const float* __restrict__ part, void* __restrict__ y,
                                                                              int nks, int t, int n, int out_f16, PfEpi epi) {
    __shared__ float red[4];
    __shared__ float fac_s;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int chunks = n >> 10, row = blockIdx.x / chunks, chunk = blockIdx.x - row * chunks;
    if (row >= t) return;
    const bool use_fac = epi.stats_in != nullptr || (epi.in_scale != 1.0f && epi.in_scale != 0.0f);
    if (epi.stats_in != nullptr && wave == 0) {
        float sum = 0.f;
        for (int e = lane; e < epi.n_stats_in; e += 64) sum += epi.stats_in[(size_t)e * epi.ld_stats + row];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off);
        if (lane == 0) fac_s = (float)(1.0 / sqrt((double)sum * (double)epi.inv_cols_in + 1e-6)) * epi.in_scale;
    }
    if (epi.stats_in != nullptr) __syncthreads();
    const float f = !use_fac ? 1.0f : epi.stats_in != nullptr ? fac_s : epi.in_scale;
    const int col = (chunk << 10) + tid * 4;
    const size_t count = (size_t)t * (size_t)n, at = (size_t)row * n + col;
    f4_t a = *reinterpret_cast<const f4_t*>(part + at);
    for (int ks = 1; ks < nks; ks++) a += *reinterpret_cast<const f4_t*>(part + (size_t)ks * count + at);
    float p = 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        float v = a[j];
        if (use_fac) v *= f;
        if (epi.resid != nullptr) {
            v += epi.resid[at + j];
            epi.resid[at + j] = v;
        }
        if (col + j < epi.stat_cols) p = __builtin_fmaf(v, v, p);
        if (epi.nw != nullptr) v *= epi.nw[col + j];
        if (epi.out_scale != 1.0f && epi.out_scale != 0.0f) {
            v *= epi.out_scale;
            asm volatile("" : "+v"(v));
        }
        a[j] = v;
    }
    if (out_f16) {
        h4_t o = {(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3]};
        *reinterpret_cast<h4_t*>(reinterpret_cast<_Float16*>(y) + at) = o;
    } else {
        *reinterpret_cast<f4_t*>(reinterpret_cast<float*>(y) + at) = a;
    }
    if (epi.stats_out != nullptr) {
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
        if (lane == 0) red[wave] = p;
        __syncthreads();
        if (tid == 0 && (chunk << 10) < epi.stat_cols) epi.stats_out[(size_t)chunk * epi.ld_stats + row] = ((red[0] + red[1]) + red[2]) + red[3];
    }
}

PREFILL_KERNEL(w4a16_prefill_g32_f16, 32, false, 4, 2)
PREFILL_KERNEL(w4a16_prefill_g32_bf16, 32, true, 4, 2)
PREFILL_KERNEL(w4a16_prefill_g32_f16_m64, 32, false, 2, 3)
PREFILL_KERNEL(w4a16_prefill_g32_bf16_m64, 32, true, 2, 3)
PREFILL_KERNEL(w4a16_prefill_g32_f16_m96, 32, false, 3, 3)
PREFILL_KERNEL(w4a16_prefill_g32_bf16_m96, 32, true, 3, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_f16_glu, 32, false, 4, 2)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_bf16_glu, 32, true, 4, 2)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_f16_m64_glu, 32, false, 2, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_bf16_m64_glu, 32, true, 2, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_f16_m96_glu, 32, false, 3, 3)
PREFILL_GLU_KERNEL(w4a16_prefill_g32_bf16_m96_glu, 32, true, 3, 3)
PREFILL_KG_FAMILY(w4a16_prefill_g32_f16, 32, false)
PREFILL_KG_FAMILY(w4a16_prefill_g32_bf16, 32, true)
PREFILL_MOE_KERNEL(w4a16_moe_g128_f16_pf_glu, 128, false, 1)
PREFILL_MOE_KERNEL(w4a16_moe_g128_f16_pf_lin, 128, false, 2)
PREFILL_MOE_KERNEL(w4a16_moe_g128_bf16_pf_glu, 128, true, 1)
PREFILL_MOE_KERNEL(w4a16_moe_g128_bf16_pf_lin, 128, true, 2)
PREFILL_MOE_KERNEL(w4a16_moe_g32_f16_pf_glu, 32, false, 1)
PREFILL_MOE_KERNEL(w4a16_moe_g32_f16_pf_lin, 32, false, 2)
PREFILL_MOE_BUILD(w4a16_moe_g32_f16x_pf_glu, 32, false, 1, true)
PREFILL_MOE_BUILD(w4a16_moe_g32_f16x_pf_lin, 32, false, 2, true)
PREFILL_MOE_KERNEL(w4a16_moe_g32_bf16_pf_glu, 32, true, 1)
PREFILL_MOE_KERNEL(w4a16_moe_g32_bf16_pf_lin, 32, true, 2)
#endif
