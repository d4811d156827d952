// Dense linears at 17..64 activation rows (and any number of rows for scales the MFMA-tiled kernel cannot divide by):
// y[t][n] = x[t][k] * W^T, weights streamed once, several 16-row token blocks per unpacked weight.  Role of the reference's
// gemm_launch below its prefill tiles (w4a16_dec/kernels/gemm.rs:4-51) and, gated, of lin_forward + ew
// (w4a16_dec/prefill.rs:148-207, assets/ew.cu:9-57).
//
// What bounds it: at these row counts neither HBM (92 MB of the 27B gate|up in 14 us) nor the matrix pipe (64 rows: 15 us at
// the rate two waves per SIMD reach) but the way x gets to the waves.  x (64 rows x 5120: 655 KB) is read by every
// workgroup, through an L1 of 64 B per clock and an LDS of 128 B per clock, and a k tile of a wave is a chain load -> LDS ->
// MFMA -> scaled sum that only other waves on the SIMD can hide.  Hence
//   * a workgroup = WN waves along n, each with a unit of two row blocks (gated: gate and up block), times WK groups along k.
//     The WN waves of a group share its staged x tile; the WK groups bring the waves that hide latency without more x.  WN is
//     chosen so that one generation of workgroups covers the output evenly (the plan in w4a16_moe.cc); a grid a little over one
//     workgroup per CU costs a second one (34816 x 5120 gated at t = 64: four waves along n 48 us, five 34);
//   * x by LDS DMA, one k tile ahead, no registers held; a lone wave along n (narrow outputs) stages its x through registers
//     instead and needs no barrier and half the LDS.  LDS sets how many waves a CU holds (at four token blocks: n5k2 160 KiB, ten
//     waves; n4k2, n2k4 128 KiB, eight; n3k4 128 KiB, twelve; n1k4 68 KiB and n4k1 64 KiB, two workgroups, eight), two or three
//     per SIMD; registers (at most 132, a lone wave 212) would allow as many;
//   * scales: group 128 one load for both row blocks of a k tile (a quad's lanes fetch them alternately, DPP broadcasts).
// Sums: a slice's k tiles are cut into MID_PARTS runs, each summed from zero and added in order.  WK groups take whole runs, so
// every launch shape gives the same bits, and so do the gated and the plain launch and a slice of a split one.
// Measured against the grouped expert kernel that served these rows before (us, before / now): gated 34816 x 5120 t = 64
// 49.8 / 34.7, t = 32 34.3 / 27.8; gated 22016 x 4096 t = 64 30.3 / 20.9; 16384 x 4096 t = 40 21.7 / 15.5; 5120 x 5120 t = 64
// 18.6 / 14.5; 5120 x 2048 group 32 t = 37 12.8 / 7.1; 17408 x 5120 t = 64 35.8 / 24.9; 512 x 17408 t = 40 20.4 / 10.7.
// FOLD (group 32, bf16 scales; rule at the launch, w4a16_moe.cc): scales multiplied into the weights (w4_deq8_scaled), a k tile's four
// MFMAs summed from zero and added once, a quarter of the additions and no scale to spread over the accumulators.  us, scaled sums /
// folded: 34816 x 5120 t = 64 52.5 / 45.5, t = 48 43.3 / 36.9, t = 20 33.4 / 30.9; gated 22016 x 4096 t = 40 20.9 / 18.9; 7168 x 5120
// t = 30 10.66 / 10.65.
// (The full wait at the barriers costs the gated 34816 x 5120 at t = 64 1 us, the other shapes of the timing cases nothing.)
#include "w4a16_common.hpp"

#define MOE_LDX 136  // halves per staged x row: 128 + 8 padding (272-byte stride: 16-lane b128 reads hit all banks once)
#define MOE_MAX_KSPLIT 8  // k slices across workgroups; the host clamps to this
#define MID_PARTS 4       // runs of a slice's k tiles, each summed from zero

template <int W>
__device__ __forceinline__ unsigned mid_quad_bcast(unsigned v) {
    return __builtin_amdgcn_update_dpp(0u, v, W * 0x55, 0xF, 0xF, true);
}

template <bool SBF>
__device__ __forceinline__ f4_t mid_scale4(unsigned d0, unsigned d1) {
    f4_t r;
    r[0] = w4_scale_fast<SBF>(d0 & 0xFFFFu);
    r[1] = w4_scale_fast<SBF>(d0 >> 16);
    r[2] = w4_scale_fast<SBF>(d1 & 0xFFFFu);
    r[3] = w4_scale_fast<SBF>(d1 >> 16);
    return r;
}

// gp = workgroups of one segment of 16 * TT rows; blockIdx.x = segment * gp + group of WN units, blockIdx.y = k slice.
// ws, tickets: workspace and zeroed counters of a launch split over k ([slice][block][wave along n][2 * TT] partial tiles, one
// counter per wave); act_kind: W4A16_ACT_* (gated form).
#define MID_PARAMS                                                                                                      \
    const u4_t *__restrict__ qt, const uint16_t *__restrict__ st, const uint16_t *__restrict__ x, void *__restrict__ y, \
        int row_blocks, int k, int n, int t, int out_f16, int act_kind, f4_t *ws, int *tickets, int nks, int gp
#define MID_ARGS qt, st, x, y, row_blocks, k, n, t, out_f16, act_kind, ws, tickets, nks, gp

template <int G, bool SBF, bool GLU, int TT, int WN, int WK, bool FOLD>
__device__ __forceinline__ void mid_body(MID_PARAMS) {
    extern __shared__ __attribute__((aligned(16))) _Float16 xs[];
    constexpr int GPT = W4_TILE_K / G, ROWS = 16 * TT, XL = (4 * TT + WN - 1) / WN, NBUF = WN > 1 ? 2 : 1;
    static_assert(WK == 1 || WK == 2 || WK == MID_PARTS, "groups along k take whole parts");
    constexpr int SL = G == 128 ? 1 : 2;  // scale loads per k tile
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kg = wave / WN, wn = wave % WN;
    const int units = GLU ? row_blocks >> 1 : (row_blocks + 1) >> 1;
    const int seg = (int)blockIdx.x >= gp ? (int)blockIdx.x / gp : 0;
    const int u_raw = ((int)blockIdx.x - seg * gp) * WN + wn;
    const bool active = u_raw < units;  // a surplus wave repeats the last unit and stores nothing
    const int u = min(u_raw, units - 1);
    const int rbA = GLU ? u : 2 * u, rbB = GLU ? u + units : min(2 * u + 1, row_blocks - 1);
    const bool haveB = GLU || 2 * u + 1 < row_blocks;
    const int kt_n = k / W4_TILE_K, kg_n = kt_n * GPT;
    const int ky = blockIdx.y;
    const int kt_lo = (kt_n * ky) / nks, kt_hi = (kt_n * (ky + 1)) / nks;
    const int per = (kt_hi - kt_lo + MID_PARTS - 1) / MID_PARTS;
    constexpr int PPW = MID_PARTS / WK;  // parts of a wave
    const int kt0 = kt_lo + kg * (PPW * per), kt1 = min(kt_hi, kt0 + PPW * per);
    const int row0 = seg * ROWS;
    const int c = lane & 15, q = lane >> 4;

    const unsigned q_bytes = (unsigned)row_blocks * (unsigned)kt_n * 1024u, s_bytes = (unsigned)row_blocks * (unsigned)kg_n * 32u,
                   x_bytes = (unsigned)t * (unsigned)k * 2u;
    const unsigned qoff[2] = {(unsigned)rbA * (unsigned)kt_n * 1024u + (unsigned)lane * 16u,
                              (unsigned)rbB * (unsigned)kt_n * 1024u + (unsigned)lane * 16u};
    // scale loads: group 128: one, lane l of a quad fetches row block l & 1; group 32: one per row block, lane l of a quad
    // fetches group l of the k tile; FOLD: one per row block, one of the k tile's 64 scales per lane
    unsigned soff[SL];
    if constexpr (FOLD) {
        soff[0] = (unsigned)rbA * (unsigned)kg_n * 32u + (unsigned)lane * 2u;
        soff[1] = (unsigned)rbB * (unsigned)kg_n * 32u + (unsigned)lane * 2u;
    } else if constexpr (G == 128) {
        soff[0] = (unsigned)((lane & 1) ? rbB : rbA) * (unsigned)kg_n * 32u + (unsigned)q * 8u;
    } else {
        soff[0] = (unsigned)rbA * (unsigned)kg_n * 32u + (unsigned)(lane & 3) * 32u + (unsigned)q * 8u;
        soff[1] = (unsigned)rbB * (unsigned)kg_n * 32u + (unsigned)(lane & 3) * 32u + (unsigned)q * 8u;
    }
    // x load l of this wave brings rows 4 * (wn + l * WN) ..+3 of the group's tile, 16 lanes x 16 B to a row.
    // WN > 1: by LDS DMA into unpadded rows of 256 B whose 16-byte chunks are swizzled, chunk p of row r at position p ^ (r & 15),
    // so that the 16 rows of a B operand's read fall into distinct banks; a lone wave: through registers into padded rows.
    unsigned xoff[XL];
#pragma unroll
    for (int l = 0; l < XL; l++) {
        const int r = 4 * (wn + l * WN) + q, row = row0 + r;
        const int piece = WN > 1 ? c ^ (r & 15) : c;
        xoff[l] = row < t ? ((unsigned)row * (unsigned)k + (unsigned)piece * 8u) * 2u : W4_OOB;
    }
    constexpr int LDX = WN > 1 ? 128 : MOE_LDX;
    _Float16* const xg = xs + kg * (NBUF * ROWS * LDX);
    _Float16* const x_put = xg + (4 * wn + q) * LDX + c * 8;
    unsigned x_get[4];  // halves: operand of MFMA w, row c of a 16-row block
#pragma unroll
    for (int w = 0; w < 4; w++) x_get[w] = (unsigned)(c * LDX + (WN > 1 ? (w * 4 + q) ^ c : w * 4 + q) * 8);
    typedef __attribute__((address_space(3))) char lds_char_t;

    struct Stage {
        u4_t q[2];
        u2_t s[SL];
    } stage[2];
    u4_t xreg[WN > 1 ? 1 : XL];
    auto load_w = [&](Stage& s_, int kt) {
        const bool live = kt < kt1;
        const __amdgpu_buffer_rsrc_t qr = w4_make_rsrc(qt, live ? q_bytes : 0u), sr = w4_make_rsrc(st, live ? s_bytes : 0u);
#pragma unroll
        for (int rb = 0; rb < 2; rb++) s_.q[rb] = __builtin_amdgcn_raw_buffer_load_b128(qr, qoff[rb], kt * 1024, 2);
#pragma unroll
        for (int l = 0; l < SL; l++) {
            if constexpr (FOLD) s_.s[l][0] = __builtin_amdgcn_raw_buffer_load_b16(sr, soff[l], kt * (GPT * 32), 0);
            else s_.s[l] = __builtin_amdgcn_raw_buffer_load_b64(sr, soff[l], kt * (GPT * 32), 0);
        }
    };
    auto load_x = [&](int kt, int buf) {
        const __amdgpu_buffer_rsrc_t xr = w4_make_rsrc(x, kt < kt1 ? x_bytes : 0u);
#pragma unroll
        for (int l = 0; l < XL; l++) {
            if constexpr (WN > 1) {
                if (4 * TT % WN == 0 || wn + l * WN < 4 * TT)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(
                        xr, (__attribute__((address_space(3))) void*)((lds_char_t*)xg + (buf * ROWS + 4 * (wn + l * WN)) * 256), 16, xoff[l],
                        kt * (W4_TILE_K * 2), 0, 0);
            } else {
                xreg[l] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[l], kt * (W4_TILE_K * 2), 0);
            }
        }
    };
    auto store_x = [&]() {
#pragma unroll
        for (int l = 0; l < XL; l++) *reinterpret_cast<u4_t*>(x_put + l * 4 * LDX) = xreg[l];
    };
    f4_t acc[2][TT];
#pragma unroll
    for (int rb = 0; rb < 2; rb++)
#pragma unroll
        for (int tt = 0; tt < TT; tt++) acc[rb][tt] = (f4_t){0.f, 0.f, 0.f, 0.f};

    auto compute = [&](const Stage& s_, int buf) {
        const _Float16* xb = xg + buf * (ROWS * LDX);
        const f4_t zero = {0.f, 0.f, 0.f, 0.f};
        f4_t part[2][TT];
        unsigned fold[2][4];  // FOLD: f16 scales of the lane's weight row, per row block and MFMA
        if constexpr (FOLD) {
#pragma unroll
            for (int rb = 0; rb < 2; rb++) w4_spread_groups(SBF ? w4_bf16_to_f16(s_.s[rb][0]) : s_.s[rb][0], fold[rb]);
        }
        auto scaled = [&](int rb, unsigned d0, unsigned d1) {
            const f4_t sc = mid_scale4<SBF>(d0, d1);
#pragma unroll
            for (int tt = 0; tt < TT; tt++) acc[rb][tt] = w4_fma4(sc, part[rb][tt], acc[rb][tt]);
        };
#pragma unroll
        for (int w = 0; w < 4; w++) {
            h8_t b[TT];
#pragma unroll
            for (int tt = 0; tt < TT; tt++) b[tt] = *reinterpret_cast<const h8_t*>(xb + x_get[w] + tt * 16 * LDX);
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                if constexpr (FOLD) {
                    const h8_t a = w4_deq8_scaled(s_.q[rb][w], fold[rb][w]);
#pragma unroll
                    for (int tt = 0; tt < TT; tt++)
                        part[rb][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[tt], w == 0 ? zero : part[rb][tt], 0, 0, 0);
                    continue;
                }
                const h8_t a = w4_deq8(s_.q[rb][w]);
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
                    part[rb][tt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[tt], (G == 32 || w == 0) ? zero : part[rb][tt], 0, 0, 0);
            }
            if constexpr (G == 32 && !FOLD) {
#pragma unroll
                for (int rb = 0; rb < 2; rb++) {
                    const u2_t s2 = s_.s[rb];
                    unsigned d0, d1;
                    if (w == 0) d0 = mid_quad_bcast<0>(s2[0]), d1 = mid_quad_bcast<0>(s2[1]);
                    if (w == 1) d0 = mid_quad_bcast<1>(s2[0]), d1 = mid_quad_bcast<1>(s2[1]);
                    if (w == 2) d0 = mid_quad_bcast<2>(s2[0]), d1 = mid_quad_bcast<2>(s2[1]);
                    if (w == 3) d0 = mid_quad_bcast<3>(s2[0]), d1 = mid_quad_bcast<3>(s2[1]);
                    scaled(rb, d0, d1);
                }
            }
        }
        if constexpr (FOLD) {
#pragma unroll
            for (int rb = 0; rb < 2; rb++)
#pragma unroll
                for (int tt = 0; tt < TT; tt++) acc[rb][tt] += part[rb][tt];
        }
        if constexpr (G == 128) {
            scaled(0, mid_quad_bcast<0>(s_.s[0][0]), mid_quad_bcast<0>(s_.s[0][1]));
            scaled(1, mid_quad_bcast<1>(s_.s[0][0]), mid_quad_bcast<1>(s_.s[0][1]));
        }
    };

    // Parts: the slice's k tiles in MID_PARTS equal runs, each summed from zero, the sums added in order.  A wave with
    // several parts keeps the sum of the finished ones in its LDS slot.
    constexpr unsigned XB = (unsigned)(WK * NBUF * ROWS * LDX) * 2u, OB = WK > 1 ? WK * WN * 2 * TT * 1024u : 0u;
    f4_t* const red = reinterpret_cast<f4_t*>(xs);
    f4_t* const slot = red + (XB > OB ? XB : OB) / 16 + wave * (2 * TT * 64) + lane;
    int done = 0, left = per;
    auto part_end = [&]() {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                f4_t* const p = slot + (rb * TT + tt) * 64;
                if (done == 0) *p = acc[rb][tt];
                else *p = *p + acc[rb][tt];
                acc[rb][tt] = (f4_t){0.f, 0.f, 0.f, 0.f};
            }
        done++;
        left = per;
    };
    const int iters = PPW * per;
    if constexpr (WN > 1) {
        // one k tile ahead: its DMA and weights are issued ahead of this tile's MFMAs and all waited for at the barrier that
        // ends them
        load_x(kt0, 0);
        load_w(stage[0], kt0);
        w4_dma_barrier();
        for (int i0 = 0; i0 < iters; i0 += 2) {
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const int kt = kt0 + i0 + d;
                load_x(kt + 1, d ^ 1);
                load_w(stage[d ^ 1], kt + 1);
                __builtin_amdgcn_sched_barrier(0);
                if (kt < kt1) compute(stage[d], d);
                if (PPW > 1 && --left == 0 && done < PPW - 1) part_end();
                w4_dma_barrier();
            }
        }
    } else {
        static_assert(WN > 1 || PPW == 1, "a lone wave has one part");
        // a wave alone in its group reads what it wrote: its LDS operations run in order, no barrier
        load_x(kt0, 0);
        __builtin_amdgcn_sched_barrier(0);
        load_w(stage[0], kt0);
        load_w(stage[1], kt0 + 1);
        __builtin_amdgcn_sched_barrier(0);
        store_x();
        load_x(kt0 + 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
        for (int i0 = 0; i0 < iters; i0 += 2) {
#pragma unroll
            for (int d = 0; d < 2; d++) {
                const int kt = kt0 + i0 + d;
                if (kt < kt1) compute(stage[d], 0);
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
                store_x();
                load_x(kt + 2, 0);
                __builtin_amdgcn_sched_barrier(0);
                load_w(stage[d], kt + 2);
                __builtin_amdgcn_sched_barrier(0);
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
            }
        }
        __syncthreads();
    }
    // add the parts in order: a wave takes the token blocks tt = kg, kg + WK, .. of its unit
    if (PPW > 1 && kg == 0) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) acc[rb][tt] = slot[(rb * TT + tt) * 64] + acc[rb][tt];
    }
    if constexpr (WK > 1) {
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
                if (tt % WK != kg) red[((wave * 2 + rb) * TT + tt) * 64 + lane] = acc[rb][tt];
        __syncthreads();
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            if (tt % WK != kg) continue;
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                const f4_t mine = acc[rb][tt];
                f4_t sum;
#pragma unroll
                for (int g2 = 0; g2 < WK; g2++) {
                    const int at = (((g2 * WN + wn) * 2 + rb) * TT + tt) * 64 + lane;
                    if (PPW == 2 && g2 == 1) sum += red[(XB > OB ? XB : OB) / 16 + at];  // the second wave's first part
                    const f4_t v = g2 == kg ? mine : red[at];
                    sum = g2 == 0 ? v : sum + v;
                }
                acc[rb][tt] = sum;
            }
        }
    }
    if (!active) return;
    if (nks > 1) {
        // Hand-over between workgroups as in the decode kernel (decode.hip): device-scope stores, complete before the
        // agent-scope ticket is drawn; the wave with the last ticket reads behind an acquire fence and adds in slice order.
        // The slice offset travels in the vector offset of the stores (scalar offset 0: the compiler then inserts the wait
        // state a write to the data registers of a 16-byte store needs) and the tiles stay live until they have completed.
        const unsigned per_slice = gridDim.x * (unsigned)(WN * 2 * TT) * 1024u;
        const __amdgpu_buffer_rsrc_t wr = w4_make_rsrc(ws, per_slice * (unsigned)nks);
        const unsigned blk = blockIdx.x;
        const unsigned mine = (blk * WN + (unsigned)wn) * (2u * TT * 1024u) + (unsigned)lane * 16u;
        const unsigned park = mine + (unsigned)ky * per_slice;
        constexpr int DEV = 16;
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
                if (tt % WK == kg)
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4_t, acc[rb][tt]), wr, park + (unsigned)(rb * TT + tt) * 1024u, 0, DEV);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
        for (int rb = 0; rb < 2; rb++)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) asm volatile("" ::"v"(acc[rb][tt]));
        int ticket = 0;
        int* const tk = tickets + blk * (unsigned)(WN * WK) + wave;
        if (lane == 0) ticket = __hip_atomic_fetch_add(tk, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        ticket = __builtin_amdgcn_readfirstlane(ticket);
        if (ticket != nks - 1) return;
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
            if (tt % WK != kg) continue;
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                f4_t part[MOE_MAX_KSPLIT];
#pragma unroll
                for (int s_ = 0; s_ < MOE_MAX_KSPLIT; s_++)
                    part[s_] = __builtin_bit_cast(f4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                            s_ < nks ? wr : w4_make_rsrc(ws, 0u),
                                                            mine + (unsigned)(rb * TT + tt) * 1024u, s_ * per_slice, DEV));
                f4_t sum = part[0];
#pragma unroll
                for (int s_ = 1; s_ < MOE_MAX_KSPLIT; s_++) sum += part[s_];
                acc[rb][tt] = sum;
            }
        }
        if (lane == 0) __hip_atomic_store(tk, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
        if (tt % WK != kg) continue;
        const int m = row0 + tt * 16 + c;
        if (m >= t) continue;
        if constexpr (GLU) {
            h4_t o;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float v = w4_act_mul(acc[0][tt][i], acc[1][tt][i], act_kind);
                asm volatile("" : "+v"(v));  // the product is rounded to f32 before the f16 conversion
                o[i] = (_Float16)v;
            }
            *reinterpret_cast<h4_t*>(reinterpret_cast<_Float16*>(y) + (size_t)m * (n >> 1) + u * 16 + 4 * q) = o;
        } else {
#pragma unroll
            for (int rb = 0; rb < 2; rb++) {
                if (rb == 1 && !haveB) break;
                const f4_t a = acc[rb][tt];
                const int row = (rb == 0 ? rbA : rbB) * 16 + 4 * q;
                if (out_f16) {
                    _Float16* yo = reinterpret_cast<_Float16*>(y) + (size_t)m * n + row;
                    if (row + 3 < n) {
                        h4_t v = {(_Float16)a[0], (_Float16)a[1], (_Float16)a[2], (_Float16)a[3]};
                        *reinterpret_cast<h4_t*>(yo) = v;
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            if (row + i < n) yo[i] = (_Float16)a[i];
                    }
                } else {
                    float* yo = reinterpret_cast<float*>(y) + (size_t)m * n + row;
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
}

#define MID_KERNEL(NAME, G, SBF, GLU, TT, WN, WK, FOLD)                                                                \
    extern "C" __global__ __launch_bounds__(WN * WK * 64) __attribute__((amdgpu_waves_per_eu(MID_WPE(WN, WK)))) void NAME( \
        MID_PARAMS) {                                                                                                      \
        mid_body<G, SBF, GLU, TT, WN, WK, FOLD>(MID_ARGS);                                                                       \
    }
#define MID_WPE(WN, WK) (WN * WK > 8 ? 3 : 2)
#define MID_FAMILY(PFX, G, SBF, TT, FOLD)                         \
    MID_KERNEL(PFX##_t##TT##_n1k4, G, SBF, false, TT, 1, 4, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n1k4_glu, G, SBF, true, TT, 1, 4, FOLD)    \
    MID_KERNEL(PFX##_t##TT##_n2k4, G, SBF, false, TT, 2, 4, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n2k4_glu, G, SBF, true, TT, 2, 4, FOLD)    \
    MID_KERNEL(PFX##_t##TT##_n3k4, G, SBF, false, TT, 3, 4, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n3k4_glu, G, SBF, true, TT, 3, 4, FOLD)    \
    MID_KERNEL(PFX##_t##TT##_n4k1, G, SBF, false, TT, 4, 1, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n4k1_glu, G, SBF, true, TT, 4, 1, FOLD)    \
    MID_KERNEL(PFX##_t##TT##_n4k2, G, SBF, false, TT, 4, 2, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n4k2_glu, G, SBF, true, TT, 4, 2, FOLD)    \
    MID_KERNEL(PFX##_t##TT##_n5k2, G, SBF, false, TT, 5, 2, FOLD)       \
    MID_KERNEL(PFX##_t##TT##_n5k2_glu, G, SBF, true, TT, 5, 2, FOLD)
#define MID_FAMILIES(PFX, G, SBF, FOLD) MID_FAMILY(PFX, G, SBF, 2, FOLD) MID_FAMILY(PFX, G, SBF, 3, FOLD) MID_FAMILY(PFX, G, SBF, 4, FOLD)
MID_FAMILIES(w4a16_mid_g128_f16, 128, false, false)
MID_FAMILIES(w4a16_mid_g128_bf16, 128, true, false)
MID_FAMILIES(w4a16_mid_g32_f16, 32, false, false)
MID_FAMILIES(w4a16_mid_g32_bf16, 32, true, false)
MID_FAMILIES(w4a16_mid_g32_bf16x, 32, true, true)
