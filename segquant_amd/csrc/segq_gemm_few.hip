// Instances of the GEMM kernel for launches of few tiles.
#include <type_traits>
#include "segq_gemm_few.h"
namespace segq {

// Tile for a launch of few tiles, or -1 where the other kernels serve it better.  Both sides are estimated in us from
// launches with weights from memory; K in steps of 128.  The constants were fitted over 220 launches of 8-bit codes of 24 to
// 700 rows, 1152 to 9216 columns and K of 1152 to 12288, and 170 of int4 codes: on other sizes the choice is 3.0 % from the best on
// the mean, int4 1.6 %, with group factors 5.4 % (the fitted ones 18 % and int4 6 % with constants of one tile a CU:
// 200 x 1536 x 6144 44.6 -> 14.2 us, 128 x 4096 x 4096 22.1 -> 13.3, e4m3 500 x 2048 x 2048 17.9 -> 10.7, int4 154 x 2560 x 2560
// 11.8 -> 8.5, 320 x 6144 x 3072 30.4 -> 24.3).  `other_us`: what the 8-wave tiles for a ragged K would take, where they serve it.
int choose_few(int64_t m, int64_t n, int64_t batch, int64_t k, int fmt, bool b4, bool grp, double other_us) {
    const int64_t cus = device_cus(), steps = (k + 127) / 128;
    auto tiles = [&](int64_t bm, int64_t bn) { return (m + bm - 1) / bm * ((n + bn - 1) / bn) * batch; };
    if (tiles(32, 64) > 32 * cus) return -1;
    // this kernel: a launch, rounds of the CUs (half way from the exact share to whole rounds: two workgroups run on a CU, but
    // not every CU has two), each with a start and the tile's operand bytes, and the weights from memory.  Three ways the units
    // of a wave come in: two in flight in all, all three or four, a loop.
    struct Fit { double start, round, per_kb, per_mb; };
    static constexpr Fit FITS[3][4][3] = {
        {{{2.0, 2.0, 0.0068, 0.13}, {2.1, 2.1, 0.0070, 0.14}, {2.2, 2.2, 0.0124, 0.193}},          // 8-bit weights: 16 x 32
         {{3.4, 2.05, 0.003, 0.144}, {2.1, 2.2, 0.0126, 0.213}, {3.7, 1.7, 0.0121, 0.258}},        // 16 x 64
         {{3.05, 1.7, 0.0047, 0.12}, {3.3, 0.45, 0.015, 0.152}, {4.05, 1.45, 0.0153, 0.207}},      // 32 x 32
         {{3.7, 2.35, 0.0042, 0.152}, {1.8, 4.95, 0.0066, 0.21}, {2.75, 1.8, 0.0153, 0.172}}},     // 32 x 64
        {{{3.1, 0.6, 0.0105, 0.089}, {3.6, 0.05, 0.0219, 0.004}, {3.1, 0.85, 0.0128, 0.105}},      // int4 weights
         {{3.1, 0.95, 0.0131, 0.096}, {4.7, 0.55, 0.0162, 0.017}, {4.9, 1.15, 0.0112, 0.128}},
         {{3.15, 0.8, 0.0121, 0.071}, {3.9, 0.95, 0.0133, 0.0}, {4.05, 1.1, 0.0113, 0.084}},
         {{2.85, 1.6, 0.0141, 0.087}, {4.0, 4.35, 0.0087, 0.034}, {1.4, 4.45, 0.0129, 0.128}}},
        {{{3.05, 0.55, 0.0166, 0.11}, {3.35, 0.9, 0.0154, 0.072}, {4.0, 0.5, 0.017, 0.062}},       // ... with group factors
         {{3.15, 0.8, 0.0215, 0.105}, {3.1, 0.0, 0.0369, 0.033}, {3.05, 3.95, 0.0119, 0.177}},
         {{3.0, 0.8, 0.0178, 0.033}, {3.55, 0.0, 0.0257, 0.041}, {2.8, 3.3, 0.0124, 0.114}},
         {{3.5, 0.35, 0.0331, 0.128}, {1.3, 7.1, 0.0, 0.129}, {2.4, 3.8, 0.0189, 0.069}}}};
    int best = -1;
    double cost = 0;
    for (int c = FIRST_FEW_CFG; c < FIRST_KT_CFG; ++c) {
        const int tm = TILE_CFGS[c].bm / 16, tn = TILE_CFGS[c].bn / 16;
        if (m <= 16 && tm > 1) continue;  // rows of padding
        const int64_t t = tiles(TILE_CFGS[c].bm, TILE_CFGS[c].bn), per_wave = (steps + FEW_WAVES - 1) / FEW_WAVES;
        const int units = per_wave <= few_depth(tm, tn, b4, grp) ? (int)per_wave : 0;
        const double bytes = (TILE_CFGS[c].bm + TILE_CFGS[c].bn * (b4 ? 0.5 : 1.0)) * 128.0 * steps, share = (double)t / cus;
        const Fit& f = FITS[b4 ? grp ? 2 : 1 : 0][c - FIRST_FEW_CFG][units == 0 ? 2 : units > 2 ? 1 : 0];
        const double rounds = share > 1.0 ? 0.5 * (share + (double)((t + cus - 1) / cus)) : 1.0;
        const double us = f.start + rounds * (f.round + f.per_kb * bytes * 1e-3) + f.per_mb * (double)n * k * batch * 1e-6;
        if (best < 0 || us < cost) {
            best = c;
            cost = us;
        }
    }
    // the others: so much per K step and round of the CUs
    const int64_t t128 = tiles(128, 128), rounds = (t128 + cus - 1) / cus;
    if (b4) {  // with the expansion of the weights in front
        const double nk = (double)n * k * batch;
        return cost < 0.95 * (grp ? 7.0 + 0.72 * steps * (double)((t128 + 2 * cus - 1) / (2 * cus)) + nk / 2.5e6 : 6.5 + 0.62 * steps * rounds + nk / 2.2e6) ? best : -1;
    }
    const double full = (double)tiles(64, 128) / (1.5 * cus);
    double other = 8.0 + 0.75 * steps * (full > 1.0 ? full : 1.0);  // the general kernel, 64 x 128
    if (k % 128 == 0) {
        // the 8-wave kernels: int8 that fits the CUs once has four or five stages of LDS, and 96 columns where they divide n
        double area = (steps + 6.0) * 64 * 128 / 0.5, keep = 0.92;
        if (t128 >= 32) {
            const bool stages = fmt == GEMM_I8 && rounds == 1, narrow = stages && n % 96 == 0 && (m + 127) / 128 * (n / 96) * batch <= cus;
            other = 6.0 + (stages ? 0.5 : fmt == GEMM_F8 ? 0.8 : 0.6) * steps * rounds;
            area = (steps + 6.0) * 128 * (narrow ? 96 : 128) / 0.7 * rounds;
            if (stages && steps <= 12) keep = 0.72;  // 256 x 2176 x 1536 is asserted to stay: 9.7 us, 8.2 here
        }
        // ... and in K shares, where their rule takes those (the sums of the shares pass through memory)
        const int64_t t = m <= 128 ? t128 : tiles(256, 192), fit = cus / t < steps / 8 ? cus / t : steps / 8, s = fit < 16 ? fit : 16;
        if (batch == 1 && steps >= 16 && s >= 2 && ((double)steps / s + 14.0) * (m <= 128 ? 128 * 128 / 0.7 : 256 * 192 / 0.95) < area) {
            other = 13.0 + (m <= 128 ? 0.45 : 0.9) * steps / s + (double)n * k / 5.5e6 + (double)s * m * n / 0.75e6;
            // asserted to stay in shares: 64 x 9216 x 3072 in three (18 us, 14 here), 512 x 1024 x 8192 in eight (29 and 14)
            keep = s <= 3 || (m > 256 && steps >= 64) ? 0.65 : 0.92;
        }
        other *= keep;
    }
    if (other_us < other) other = other_us;
    return cost < other ? best : -1;
}

int launch_gemm_few(const GemmParams& g, int fmt, bool b4, int cfg, int64_t batch, hipStream_t st, const segq_quant_desc* q) {
    if (g.dry) return SEGQ_OK;
    const KRange& r = g.r[0];
    FewParams p = {r.a_sel == 1 ? g.A2 : g.A, g.B, g.C, r.sx, r.sw, g.bias, g.addend, g.grw,
                         g.lda, g.ldb, g.ldc, g.ldadd, g.grw_gs, g.bsA, g.bsB, g.bsC, g.bsSx, g.bsSw,
                         g.M, g.N, r.k0, r.k1, r.sx_rs, r.sw_cs, g.tiles_m, g.tiles_n, g.out_dtype, g.bias_dtype, g.vec_store, g.vec_add,
                   nullptr, nullptr, nullptr, 0, 0, 0, 0, 0, 0};
    if (q) {
        p.X = q->x;
        p.q_scale = q->scale;
        p.codes = static_cast<uint8_t*>(q->codes);
        p.ldx = q->ldx;
        p.ld_codes = q->ld_codes;
        p.x_dtype = q->x_dtype;
        p.q_rs = (int32_t)q->row_stride;
        p.dynamic = q->dynamic;
    }
    const int f = cfg - FIRST_FEW_CFG;
    if (fmt == GEMM_F8) return launch_few_format<GEMM_F8, false, false>(p, f, batch, st);
    if (!b4) return launch_few_format<GEMM_I8, false, false>(p, f, batch, st);
    return p.grw ? launch_few_format<GEMM_I8, true, true>(p, f, batch, st) : launch_few_format<GEMM_I8, true, false>(p, f, batch, st);
}
}  // namespace segq
