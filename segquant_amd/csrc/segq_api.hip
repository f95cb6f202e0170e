// C ABI of libsegq: argument checks, kernel selection, launches.
#include "segq_gemm_kernel.h"
#include <string.h>
#include <atomic>

namespace segq {

static thread_local char g_err[512] = "";

int fail(int status, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return status;
}

int check_launch(const char* what) {
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(SEGQ_ERR_LAUNCH, "%s: %s", what, hipGetErrorString(e));
    return SEGQ_OK;
}

int device_cus() {
    static std::atomic<int> cus[64];
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
    int n = cus[dev].load(std::memory_order_relaxed);
    if (n == 0) {
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cus[dev].store(n, std::memory_order_relaxed);
    }
    return n;
}

int reserve_lds(const void* kern, int bytes, unsigned long long* done) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) dev = 0;
    const unsigned long long bit = 1ull << (dev & 63);
    if (__atomic_load_n(done, __ATOMIC_ACQUIRE) & bit) return SEGQ_OK;
    // (the call is idempotent: two threads that both find the bit clear both make it)
    if (hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess)
        return fail(SEGQ_ERR_LAUNCH, "segq_gemm: cannot reserve %d bytes of LDS", bytes);
    __atomic_fetch_or(done, bit, __ATOMIC_RELEASE);
    return SEGQ_OK;
}

int quantize_impl(const segq_quant_desc* d, hipStream_t st, const float* scale_by_value);
int quantize_check(const segq_quant_desc* d);
int quantize_many_impl(const segq_quant_desc* descs, int32_t n, hipStream_t st);
int fake_e4m3_impl(const void* x, void* out, int32_t dtype, int64_t numel, hipStream_t st);
int quantize_groups_impl(const void* w, int32_t w_dtype, int64_t n, int64_t k, void* codes, int32_t fmt, const float* scales,
                         int64_t group, hipStream_t st);
int lowrank_rows_impl(const void* x, int64_t ldx, const void* l1t, int64_t ldl, void* t, int64_t ldt, int64_t m, int64_t k, int64_t r, int32_t dtype,
                      hipStream_t st);
int repack_i4_impl(const void* colpacked, void* rowpacked, int64_t out, int64_t cols, hipStream_t st);

static bool is_float_dtype(int t) { return t == SEGQ_F32 || t == SEGQ_F16 || t == SEGQ_BF16; }
static bool al(const void* p, uintptr_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// Tile choice when the caller leaves it to the library.  The 8-wave kernels need
// K in whole 128-byte steps and 32-bit row offsets.  A launch runs in rounds of
// one tile per CU, so its time goes as rounds x tile area x a per-tile weight
// (smaller tiles move more operand bytes per MAC: measured on M = 4608, 216
// tiles of 256 x 256 beat 432 tiles of 256 x 128 by 30 %).  The 192 x 288 and
// 288 x 192 tiles exist because 4608 rows of FLUX tokens make whole rounds with
// them where 256 x 256 leaves the last round half empty.
static int choose_tile(int64_t m, int64_t n, int64_t batch, bool fold, bool wide_ok, bool plain8, int64_t k_steps = 1 << 20,
                       bool big_ok = false) {  // fold: needs a second accumulator set; big_ok: 384 x 192 serves this launch
    auto tiles = [&](int cfg) {
        const TileCfg& c = TILE_CFGS[cfg];
        return ((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * batch;
    };
    // (plain 8-bit operands go to the 8-wave kernels from 32 tiles of 128 x 128 up: 64 x 9216 x 3072 runs
    // 24.9 us there against 35.2 us on the general kernel; with a second accumulator set, both ranges of a
    // DualScale 512 x 1024 x 1024 17.9 against 25.8 us, quantising included, and 512 x 1024 x 256 10.5 against 14.2)
    if (wide_ok && tiles(FIRST_WIDE_CFG + 3) >= (plain8 ? 32 : 96)) {
        // Short contractions of middling size: the plain 128 x 128 kernel needs ~100 registers, so two
        // workgroups share a CU and each one's prologue and epilogue (most of a tile's time at a dozen
        // K steps) run under the other's MFMAs.  Measured at K = 1280 .. 1536: 2048 x 10240 34.5 vs 45.5 us
        // and 4096 x 6144 44.7 vs 47-50 us for the rule below's choice; 8192 x 10240 (1280 tiles of
        // 256 x 256, five whole rounds) stays 20 % better on the big tile.
        if (plain8 && !fold && k_steps <= 12 && tiles(FIRST_WIDE_CFG) <= 512 && tiles(FIRST_WIDE_CFG + 3) >= 512) {
            // ... unless 256 x 192 tiles make whole rounds of the CUs exactly (4096 x 6144 x 1536: 512 tiles,
            // 46.4 against 50.8 us in e4m3, 48.5 against 50.8 in int8)
            const int c = FIRST_WIDE_CFG + 6;
            if (m % TILE_CFGS[c].bm == 0 && n % TILE_CFGS[c].bn == 0 && tiles(c) % device_cus() == 0) return c;
            return FIRST_WIDE_CFG + 3;
        }
        static const double weight[6] = {1.0, 1.18, 1.18, 1.45, 1.04, 1.04};
        const int64_t cus = device_cus();
        int best = -1;
        double best_cost = 0;
        for (int i = 0; i < 6; ++i) {
            if (i == 0 && fold) continue;                  // no 256 x 256 with a second accumulator set
            if (i >= 4 && (fold || !plain8)) continue;  // plain int8 or e4m3 operands, one range only
            const int cfg = FIRST_WIDE_CFG + i;
            const int64_t rounds = (tiles(cfg) + cus - 1) / cus;
            const double cost = (double)rounds * TILE_CFGS[cfg].bm * TILE_CFGS[cfg].bn * weight[i];
            if (best < 0 || cost < best_cost) {
                best = cfg;
                best_cost = cost;
            }
        }
        // 384 x 192, eight wave tiles of 96 x 96 (the fewest LDS bytes per MFMA of all tiles): taken when
        // it tiles the output exactly, in whole rounds of the CUs, and with no more rounds x area than
        // the choice above.  4608 x 12288 x 3072: three rounds instead of four of 288 x 192, e4m3 165 ->
        // 140 us; 8192^3, which it does not tile exactly, is 12 % slower on it than on 256 x 256
        const int big = FIRST_WIDE_CFG + 9;
        if (big_ok && plain8 && !fold && batch == 1 && m % TILE_CFGS[big].bm == 0 && n % TILE_CFGS[big].bn == 0 && tiles(big) % cus == 0) {
            const TileCfg& t = TILE_CFGS[best];
            const int64_t rounds = (tiles(best) + cus - 1) / cus;
            if (tiles(big) / cus * TILE_CFGS[big].bm * TILE_CFGS[big].bn <= rounds * t.bm * t.bn) return big;
        }
        return best;
    }
    return tiles(2) >= 256 ? 2 : 3;
}

// A tile that walks K once (segq_gemm_wide.h, launch_walk) and what the launch takes with it, in us, from times on 60 shapes
// (within 20 %): so much per step of 128 and per round of the CUs.
struct Walk {
    int cfg;
    double us;
};

static int64_t tiles_of_cfg(int cfg, int64_t m, int64_t n, int64_t batch) {
    const TileCfg& c = TILE_CFGS[cfg];
    return (m + c.bm - 1) / c.bm * ((n + c.bn - 1) / c.bn) * batch;
}

// One range, K not in whole steps.  (Rows of such a K start anywhere in a cache line: a step costs more than an aligned one's.)
//   us, general kernel before / 256 x 256 / 256 x 192 / 128 x 128:  4900 x 5900 x 4912 270 / 170 / 209 / 231;
//   4000 x 3000 x 2064 66 / 41 / 37 / 46;  2000 x 3000 x 1008 25.1 / 25.2 / 20.6 / 15.3;  1200 x 3000 x 800 16.2 / 25.4 / 18.8 / 11.1
// `scattered`: fp32 outputs whose rows do not start on the boundaries of whole stores are written value by value, which costs a
// 128 x 128 tile of these kernels more than one of the general kernel (64 x 128): a short K stays with that (cfg -1) while its tiles
// fit the CUs once.  us, 128 x 128 / general: 748 x 383 x 208 9.0 / 7.6; 869 x 479 x 160 9.2 / 7.9; 762 x 2595 x 1264 18.5 / 20.6.
// Of 971 such launches 2.8 % are slower than on the general kernel by 3 % or more, 42 % without this line (16-bit outputs: 0.4 %).
static Walk choose_ragged(int64_t m, int64_t n, int64_t batch, int64_t k, bool scattered) {
    const double steps = (double)((k + 127) / 128);
    const int64_t cus = device_cus();
    auto rounds = [&](int cfg) { return (double)((tiles_of_cfg(cfg, m, n, batch) + cus - 1) / cus); };
    Walk w{FIRST_KT_CFG + 2, 4.2 + 0.72 * steps * rounds(FIRST_KT_CFG + 2)};
    const bool full = tiles_of_cfg(FIRST_KT_CFG + 1, m, n, batch) * 4 > cus * 3;
    // (idle CUs, and at most two rounds of 128 x 128 tiles: 722 x 5554 x 2320 45 us on 256 x 192, 34 on 128 x 128 and 43 on the
    // general kernel; 415 launches that go to 128 x 128 by this are 0.1 % from the best tile, 20 % with 1.15)
    const bool two = tiles_of_cfg(FIRST_KT_CFG + 2, m, n, batch) <= 2 * cus;
    const double us192 = rounds(FIRST_KT_CFG + 1) * ((full ? 1.72 : two ? 1.42 : 1.15) * steps + 9.0);
    if (us192 < w.us) w = Walk{FIRST_KT_CFG + 1, us192};
    const double us256 = rounds(FIRST_KT_CFG) * (2.0 * steps + 6.0);
    if (us256 < w.us) w = Walk{FIRST_KT_CFG, us256};
    if (scattered && w.cfg == FIRST_KT_CFG + 2 && tiles_of_cfg(3, m, n, batch) <= cus) {
        auto rows = [&](int cfg) { return m < TILE_CFGS[cfg].bm ? (double)m / TILE_CFGS[cfg].bm : 1.0; };  // of a tile, that are stored
        if (1.03 * (6.2 + 1.04 * steps + rows(3)) < 4.8 + 0.83 * steps + 3.7 * rows(w.cfg)) w.cfg = -1;
    }
    return w;
}

// DualScale's two ranges.  us, second register set before / 128 x 192 / 64 x 128:  2 x 2048 x 1536 x 3072 54.8 / 35.6 / 43.1;
//   3000 x 3000 x 1024 46.3 / 30.8 / 28.4;  2 x 500 x 2000 x 2048 24.9 / 22.5 / 15.4;  merged tensor before, K not in whole
//   steps: 3 x 2800 x 2000 x 960 166 / 53.6 / 52.6;  2 x 200 x 1000 x 992 21.9 / 14.7 / 8.4.  Below 257 or, in whole steps, 513
//   the ranges stay in turn (3000 x 2000 x 512 20.1, 64 x 128 15.7): the tests assert the tiles of those launches
static Walk choose_dual(int64_t m, int64_t n, int64_t batch, int64_t k) {
    const double steps = (double)((k + 127) / 128);
    const int64_t cus = device_cus(), t64 = tiles_of_cfg(FIRST_DUAL_CFG + 1, m, n, batch), t192 = tiles_of_cfg(FIRST_DUAL_CFG, m, n, batch);
    Walk w{FIRST_DUAL_CFG + 1, 4.0 + (double)((t64 + cus - 1) / cus) * ((t64 <= cus ? 0.6 : 0.5) * steps + 0.8)};
    const double us192 = (double)((t192 + cus - 1) / cus) * (1.3 * steps + 5.5);
    if (us192 < w.us) w = Walk{FIRST_DUAL_CFG, us192};
    return w;
}

// K shares of the steps of `cfg`'s tiles, and the tile that takes them (cfg and 1: none).
// Whole tiles would leave more than a tenth of the CUs idle: look for a big tile and a
// number of shares that fill them.  Measured (us, random codes, 256 CUs):
//   1024 x 3072, K 13824 twice (DualScale):  e4m3  256x192 x4 99 | 256x256 x5 130 | 128x128 176
//                                            int8  256x192 x4 108 | 256x256 x4 125 | 128x128 184
//   4096 x 1536, K 6144 twice:               e4m3  256x192 x2 85 | 256x256 x2 94 | 256x128 123
// The choice minimises rounds x (K steps per share + fixed cost) x tile area / efficiency:
// about 6 steps' worth of prologue and epilogue per workgroup, 8 more for the shares' trip
// through memory; big tiles get more out of every byte they stream.
struct Shares {
    int cfg, n;
};

static Shares choose_shares(int64_t m, int64_t n, int64_t total_steps, int cfg, bool big_ok, bool sep, bool parks) {
    const int64_t cus = device_cus();
    Shares pick{cfg, 1};
    if (total_steps < 16 || tiles_of_cfg(cfg, m, n, 1) * 10 >= cus * 9) return pick;
    auto eff = [](int c) {
        const int area = TILE_CFGS[c].bm * TILE_CFGS[c].bn;
        return c < FIRST_WIDE_CFG ? 0.5 : area >= 256 * 256 ? 1.0 : area >= 256 * 192 ? 0.95 : area >= 256 * 128 ? 0.85 : 0.7;
    };
    auto cost = [&](int c, int64_t s_) {
        const int64_t wgs = tiles_of_cfg(c, m, n, 1) * s_;
        return (double)((wgs + cus - 1) / cus) * ((double)total_steps / s_ + 6.0 + (s_ > 1 ? 8.0 : 0.0)) *
               TILE_CFGS[c].bm * TILE_CFGS[c].bn / eff(c);
    };
    // (the 128 x 128 tile joins for very few tokens: 64 x 9216 x 3072 in two or three shares
    // 19 us against 25 us whole)
    const int cands[4] = {FIRST_WIDE_CFG + 6, FIRST_WIDE_CFG, FIRST_WIDE_CFG + 7, FIRST_WIDE_CFG + 3};
    double best = cost(cfg, 1);
    for (int i = 0; i < (big_ok ? 4 : sep ? 2 : 1); ++i) {
        const int c = big_ok ? cands[i] : FIRST_WIDE_CFG + (i == 0 ? 1 : 3);
        if (c == FIRST_WIDE_CFG + 3 && (m > 128 || parks)) continue;
        int64_t s_ = cus / tiles_of_cfg(c, m, n, 1);
        if (s_ > total_steps / 8) s_ = total_steps / 8;
        if (s_ > 16) s_ = 16;
        if (s_ < 2) continue;
        if (cost(c, s_) < best) {
            best = cost(c, s_);
            pick = Shares{c, (int)s_};
        }
    }
    return pick;
}

// Group factors: us, of what the outputs take (x: rounds of the CUs that they would be without ragged tiles) and of the rounds that
// the tiles take, per step and beside the steps; fp32 outputs are bound by their stores as well, and a tile with ragged columns
// takes longer than whole ones.  Fitted to 1379 shapes of 200 to 8192 rows (rms 5 to 7 %).  Two workgroups of 128 x 128 share
// a CU and flow on from round to round, so their rounds count by halves.  A big tile has to be ahead by more than the fit is off where
// it matters, fp32 by more: of the shapes 20 are then slower than 128 x 128 by 2 % (at most 11 %), and all 2 to 3 % faster in the mean (52
// and 21 % with rounds alone in the sum).  us, 128 x 128 / 256 x 256 / 256 x 192 / 192 x 256:  8192 x 10240 x 1280 166 / 155 / 160 / 158;
// 8192 x 1280 x 5120 81 / 85 / 75 / 69;  4096 x 12288 x 1536 117 / 108 / 117 / 128;  2048 x 10240 x 1280 50 / 59 / 53 / 53;  2048 x 1280 x 5120 37 / 83 /
// 70 / 65;  4774 x 7680 x 384 35 / 45 / 36 / 42;  6105 x 6912 x 2176 fp32 141 / 151 / 151 / 161.
// (256 x 128 and 128 x 256, by id: never the best by more than 3 %.)
static int choose_groups(int64_t m, int64_t n, int64_t k_steps, bool fold, bool f32) {
    const int64_t cus = device_cus(), t128 = tiles_of_cfg(FIRST_WIDE_CFG + 3, m, n, 1);
    if (fold || 8 * t128 <= 5 * cus) return FIRST_WIDE_CFG + 3;
    const double s = (double)k_steps, outs = (double)m * (double)n / (double)cus, f = f32 ? 1.0 : 0.0;
    const double x128 = outs / (2 * 128 * 128), half = 0.5 * (double)((t128 + cus - 1) / cus);
    double us = (f32 ? 0.94 : 0.985) * ((0.37 * s + 3.32 + 3.76 * f) * x128 + (0.84 * s + 0.27) * half + 5.3);
    int best = FIRST_WIDE_CFG + 3;
    static const struct { int tile; double x_step, x, x_f32, step, tail, ragged; } big[3] = {
        {0, 0.63, 0.71, 7.58, 1.56, 9.14, 2.5}, {6, 0.36, 0.0, 5.16, 1.24, 8.47, 1.18}, {7, 0.42, 0.0, 5.83, 1.11, 8.66, 1.09}};
    for (const auto& b : big) {
        const TileCfg& c = TILE_CFGS[FIRST_WIDE_CFG + b.tile];
        const double x = outs / (c.bm * c.bn), rounds = (double)((tiles_of_cfg(FIRST_WIDE_CFG + b.tile, m, n, 1) + cus - 1) / cus);
        const double t = (b.x_step * s + b.x + b.x_f32 * f) * x + (b.step * s + b.tail) * rounds + (n % c.bn ? b.ragged * (1.0 + f) : 0.0);
        if (t < us) {
            us = t;
            best = FIRST_WIDE_CFG + b.tile;
        }
    }
    return best;
}

// Workgroups that could share the K steps of each of a launch's tiles (1: none).
static int64_t k_shares(int64_t m, int64_t n, int64_t steps, int cfg) {
    const int64_t cus = device_cus(), t = tiles_of_cfg(cfg, m, n, 1);
    if (t * 10 >= cus * 9) return 1;
    int64_t s = cus / t < steps / 8 ? cus / t : steps / 8;
    if (s > 16) s = 16;
    return s > 1 ? s : 1;
}

// The same two ranges in turn, rescaled in place (e4m3) or, with a workspace, in K shares or parked.  us: 4608 x 3072 x 12288 e4m3
// 265 in place, 321 in one walk; 400 x 3072 x 12288 52 in eight shares, 80 in one walk; 4096 x 1536 x 6144 78 in two shares, 62 in
// one walk, int8 88 and 65; 2000 x 2048 x 8192 96 and 61, int8 101 and 63.
static double in_turn_us(int64_t m, int64_t n, int64_t steps, bool f8, bool ws) {
    const int64_t cus = device_cus();
    double us = 1e30;
    if (ws) {
        const bool small = m <= 128 && f8;
        const int64_t s = k_shares(m, n, steps, small ? FIRST_WIDE_CFG + 3 : FIRST_WIDE_CFG + 6);
        if (s > 1) us = 12.0 + (small ? 0.6 : 1.1) * steps / s + (double)m * n * s * 8.0 / 4e6;
    }
    if (f8 || ws) {
        double fill = 0.0;  // of the largest tiles
        for (int c : {FIRST_WIDE_CFG, FIRST_WIDE_CFG + 4, FIRST_WIDE_CFG + 5}) {
            const double rounds = (double)((tiles_of_cfg(c, m, n, 1) + cus - 1) / cus);
            const double f = (double)m * n / (rounds * cus * TILE_CFGS[c].bm * TILE_CFGS[c].bn);
            if (f > fill) fill = f;
        }
        const double whole = 8.0 + (double)m * n * 256.0 * steps / (f8 ? 2.6e9 : 2.2e9) / fill;
        if (whole < us) us = whole;
    }
    return us;
}

// What a GEMM of few tiles takes longer, in us, if each of its workgroups reads and encodes the rows of x itself: so much per
// round of the CUs, more for more bytes and rows, and less where that passes under the wait for the weights.  Fitted over 1400
// launches (rms 0.8).  A quantise launch takes 2 us of the GPU and 3.8 of the host, which small layers wait for: up to the sum
// of the two the linear stays in one launch.  us, one launch / two, on the GPU alone: 8 x 9216 x 1536 int4 bf16 6.7 / 7.9 (1.9 by
// this estimate); 16 x 9216 x 1536 fp32 dynamic 10.1 / 8.0 (5.9); 16 x 36864 x 3072 e4m3 bf16 44 / 27 (17).
static double quantise_in_gemm_us(const segq_quant_desc* q, int64_t tiles) {
    const int64_t cus = device_cus();
    const double rounds = (double)((tiles + cus - 1) / cus), k = q->cols / 1024.0;
    const bool f32 = q->x_dtype == SEGQ_F32, second = q->rows > 8;
    return rounds * (q->dynamic ? 0.9 : 0.1) + k * (rounds * (0.83 + (second ? 0.36 : 0.0) + (f32 ? second ? 0.44 : 0.12 : 0.0)) - 0.55);
}

struct MixPick {
    int cfg, shares;
    double us;
};

// Workspace of a launch in K shares on one of the MIX tiles: two tile-sized shares and a word per tile, or the partial results.
static int64_t mix_bytes(int64_t m, int64_t n, int cfg, int shares) {
    const int64_t tiles = tiles_of_cfg(cfg, m, n, 1);
    if (shares == 2) return tiles * 2 * TILE_CFGS[cfg].bm * TILE_CFGS[cfg].bn * 4 + ((tiles * 4 + 255) & ~(int64_t)255);
    return (shares * m * n * 4 + 255) & ~(int64_t)255;
}

// Tile and K shares of a DualScale pair and the plain range beside it (or none): us of rounds of the CUs, each so much per step,
// the last one less the emptier it is, a launch of one round an eighth quicker (the clock), and what shares cost.  Fitted to 50
// shapes: within 5 % of the best of three tiles and up to 12 shares on 45 of them, 12 % at most.  us, ranges in turn before / this,
// int8 | e4m3:  9216 x 3072 x (3072 + 12288) 745 / 601 | 643 / 574;  4608 361 / 316 | 299 / 296;  2048 187 / 131 | 153 / 123;
// 1024 119 / 79 | 82 / 74;  300 57 / 45 | 43 / 43;  4012 x 1536 x (1536 + 6144) 118 / 70 | 79 / 65;  366 42 / 27 | 31 / 27
static MixPick choose_mix(int64_t m, int64_t n, int64_t steps, int64_t plain, int max_shares) {
    static const struct { double full, few, tail; } fit[3] = {{1.80, 1.29, 7.0}, {1.57, 1.20, 7.0}, {1.25, 0.93, 6.5}};
    const int64_t cus = device_cus();
    const double e = (double)steps + 0.6 * (double)plain;
    MixPick best{-1, 1, 1e30};
    for (int i = 0; i < 3; ++i) {
        const int64_t tiles = tiles_of_cfg(FIRST_MIX_CFG + i, m, n, 1);
        for (int sh = 1; sh <= max_shares && (sh == 1 || (tiles * sh <= cus && e >= 8.0 * sh)); ++sh) {
            const double full = (tiles * sh <= cus ? 0.92 : 1.0) * (fit[i].full * e / sh + fit[i].tail), few = fit[i].few * e / sh + fit[i].tail;
            const double rest = (double)(tiles * sh % cus) / (double)cus;
            double us = (double)(tiles * sh / cus) * full + (rest > 0.0 ? few + rest * rest * (full - few) : 0.0);
            if (sh == 2) us += i == 2 ? 5.0 : 9.0;
            else if (sh > 2) us += 4.0 + (double)m * n * sh / 0.8e6;
            if (us < best.us) best = MixPick{FIRST_MIX_CFG + i, sh, us};
        }
    }
    return best;
}

// e4m3, DualScale beside a plain range.  One walk multiplies a step of the plain range on half of its rows' registers; the ranges in turn,
// rescaled in place, have their tiles whole for it and walk the pair twice.  us of both, for steps and output tiles in whole
// rounds and beside them, fitted to 1169 shapes of 129 to 9216 rows (rms 6 % and 5 %).  us, one walk / in turn: 1479 x 6336 x (3328 + 256)
// 62 / 45;  8950 x 1408 x (3072 + 256) fp32 77 / 56;  7940 x 4736 x (3328 + 640) fp32 245 / 203;  472 x 7424 x (3200 + 512) 32 / 26;  425 x 1280 x (256 + 256)
// 11.1 / 9.9;  4608 x 3072 x (3072 + 12288) 296 / 299.  Of the shapes 234 were slower by 2 % or more on the one walk, by up to 39 %; with this line 30 are, by up to 24 %.
// (int8 parks in turn: of 155 shapes two were slower on the one walk, by 4 %.)
static double mix_beside_us(int64_t m, int64_t n, int64_t steps, int64_t plain, const MixPick& pick, bool f32) {
    if (pick.shares > 1) return pick.us;
    static const struct { double xs, xp, rs, rp, x, r, one, x_f32; } fit[3] = {
        {0.35, 0.61, 1.11, 0.37, 0.0, 9.6, 1.1, 4.5}, {0.49, 0.43, 0.84, 0.54, 0.4, 7.3, 2.9, 4.25}, {0.08, 0.12, 0.81, 0.61, 1.2, 5.3, 2.5, 4.65}};
    const auto& w = fit[pick.cfg - FIRST_MIX_CFG];
    const TileCfg& c = TILE_CFGS[pick.cfg];
    const double cus = (double)device_cus(), s = (double)steps, p = (double)plain;
    const double x = (double)m * (double)n / (cus * c.bm * c.bn), r = std::ceil((double)tiles_of_cfg(pick.cfg, m, n, 1) / cus);
    return (w.xs * s + w.xp * p + w.x + (f32 ? w.x_f32 : 0.0)) * x + (w.rs * s + w.rp * p + w.r) * r + w.one;
}

static double beside_in_turn_us(int64_t m, int64_t n, int64_t all_steps, int cfg, bool f32) {
    static const struct { double xs, rs, x, r, one, x_f32; } fit[4] = {
        {0.0, 1.7, 4.5, 0.0, 7.1, 0.0}, {0.0, 1.15, 4.1, 0.52, 6.7, 3.9}, {0.3, 0.59, 0.0, 11.3, 0.0, 3.1}, {0.56, 0.8, 3.6, 10.1, 1.3, 6.5}};
    const TileCfg& c = TILE_CFGS[cfg];
    const int area = c.bm * c.bn;
    if (area > 192 * 288 || cfg >= NUM_TILE_CFG) return 1e30;
    const auto& w = fit[area <= 64 * 128 ? 0 : area <= 128 * 128 ? 1 : area <= 256 * 128 ? 2 : 3];
    // (two workgroups of the smaller tiles share a CU and flow on from round to round: rounds by halves)
    const double cus = (double)device_cus(), room = area <= 128 * 128 ? 2.0 * cus : cus, part = area <= 128 * 128 ? 2.0 : 1.0;
    const double x = (double)m * (double)n / (room * area), r = std::ceil(part * (double)tiles_of_cfg(cfg, m, n, 1) / room) / part;
    return (w.xs * (double)all_steps + w.x + (f32 ? w.x_f32 : 0.0)) * x + (w.rs * (double)all_steps + w.r) * r + w.one;
}

// int4 weight rows (two values per byte, even k in the low nibble) -> int8 rows.
// One thread expands 16 packed bytes to 32 values.
__global__ void __launch_bounds__(256) expand_i4_kernel(const uint8_t* src, int64_t ld_src, uint8_t* dst, int64_t ld_dst,
                                                        int64_t rows, int64_t chunks_per_row) {
    const int64_t total = rows * chunks_per_row;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
        const int64_t row = i / chunks_per_row, c = i - row * chunks_per_row;
        const uint4 v = *reinterpret_cast<const uint4*>(src + row * ld_src + c * 16);
        const uint32_t in[4] = {v.x, v.y, v.z, v.w};
        uint32_t out[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            uint32_t e = in[j] & 0x0F0F0F0Fu, o = (in[j] >> 4) & 0x0F0F0F0Fu;
            e |= (e & 0x08080808u) * 0x1Eu;  // sign-extend each nibble into its byte
            o |= (o & 0x08080808u) * 0x1Eu;
            out[2 * j] = __builtin_amdgcn_perm(o, e, 0x05010400u);      // k0 k1 k2 k3
            out[2 * j + 1] = __builtin_amdgcn_perm(o, e, 0x07030602u);  // k4 k5 k6 k7
        }
        uint4* q = reinterpret_cast<uint4*>(dst + row * ld_dst + c * 32);
        q[0] = make_uint4(out[0], out[1], out[2], out[3]);
        q[1] = make_uint4(out[4], out[5], out[6], out[7]);
    }
}

// Sum of the fp32 partial results of a split-K launch, plus bias, rounded once to the
// output type.  VEC: four columns per thread.
template <bool VEC>
__global__ void __launch_bounds__(256) splitk_reduce_kernel(const float* part, int splits, int64_t m, int64_t n, const void* bias,
                                                            int bias_dtype, void* out, int out_dtype, int64_t ldo,
                                                            const void* addend, int64_t ldadd) {
    constexpr int W = VEC ? 4 : 1;
    const int64_t per_row = n / W;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= m * per_row) return;
    const int64_t row = i / per_row, col = (i - row * per_row) * W;
    float acc[W];
#pragma unroll
    for (int v = 0; v < W; ++v) acc[v] = 0.0f;
    for (int z = 0; z < splits; ++z) {
        const float* q = part + ((int64_t)z * m + row) * n + col;
        if constexpr (VEC) {
            const float4 t = *reinterpret_cast<const float4*>(q);
            acc[0] += t.x; acc[1] += t.y; acc[2] += t.z; acc[3] += t.w;
        } else {
            acc[0] += q[0];
        }
    }
    if (bias) {
#pragma unroll
        for (int v = 0; v < W; ++v) acc[v] += load_bias(bias, bias_dtype, col + v);
    }
    if (addend) {  // same dtype as the output
        const int64_t ea = row * ldadd + col;
#pragma unroll
        for (int v = 0; v < W; ++v) acc[v] += load_bias(addend, out_dtype, ea + v);
    }
    const int64_t e = row * ldo + col;
    if (out_dtype == SEGQ_F32) {
#pragma unroll
        for (int v = 0; v < W; ++v) static_cast<float*>(out)[e + v] = acc[v];
    } else if constexpr (VEC) {
        const bool bf = out_dtype == SEGQ_BF16;
        *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + e) =
            make_uint2(bf ? pack2_bf16(acc[0], acc[1]) : pack2_f16(acc[0], acc[1]), bf ? pack2_bf16(acc[2], acc[3]) : pack2_f16(acc[2], acc[3]));
    } else {
        const uint32_t two = out_dtype == SEGQ_BF16 ? pack2_bf16(acc[0], 0.0f) : pack2_f16(acc[0], 0.0f);
        static_cast<uint16_t*>(out)[e] = (uint16_t)(two & 0xffffu);
    }
}

// What a launch would do, for callers that ask before (or instead of) launching.
struct GemmPlan {
    int64_t bytes;  // workspace it would use
    int tile;       // tile id (1-based, as in segq_gemm_desc.tile)
    int splits;     // workgroups sharing the K steps of a tile (1: none)
    int parked;     // finished ranges parked in the workspace
};

// plan != nullptr: nothing is launched; *plan says what the launch would do if the caller lent
// as much workspace as the library can make use of (probe) or with d's own workspace (!probe).
// q: a quantise step that the launch may do by itself; *fused says whether it did.  If it does not, nothing is launched.
static int gemm_impl(const segq_gemm_desc* d, hipStream_t st, GemmPlan* plan = nullptr, bool probe = true, const segq_quant_desc* q = nullptr,
                     bool* fused = nullptr) {
    const bool need = plan != nullptr && probe;
    if (plan) *plan = GemmPlan{0, 0, 1, 0};
    if (!d) return fail(SEGQ_ERR_ARG, "segq_gemm: null descriptor");
    if (d->m < 0 || d->n < 0 || d->batch < 1) return fail(SEGQ_ERR_ARG, "segq_gemm: bad sizes");
    if (d->m == 0 || d->n == 0) return SEGQ_OK;
    if (d->m > 0x7fffffff / 2 || d->n > 0x7fffffff / 2) return fail(SEGQ_ERR_ARG, "segq_gemm: m or n too large");
    const bool codes_out = d->out_codes != nullptr;
    if (!d->a || !d->b || (!d->out && !codes_out)) return fail(SEGQ_ERR_ARG, "segq_gemm: null a, b or out");
    if (codes_out) {
        if ((d->out_dtype != SEGQ_BF16 && d->out_dtype != SEGQ_F16) || d->batch != 1 || !d->out_scale || d->ld_out_codes < d->n || d->split_k > 1 ||
            (d->out_code_fmt != SEGQ_CODE_I8 && d->out_code_fmt != SEGQ_CODE_E4M3) || d->out_pre_op < 0 || d->out_pre_op > SEGQ_PRE_SILU ||
            (d->out_scale_neg != nullptr) != (d->out_codes_neg != nullptr))
            return fail(SEGQ_ERR_ARG, "segq_gemm: out_codes needs out_dtype F16 or BF16, batch == 1, ld_out_codes >= n, int8 or e4m3 codes, "
                                      "out_scale, and out_scale_neg together with out_codes_neg");
    }
    if (d->n_ranges < 1 || d->n_ranges > SEGQ_MAX_RANGES) return fail(SEGQ_ERR_ARG, "segq_gemm: n_ranges %d out of range", d->n_ranges);
    const bool i8 = d->a_fmt == SEGQ_CODE_I8 && d->b_fmt == SEGQ_CODE_I8;
    const bool f8 = d->a_fmt == SEGQ_CODE_E4M3 && d->b_fmt == SEGQ_CODE_E4M3;
    const bool w4 = d->a_fmt == SEGQ_CODE_I8 && d->b_fmt == SEGQ_CODE_I4;
    if (!i8 && !f8 && !w4) return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: no kernel for a_fmt %d with b_fmt %d", d->a_fmt, d->b_fmt);
    if (d->out_dtype != SEGQ_ACC && !is_float_dtype(d->out_dtype)) return fail(SEGQ_ERR_ARG, "segq_gemm: bad out_dtype %d", d->out_dtype);
    if (d->bias && !is_float_dtype(d->bias_dtype)) return fail(SEGQ_ERR_ARG, "segq_gemm: bad bias_dtype %d", d->bias_dtype);
    if (d->out_dtype == SEGQ_ACC && d->n_ranges != 1) return fail(SEGQ_ERR_ARG, "segq_gemm: raw accumulators need exactly one range");
    if (d->lda % 16 || d->ldb % 16 || !al(d->a, 16) || !al(d->b, 16) || (d->a_neg && !al(d->a_neg, 16)) ||
        d->batch_stride_a % 16 || d->batch_stride_b % 16)
        return fail(SEGQ_ERR_ARG, "segq_gemm: a and b need 16-byte aligned bases and row strides");
    if (!codes_out && d->ldo < d->n) return fail(SEGQ_ERR_ARG, "segq_gemm: ldo smaller than n");
    if (d->addend && (d->out_dtype == SEGQ_ACC || d->ld_addend < d->n))
        return fail(SEGQ_ERR_ARG, "segq_gemm: an addend needs a float output and ld_addend >= n");
    const bool lowrank = d->lowrank_t != nullptr || d->lowrank_rank != 0;
    if (lowrank) {
        if (!d->lowrank_t || !d->lowrank_l2t || d->lowrank_rank <= 0 || d->lowrank_rank % 32 || d->lowrank_rank > 512)
            return fail(SEGQ_ERR_ARG, "segq_gemm: the low-rank branch needs both matrices and a rank that is a multiple of 32, at most 512");
        if (d->out_dtype != SEGQ_BF16 && d->out_dtype != SEGQ_F16)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: the low-rank branch runs in the output's 16-bit dtype (out_dtype F16 or BF16)");
        if (d->ld_lowrank_t < d->lowrank_rank || d->ld_lowrank_l2t < d->lowrank_rank || d->ld_lowrank_t % 8 || d->ld_lowrank_l2t % 8 ||
            !al(d->lowrank_t, 16) || !al(d->lowrank_l2t, 16))
            return fail(SEGQ_ERR_ARG, "segq_gemm: low-rank matrices need 16-byte aligned rows of at least lowrank_rank elements");
        if (d->batch != 1 || d->split_k > 1)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: the low-rank branch needs batch == 1 and no split_k");
    }
    const bool groups = d->group_dequant != nullptr;
    if (groups) {
        if (!(i8 || w4) || d->batch != 1 || d->out_dtype == SEGQ_ACC || d->group_dequant_stride < d->n || !al(d->group_dequant, 4))
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors need int8 activations, one problem, a float output "
                                              "and a stride of at least n");
    }

    void* const ws = need ? reinterpret_cast<void*>(uintptr_t(256)) : d->workspace;
    const int64_t ws_bytes = need ? (int64_t)1 << 60 : d->workspace_bytes;
    GemmParams p;
    memset(&p, 0, sizeof(p));
    const int64_t kalign = w4 ? 32 : 16;
    int64_t kmax = 0, ktotal = 0;
    for (int i = 0; i < d->n_ranges; ++i) {
        const segq_krange& r = d->ranges[i];
        // the K rule of the reference's GEMM (segquant/src/real_quant/real_gemm.cu:237-247)
        if (r.k_begin < 0 || r.k_len <= 0 || r.k_begin % kalign || r.k_len % kalign)
            return fail(SEGQ_ERR_ARG, "segq_gemm: range %d: k_begin %lld and k_len %lld must be positive multiples of %lld",
                        i, (long long)r.k_begin, (long long)r.k_len, (long long)kalign);
        if (r.a_sel < 0 || r.a_sel > 3) return fail(SEGQ_ERR_ARG, "segq_gemm: range %d: bad a_sel %d", i, r.a_sel);
        if (r.a_sel == 1 && !d->a_neg) return fail(SEGQ_ERR_ARG, "segq_gemm: range %d reads a_neg, which is null", i);
        if (d->out_dtype != SEGQ_ACC && (!r.sx || !r.sw)) return fail(SEGQ_ERR_ARG, "segq_gemm: range %d has a null scale", i);
        if ((r.sx_row_stride | 1) != 1 || (r.sw_col_stride | 1) != 1) return fail(SEGQ_ERR_ARG, "segq_gemm: range %d: scale strides are 0 or 1", i);
        KRange& o = p.r[i];
        o.k0 = (int32_t)r.k_begin;
        o.k1 = (int32_t)(r.k_begin + r.k_len);
        o.a_sel = r.a_sel;
        o.sx_rs = r.sx_row_stride;
        o.sw_cs = r.sw_col_stride;
        o.sx = r.sx;
        o.sw = r.sw;
        if (r.k_begin + r.k_len > kmax) kmax = r.k_begin + r.k_len;
        ktotal += r.k_len;
    }
    if (kmax > d->lda || (w4 ? (kmax / 2 > d->ldb) : (kmax > d->ldb)))
        return fail(SEGQ_ERR_ARG, "segq_gemm: a range ends at %lld, beyond the row stride", (long long)kmax);
    // int4 weights are staged as value*16: keep |acc| below 2^31
    if (w4 && ktotal > 131071) return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: K too large for int4 weights");
    if (kmax > 0x7fffff00) return fail(SEGQ_ERR_ARG, "segq_gemm: K too large");

    const int64_t osz = (d->out_dtype == SEGQ_F32 || d->out_dtype == SEGQ_ACC) ? 4 : 2;
    const bool vec_store = ((d->ldo * osz) % (4 * osz) == 0) && ((d->batch_stride_out * osz) % (4 * osz) == 0) && al(d->out, 4 * osz);

    // One walk of K: one range whose end is ragged, or DualScale's two ranges over the same run (a, then a_neg)
    Walk walk{-1, 1e30};
    {
        const segq_krange &r = d->ranges[0], &s = d->ranges[d->n_ranges - 1];
        const bool base = (i8 || f8) && !lowrank && !codes_out && !groups && d->split_k <= 1 && d->m * d->lda < (int64_t)1 << 32 && d->n * d->ldb < (int64_t)1 << 32;
        const bool one = base && d->n_ranges == 1 && r.a_sel < 2;
        const bool pair = base && d->n_ranges == 2 && r.k_begin == s.k_begin && r.k_len == s.k_len, two = pair && r.a_sel == 0 && s.a_sel == 1;
        // (codes of both signs in one tensor: what two tensors would do, for the choice below)
        const bool merged = pair && d->finite_scales && r.a_sel == 2 && s.a_sel == 3;
        if (d->tile > FIRST_KT_CFG && d->tile <= FIRST_MIX_CFG) {
            if (!(d->tile > FIRST_DUAL_CFG ? two : one))
                return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tiles %d to %d serve one range, tiles %d to %d two over the same run of K from a and a_neg, in plain "
                                                  "8-bit codes, without group factors, a low-rank branch, codes out or split_k",
                            FIRST_KT_CFG + 1, FIRST_DUAL_CFG, FIRST_DUAL_CFG + 1, FIRST_MIX_CFG);
            walk.cfg = (int)d->tile - 1;
        } else if (d->tile == 0 && d->out_dtype != SEGQ_ACC) {
            if (one && r.k_len % 128) walk = choose_ragged(d->m, d->n, d->batch, r.k_len, osz == 4 && !vec_store);
            if ((two || merged) && (r.own_sum || d->finite_scales) && r.k_len > (r.k_len % 128 ? 256 : 512)) {
                walk = choose_dual(d->m, d->n, d->batch, r.k_len);
                const bool lent = d->split_k != 1 && ws && al(ws, 16), in_turn = r.k_len % 128 == 0 && d->batch == 1;
                const int64_t steps = r.k_len / 64;  // of both ranges in turn
                if (in_turn && !r.own_sum) {  // (0.85: the estimates)
                    if (0.85 * in_turn_us(d->m, d->n, steps, f8, lent) < walk.us) walk.cfg = -1;
                } else if (in_turn && lent && k_shares(d->m, d->n, steps, FIRST_WIDE_CFG + 6) > 2) {
                    walk.cfg = -1;  // a workspace lent to ranges summed on their own is lent for K shares
                }
            }
        }
    }
    // ... or a DualScale pair with one plain range beside it (at any place), in whole steps
    struct { int cfg = -1, shares = 1, pos = 0, neg = 1, plain = -1; } mix;
    if (d->n_ranges == 2 || d->n_ranges == 3) {
        bool ok = (i8 || f8) && !lowrank && !codes_out && !groups && d->batch == 1 && d->out_dtype != SEGQ_ACC &&
                  d->m * d->lda < (int64_t)1 << 32 && d->n * d->ldb < (int64_t)1 << 32;
        mix.neg = -1;
        for (int i = 0; i < d->n_ranges; ++i) {
            const segq_krange& r = d->ranges[i];
            ok = ok && r.k_begin % 128 == 0 && r.k_len % 128 == 0;
            if (r.a_sel == 1 || r.a_sel == 3) {
                ok = ok && mix.neg < 0;
                mix.neg = i;
            }
        }
        mix.pos = -1;
        for (int i = 0; ok && mix.neg >= 0 && i < d->n_ranges; ++i) {
            const segq_krange &r = d->ranges[i], &s = d->ranges[mix.neg];
            if (i == mix.neg) continue;
            if (mix.pos < 0 && r.k_begin == s.k_begin && r.k_len == s.k_len && r.a_sel == s.a_sel - 1) mix.pos = i;
            else if (r.a_sel == 0) mix.plain = i;
            else ok = false;
        }
        ok = ok && mix.neg >= 0 && mix.pos >= 0;
        const bool lent = ws && al(ws, 16);
        auto shares_fit = [&](int c, int n_) { return lent && ws_bytes >= mix_bytes(d->m, d->n, c, n_); };
        const int64_t steps = ok ? d->ranges[mix.neg].k_len / 128 : 0, plain = ok && mix.plain >= 0 ? d->ranges[mix.plain].k_len / 128 : 0;
        if (d->tile > FIRST_MIX_CFG && d->tile <= FIRST_LR_CFG) {
            if (!ok)
                return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tiles %d to %d serve two ranges over the same run of K from a and a_neg, and one plain range "
                                                  "beside them, in plain 8-bit codes and whole steps of 128, one problem, without group factors, a low-rank "
                                                  "branch or codes out", FIRST_MIX_CFG + 1, FIRST_LR_CFG);
            mix.cfg = (int)d->tile - 1;
            if (d->split_k > 1) {
                mix.shares = (int)(d->split_k < steps + plain / 2 ? d->split_k : steps + plain / 2);  // (a step at least for each)
                if (mix.shares > 1 && !shares_fit(mix.cfg, mix.shares)) return fail(SEGQ_ERR_ARG, "segq_gemm: workspace too small for split_k");
            }
        } else if (ok && d->tile == 0 && d->finite_scales && !d->ranges[0].own_sum && d->split_k <= 1 && (mix.plain >= 0 || steps > 4)) {
            const bool share = lent && d->split_k != 1;
            MixPick pick = choose_mix(d->m, d->n, steps, plain, share ? 16 : 1);
            while (pick.shares > 1 && !shares_fit(pick.cfg, pick.shares)) pick = choose_mix(d->m, d->n, steps, plain, pick.shares - 1);
            // (Codes of both signs in one tensor have no other way than this but the general kernel, far behind it: the lines below are
            // for two tensors, and for the caller that may still make two of them, a_neg.)
            // Up to 128 rows K shares of the ranges in turn are ahead, from where there are enough of them.  us a pass, that / this:
            // 32 x 1536 x (1536 + 6144) e4m3 18.7 / 23.4, 128 rows 22.0 / 25.1, int8 27.0 / 25.4.  Beside a plain range e4m3 takes
            // 128 x 128 tiles in three shares and more: 1 x 512 x (512 + 2048) 18.2 / 22.0, 128 rows 20.6 / 25.2, 1 x 4096 x (1024 +
            // 1024) 15.7 / 21.7, 128 x 4096 x (1024 + 2816) 26.0 / 30.0; two shares 1 x 2048 x (512 + 1024) 29.7 / 19.9, and
            // many outputs, whose shares are a trip through memory, 128 x 9216 x (384 + 1536) 27.6 / 24.2.  int8, which parks, has
            // 256 x 192 tiles: 1 x 512 x (512 + 3072) 20.7 / 22.4, 32 x 512 x (1024 + 2816) 23.7 / 25.9, 64 rows 25.9 / 26.1, 128 x 768 x
            // (768 + 3072) 27.0 / 26.4, 16 x 3072 24.7 / 24.0, 1 x 640 x (640 + 2560), which is not shared, 49.6 / 24.3.
            const int64_t all = 2 * steps + plain;
            const bool in_shares = steps + plain >= 32 || (mix.plain >= 0 && (f8 ? all >= 24 && d->m * d->n <= 540000 : all >= 52 && d->m <= 32 && d->n <= 1024));
            const bool part = d->ranges[mix.pos].a_sel == 2;
            bool take = d->m > 128 || !share || !in_shares;
            // The pair alone: against one walk of tiles 29 and 30, or the ranges in turn.  us, that / this: 2500 x 3072 x 12288 161 / 143,
            // 600 x 2048 x 8192 44 / 34, 4608 x 3072 x 12288 int8 310 / 266; 4096 x 1536 x 6144 57 / 60, 2600 x 1152 x 4608 30 / 34.
            if (mix.plain < 0) {
                const double cus = device_cus(), t64 = (double)tiles_of_cfg(FIRST_DUAL_CFG + 1, d->m, d->n, 1) / cus, k = (double)steps;
                const double now = walk.cfg < 0 ? in_turn_us(d->m, d->n, 2 * steps, f8, share)
                                   : walk.cfg == FIRST_DUAL_CFG ? std::ceil((double)tiles_of_cfg(FIRST_DUAL_CFG, d->m, d->n, 1) / cus) * (1.1 * k + 5.0)
                                   : t64 <= 1.0 ? 4.8 + 0.6 * k : 4.0 + t64 * (0.44 * k + 0.8);
                // (one tensor: with what the quantise step, which asks for this plan, then does not write.  Feed-forward of 4096
                // rows, 1536 x 6144 e4m3 through the epilogue that writes codes: two tensors 125 us a pass, one 121)
                double most = part ? now + (double)d->m * steps * 128 / 5e6 : 0.95 * now;
                // Where the two estimates meet these are short of what the launches take: int8 beside whole tiles of 128 x 192 with fewer than
                // twice as many rows as columns, so that what one tensor saves is not the most of what is loaded (1552 x 3008 x 5760
                // 58.4 us a pass, here 64.7; of 28 such shapes 27 were slower here, by 3 % in the middle; 4096 x 1536 x 6144 76.2 / 74.5), and three
                // or four shares of a short K beside one round of 64 x 128 (605 x 1088 x 3968 27.2 / 30.9, 800 x 1152 x 4608 32.1 / 33.9).
                if (i8 && walk.cfg == FIRST_DUAL_CFG && d->m < 2 * d->n) most = 0.92 * now;
                if (walk.cfg == FIRST_DUAL_CFG + 1 && t64 <= 1.0 && pick.shares > 2 && steps < 40) most = 0.85 * now;
                take = take && pick.us < most;
            }
            // Beside a plain range, e4m3: where whole tiles in turn are ahead (not those that would be shared along K: one walk is).
            // One tensor: with what the quantise step then does not write.
            if (mix.plain >= 0 && f8) {
                const int turn = choose_tile(d->m, d->n, 1, false, true, true, all, true);
                const bool whole = !share || choose_shares(d->m, d->n, all, turn, true, false, false).n == 1;
                const double more = part ? (double)d->m * steps * 128 / 5e6 : 0.0;
                if (whole && beside_in_turn_us(d->m, d->n, all, turn, osz == 4) + more < 1.03 * mix_beside_us(d->m, d->n, steps, plain, pick, osz == 4)) take = false;
            }
            if (take || (part && !d->a_neg)) {
                walk.cfg = -1;
                mix.cfg = pick.cfg;
                mix.shares = pick.shares;
            }
        }
    }
    if (walk.cfg >= FIRST_DUAL_CFG && d->ranges[0].a_sel != 0) walk.cfg = -1;
    const int few = [&]() -> int {
        const int64_t reach = (int64_t)1 << 31;  // a tile's rows are addressed with 31 bits
        const segq_krange& r = d->ranges[0];
        const bool ok = d->n_ranges == 1 && r.a_sel < 2 && d->m < reach >> 4 && d->n < reach >> 4 && !lowrank && !codes_out && d->split_k <= 1 && 64 * d->lda + kmax < reach && 64 * d->ldb + kmax < reach &&
                        (!groups || (w4 && r.k_begin % 128 == 0 && r.k_len % 128 == 0 && d->n % 4 == 0 && d->group_dequant_stride % 4 == 0 &&
                                     al(d->group_dequant, 16) && kmax / 128 * d->group_dequant_stride < reach / 4));
        if (d->tile != 0) return d->tile > FIRST_FEW_CFG && d->tile <= FIRST_KT_CFG ? (ok ? (int)d->tile - 1 : -2) : -1;
        // (raw accumulators are for checks of the integers and keep the route, and the workspace, that they had)
        return ok && d->out_dtype != SEGQ_ACC ? choose_few(d->m, d->n, d->batch, r.k_len, f8 ? GEMM_F8 : GEMM_I8, w4, groups, walk.us) : -1;
    }();
    if (q) {
        *fused = few >= FIRST_FEW_CFG && TILE_CFGS[few].bm == 16 && d->m <= 16 && d->ranges[0].k_len <= 128 * 8 * (TILE_CFGS[few].bn == 32 ? 4 : 3) &&
                 quantise_in_gemm_us(q, tiles_of_cfg(few, d->m, d->n, 1)) <= 5.8;
        if (!*fused) return SEGQ_OK;
    }
    if (few == -2)
        return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tiles %d to %d serve one range without a sign selection, a low-rank branch, codes out or split_k "
                                          "(and group factors of int4 weights)", FIRST_FEW_CFG + 1, FIRST_KT_CFG);
    if (groups && w4) {
        const int64_t kp = (kmax + 31) & ~(int64_t)31;
        if (!ws || !al(ws, 16) || ws_bytes < d->n * kp)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors with int4 weights need %lld bytes of workspace",
                        (long long)(d->n * kp));
    }
    if (few < 0 && w4 && ws) {
        // expand b to int8 in the caller's workspace and run the int8 kernels on it
        const int64_t kp = (kmax + 31) & ~(int64_t)31;  // whole 16-byte packed chunks
        if (al(ws, 16) && ws_bytes >= d->batch * d->n * kp && kp / 2 <= d->ldb) {
            if (plan) {  // the plan of the int8 launch on the expanded weights, plus the expansion's room
                segq_gemm_desc d8 = *d;
                d8.b_fmt = SEGQ_CODE_I8;
                d8.b = ws;
                d8.ldb = kp;
                d8.batch_stride_b = d->n * kp;
                d8.workspace = nullptr;
                d8.workspace_bytes = 0;
                const int rc = gemm_impl(&d8, st, plan, false);
                plan->bytes = d->batch * d->n * kp;
                return rc;
            }
            const int64_t chunks = kp / 32;
            for (int64_t zb = 0; zb < d->batch; ++zb) {
                const int64_t total = d->n * chunks;
                const unsigned blocks = (unsigned)((total + 255) / 256 < 4096 ? (total + 255) / 256 : 4096);
                hipLaunchKernelGGL(expand_i4_kernel, dim3(blocks), dim3(256), 0, st,
                                   static_cast<const uint8_t*>(d->b) + zb * d->batch_stride_b, d->ldb,
                                   static_cast<uint8_t*>(d->workspace) + zb * d->n * kp, kp, d->n, chunks);
            }
            const int rc = check_launch("segq_gemm (int4 expansion)");
            if (rc != SEGQ_OK) return rc;
            segq_gemm_desc d8 = *d;
            d8.b_fmt = SEGQ_CODE_I8;
            d8.b = d->workspace;
            d8.ldb = kp;
            d8.batch_stride_b = d->n * kp;
            d8.workspace = nullptr;
            d8.workspace_bytes = 0;
            return gemm_impl(&d8, st);
        }
    }

    p.A = static_cast<const uint8_t*>(d->a);
    p.A2 = static_cast<const uint8_t*>(d->a_neg);
    p.B = static_cast<const uint8_t*>(d->b);
    p.C = d->out;
    p.bias = d->out_dtype == SEGQ_ACC ? nullptr : d->bias;
    p.M = (int32_t)d->m;
    p.N = (int32_t)d->n;
    p.lda = d->lda; p.ldb = d->ldb; p.ldc = d->ldo;
    p.bsA = d->batch_stride_a; p.bsB = d->batch_stride_b; p.bsC = d->batch_stride_out;
    p.bsSx = d->batch_stride_sx; p.bsSw = d->batch_stride_sw;
    p.out_dtype = d->out_dtype; p.bias_dtype = d->bias_dtype;
    {
        const int64_t asz = d->out_dtype == SEGQ_F32 ? 4 : 2;
        p.addend = d->addend;
        p.ldadd = d->ld_addend;
        p.vec_add = d->addend && (d->ld_addend * asz) % (4 * asz) == 0 && (d->batch_stride_out * asz) % (4 * asz) == 0 && al(d->addend, 4 * asz);
    }
    p.vec_store = vec_store;
    p.vec_store16 = osz == 2 && d->ldo % 8 == 0 && d->batch_stride_out % 8 == 0 && al(d->out, 16);
    p.nr = d->n_ranges;
    if (few >= 0) {
        const TileCfg& c = TILE_CFGS[few];
        const int64_t tm = (d->m + c.bm - 1) / c.bm, tn = (d->n + c.bn - 1) / c.bn;
        if (tm * tn > 0x7fffffff || d->batch > 65535) return fail(SEGQ_ERR_ARG, "segq_gemm: grid too large");
        p.tiles_m = (int32_t)tm;
        p.tiles_n = (int32_t)tn;
        p.grw = d->group_dequant;
        p.grw_gs = d->group_dequant_stride;
        if (plan) {
            plan->tile = few + 1;
            if (groups) plan->bytes = d->n * ((kmax + 31) & ~(int64_t)31);  // asked for above, whatever the tile
            p.dry = 1;
        }
        return launch_gemm_few(p, f8 ? GEMM_F8 : GEMM_I8, w4, few, d->batch, st, q);
    }
    // K shares in d's workspace: two that meet in the launch, or any number that a second kernel sums
    auto launch_met = [&](int cfg, bool fold) -> int {
        const TileCfg& c = TILE_CFGS[cfg];
        p.splits = 2;
        p.part = static_cast<float*>(d->workspace);
        const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
        p.arrived = reinterpret_cast<unsigned int*>(static_cast<uint8_t*>(d->workspace) + tiles * 2 * c.bm * c.bn * 4);
        p.bsA = p.bsB = p.bsC = p.bsSx = p.bsSw = 0;  // blockIdx.y counts shares here, not problems
        static unsigned int g_stamp = 0x5e690000u;
        if (!p.dry) do p.stamp = __atomic_add_fetch(&g_stamp, 1u, __ATOMIC_RELAXED); while (p.stamp == 0u);  // 0 means "cleared"
        return i8 ? launch_gemm_i8(p, cfg, fold, 2, st) : launch_gemm_f8(p, cfg, fold, 2, st);
    };
    auto launch_shares = [&](int cfg, bool fold, int splits) -> int {
        p.splits = splits;
        p.C = d->workspace;
        p.ldc = d->n;
        p.bsC = d->m * d->n;
        p.bsA = p.bsB = p.bsSx = p.bsSw = 0;
        p.out_dtype = SEGQ_F32;
        p.bias = nullptr;
        p.addend = nullptr;
        p.vec_store = d->n % 4 == 0;
        p.vec_store16 = 0;
        const int rc = i8 ? launch_gemm_i8(p, cfg, fold, splits, st) : launch_gemm_f8(p, cfg, fold, splits, st);
        if (rc != SEGQ_OK || p.dry) return rc;
        const bool vec = d->n % 4 == 0 && d->ldo % 4 == 0 && al(d->out, 16);
        const int64_t items = d->m * (vec ? d->n / 4 : d->n);
        const dim3 grid((unsigned)((items + 255) / 256));
        if (vec)
            hipLaunchKernelGGL(splitk_reduce_kernel<true>, grid, dim3(256), 0, st, static_cast<const float*>(d->workspace), splits,
                               d->m, d->n, d->bias, d->bias_dtype, d->out, d->out_dtype, d->ldo, d->addend, d->ld_addend);
        else
            hipLaunchKernelGGL(splitk_reduce_kernel<false>, grid, dim3(256), 0, st, static_cast<const float*>(d->workspace), splits,
                               d->m, d->n, d->bias, d->bias_dtype, d->out, d->out_dtype, d->ldo, d->addend, d->ld_addend);
        return check_launch("segq_gemm (split-K sum)");
    };
    if (walk.cfg >= 0) {
        const TileCfg& c = TILE_CFGS[walk.cfg];
        const int64_t tm = (d->m + c.bm - 1) / c.bm, tn = (d->n + c.bn - 1) / c.bn;
        if (tm * tn > 0x7fffffff || d->batch > 65535) return fail(SEGQ_ERR_ARG, "segq_gemm: grid too large");
        p.tiles_m = (int32_t)tm;
        p.tiles_n = (int32_t)tn;
        p.group_m = 8;
        if (plan) {
            plan->tile = walk.cfg + 1;
            p.dry = 1;
        }
        return i8 ? launch_gemm_i8(p, walk.cfg, false, d->batch, st) : launch_gemm_f8(p, walk.cfg, false, d->batch, st);
    }
    if (mix.cfg >= 0) {
        const TileCfg& c = TILE_CFGS[mix.cfg];
        p.tiles_m = (int32_t)((d->m + c.bm - 1) / c.bm);
        p.tiles_n = (int32_t)((d->n + c.bn - 1) / c.bn);
        if ((int64_t)p.tiles_m * p.tiles_n > 0x7fffffff) return fail(SEGQ_ERR_ARG, "segq_gemm: grid too large");
        p.group_m = 8;
        // the pair first, positive codes in front, then the plain range
        const KRange pos = p.r[mix.pos], neg = p.r[mix.neg], plain = p.r[mix.plain >= 0 ? mix.plain : 0];
        p.r[0] = pos;
        p.r[1] = neg;
        p.r[2] = plain;
        if (plan) {
            plan->bytes = mix.shares > 1 ? mix_bytes(d->m, d->n, mix.cfg, mix.shares) : 0;
            plan->tile = mix.cfg + 1;
            plan->splits = mix.shares;
            p.dry = 1;
        }
        if (mix.shares == 2) return launch_met(mix.cfg, false);
        if (mix.shares > 2) return launch_shares(mix.cfg, false, mix.shares);
        return i8 ? launch_gemm_i8(p, mix.cfg, false, 1, st) : launch_gemm_f8(p, mix.cfg, false, 1, st);
    }
    const bool fold = d->n_ranges > 1;
    bool wide_ok = d->m * d->lda < (int64_t)1 << 32 && d->n * d->ldb < (int64_t)1 << 32;
    for (int i = 0; i < d->n_ranges; ++i) wide_ok = wide_ok && d->ranges[i].k_begin % 128 == 0 && d->ranges[i].k_len % 128 == 0;
    int cfg;
    bool plain8 = i8 || f8;  // both operands straight to LDS: no sign selection, no int4 unpacking
    for (int i = 0; i < d->n_ranges; ++i) plain8 = plain8 && d->ranges[i].a_sel < 2;
    // several ranges cost a second (fp32) accumulator set, and with it the biggest tiles,
    // unless the accumulators are fp32 already (plain e4m3: rescaled in place, which takes the ratio of two
    // ranges' scales and is not for callers whose scales may be infinite: own_sum)
    p.sep = f8 && fold && plain8 && d->ranges[0].own_sum != 0;
    const bool fold2 = fold && !(f8 && plain8 && !p.sep);
    if (groups) {
        bool ok = wide_ok && plain8;
        for (int i = 0; i < d->n_ranges; ++i) ok = ok && d->ranges[i].a_sel < 2;
        if (!ok) return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors need ranges of whole 128-column groups and a_sel 0 or 1");
        p.grw = d->group_dequant;
        p.grw_gs = d->group_dequant_stride;
    }
    // int8 with several ranges keeps the big tiles if the caller lends a workspace to park
    // finished ranges in: one fp32 tile per workgroup
    bool park = i8 && plain8 && fold && !groups && wide_ok && d->batch == 1 && d->out_dtype != SEGQ_ACC && ws && al(ws, 16);
    auto park_fits = [&](int c) {
        if (c < FIRST_WIDE_CFG || c >= NUM_TILE_CFG) return false;
        const TileCfg& t = TILE_CFGS[c];
        const int64_t tiles = ((d->m + t.bm - 1) / t.bm) * ((d->n + t.bn - 1) / t.bn);
        return ws_bytes >= tiles * t.bm * t.bn * 4;
    };
    if (d->tile == 0) {
        if (groups) {
            cfg = choose_groups(d->m, d->n, ktotal / 128, fold, d->out_dtype == SEGQ_F32);
        } else {
            cfg = park ? choose_tile(d->m, d->n, d->batch, false, wide_ok, plain8) : -1;
            park = park && park_fits(cfg);
            if (!park) cfg = choose_tile(d->m, d->n, d->batch, fold2, wide_ok, plain8, ktotal / 128, (!fold || (f8 && !p.sep)) && !lowrank);
        }
    }
    else if (d->tile >= 1 && d->tile <= NUM_TILE_CFG) cfg = d->tile - 1;
    else return fail(SEGQ_ERR_ARG, "segq_gemm: tile %d is not in 0..%d", d->tile, NUM_TILE_CFG);
    if (cfg >= FIRST_MIX_CFG && (cfg < FIRST_LR_CFG || !lowrank || fold))
        return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tiles %d to %d serve a low-rank branch beside one range, %d to %d DualScale", FIRST_LR_CFG + 1, NUM_TILE_CFG,
                    FIRST_MIX_CFG + 1, FIRST_LR_CFG);
    // Few tokens: when the 128 x 128 tiles do not even fill the CUs once, a workgroup has its CU to
    // itself and waits on HBM latency: the int8 kernel with four LDS stages keeps three K steps in
    // flight instead of one (256 x 9216 x 1536: 14.8 -> 12.9 us, 512 x 6144 x 3072: 25.5 -> 20.4 us)
    if (d->tile == 0 && cfg == FIRST_WIDE_CFG + 3 && i8 && plain8 && !fold && !groups && !lowrank && wide_ok &&
        ((d->m + 127) / 128) * ((d->n + 127) / 128) * d->batch <= device_cus() && ktotal / 128 >= 6) {
        cfg = FIRST_WIDE_CFG + 8;
        // ... and where 128 x 96 tiles still fit the CUs once and tile the columns exactly, a third more
        // workgroups pull from memory, each with four K steps in flight (five stages)
        if (d->n % 96 == 0 && ((d->m + 127) / 128) * (d->n / 96) * d->batch <= device_cus()) cfg = FIRST_WIDE_CFG + 10;
    }
    // the 8-wave tiles that exist with the finish in output units (low-rank branch, two-way K split)
    auto tail_tile = [](int c) {
        const int w = c - FIRST_WIDE_CFG;
        return w == 0 || w == 1 || w == 3 || w == 6 || w == 7;
    };
    if (lowrank && d->tile == 0 && cfg >= FIRST_WIDE_CFG && !tail_tile(cfg)) {
        cfg = cfg == FIRST_WIDE_CFG + 2 ? FIRST_WIDE_CFG + 1 : FIRST_WIDE_CFG;
        park = park && park_fits(cfg);
    }
    // Split K: few tiles and a long contraction.  The K steps of every tile are shared by
    // `splits` workgroups (grid.y).
    //  * Two shares are finished inside the launch: each workgroup leaves its fp32 share in the
    //    workspace, and the second to arrive adds the two, adds the bias and rounds.  Workspace:
    //    two tile-sized shares per tile, one word per tile in which the first to arrive leaves the
    //    launch's stamp (a per-process counter: no clearing between launches, and a fresh workspace
    //    may hold anything) and which the second clears (so that a captured graph, which replays
    //    the launch with the stamp it was recorded with, works too).
    //  * More shares: each workgroup writes an fp32 partial result, a second kernel sums them in the
    //    order of the shares.  Workspace: the partial results.
    // Either way the parking slots of all those workgroups follow (int8 with several ranges).
    // (No instance with a second register set of e4m3 sums meets in the launch: two shares of it take the second kernel.)
    int splits = 1;
    int64_t part_bytes = 0;
    auto meet = [&](int s_, int c) { return s_ == 2 && tail_tile(c) && !p.sep; };
    {
        const bool can = plain8 && wide_ok && d->batch == 1 && !groups && !lowrank && d->out_dtype != SEGQ_ACC && ws && al(ws, 16) &&
                         d->split_k != 1 && (d->tile == 0 || cfg >= FIRST_WIDE_CFG) && !codes_out;
        const int64_t total_steps = ktotal / 128;
        if (d->split_k > 1 && !can)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: split_k needs plain 8-bit codes, K ranges in multiples of 128, one problem, "
                                              "a float output, an 8-wave tile and a workspace");
        if (can) {
            int want = 1, scfg = cfg;
            const bool big_ok = !fold2 || park;  // the 256 x 256 tile, or 256 x 128 with a second register set
            auto tiles_of = [&](int c) { return ((d->m + TILE_CFGS[c].bm - 1) / TILE_CFGS[c].bm) * ((d->n + TILE_CFGS[c].bn - 1) / TILE_CFGS[c].bn); };
            if (d->split_k > 1) {
                want = (int)(d->split_k < total_steps ? d->split_k : total_steps);
                if (d->tile == 0) scfg = big_ok ? FIRST_WIDE_CFG : FIRST_WIDE_CFG + 1;
            } else if (d->tile == 0) {
                const Shares pick = choose_shares(d->m, d->n, total_steps, cfg, big_ok, p.sep, i8 && fold);
                scfg = pick.cfg;
                want = pick.n;
            }
            const TileCfg& t = TILE_CFGS[scfg];
            const int64_t tiles = tiles_of(scfg);
            const bool need_park = i8 && fold && scfg != FIRST_WIDE_CFG + 1 && scfg != FIRST_WIDE_CFG + 2 && scfg != FIRST_WIDE_CFG + 3;
            auto shares_for = [&](int s_) {
                if (meet(s_, scfg)) return tiles * 2 * t.bm * t.bn * 4 + ((tiles * 4 + 255) & ~(int64_t)255);
                return (((int64_t)s_ * d->m * d->n * 4) + 255) & ~(int64_t)255;
            };
            auto bytes_for = [&](int s_) { return shares_for(s_) + (need_park || park ? (int64_t)s_ * tiles * t.bm * t.bn * 4 : 0); };
            while (want > 1 && bytes_for(want) > ws_bytes) --want;
            if (d->split_k > 1 && want < 2) return fail(SEGQ_ERR_ARG, "segq_gemm: workspace too small for split_k");
            if (want > 1) {
                splits = want;
                cfg = scfg;
                part_bytes = shares_for(splits);
                park = (need_park || park) && i8 && fold;
            }
        }
    }
    if (splits == 1 && d->tile != 0) park = park && park_fits(cfg);
    if (park) p.park = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + part_bytes);
    if (park) {
        // every 8-wave tile serves several ranges this way
    } else if (cfg >= FIRST_WIDE_CFG) {
        if (!wide_ok) return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tile %d needs K ranges in multiples of 128", cfg + 1);
        if ((fold2 || (groups && fold)) && cfg == FIRST_WIDE_CFG) cfg = FIRST_WIDE_CFG + 1;
        if (groups && cfg > FIRST_WIDE_CFG + 3 && (fold || (cfg != FIRST_WIDE_CFG + 6 && cfg != FIRST_WIDE_CFG + 7)))
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors run on tiles %d to %d, and with one range on %d and %d",
                        FIRST_WIDE_CFG + 1, FIRST_WIDE_CFG + 4, FIRST_WIDE_CFG + 7, FIRST_WIDE_CFG + 8);
    } else if (groups) {
        return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors run on tiles %d to %d, and with one range on %d and %d", FIRST_WIDE_CFG + 1,
                    FIRST_WIDE_CFG + 4, FIRST_WIDE_CFG + 7, FIRST_WIDE_CFG + 8);
    } else if (cfg >= FIRST_BIG_CFG) {
        if (!wide_ok || w4 || fold)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tile %d needs one range, 8-bit weights and K in multiples of 128", cfg + 1);
    }
    if (lowrank) {
        // small problems, which would otherwise go to the general kernel: the smallest 8-wave tile
        if (d->tile == 0 && cfg < FIRST_WIDE_CFG && plain8 && wide_ok && splits == 1) cfg = FIRST_WIDE_CFG + 3;
        if (cfg < FIRST_WIDE_CFG || !plain8 || !wide_ok)
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: the low-rank branch needs plain 8-bit codes on both sides, K ranges in multiples "
                                              "of 128 and a shape the 8-wave kernels serve; pass the product as addend instead");
        p.lr_t = static_cast<const uint16_t*>(d->lowrank_t);
        p.lr_l2 = static_cast<const uint16_t*>(d->lowrank_l2t);
        p.lr_ldt = d->ld_lowrank_t;
        p.lr_ldl = d->ld_lowrank_l2t;
        p.lr_rank = d->lowrank_rank;
    }
    if (codes_out) {
        // the epilogue that writes codes is built into two tiles of the pipelined kernels
        if (!(plain8 && wide_ok && !fold && !groups && !lowrank && splits == 1))
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: out_codes needs plain int8 or e4m3 codes on both sides and one K range in "
                                              "multiples of 128; no group factors, low-rank branch or split_k");
        // 128 x 128: two workgroups share a CU, so one's epilogue (all VALU: ~40 instructions per element
        // with a GELU and two code tensors) can run under the other's MFMAs.  Measured on 4096 x 1536 ->
        // 6144 e4m3, GELU(tanh), DualScale: 66 us against 104 us on 256 x 256, one workgroup per CU
        if (d->tile == 0) cfg = FIRST_WIDE_CFG + 3;
        p.oc = d->out_codes;
        p.oc_neg = d->out_codes_neg;
        p.ldoc = d->ld_out_codes;
        p.oc_scale = d->out_scale;
        p.oc_scale_neg = d->out_scale_neg;
        p.oc_fmt = d->out_code_fmt;
        p.oc_pre = d->out_pre_op;
        p.oc_vec = d->ld_out_codes % 8 == 0 && al(d->out_codes, 8) && (!d->out_codes_neg || al(d->out_codes_neg, 8));
    }
    const TileCfg& c = TILE_CFGS[cfg];
    p.tiles_m = (int32_t)((d->m + c.bm - 1) / c.bm);
    p.tiles_n = (int32_t)((d->n + c.bn - 1) / c.bn);
    if (plan) {
        plan->bytes = part_bytes + (park ? (int64_t)splits * p.tiles_m * p.tiles_n * c.bm * c.bn * 4 : 0);
        plan->tile = cfg + 1;
        plan->splits = splits;
        plan->parked = park ? 1 : 0;
        // walk the same dispatch the launch takes, down to the kernel instance, and launch nothing:
        // the plan is refused exactly when the launch would be
        p.dry = 1;
    }
    // tiles are numbered down groups of this many tile rows, so that the 32 tiles an XCD holds at a time
    // share few operand panels; 384-row tiles reach that with half as many rows (e4m3 4608 x 12288 x 3072
    // 140.7 -> 136.2 us; other heights between 2 and 16 measured the same or worse on the 4608-token shapes)
    p.group_m = (cfg == FIRST_WIDE_CFG + 9 || cfg == FIRST_LR_CFG + 2) ? 4 : 8;
    {
        // e4m3 rescaled in place only (4608 x 15360 x 3072 in three ranges: 350 -> 338 us); int8, which parks its
        // sums at the boundaries, loses more to the XCDs reading different operand columns at a time than it gains
        // from spreading its stores (385 -> 397 us), and keeps the common order
        p.rot = (d->n_ranges > 1 && splits == 1 && f8 && !p.sep) ? 1 : 0;
    }
    if ((int64_t)p.tiles_m * p.tiles_n > 0x7fffffff || d->batch > 65535) return fail(SEGQ_ERR_ARG, "segq_gemm: grid too large");
    if (meet(splits, cfg)) return launch_met(cfg, fold);
    if (splits > 1) return launch_shares(cfg, fold, splits);
    if (i8) return launch_gemm_i8(p, cfg, fold, d->batch, st);
    if (f8) return launch_gemm_f8(p, cfg, fold, d->batch, st);
    return launch_gemm_w4(p, cfg, fold, d->batch, st);
}

static bool overlap(const void* a, int64_t a_bytes, const void* b, int64_t b_bytes) {
    const uintptr_t pa = reinterpret_cast<uintptr_t>(a), pb = reinterpret_cast<uintptr_t>(b);
    return pa < pb + (uintptr_t)b_bytes && pb < pa + (uintptr_t)a_bytes;
}

// Whether the GEMM may do the quantise step of a linear by itself: up to 16 rows with one scale or one per row, no producer
// fused in front, and, dynamic, the scales it divides by are the ones it makes.  Every workgroup of that launch reads all of x
// while others store already, so nothing it writes may lie over x; the two launches have read all of x before the first store.
static bool one_launch(const segq_quant_desc* q, const segq_gemm_desc* g) {
    const segq_krange& r = g->ranges[0];
    const int64_t xsz = q->x_dtype == SEGQ_F32 ? 4 : 2, osz = g->out_dtype == SEGQ_F32 ? 4 : 2;
    const int64_t x_bytes = ((q->rows - 1) * q->ldx + q->cols) * xsz;
    if (overlap(q->x, x_bytes, g->out, ((g->m - 1) * g->ldo + g->n) * osz) || overlap(q->x, x_bytes, q->codes, (q->rows - 1) * q->ld_codes + q->cols))
        return false;
    return q->rows > 0 && q->rows <= 16 && g->n_ranges == 1 && g->batch == 1 && r.a_sel == 0 && r.k_begin == 0 && r.k_len == q->cols && !q->dual && q->n_kseg == 1 &&
           q->pre_op == SEGQ_PRE_NONE && !q->gate && !q->col_div && (q->seg_rows <= 0 || q->seg_rows >= q->rows) && (q->row_stride | 1) == 1 &&
           (q->code_fmt == SEGQ_CODE_I8 || q->code_fmt == SEGQ_CODE_E4M3) && g->tile == 0 && g->out_dtype != SEGQ_ACC && q->ldx < (int64_t)1 << 24 &&
           (!q->dynamic || (r.sx == q->scale && (q->rows == 1 || (q->row_stride == 1 && r.sx_row_stride == 1))));
}

// ---- the library's own scratch memory, for segq_gemm_noalloc -------------------------------
// One array per GPU the library runs on, held until the process ends.  In host code the name
// `scratch` is only a handle for hipGetSymbolAddress: the device address it resolves to (one per
// device, each GPU holding its own copy) is what kernels, copies and fills are given.
constexpr int64_t SCRATCH_BYTES = SEGQ_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];
static void* g_scratch_ptr[64];  // resolved address per device ordinal

static int scratch_address(void** out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
        return fail(SEGQ_ERR_LAUNCH, "segq: cannot tell the current device (or its ordinal is above 63)");
    void* ptr = __atomic_load_n(&g_scratch_ptr[dev], __ATOMIC_ACQUIRE);
    if (!ptr) {
        const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr)
            return fail(SEGQ_ERR_LAUNCH, "segq: cannot resolve the scratch array on device %d: %s", dev, hipGetErrorString(e));
        __atomic_store_n(&g_scratch_ptr[dev], ptr, __ATOMIC_RELEASE);
    }
    *out = ptr;
    return SEGQ_OK;
}

}  // namespace segq

using namespace segq;

// only the C ABI leaves the library: everything else is built with hidden visibility
#pragma GCC visibility push(default)
extern "C" {

int segq_version(void) { return 100; }

const char* segq_last_error(void) { return g_err; }

int segq_quantize(const segq_quant_desc* d, segq_stream_t stream) {
    return quantize_impl(d, static_cast<hipStream_t>(stream), nullptr);
}

int segq_quantize_many(const segq_quant_desc* descs, int32_t n, segq_stream_t stream) {
    return quantize_many_impl(descs, n, static_cast<hipStream_t>(stream));
}

static void weight_desc(segq_quant_desc* q, const void* w, int32_t w_dtype, int64_t n, int64_t k, void* codes, int32_t fmt) {
    memset(q, 0, sizeof(*q));
    q->x = w; q->x_dtype = w_dtype; q->code_fmt = fmt;
    q->rows = n; q->cols = k; q->ldx = k;
    q->codes = codes; q->ld_codes = fmt == SEGQ_CODE_I4 ? k / 2 : k;
    q->n_kseg = 1;
}

int segq_quantize_weights_scalar(const void* weights, int32_t w_dtype, int64_t n, int64_t k, void* codes,
                                 int32_t code_fmt, float scale_w, segq_stream_t stream) {
    segq_quant_desc q;
    weight_desc(&q, weights, w_dtype, n, k, codes, code_fmt);
    return quantize_impl(&q, static_cast<hipStream_t>(stream), &scale_w);
}

int segq_quantize_weights_rows(const void* weights, int32_t w_dtype, int64_t n, int64_t k, void* codes,
                               int32_t code_fmt, const float* scale_w_rows, segq_stream_t stream) {
    segq_quant_desc q;
    weight_desc(&q, weights, w_dtype, n, k, codes, code_fmt);
    q.scale = const_cast<float*>(scale_w_rows);
    q.row_stride = 1;
    return quantize_impl(&q, static_cast<hipStream_t>(stream), nullptr);
}

int segq_quantize_weights_groups(const void* weights, int32_t w_dtype, int64_t n, int64_t k, void* codes, int32_t code_fmt,
                                 const float* scales, int64_t group, segq_stream_t stream) {
    return quantize_groups_impl(weights, w_dtype, n, k, codes, code_fmt, scales, group, static_cast<hipStream_t>(stream));
}

int segq_repack_int4_cols_to_rows(const void* colpacked, void* rowpacked, int64_t out, int64_t cols, segq_stream_t stream) {
    return repack_i4_impl(colpacked, rowpacked, out, cols, static_cast<hipStream_t>(stream));
}

int segq_lowrank_rows(const void* x, int64_t ldx, const void* l1t, int64_t ld_l1t, void* t, int64_t ldt, int64_t m, int64_t k, int64_t r, int32_t dtype,
                      segq_stream_t stream) {
    return lowrank_rows_impl(x, ldx, l1t, ld_l1t, t, ldt, m, k, r, dtype, static_cast<hipStream_t>(stream));
}

int segq_gemm(const segq_gemm_desc* d, segq_stream_t stream) { return gemm_impl(d, static_cast<hipStream_t>(stream)); }

int segq_gemm_tile_count(void) { return NUM_TILE_CFG; }

int segq_gemm_workspace_bytes(const segq_gemm_desc* d, int64_t* bytes) {
    if (!bytes) return fail(SEGQ_ERR_ARG, "segq_gemm_workspace_bytes: null result pointer");
    GemmPlan plan;
    const int rc = gemm_impl(d, nullptr, &plan);
    *bytes = plan.bytes;
    return rc;
}

int segq_gemm_plan(const segq_gemm_desc* d, int32_t* tile, int32_t* splits, int32_t* parked) {
    GemmPlan plan;
    const int rc = gemm_impl(d, nullptr, &plan, false);
    if (tile) *tile = plan.tile;
    if (splits) *splits = plan.splits;
    if (parked) *parked = plan.parked;
    return rc;
}

int segq_init(void) {
    void* ptr = nullptr;
    (void)device_cus();
    return scratch_address(&ptr);
}

int64_t segq_noalloc_scratch_bytes(void) { return SCRATCH_BYTES; }

int segq_device_info(int32_t* compute_units, int32_t* max_engine_clock_khz) {
    int dev = 0, cus = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeClockRate, dev) != hipSuccess)
        return fail(SEGQ_ERR_LAUNCH, "segq_device_info: cannot read the current device's attributes");
    if (compute_units) *compute_units = cus;
    if (max_engine_clock_khz) *max_engine_clock_khz = khz;
    return SEGQ_OK;
}

int segq_gemm_noalloc(const segq_gemm_desc* d, segq_stream_t stream) {
    GemmPlan plan;
    int rc = gemm_impl(d, nullptr, &plan);
    if (rc != SEGQ_OK) return rc;
    const int64_t wish = plan.bytes;  // what the launch would use of an unlimited workspace
    segq_gemm_desc c = *d;
    c.workspace = nullptr;
    c.workspace_bytes = 0;
    if (wish > 0) {
        void* ptr = nullptr;
        rc = scratch_address(&ptr);  // resolved once per device (segq_init does it ahead of time)
        if (rc != SEGQ_OK) return rc;
        c.workspace = ptr;
        c.workspace_bytes = SCRATCH_BYTES;
    }
    // a launch that could use more than the array holds runs with what fits, as segq_gemm does with
    // a workspace of that size (fewer K shares, a second register set instead of parked sums); it
    // is refused only where it cannot run with less
    rc = gemm_impl(&c, static_cast<hipStream_t>(stream));
    if (rc != SEGQ_OK && wish > SCRATCH_BYTES) {
        char why[256];
        snprintf(why, sizeof(why), "%s", g_err);
        return fail(rc, "segq_gemm_noalloc: this launch needs more workspace than the library's scratch array holds (%lld bytes; "
                        "it could use %lld): %s; use segq_gemm with a workspace of the caller's",
                    (long long)SCRATCH_BYTES, (long long)wish, why);
    }
    return rc;
}

int segq_linear(const segq_quant_desc* q, const segq_gemm_desc* g, segq_stream_t stream) {
    if (!q || !g) return fail(SEGQ_ERR_ARG, "segq_linear: null descriptor");
    if (q->rows == 0 && g->m == 0) return SEGQ_OK;  // no token rows: nothing to quantise, nothing to multiply
    // the GEMM must consume exactly what the quantise step produces
    if (q->codes != g->a) return fail(SEGQ_ERR_ARG, "segq_linear: the GEMM must read the codes the quantise step writes");
    if (g->n_ranges < 1 || g->n_ranges > SEGQ_MAX_RANGES) return fail(SEGQ_ERR_ARG, "segq_linear: n_ranges %d out of range", g->n_ranges);
    bool reads_neg = false;
    for (int i = 0; i < g->n_ranges; ++i) reads_neg = reads_neg || g->ranges[i].a_sel == 1;
    if (reads_neg && (!q->codes_neg || q->codes_neg != g->a_neg))
        return fail(SEGQ_ERR_ARG, "segq_linear: a range reads a_neg, which is not the second code tensor the quantise step writes");
    if (q->ld_codes != g->lda || q->rows != g->m * g->batch)
        return fail(SEGQ_ERR_ARG, "segq_linear: the code tensor's rows (%lld, stride %lld) do not match the GEMM's (%lld, stride %lld)",
                    (long long)q->rows, (long long)q->ld_codes, (long long)(g->m * g->batch), (long long)g->lda);
    if (q->code_fmt != g->a_fmt) return fail(SEGQ_ERR_ARG, "segq_linear: code formats differ (%d written, %d read)", q->code_fmt, g->a_fmt);
    if (q->dynamic && g->out_dtype != SEGQ_ACC) {
        // dynamic scales are outputs of the first step: every range must divide by one of them
        const int64_t seg_rows = q->seg_rows > 0 ? q->seg_rows : q->rows;
        const int64_t extent = (seg_rows > 0 ? (q->rows - 1) / seg_rows : 0) * q->seg_stride + (seg_rows - 1) * q->row_stride +
                               (int64_t)(q->n_kseg - 1) * q->kseg_stride + 1;
        for (int i = 0; i < g->n_ranges; ++i) {
            const float* sx = g->ranges[i].sx;
            const bool in_pos = q->scale && sx >= q->scale && sx < q->scale + extent;
            const bool in_neg = q->scale_neg && sx >= q->scale_neg && sx < q->scale_neg + extent;
            if (!in_pos && !in_neg)
                return fail(SEGQ_ERR_ARG, "segq_linear: range %d divides by scales the dynamic quantise step does not write", i);
        }
    }
    if (one_launch(q, g)) {
        const int rc = quantize_check(q);
        if (rc != SEGQ_OK) return rc;
        bool fused = false;
        const int rc2 = gemm_impl(g, static_cast<hipStream_t>(stream), nullptr, true, q, &fused);
        if (rc2 != SEGQ_OK || fused) return rc2;
    }
    const int rc = quantize_impl(q, static_cast<hipStream_t>(stream), nullptr);
    if (rc != SEGQ_OK) return rc;
    return gemm_impl(g, static_cast<hipStream_t>(stream));
}

int segq_fake_e4m3(const void* x, void* out, int32_t dtype, int64_t numel, segq_stream_t stream) {
    return fake_e4m3_impl(x, out, dtype, numel, static_cast<hipStream_t>(stream));
}

}  // extern "C"
#pragma GCC visibility pop
