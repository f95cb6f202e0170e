// Segmented GEMM for launches of few tiles: few tokens, few output columns, any K in sixteens.
//
// Such a launch is a chain of memory round trips on a chip that is mostly idle, so everything here
// is about loads in flight.  The tile is small (16 x 32 to 32 x 64 outputs, many workgroups) and the
// eight waves of a workgroup share its K: wave w takes every eighth unit of 128 values, keeps a few
// units in flight in registers, and never meets the other waves before its share is done.  No barrier
// in the K loop, no chain from one K step to the next beyond the accumulators.  The shares meet once,
// in LDS, in the order of the waves; every wave finishes some of the tile's 16 x 16 blocks.
//
// A unit passes through a patch of LDS of the wave's own between its load and its MFMAs.  An MFMA
// fragment wants 16 rows in 16 neighbouring lanes; loaded like that, every lane is a cache line of its
// own and an instruction takes 64 clocks of the vector cache (measured: 34 bytes per ns and CU, the
// 64 x 64 tile on K 3072 16 us whatever the rest does).  Loaded as eight lanes to a 128-byte row it
// moves whole lines, and the patch gives each lane its fragment.
//
// Operands are read through buffer resources: a lane past the end of K (a ragged last unit, or a wave
// without a unit left) is given an offset past the end of the resource, reads zero and costs no
// traffic, so that no load hangs on a branch and each unit is waited for alone.
#pragma once
#include "segq_gemm_kernel.h"
#include "segq_encode.h"

namespace segq {

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

constexpr int FEW_WAVES = 8;

// What a launch needs of GemmParams, whose range table alone is 2.5 KB: every workgroup begins with the round trip
// that fetches its arguments.
struct FewParams {
    const uint8_t* A;
    const uint8_t* B;
    void* C;
    const float* sx;
    const float* sw;
    const void* bias;
    const void* addend;
    const float* grw;
    int64_t lda, ldb, ldc, ldadd, grw_gs;
    int64_t bsA, bsB, bsC, bsSx, bsSw;
    int32_t M, N, k0, k1;
    int32_t sx_rs, sw_cs;
    int32_t tiles_m, tiles_n;
    int32_t out_dtype, bias_dtype;
    int32_t vec_store, vec_add;
    // the quantise step in front of up to 16 rows (QE instances; A is not read): x, its codes and, dynamic, its scales
    const void* X;
    float* q_scale;
    uint8_t* codes;
    int64_t ldx, ld_codes;
    int32_t x_dtype, q_rs, dynamic, pad_;
};

// Registers of a unit of operands, and units of K in flight per wave: of a short K all of them (at most four, and no more
// than fit beside the accumulators with two waves per SIMD), of a longer one two.
constexpr int few_unit(int tm, int tn, bool b4, bool grp) { return tm * 8 + tn * (b4 ? 4 : 8) + (grp ? tn * 4 : 0); }
constexpr int few_depth(int tm, int tn, bool b4, bool grp) {
    const int room = (176 - tm * tn * 4) / few_unit(tm, tn, b4, grp);
    return room >= 4 ? 4 : room >= 3 ? 3 : 2;
}
// Whether a second workgroup fits the CU: 128 registers per lane.  (`iter`: units per wave all in flight, 0: a loop.)
constexpr bool few_two(int tm, int tn, bool b4, bool grp, int iter) {
    return 34 + few_unit(tm, tn, b4, grp) * (iter > 0 ? iter : 2) <= 130 && (iter > 0 || (tn == 2 && !(grp && tm == 2)));
}

// LDS of one wave: the unit's activations and one block of its weights, and then the wave's share of the sums.
template <int TM, int TN, bool B4> constexpr int few_patch() {
    constexpr int operands = TM * 2048 + (B4 ? 1024 : 2048), sums = TM * TN * 1024;
    return operands > sums ? operands : sums;
}

// ITER: units per wave of a short K, all asked for at once (no loop, and registers for no more than these); 0: any number.
// QE: the linear's quantise step runs here as well (2, 4: bytes of an element of x): a wave loads the floats of its units and
// encodes each on its way to the patch, so that the linear is one launch and the codes need no trip through memory.  Every
// workgroup encodes all of its 16 rows, which is why it serves no more; the first column of tiles also leaves the codes
// and the dynamic scales where the quantise launch would have.  2 x 1536 -> 9216 fp16: both launches 9.4 us
// and the gap between them, this 7.6; dynamic 8 x 3072 -> 6144 10.0 and 8.4.  (Wide layers and long rows: quantise_in_gemm_us().)
template <int TM, int TN, int FMT, bool B4, bool GRP, int ITER, int QE = 0>
__global__ void __launch_bounds__(FEW_WAVES * 64, QE == 0 && few_two(TM, TN, B4, GRP, ITER) ? 4 : 2) gemm_few_kernel(const FewParams p) {
    constexpr int NW = FEW_WAVES, BM = TM * 16, BN = TN * 16, NB = TM * TN;
    constexpr bool F8 = FMT == GEMM_F8;
    constexpr int UNIT = 128;               // K of one unit
    constexpr int LA = 2, LB = B4 ? 1 : 2;  // 16-byte pieces per lane, 16 rows and unit
    constexpr int DEPTH = ITER > 0 ? ITER : 2;
    constexpr int PATCH = few_patch<TM, TN, B4>();
    constexpr int OWN = (NB + NW - 1) / NW;  // 16 x 16 blocks a wave finishes
    static_assert(!B4 || !F8, "int4 weights pair with int8 activations");
    static_assert(QE == 0 || (TM == 1 && ITER > 0), "quantising: 16 rows, all of K in registers");
    constexpr int XL = QE == 0 ? 1 : QE;  // 16-byte loads for 16 elements
    typedef typename AccT<FMT>::type acc_t;
    typedef typename std::conditional<GRP, v4f, acc_t>::type sum_t;

    extern __shared__ __align__(16) uint8_t smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 15, lgrp = lane >> 4;

    // Tiles are numbered down the rows first and dealt to the XCDs in runs: the tiles that read the same
    // weight rows sit behind one L2.
    int bid = blockIdx.x;
    {
        const int nb = p.tiles_m * p.tiles_n, q = nb >> 3, r = nb & 7, x = bid & 7;
        bid = x * q + min(x, r) + (bid >> 3);
    }
    const int tile_n = bid / p.tiles_m, tile_m = bid - tile_n * p.tiles_m;
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int64_t z = blockIdx.y;
    const int k0 = p.k0, k1 = p.k1;

    // Resources that start at the tile's first row and end with its last row's last code (the host has checked
    // that a tile's rows span less than 2^31 bytes).
    constexpr uint32_t NOWHERE = 0x80000000u;  // past the end of any of them
    const uint8_t* const Ab = QE ? nullptr : p.A + z * p.bsA + (int64_t)m0 * p.lda;
    const uint8_t* const Bb = p.B + z * p.bsB + (int64_t)n0 * p.ldb;
    const int rows_a = min(BM, p.M - m0), rows_b = min(BN, p.N - n0);
    const __amdgpu_buffer_rsrc_t rsa = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(Ab), 0, (int)((rows_a - 1) * (uint32_t)p.lda + (uint32_t)k1), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(Bb), 0, (int)((rows_b - 1) * (uint32_t)p.ldb + (uint32_t)(B4 ? k1 >> 1 : k1)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsg = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(p.grw), 0, GRP ? (int)((((k1 >> 7) - 1) * (uint32_t)p.grw_gs + (uint32_t)p.N) * 4) : 0, 0x00020000);
    // Lane to 16 bytes of a row: eight lanes a row and two loads for 16 rows, or, packed int4, four lanes and one load.
    const int a_row = lane >> 3, a_pc = lane & 7;
    const int b_row = B4 ? lane >> 2 : a_row, b_pc = B4 ? lane & 3 : a_pc;
    uint32_t a_off[TM * LA], b_off[TN * LB];
#pragma unroll
    for (int i = 0; i < TM * LA; ++i) a_off[i] = (uint32_t)min(i * 8 + a_row, rows_a - 1) * (uint32_t)p.lda + a_pc * 16;
#pragma unroll
    for (int i = 0; i < TN * LB; ++i) b_off[i] = (uint32_t)min(i * (16 / LB) + b_row, rows_b - 1) * (uint32_t)p.ldb + b_pc * 16;

    // QE: 16 elements of a row per lane instead of their 16 codes; rows past M read as zeros
    const __amdgpu_buffer_rsrc_t rsx = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<void*>(p.X), 0, QE ? (int)(((rows_a - 1) * (uint32_t)p.ldx + (uint32_t)k1) * QE) : 0, 0x00020000);
    uint32_t x_off[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) x_off[i] = i * 8 + a_row < rows_a ? ((uint32_t)(i * 8 + a_row) * (uint32_t)p.ldx + a_pc * 16) * QE : NOWHERE;

    // Unit u in registers.
    const int units = (k1 - k0 + UNIT - 1) / UNIT;
    v4u qx[QE ? DEPTH : 1][2][XL];
    v4u qa[QE ? 1 : DEPTH][TM * LA], qb[DEPTH][TN * LB];
    v4f qg[GRP ? DEPTH : 1][GRP ? TN : 1];
    auto load_unit = [&](int u, v4u (&a)[TM * LA], v4u (&b)[TN * LB], v4f (&g)[GRP ? TN : 1], v4u (&x)[2][XL]) __attribute__((always_inline)) {
        const int k = min(k0 + min(u, units) * UNIT, k1);  // (uniform: the scalar offset of the loads)
        const bool a_in = k + a_pc * 16 < k1, b_in = k + b_pc * (B4 ? 32 : 16) < k1;
#pragma unroll
        for (int i = 0; i < TM * LA; ++i) {
            if constexpr (QE) {
#pragma unroll
                for (int j = 0; j < XL; ++j) x[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rsx, a_in && x_off[i] != NOWHERE ? x_off[i] + j * 16 : NOWHERE, k * QE, 0);
            } else {
                a[i] = __builtin_amdgcn_raw_buffer_load_b128(rsa, a_in ? a_off[i] : NOWHERE, k, 0);
            }
        }
#pragma unroll
        for (int i = 0; i < TN * LB; ++i) b[i] = __builtin_amdgcn_raw_buffer_load_b128(rsb, b_in ? b_off[i] : NOWHERE, B4 ? k >> 1 : k, 0);
        if constexpr (GRP) {  // four factors at a time (the host has checked that columns and rows come in fours)
#pragma unroll
            for (int i = 0; i < TN; ++i)
                g[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(rsg, min(n0 + i * 16 + 4 * lgrp, p.N - 4) * 4, (min(k, k1 - UNIT) >> 7) * (int)p.grw_gs * 4, 0));
        }
    };

    sum_t acc[TN][TM];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = sum_t{0, 0, 0, 0};

    // Registers -> the wave's patch -> fragments -> MFMAs.  LDS operations of a wave complete in order, so the patch
    // needs no barrier.  A 128-byte row has its 16-byte pieces swizzled by the row as in the other kernels, a 64-byte row of
    // packed int4 by its quarter of the 16 rows: writes and reads are free of bank conflicts.
    // Lane group g of a fragment holds pieces g and 4 + g of its row; with int4 weights packed piece g, which is 32
    // values, and activation pieces 2 g and 2 g + 1.
    uint8_t* const patch = smem + wave * PATCH;
    const int a_st = a_row * BK + ((a_pc ^ swz(a_row)) << 4), b_st = B4 ? b_row * 64 + ((b_pc ^ (b_row >> 2)) << 4) : a_st;
    const int f0 = lrow * BK + (((B4 ? 2 * lgrp : lgrp) ^ swz(lrow)) << 4);
    const int f1 = lrow * BK + (((B4 ? 2 * lgrp + 1 : 4 + lgrp) ^ swz(lrow)) << 4);
    const int f4 = lrow * 64 + ((lgrp ^ (lrow >> 2)) << 4);
    auto multiply = [&](const v4u (&qa_)[TM * LA], const v4u (&qb_)[TN * LB], const v4f (&g)[GRP ? TN : 1]) __attribute__((always_inline)) {
        uint8_t* const pb = patch + TM * 2048;
#pragma unroll
        for (int i = 0; i < TM * LA; ++i)  // (rows 8 apart: the swizzle's top bit flips)
            *reinterpret_cast<v4u*>(patch + i * 1024 + ((i & 1) ? a_st ^ 64 : a_st)) = qa_[i];
        __builtin_amdgcn_wave_barrier();  // what a lane reads, others have written: no reordering across here
        v4i a0[TM], a1[TM];
#pragma unroll
        for (int s = 0; s < TM; ++s) {
            a0[s] = *reinterpret_cast<const v4i*>(patch + s * 2048 + f0);
            a1[s] = *reinterpret_cast<const v4i*>(patch + s * 2048 + f1);
        }
#pragma unroll
        for (int t = 0; t < TN; ++t) {
            // (one block of weights after the other through the same place: a smaller patch, and a second workgroup on the CU)
#pragma unroll
            for (int i = 0; i < LB; ++i) *reinterpret_cast<v4u*>(pb + i * 1024 + ((!B4 && i == 1) ? b_st ^ 64 : b_st)) = qb_[t * LB + i];
            __builtin_amdgcn_wave_barrier();
            v4i b0, b1;
            if constexpr (B4) {
                const v4u w4 = *reinterpret_cast<const v4u*>(pb + f4);
                uint32_t o[8];
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // eight nibbles -> eight bytes holding value * 16, in the order of k
                    const uint32_t ev = (w4[j] << 4) & 0xF0F0F0F0u, od = w4[j] & 0xF0F0F0F0u;
                    o[2 * j] = __builtin_amdgcn_perm(od, ev, 0x05010400u);
                    o[2 * j + 1] = __builtin_amdgcn_perm(od, ev, 0x07030602u);
                }
                b0 = v4i{(int)o[0], (int)o[1], (int)o[2], (int)o[3]};
                b1 = v4i{(int)o[4], (int)o[5], (int)o[6], (int)o[7]};
            } else {
                b0 = *reinterpret_cast<const v4i*>(pb + f0);
                b1 = *reinterpret_cast<const v4i*>(pb + f1);
            }
#pragma unroll
            for (int s = 0; s < TM; ++s) {
                if constexpr (F8) {
                    acc[t][s] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(v8i{b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w},
                                                                                 v8i{a0[s].x, a0[s].y, a0[s].z, a0[s].w, a1[s].x, a1[s].y, a1[s].z, a1[s].w},
                                                                                 acc[t][s], 0, 0, 0, 0, 0, 0);
                } else {
                    v4i c = {0, 0, 0, 0};
                    if constexpr (!GRP) c = acc[t][s];
                    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b0, a0[s], c, 0, 0, 0);
                    c = __builtin_amdgcn_mfma_i32_16x16x64_i8(b1, a1[s], c, 0, 0, 0);
                    if constexpr (GRP) acc[t][s] += __builtin_convertvector(c, v4f) * g[t];
                    else acc[t][s] = c;
                }
            }
        }
    };

    // ---- this wave's units: wave, wave + NW, ...
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load_unit(wave + d * NW, qa[QE ? 0 : d], qb[d], qg[GRP ? d : 0], qx[QE ? d : 0]);

    // What this wave finishes: block i of the tile is column block i / TM, row block i % TM.  Its scales and
    // bias are asked for behind the first operands, so that the end of the launch waits for no memory; loads that
    // do not apply (no bias, the other bias type, raw accumulators) go to empty resources instead of round a branch.
    const bool scaled = p.out_dtype != SEGQ_ACC;
    auto rsrc = [](const void* base, bool there) __attribute__((always_inline)) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, there ? 0x7fffffff : 0, 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t rs_sx = rsrc(p.sx + z * p.bsSx, scaled), rs_sw = rsrc(p.sw + z * p.bsSw, scaled);
    const __amdgpu_buffer_rsrc_t rs_b32 = rsrc(p.bias, p.bias && p.bias_dtype == SEGQ_F32), rs_b16 = rsrc(p.bias, p.bias && p.bias_dtype != SEGQ_F32);
    uint32_t sx_raw[OWN], sw_raw[OWN][4], b32_raw[OWN][4], b16_raw[OWN][4];
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int blk = min(i * NW + wave, NB - 1);
        const int n = n0 + blk / TM * 16 + 4 * lgrp;
        sx_raw[i] = __builtin_amdgcn_raw_buffer_load_b32(rs_sx, min(m0 + blk % TM * 16 + lrow, p.M - 1) * p.sx_rs * 4, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int nv = min(n + v, p.N - 1);
            sw_raw[i][v] = __builtin_amdgcn_raw_buffer_load_b32(rs_sw, nv * p.sw_cs * 4, 0, 0);
            b32_raw[i][v] = __builtin_amdgcn_raw_buffer_load_b32(rs_b32, nv * 4, 0, 0);
            b16_raw[i][v] = __builtin_amdgcn_raw_buffer_load_b16(rs_b16, nv * 2, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    [[maybe_unused]] float own_scale = 0.0f;  // dynamic: of row lrow
    if constexpr (QE != 0) {
        auto floats = [&](const v4u (&x)[XL], float (&v)[16]) __attribute__((always_inline)) {
            if constexpr (QE == 4) {
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = __uint_as_float(x[i / 4][i % 4]);
            } else if (p.x_dtype == SEGQ_BF16) {
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = __uint_as_float((i & 1) ? x[i / 8][i / 2 % 4] & 0xffff0000u : x[i / 8][i / 2 % 4] << 16);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) v[i] = f16_bits_to_f32((i & 1) ? x[i / 8][i / 2 % 4] >> 16 : x[i / 8][i / 2 % 4] & 0xffffu);
            }
        };
        const int halves = rows_a > 8 ? 2 : 1;  // of the 16 rows; what is not there is zeros already
        float s[2];
        if (p.dynamic) {
            // the quantise kernels' maximum and scale: non-negative floats are ordered like their bits, and a NaN wins
            uint32_t amax[2] = {0, 0};
#pragma unroll
            for (int d = 0; d < DEPTH; ++d)
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    if (i >= halves) continue;
                    float v[16];
                    floats(qx[d][i], v);
#pragma unroll
                    for (int j = 0; j < 16; ++j) amax[i] = max(amax[i], __float_as_uint(fabsf(v[j])));
                }
            uint32_t* const red = reinterpret_cast<uint32_t*>(smem);  // [NW][16]
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int o = 4; o > 0; o >>= 1) amax[i] = max(amax[i], (uint32_t)__shfl_xor((int)amax[i], o, 64));
                if (a_pc == 0) red[wave * 16 + i * 8 + a_row] = amax[i];
            }
            __syncthreads();
            auto scale_of = [&](int row) {
                uint32_t t = 0;
#pragma unroll
                for (int w = 0; w < NW; ++w) t = max(t, red[w * 16 + row]);
                return (F8 ? 448.0f : 127.0f) / __uint_as_float(max(t, 0x33800000u));  // 2^-24
            };
            s[0] = scale_of(a_row);
            s[1] = scale_of(8 + a_row);
            own_scale = scale_of(lrow);
            __syncthreads();  // (the patches lie over the maxima)
            if (tile_n == 0 && wave == 0 && a_pc == 0) {
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    if (i * 8 + a_row < rows_a) p.q_scale[(int64_t)(i * 8 + a_row) * p.q_rs] = s[i];
            }
        } else {
            s[0] = p.q_scale[(int64_t)min(a_row, rows_a - 1) * p.q_rs];
            s[1] = p.q_scale[(int64_t)min(8 + a_row, rows_a - 1) * p.q_rs];
        }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            // (unpacked again: kept from the maximum on, the floats would take twice the registers)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < XL; ++j) asm volatile("" : "+v"(qx[d][i][j]));
            v4u c[2] = {{0, 0, 0, 0}, {0, 0, 0, 0}};
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (i >= halves) continue;
                float v[16];
                floats(qx[d][i], v);
#pragma unroll
                for (int j = 0; j < 16; ++j) v[j] *= s[i];
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    c[i][j] = F8 ? pack4_e4m3(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]) : pack4_i8(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
            }
            const int k = k0 + (wave + d * NW) * UNIT + a_pc * 16;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (k >= k1 || i * 8 + a_row >= rows_a) c[i] = v4u{0, 0, 0, 0};  // (0 times an infinite scale is a NaN)
                else if (tile_n == 0) *reinterpret_cast<v4u*>(p.codes + (int64_t)(i * 8 + a_row) * p.ld_codes + k) = c[i];
            }
            if (!GRP || wave + d * NW < units) multiply(c, qb[d], qg[GRP ? d : 0]);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else if constexpr (ITER > 0) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            if (!GRP || wave + d * NW < units) multiply(qa[d], qb[d], qg[GRP ? d : 0]);
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        int left = (units + NW - 1) / NW;  // the same for all waves: past the last unit the operands are zeros
        for (int u = wave; left > 0;) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                if (!GRP || u < units) multiply(qa[d], qb[d], qg[GRP ? d : 0]);  // (a group factor may be infinite)
                if (--left <= 0) break;
                __builtin_amdgcn_sched_barrier(0);
                load_unit(u + DEPTH * NW, qa[d], qb[d], qg[GRP ? d : 0], qx[0]);
                __builtin_amdgcn_sched_barrier(0);
                u += NW;
            }
        }
    }

    // ---- the shares meet
    sum_t* const shares = reinterpret_cast<sum_t*>(smem);  // [NW][PATCH]: 64 lanes of NB blocks in front of each patch
    constexpr int SW = PATCH / 16;
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) shares[wave * SW + (a * TM + b) * 64 + lane] = acc[a][b];
    __syncthreads();

    const int64_t c_off = z * p.bsC;
#pragma unroll
    for (int i = 0; i < OWN; ++i) {
        const int blk = i * NW + wave;
        if (blk >= NB) return;
        sum_t s = shares[blk * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) s += shares[w * SW + blk * 64 + lane];
        const int m = m0 + blk % TM * 16 + lrow, n = n0 + blk / TM * 16 + 4 * lgrp;
        if (m >= p.M || n >= p.N) continue;
        const int64_t e = c_off + (int64_t)m * p.ldc + n;
        const bool vec = p.vec_store && n + 3 < p.N;
        if (p.out_dtype == SEGQ_ACC) {
            if constexpr (!GRP) {
                if constexpr (B4) { s[0] >>= 4; s[1] >>= 4; s[2] >>= 4; s[3] >>= 4; }
                typename AccT<FMT>::elem* const dst = static_cast<typename AccT<FMT>::elem*>(p.C) + e;
                if (vec) *reinterpret_cast<acc_t*>(dst) = s;
                else
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < p.N) dst[v] = s[v];
            }
            continue;
        }
        const float rx = 1.0f / (QE && p.dynamic ? own_scale : __uint_as_float(sx_raw[i]));
        float o[4];
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const float rw = (B4 ? 0.0625f : 1.0f) / __uint_as_float(sw_raw[i][v]);  // (the factor 16 of the unpacked weights is exact)
            const float b16 = p.bias_dtype == SEGQ_BF16 ? bf16_bits_to_f32(b16_raw[i][v]) : f16_bits_to_f32(b16_raw[i][v]);
            const float bv = p.bias_dtype == SEGQ_F32 ? __uint_as_float(b32_raw[i][v]) : b16;  // (zeros without a bias)
            o[v] = dequant_bias((float)s[v], rx, rw, bv);
        }
        add_addend4(p, z, m, n, o);
        if (p.out_dtype == SEGQ_F32) {
            float* const dst = static_cast<float*>(p.C) + e;
            if (vec) *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
            else
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < p.N) dst[v] = o[v];
        } else {
            const bool bf = p.out_dtype == SEGQ_BF16;
            const uint32_t lo = bf ? pack2_bf16(o[0], o[1]) : pack2_f16(o[0], o[1]), hi = bf ? pack2_bf16(o[2], o[3]) : pack2_f16(o[2], o[3]);
            uint16_t* const dst = static_cast<uint16_t*>(p.C) + e;
            if (vec) {
                *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
            } else {
                const uint32_t h[4] = {lo & 0xffffu, lo >> 16, hi & 0xffffu, hi >> 16};
#pragma unroll
                for (int v = 0; v < 4; ++v)
                    if (n + v < p.N) dst[v] = (uint16_t)h[v];
            }
        }
    }
}

template <int TM, int TN, int FMT, bool B4, bool GRP, int ITER, int QE = 0>
int launch_few_instance(const FewParams& p, int64_t batch, hipStream_t st) {
    auto kern = gemm_few_kernel<TM, TN, FMT, B4, GRP, ITER, QE>;
    constexpr int lds = FEW_WAVES * few_patch<TM, TN, B4>();
    static unsigned long long attr_done = 0;
    if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds, &attr_done)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.tiles_m * p.tiles_n), (unsigned)batch), dim3(FEW_WAVES * 64), lds, st, p);
    return check_launch("segq_gemm");
}

template <int TM, int TN, int FMT, bool B4, bool GRP>
int launch_few_tile(const FewParams& p, int64_t batch, hipStream_t st) {
    constexpr int DEPTH = few_depth(TM, TN, B4, GRP);
    const int per_wave = ((p.k1 - p.k0 + 127) / 128 + FEW_WAVES - 1) / FEW_WAVES;
    if constexpr (TM == 1) {
        if (p.X) {  // (the host has checked: four units per wave at most)
            const bool f32 = p.x_dtype == SEGQ_F32;
#define SEGQ_QE(ITER_) return f32 ? launch_few_instance<TM, TN, FMT, B4, GRP, ITER_, 4>(p, batch, st) : launch_few_instance<TM, TN, FMT, B4, GRP, ITER_, 2>(p, batch, st)
            if (per_wave == 1) SEGQ_QE(1);
            if (per_wave == 2) SEGQ_QE(2);
            if (per_wave == 3) SEGQ_QE(3);
            if constexpr (TN == 2) SEGQ_QE(4);
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_linear: K too long for a quantise step in the GEMM");  // (not reached)
#undef SEGQ_QE
        }
    }
    if (per_wave > DEPTH) return launch_few_instance<TM, TN, FMT, B4, GRP, 0>(p, batch, st);
    if (per_wave == 1) return launch_few_instance<TM, TN, FMT, B4, GRP, 1>(p, batch, st);
    if (per_wave == 2) return launch_few_instance<TM, TN, FMT, B4, GRP, 2>(p, batch, st);
    if constexpr (DEPTH >= 3) {
        if (per_wave == 3) return launch_few_instance<TM, TN, FMT, B4, GRP, 3>(p, batch, st);
    }
    return launch_few_instance<TM, TN, FMT, B4, GRP, DEPTH>(p, batch, st);
}

template <int FMT, bool B4, bool GRP>
int launch_few_format(const FewParams& p, int fcfg, int64_t batch, hipStream_t st) {
    switch (fcfg) {
        case 0: return launch_few_tile<1, 2, FMT, B4, GRP>(p, batch, st);
        case 1: return launch_few_tile<1, 4, FMT, B4, GRP>(p, batch, st);
        case 2: return launch_few_tile<2, 2, FMT, B4, GRP>(p, batch, st);
        case 3: return launch_few_tile<2, 4, FMT, B4, GRP>(p, batch, st);
    }
    return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: no kernel for tile %d", FIRST_FEW_CFG + fcfg + 1);
}

}  // namespace segq
