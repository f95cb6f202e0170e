// Segmented GEMM, main kernel: eight waves per workgroup, K walked in whole
// 128-byte steps, operands streamed global -> LDS without passing through
// registers wherever no per-byte transform is needed.
//
// Design points, each backed by a measurement on MI355X:
//  * Two waves per SIMD.  The 4-pass v_mfma_i32_16x16x64_i8 issued back to back
//    from ONE wave reaches 56 % of the matrix pipe's rate, from two waves 90 %.
//  * global_load_lds_dwordx4 for plain operands: no staging VGPRs, no ds_write
//    instructions (ds_write_b128 moves ~80 B/clk/CU, a third of what reads do),
//    and nothing in the loop consumes a loaded value, so the loads of step k+1
//    really overlap the MFMAs of step k.  The LDS side of such a load is
//    lane-linear, so the bank swizzle is applied to the global address instead.
//  * int4 weights, and DualScale codes of both signs in one tensor on the tiles that
//    cannot part them behind LDS (MERGE, below, does), go through registers on their
//    way there; their transform is branch-free.
//  * Epilogue through LDS for 16-bit outputs: each lane owns 4 consecutive
//    columns of 16 different rows, which as direct stores are 32-byte pieces of
//    16 lines per instruction (measured 1.7 TB/s); transposed through a private
//    LDS patch every store instruction writes four full 256-byte row pieces.
#pragma once
#include "segq_gemm_kernel.h"
#include "segq_encode.h"
#include <type_traits>

namespace segq {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* glb_ptr_t;

// One lane's 16 bytes from global memory to LDS at lds_base + lane * 16.
__device__ __forceinline__ void load16_to_lds(const uint8_t* g, uint8_t* lds_base) {
    __builtin_amdgcn_global_load_lds((glb_ptr_t)g, (lds_ptr_t)lds_base, 16, 0, 0);
}

// Four consecutive outputs of one row, rounded once to the output type.
template <int OUT>
__device__ __forceinline__ void store4(void* C, int64_t e, const float (&o)[4], bool vec, int n_left) {
    if constexpr (OUT == SEGQ_F32) {
        float* dst = static_cast<float*>(C) + e;
        if (vec) {
            *reinterpret_cast<float4*>(dst) = make_float4(o[0], o[1], o[2], o[3]);
        } else {
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (v < n_left) dst[v] = o[v];
        }
    } else {
        const uint32_t lo = (OUT == SEGQ_BF16) ? pack2_bf16(o[0], o[1]) : pack2_f16(o[0], o[1]);
        const uint32_t hi = (OUT == SEGQ_BF16) ? pack2_bf16(o[2], o[3]) : pack2_f16(o[2], o[3]);
        uint16_t* dst = static_cast<uint16_t*>(C) + e;
        if (vec) {
            *reinterpret_cast<uint2*>(dst) = make_uint2(lo, hi);
        } else {
            const uint32_t h[4] = {lo & 0xffffu, lo >> 16, hi & 0xffffu, hi >> 16};
#pragma unroll
            for (int v = 0; v < 4; ++v)
                if (v < n_left) dst[v] = (uint16_t)h[v];
        }
    }
}


// Four codes of fmt from four values (already scaled), low byte first.
__device__ __forceinline__ uint32_t pack4_codes(int fmt, float a, float b, float c, float d) {
    return fmt == SEGQ_CODE_I8 ? pack4_i8(a, b, c, d) : pack4_e4m3(a, b, c, d);
}

// The epilogue that writes CODES: what a quantise launch with a static per-tensor scale (or a
// DualScale pair, two code tensors) and a fused activation function would have made of this
// GEMM's 16-bit output, bit for bit: the de-quantised sum plus bias (and addend) is rounded to
// out_dtype, the activation function applied in fp32 and rounded to out_dtype again, then
// scaled and encoded.  The float output itself is never written to memory: every wave passes
// 16 rows at a time through its own LDS patch in out_dtype (which is also the transposition that
// gives each lane eight consecutive columns of one row), reads them back, and stores eight
// codes per lane.  epi: the tile's vectors parked in LDS, [1/sx BM | 1/sw BN | bias BN].
template <int BM, int BN, int WGM, int WGN, int FMT>
__device__ __forceinline__ void codes_epilogue(const GemmParams& p, typename AccT<FMT>::type (&acc)[BN / WGN / 16][BM / WGM / 16],
                                               uint8_t* smem, int m0, int n0, int wave, int lane, const float* epi) {
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int TM = WM / 16, TN = WN / 16;
    const int wm = wave % WGM, wn = wave / WGM;
    const int lrow = lane & 15, lgrp = lane >> 4;
    const int m_base = m0 + wm * WM + lrow;
    const int n_base = n0 + wn * WN + 4 * lgrp;
    const bool dual = p.oc_neg != nullptr, two = dual && p.oc_neg != p.oc;  // (the same tensor: codes of both signs in one)
    const float s_pos = p.oc_scale[0];
    const float s_neg = dual ? p.oc_scale_neg[0] : s_pos;
    const bool bf = p.out_dtype == SEGQ_BF16;
    const int fmt = p.oc_fmt, op = p.oc_pre;
    constexpr int RS = WN * 2 + 16;  // patch row stride in bytes; the 16 spreads the rows over the banks
    constexpr int CH = WN / 8;       // 8-element pieces per patch row
    __syncthreads();                 // the operand tiles are dead from here on
    uint8_t* const patch = smem + wave * 16 * RS;
    uint8_t* const ocp = static_cast<uint8_t*>(p.oc);
    uint8_t* const ocn = static_cast<uint8_t*>(p.oc_neg);
    // the 16 rows in the patch -> codes.  A real loop over b would have to index the accumulators, so
    // the blocks below are unrolled, each followed by this loop
    auto encode_rows = [&](int b) __attribute__((always_inline)) {
        for (int j = 0; j < (16 * CH + 63) / 64; ++j) {
            const int c = j * 64 + lane;
            const int row = c / CH, col = c % CH;
            if ((16 * CH) % 64 != 0 && c >= 16 * CH) continue;
            const uint4 raw = *reinterpret_cast<const uint4*>(patch + row * RS + col * 16);
            const uint32_t w[4] = {raw.x, raw.y, raw.z, raw.w};
            const int mm = m0 + wm * WM + b * 16 + row;
            const int n = n0 + wn * WN + col * 8;
            if (mm >= p.M || n >= p.N) continue;
            const int64_t e = (int64_t)mm * p.ldoc + n;
            float t8[8], cp[8], cn[8];
            auto widen = [&](const uint32_t (&q)[4]) __attribute__((always_inline)) {
                if (bf) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) t8[i] = __uint_as_float((i & 1) ? (q[i >> 1] & 0xffff0000u) : (q[i >> 1] << 16));
                } else {
#pragma unroll
                    for (int i = 0; i < 8; ++i) t8[i] = f16_bits_to_f32((i & 1) ? (q[i >> 1] >> 16) : (q[i >> 1] & 0xffffu));
                }
            };
            widen(w);
            if (op != SEGQ_PRE_NONE) {
                act_values(op, t8);
                uint32_t q[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) q[i] = bf ? pack2_bf16(t8[2 * i], t8[2 * i + 1]) : pack2_f16(t8[2 * i], t8[2 * i + 1]);
                widen(q);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float t = t8[i];
                // x >= 0 takes the positive scale; in two tensors the branch not taken holds code(0)
                // (segquant/src/real_quant/quantizer.cuh:193-203).  Without DualScale: one scale for both signs.
                const bool pos = t >= 0.0f;
                t *= pos ? s_pos : s_neg;
                cp[i] = pos || !two ? t : 0.0f;
                cn[i] = pos ? 0.0f : t;
            }
            const uint2 vp = make_uint2(pack4_codes(fmt, cp[0], cp[1], cp[2], cp[3]), pack4_codes(fmt, cp[4], cp[5], cp[6], cp[7]));
            uint2 vn = make_uint2(0u, 0u);
            if (two) vn = make_uint2(pack4_codes(fmt, cn[0], cn[1], cn[2], cn[3]), pack4_codes(fmt, cn[4], cn[5], cn[6], cn[7]));
            if (p.oc_vec && n + 7 < p.N) {
                *reinterpret_cast<uint2*>(ocp + e) = vp;
                if (two) *reinterpret_cast<uint2*>(ocn + e) = vn;
            } else {
                const uint64_t bp = ((uint64_t)vp.y << 32) | vp.x, bn = ((uint64_t)vn.y << 32) | vn.x;
                for (int i = 0; i < 8 && n + i < p.N; ++i) {
                    ocp[e + i] = (uint8_t)(bp >> (8 * i));
                    if (two) ocn[e + i] = (uint8_t)(bn >> (8 * i));
                }
            }
        }
    };
#pragma unroll
    for (int b = 0; b < TM; ++b) {
        const float rx = epi[wm * WM + b * 16 + lrow];
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            const v4f rw = *reinterpret_cast<const v4f*>(epi + BM + wn * WN + a * 16 + 4 * lgrp);
            const v4f bias = *reinterpret_cast<const v4f*>(epi + BM + BN + wn * WN + a * 16 + 4 * lgrp);
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) o[v] = dequant_bias((float)acc[a][b][v], rx, rw[v], bias[v]);
            if (p.addend) add_addend4(p, 0, min(m_base + b * 16, p.M - 1), n_base + a * 16, o);
            *reinterpret_cast<uint2*>(patch + lrow * RS + (a * 16 + 4 * lgrp) * 2) =
                make_uint2(bf ? pack2_bf16(o[0], o[1]) : pack2_f16(o[0], o[1]), bf ? pack2_bf16(o[2], o[3]) : pack2_f16(o[2], o[3]));
        }
        __builtin_amdgcn_wave_barrier();
        encode_rows(b);
        __builtin_amdgcn_wave_barrier();
    }
}

// Scale, add bias, round once, store.  16-bit outputs of full tiles go through a
// per-wave LDS patch so that every store instruction writes whole row pieces.
template <int BM, int BN, int WGM, int WGN, int FMT, bool B4, bool FOLD>
__device__ __forceinline__ void wide_epilogue(const GemmParams& p, typename AccT<FMT>::type (&acc)[BN / WGN / 16][BM / WGM / 16],
                                              v4f (&accf)[FOLD ? BN / WGN / 16 : 1][FOLD ? BM / WGM / 16 : 1],
                                              uint8_t* smem, int64_t z, int m0, int n0, int wave, int lane, int r_epi = 0,
                                              const float* epi = nullptr) {
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int TM = WM / 16, TN = WN / 16;
    typedef typename AccT<FMT>::type acc_t;
    typedef typename AccT<FMT>::elem acc_e;
    const int wm = wave % WGM, wn = wave / WGM;
    const int lrow = lane & 15, lgrp = lane >> 4;
    const int m_base = m0 + wm * WM + lrow;
    const int n_base = n0 + wn * WN + 4 * lgrp;
    auto range_rx = [&](int r, float (&rx)[TM]) {
        const float* sx = p.r[r].sx + z * p.bsSx;
        const int rs = p.r[r].sx_rs;
#pragma unroll
        for (int b = 0; b < TM; ++b) rx[b] = __builtin_amdgcn_rcpf(sx[(int64_t)min(m_base + b * 16, p.M - 1) * rs]);
    };
    auto range_rw = [&](int r, int a, float (&rw)[4]) {
        const float* sw = p.r[r].sw + z * p.bsSw;
        const int cs = p.r[r].sw_cs;
        const float unscale = B4 ? 0.0625f : 1.0f;
#pragma unroll
        for (int v = 0; v < 4; ++v) rw[v] = unscale * __builtin_amdgcn_rcpf(sw[(int64_t)min(n_base + a * 16 + v, p.N - 1) * cs]);
    };
    const int64_t c_off = z * p.bsC;
    if (p.out_dtype == SEGQ_ACC) {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) {
                const int m = m_base + b * 16, n = n_base + a * 16;
                if (m >= p.M) continue;
                acc_t t = acc[a][b];
                if constexpr (B4) { t[0] >>= 4; t[1] >>= 4; t[2] >>= 4; t[3] >>= 4; }
                acc_e* dst = static_cast<acc_e*>(p.C) + c_off + (int64_t)m * p.ldc + n;
                if (p.vec_store && n + 3 < p.N) {
                    *reinterpret_cast<acc_t*>(dst) = t;
                } else {
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        if (n + v < p.N) dst[v] = t[v];
                }
            }
        return;
    }
    const bool is16 = p.out_dtype != SEGQ_F32;
    const bool via_lds = is16 && p.vec_store16 && (n0 + BN <= p.N);
    float rx[TM];
    // epi: the tile's vectors parked in LDS by the caller, [1/sx BM | 1/sw BN | bias BN]
    if constexpr (!FOLD) {
        if (epi) {
#pragma unroll
            for (int b = 0; b < TM; ++b) rx[b] = epi[wm * WM + b * 16 + lrow];
        } else {
            range_rx(r_epi, rx);  // the range whose scales the accumulators are in units of
        }
    }
    if (via_lds) {
        // every wave transposes 16 rows at a time through its own patch of LDS
        constexpr int RS = WN * 2 + 16;  // row stride in bytes; the 16 spreads rows over the banks
        __syncthreads();                 // the operand tiles are dead from here on
        uint8_t* patch = smem + wave * 16 * RS;
        constexpr int CH = WN / 8;  // 16-byte pieces per patch row
        float rwv[TN][4], bvv[TN][4];
        if (epi) {
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                const v4f w = *reinterpret_cast<const v4f*>(epi + BM + wn * WN + a * 16 + 4 * lgrp);
                const v4f bb = *reinterpret_cast<const v4f*>(epi + BM + BN + wn * WN + a * 16 + 4 * lgrp);
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    rwv[a][v] = w[v];
                    bvv[a][v] = bb[v];
                }
            }
        } else {
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                if constexpr (!FOLD) range_rw(r_epi, a, rwv[a]);
#pragma unroll
                for (int v = 0; v < 4; ++v) bvv[a][v] = p.bias ? load_bias(p.bias, p.bias_dtype, n_base + a * 16 + v) : 0.0f;
            }
        }
        // (two instances, so that launches without an addend carry no trace of it)
        auto blocks = [&](auto add_c) __attribute__((always_inline)) {
            constexpr bool ADD = decltype(add_c)::value;
#pragma unroll
            for (int b = 0; b < TM; ++b) {
#pragma unroll
                for (int a = 0; a < TN; ++a) {
                    float o[4];
#pragma unroll
                    for (int v = 0; v < 4; ++v)
                        o[v] = FOLD ? accf[a][b][v] + bvv[a][v] : dequant_bias((float)acc[a][b][v], rx[b], rwv[a][v], bvv[a][v]);
                    if constexpr (ADD) add_addend4(p, z, min(m_base + b * 16, p.M - 1), n_base + a * 16, o);
                    const bool bf = p.out_dtype == SEGQ_BF16;
                    *reinterpret_cast<uint2*>(patch + lrow * RS + (a * 16 + 4 * lgrp) * 2) =
                        make_uint2(bf ? pack2_bf16(o[0], o[1]) : pack2_f16(o[0], o[1]),
                                   bf ? pack2_bf16(o[2], o[3]) : pack2_f16(o[2], o[3]));
                }
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int j = 0; j < (16 * CH + 63) / 64; ++j) {
                    const int c = j * 64 + lane;
                    const int row = c / CH, col = c % CH;
                    if ((16 * CH) % 64 != 0 && c >= 16 * CH) continue;
                    const uint4 v = *reinterpret_cast<const uint4*>(patch + row * RS + col * 16);
                    const int m = m0 + wm * WM + b * 16 + row;
                    if (m < p.M) {
                        *reinterpret_cast<uint4*>(static_cast<uint16_t*>(p.C) + c_off + (int64_t)m * p.ldc + n0 + wn * WN + col * 8) = v;
                    }
                }
                __builtin_amdgcn_wave_barrier();
            }
        };
        if (p.addend) blocks(std::true_type{});
        else blocks(std::false_type{});
        return;
    }
#pragma unroll
    for (int a = 0; a < TN; ++a) {
        float rw[4];
        float bv[4] = {0.f, 0.f, 0.f, 0.f};
        if (epi) {  // (fp32 outputs and ragged columns too: the same factors as above, and no loads behind the K loop)
            const v4f w = *reinterpret_cast<const v4f*>(epi + BM + wn * WN + a * 16 + 4 * lgrp);
            const v4f bb = *reinterpret_cast<const v4f*>(epi + BM + BN + wn * WN + a * 16 + 4 * lgrp);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                rw[v] = w[v];
                bv[v] = bb[v];
            }
        } else {
            if constexpr (!FOLD) range_rw(r_epi, a, rw);
            if (p.bias) {
#pragma unroll
                for (int v = 0; v < 4; ++v) bv[v] = load_bias(p.bias, p.bias_dtype, min(n_base + a * 16 + v, p.N - 1));
            }
        }
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            const int m = m_base + b * 16, n = n_base + a * 16;
            if (m >= p.M || n >= p.N) continue;
            float o[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (FOLD) o[v] = accf[a][b][v] + bv[v];
                else o[v] = dequant_bias((float)acc[a][b][v], rx[b], rw[v], bv[v]);
            }
            add_addend4(p, z, m, n, o);
            const int64_t e = c_off + (int64_t)m * p.ldc + n;
            const bool vec = p.vec_store && (n + 3 < p.N);
            if (p.out_dtype == SEGQ_F32) store4<SEGQ_F32>(p.C, e, o, vec, p.N - n);
            else if (p.out_dtype == SEGQ_BF16) store4<SEGQ_BF16>(p.C, e, o, vec, p.N - n);
            else store4<SEGQ_F16>(p.C, e, o, vec, p.N - n);
        }
    }
}

template <int BM, int BN, int WGM, int WGN, int FMT, bool B4, bool FOLD, bool ASEL>
__global__ void __launch_bounds__(WGM* WGN * 64) gemm_wide_kernel(const GemmParams p) {
    constexpr int NW = WGM * WGN, NT = NW * 64;
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int TM = WM / 16, TN = WN / 16;
    constexpr int A_IT = BM * 8 / NT;                 // 16-byte chunks per thread, activations
    constexpr int B_IT = (B4 ? BN * 4 : BN * 8) / NT;  // same, weights (packed chunks when int4)
    constexpr int RPI = NT / 8;                        // rows covered by one pass of all threads
    constexpr int RPI4 = NT / 4;
    static_assert(BM * 8 % NT == 0 && BN * 4 % NT == 0 && RPI % 16 == 0, "tile does not divide over the threads");
    static_assert(!B4 || FMT == GEMM_I8, "int4 weights pair with int8 activations");
    typedef typename AccT<FMT>::type acc_t;
    typedef typename AccT<FMT>::elem acc_e;
    const acc_t acc_zero = {0, 0, 0, 0};

    extern __shared__ __align__(16) uint8_t smem[];
    uint8_t* const As = smem;                // [2][BM][128]
    uint8_t* const Bs = smem + 2 * BM * BK;  // [2][BN][128]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int lrow = lane & 15, lgrp = lane >> 4;

    int bid = blockIdx.x;
    {
        const int nb = p.tiles_m * p.tiles_n;
        if ((nb & 7) == 0) bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    }
    int tile_m, tile_n;
    {
        const int gsz = p.group_m * p.tiles_n;
        const int g = bid / gsz;
        const int first_m = g * p.group_m;
        const int rows_in_group = min(p.tiles_m - first_m, p.group_m);
        const int in_g = bid - g * gsz;
        tile_m = first_m + in_g % rows_in_group;
        tile_n = in_g / rows_in_group;
    }
    const int m0 = tile_m * BM, n0 = tile_n * BN;
    const int64_t z = blockIdx.y;
    const uint8_t* const Ab = p.A + z * p.bsA;
    const uint8_t* const A2b = p.A2 ? p.A2 + z * p.bsA : nullptr;
    const uint8_t* const Bb = p.B + z * p.bsB;

    // ---- staging.  Thread t, pass i: row i * RPI + t / 8, physical chunk t % 8,
    // which holds logical chunk (t % 8) ^ swz(row).
    const int s_row = tid >> 3;
    const int s_pc = tid & 7;
    const int s_lc = s_pc ^ swz(s_row);
    uint32_t a_goff[A_IT];
#pragma unroll
    for (int i = 0; i < A_IT; ++i) a_goff[i] = (uint32_t)min(m0 + s_row + i * RPI, p.M - 1) * (uint32_t)p.lda + s_lc * 16;
    // weights: same scheme, or 4 packed chunks per row when int4
    const int b_row = B4 ? (tid >> 2) : s_row;
    const int b_pk = tid & 3;  // int4: packed chunk = 32 k = logical chunks 2 b_pk, 2 b_pk + 1
    constexpr int B_RSTEP = B4 ? RPI4 : RPI;
    uint32_t b_goff[B_IT];
#pragma unroll
    for (int i = 0; i < B_IT; ++i)
        b_goff[i] = (uint32_t)min(n0 + b_row + i * B_RSTEP, p.N - 1) * (uint32_t)p.ldb + (B4 ? b_pk : s_lc) * 16;
    const int b_sw = swz(b_row);
    const int w_lds = wave * 8 * BK;  // direct loads: the 8 rows this wave fills per pass

    uint4 ra[ASEL ? A_IT : 1], rb[B4 ? B_IT : 1];

    auto issue_loads = [&](const uint8_t* ap, int k, int buf) {
        if constexpr (ASEL) {
#pragma unroll
            for (int i = 0; i < A_IT; ++i) ra[i] = *reinterpret_cast<const uint4*>(ap + k + a_goff[i]);
        } else {
            uint8_t* as = As + buf * BM * BK + w_lds;
#pragma unroll
            for (int i = 0; i < A_IT; ++i) load16_to_lds(ap + k + a_goff[i], as + i * RPI * BK);
        }
        if constexpr (B4) {
#pragma unroll
            for (int i = 0; i < B_IT; ++i) rb[i] = *reinterpret_cast<const uint4*>(Bb + (k >> 1) + b_goff[i]);
        } else {
            uint8_t* bs = Bs + buf * BN * BK + w_lds;
#pragma unroll
            for (int i = 0; i < B_IT; ++i) load16_to_lds(Bb + k + b_goff[i], bs + i * RPI * BK);
        }
    };
    // sel_or / sel_xor: branch-free sign selection, kept = x & ((negmask ^ sel_xor) | sel_or)
    auto commit_loads = [&](int buf, uint32_t sel_or, uint32_t sel_xor) {
        if constexpr (ASEL) {
            uint8_t* as = As + buf * BM * BK + s_row * BK + s_pc * 16;
#pragma unroll
            for (int i = 0; i < A_IT; ++i) {
                uint4 v = ra[i];
                v.x &= (neg_byte_mask(v.x) ^ sel_xor) | sel_or;
                v.y &= (neg_byte_mask(v.y) ^ sel_xor) | sel_or;
                v.z &= (neg_byte_mask(v.z) ^ sel_xor) | sel_or;
                v.w &= (neg_byte_mask(v.w) ^ sel_xor) | sel_or;
                *reinterpret_cast<uint4*>(as + i * RPI * BK) = v;
            }
        }
        if constexpr (B4) {
            uint8_t* bs = Bs + buf * BN * BK + b_row * BK;
#pragma unroll
            for (int i = 0; i < B_IT; ++i) {
                uint4 lo, hi;
                unpack8_i4x16(rb[i].x, lo.x, lo.y);
                unpack8_i4x16(rb[i].y, lo.z, lo.w);
                unpack8_i4x16(rb[i].z, hi.x, hi.y);
                unpack8_i4x16(rb[i].w, hi.z, hi.w);
                uint8_t* row = bs + i * B_RSTEP * BK;
                *reinterpret_cast<uint4*>(row + (((2 * b_pk) ^ b_sw) << 4)) = lo;
                *reinterpret_cast<uint4*>(row + (((2 * b_pk + 1) ^ b_sw) << 4)) = hi;
            }
        }
        if constexpr (!ASEL || !B4) __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): direct loads have landed
    };

    acc_t acc[TN][TM];
    v4f accf[FOLD ? TN : 1][FOLD ? TM : 1];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = acc_zero;
    if constexpr (FOLD) {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) accf[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    }

    const int f_sw = swz(lrow);
    const int a_frag = (wm * WM + lrow) * BK;
    const int b_frag = (wn * WN + lrow) * BK;

    auto compute = [&](int buf) {
        const uint8_t* as = As + buf * BM * BK + a_frag;
        const uint8_t* bs = Bs + buf * BN * BK + b_frag;
        if constexpr (FMT == GEMM_I8) {
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                const int off = ((ks * 4 + lgrp) ^ f_sw) << 4;
                v4i fa[TM], fb[TN];
#pragma unroll
                for (int t = 0; t < TM; ++t) fa[t] = *reinterpret_cast<const v4i*>(as + t * 16 * BK + off);
#pragma unroll
                for (int t = 0; t < TN; ++t) fb[t] = *reinterpret_cast<const v4i*>(bs + t * 16 * BK + off);
#pragma unroll
                for (int a = 0; a < TN; ++a)
#pragma unroll
                    for (int b = 0; b < TM; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[a], fa[b], acc[a][b], 0, 0, 0);
            }
        } else {
            // (K slot g of the MFMA gets 16-byte pieces g and 4 + g of the step, for both operands:
            // the int8 path's conflict-free read pattern)
            const int off0 = (lgrp ^ f_sw) << 4;
            const int off1 = ((4 + lgrp) ^ f_sw) << 4;
            v8i fa[TM], fb[TN];
#pragma unroll
            for (int t = 0; t < TM; ++t) {
                const v4i lo = *reinterpret_cast<const v4i*>(as + t * 16 * BK + off0);
                const v4i hi = *reinterpret_cast<const v4i*>(as + t * 16 * BK + off1);
                fa[t] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
#pragma unroll
            for (int t = 0; t < TN; ++t) {
                const v4i lo = *reinterpret_cast<const v4i*>(bs + t * 16 * BK + off0);
                const v4i hi = *reinterpret_cast<const v4i*>(bs + t * 16 * BK + off1);
                fb[t] = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
            }
#pragma unroll
            for (int a = 0; a < TN; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b)
                    acc[a][b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[a], fa[b], acc[a][b], 0, 0, 0, 0, 0, 0);
        }
    };

    // lane's output coordinates: row m_base + 16 b, columns n_base + 16 a + 0..3
    const int m_base = m0 + wm * WM + lrow;
    const int n_base = n0 + wn * WN + 4 * lgrp;

    auto range_rx = [&](int r, float (&rx)[TM]) {
        const float* sx = p.r[r].sx + z * p.bsSx;
        const int rs = p.r[r].sx_rs;
#pragma unroll
        for (int b = 0; b < TM; ++b) rx[b] = __builtin_amdgcn_rcpf(sx[(int64_t)min(m_base + b * 16, p.M - 1) * rs]);
    };
    auto range_rw = [&](int r, int a, float (&rw)[4]) {
        const float* sw = p.r[r].sw + z * p.bsSw;
        const int cs = p.r[r].sw_cs;
        const float unscale = B4 ? 0.0625f : 1.0f;  // the staged int4 weights carry an exact factor 16
#pragma unroll
        for (int v = 0; v < 4; ++v) rw[v] = unscale * __builtin_amdgcn_rcpf(sw[(int64_t)min(n_base + a * 16 + v, p.N - 1) * cs]);
    };
    auto fold = [&](int r) {
        if constexpr (FOLD) {
            float rx[TM];
            range_rx(r, rx);
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                float rw[4];
                range_rw(r, a, rw);
#pragma unroll
                for (int b = 0; b < TM; ++b) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) accf[a][b][v] += (float)acc[a][b][v] * rx[b] * rw[v];
                    acc[a][b] = acc_zero;
                }
            }
        }
    };
    auto sel_masks = [&](int a_sel, uint32_t& so, uint32_t& sx) {
        so = (a_sel >= 2) ? 0u : 0xFFFFFFFFu;
        sx = (a_sel == 2) ? 0xFFFFFFFFu : 0u;
    };

    // ---- main loop over (range, k) steps; every range is whole 128-byte steps
    int r = 0, k = p.r[0].k0;
    uint32_t so, sxm;
    sel_masks(p.r[0].a_sel, so, sxm);
    issue_loads((p.r[0].a_sel == 1) ? A2b : Ab, k, 0);
    commit_loads(0, so, sxm);
    __syncthreads();
    int buf = 0;
    while (true) {
        int rn = r, kn = k + BK;
        const bool range_done = kn >= p.r[r].k1;
        if (range_done) {
            rn = r + 1;
            kn = (rn < p.nr) ? p.r[rn].k0 : 0;
        }
        const bool more = rn < p.nr;
        if (more) {
            const int sel = p.r[rn].a_sel;
            sel_masks(sel, so, sxm);
            issue_loads((sel == 1) ? A2b : Ab, kn, buf ^ 1);
        }
        compute(buf);
        if (FOLD && range_done) fold(r);
        if (!more) break;
        commit_loads(buf ^ 1, so, sxm);
        __syncthreads();
        buf ^= 1;
        r = rn;
        k = kn;
    }

    wide_epilogue<BM, BN, WGM, WGN, FMT, B4, FOLD>(p, acc, accf, smem, z, m0, n0, wave, lane);
}

// Low-rank branch of the epilogue: of[a][b] += sum_k L2T[n][k] T[m][k] over k < lr_rank, on the
// matrix cores (v_mfma_f32_16x16x32_bf16 / _f16, fp32 accumulation), for the wave's WM x WN
// patch at (m_row0, n_col0).  `of` holds the de-quantised sums in output units in the lane layout
// of the accumulators (four consecutive columns of one row per lane and block), which is also
// the result layout of these MFMAs with L2T as the first operand.  Both fragments are 16 rows of
// 32 contiguous 16-bit values: a lane reads the 16 bytes of its row at k + 8 lgrp, straight from
// memory (T and L2T are small and stay in the L2) or, the first 32 columns with one range, from the K loop's LDS.
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

// LDS: the kernel may have the wave's rows of the first 32 columns of both in LDS by then (in_lds), 64 bytes each at lds_t and lds_l.
// (A template argument: instances that never have them there spilled more registers when the code merely did not take that
// side, int8 parked 256 x 256 672 bytes a lane for 556, 192 x 256 208 for 132.)
template <bool LDS, int TM, int TN>
__device__ __forceinline__ void lowrank_accumulate(const GemmParams& p, v4f (&of)[TN][TM], int m_row0, int n_col0, int lane,
                                                   [[maybe_unused]] bool in_lds = false, [[maybe_unused]] const uint8_t* lds_t = nullptr,
                                                   [[maybe_unused]] const uint8_t* lds_l = nullptr) {
    const int lrow = lane & 15, lgrp = lane >> 4;
    const bool bf = p.out_dtype == SEGQ_BF16;
    for (int kk = 0; kk < p.lr_rank; kk += 32) {
        uint4 tf[TM];
#pragma unroll
        for (int b = 0; b < TM; ++b) {
            const int64_t m = min(m_row0 + b * 16 + lrow, p.M - 1);
            if (LDS && in_lds && kk == 0) tf[b] = *reinterpret_cast<const uint4*>(lds_t + (b * 16 + lrow) * 64 + lgrp * 16);
            else tf[b] = *reinterpret_cast<const uint4*>(p.lr_t + m * p.lr_ldt + kk + lgrp * 8);
        }
        // (half of the column blocks' loads at a time, in front of their products: one by one, every block waited for L2
        // behind the block before it; all at once, registers.  Two where the sums take half of the registers: with four the one-range
        // int8 256 x 256 instance spilled 8 bytes a lane.)
        constexpr int CH = TM * TN >= 32 ? 2 : (TN + 1) / 2;
#pragma unroll
        for (int a0 = 0; a0 < TN; a0 += CH) {
            uint4 lf[CH];
#pragma unroll
            for (int a = a0; a < TN && a < a0 + CH; ++a) {
                const int64_t n = min(n_col0 + a * 16 + lrow, p.N - 1);
                if (LDS && in_lds && kk == 0) lf[a - a0] = *reinterpret_cast<const uint4*>(lds_l + (a * 16 + lrow) * 64 + lgrp * 16);
                else lf[a - a0] = *reinterpret_cast<const uint4*>(p.lr_l2 + n * p.lr_ldl + kk + lgrp * 8);
            }
#pragma unroll
            for (int a = a0; a < TN && a < a0 + CH; ++a)
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    if (bf)
                        of[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, lf[a - a0]), __builtin_bit_cast(v8bf, tf[b]), of[a][b], 0, 0, 0);
                    else
                        of[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, lf[a - a0]), __builtin_bit_cast(v8h, tf[b]), of[a][b], 0, 0, 0);
                }
        }
    }
}

// s_waitcnt immediate for "vmcnt(n) lgkmcnt(0)" on gfx9-family encodings
constexpr int waitcnt_vm_lgkm0(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4); }

// Two workgroups share a tile.  Each leaves its share (of, in output units) in the workspace and counts itself in; the one that
// finds the other counted adds that share to its own (a + b = b + a: the result does not depend on who came last) and
// finishes the tile: true.  The two can sit on different XCDs, whose L2 caches do not see each other's lines, so the
// shares are written through and read past the caches (agent scope: what the compiler emits for a relaxed agent-scope
// atomic, but 16 bytes per lane: 1 KB contiguous per wave and instruction).  flag: a word of LDS that is read no more.
// CH: blocks whose loads are in flight at once (registers: the sums are still live).
template <int NT, int CH, int TN, int TM>
__device__ __forceinline__ bool meet_share(const GemmParams& p, v4f (&of)[TN][TM], int tile_id, int my, int tid, int* flag) {
    using v4u = __attribute__((ext_vector_type(4))) unsigned int;
    constexpr int AGENT = 16;  // the cache-policy bit for agent scope
    constexpr int SHARE = TN * TM * NT * 16;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<uint8_t*>(p.part) + (int64_t)tile_id * 2 * SHARE, 0, 2 * SHARE, 0x00020000);
#pragma unroll
    for (int i = 0; i < TN * TM; ++i)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, of[i / TM][i % TM]), rs, tid * 16, my * SHARE + i * NT * 16, AGENT);
    __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(0));  // this wave's stores have reached memory
    __syncthreads();                                  // ... and so have the other waves'
    if (tid == 0) {
        // the launch's own stamp instead of a count: whatever the word held before (an earlier
        // launch's stamp, or anything at all in a fresh workspace) reads as "nobody yet"
        const unsigned before = __hip_atomic_exchange(p.arrived + tile_id, p.stamp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *flag = before == p.stamp;
        // the second one clears the word: a replay of this very launch (a captured graph keeps
        // the stamp it was recorded with) must find "nobody yet" again
        if (before == p.stamp) __hip_atomic_store(p.arrived + tile_id, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    if (!*flag) return false;
#pragma unroll
    for (int c0 = 0; c0 < TN * TM; c0 += CH) {
        v4u other[CH];
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (c0 + i < TN * TM)
                other[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, tid * 16, (1 - my) * SHARE + (c0 + i) * NT * 16, AGENT);
#pragma unroll
        for (int i = 0; i < CH; ++i)
            if (c0 + i < TN * TM) of[(c0 + i) / TM][(c0 + i) % TM] += __builtin_bit_cast(v4f, other[i]);
    }
    return true;
}

// Software-pipelined variant for plain 8-bit operands (both straight to LDS) with
// NS LDS stages.  Two are what nearly all instances have: on FLUX shapes three and
// four stages measured slower (they cost a co-resident workgroup or buy nothing,
// the global -> LDS path being throughput- rather than latency-bound: ~31 of a
// measured ~55 B/clk/CU).  MERGE instances have three (launch_mix), launches of few
// tiles four and five (128 x 128 and 128 x 96, int8).  The K step is split at its one barrier:
//
//   barrier (tile s landed, tile s-1 fully in registers)
//     DMA tile s+1 into the buffer of tile s-1      <- a whole step of latency cover
//     LDS -> fragments F0 of tile s
//     MFMAs on fragments F1 of tile s-1             <- hides the F0 reads
//     LDS -> fragments F1 of tile s
//     MFMAs on F0 of tile s                         <- hides the F1 reads
//   wait own DMA and LDS reads, barrier
//
// so fragment reads never stand between an MFMA group and the one before it.

// 1 / x for the second register set of int8 ranges: v_rcp_f32 (1 ulp) and one Newton step, with which the sums lie as
// close to the exact ones as with correctly rounded quotients, which the general kernel takes for the same launches when
// they are small or ragged; v_rcp_f32 through a ratio of two scales put them 1.4 times as far (rms).  0, infinities and
// NaN have no finite residual and keep v_rcp_f32's value.  512 x 1024 x 512, two ranges, with the quantise launch: v_rcp_f32 13.4 us, this
// 13.8, divisions 14.6.  e4m3 keeps v_rcp_f32: the matrix cores' own sums are off by hundreds of times as much; parked
// sums too, whose launches are the layers' long ones (9216 x 15360 x 3072: 0.2 % more with the Newton step).
template <int FMT>
__device__ __forceinline__ float recip(float x) {
    const float y = __builtin_amdgcn_rcpf(x);
    if constexpr (FMT == GEMM_F8) return y;
    const float e = __builtin_fmaf(-x, y, 1.0f);
    return __builtin_fabsf(e) < 1.0f ? __builtin_fmaf(y, e, y) : y;
}

template <int BM, int BN, int WGM, int WGN, int FMT, bool FOLD, int NS, bool GRP = false, bool PARK = false, bool FINISH = false,
          bool CODES = false,  // CODES: the epilogue writes the next linear's codes instead of floats (one range)
          bool SEP = false,    // SEP (e4m3, several ranges): a second register set, as int8 has it, instead of rescaling in place
          bool KT = false,     // KT: K ends anywhere in sixteens (one walk of K)
          bool DUAL = false,   // DUAL: two ranges over one run of K, from the two code tensors, in one walk
          bool MIX = false,    // MIX (DUAL): whole steps of K, behind them those of a plain range, K shares
          bool MERGE = false>  // MERGE (MIX): both signs in one code tensor, parted in registers
__global__ void __launch_bounds__(WGM* WGN * 64) gemm_pipe_kernel(const GemmParams p) {
    static_assert(!CODES || (!FOLD && !GRP && !PARK && !FINISH), "codes out: plain operands, one range");
    static_assert(!KT || (!FOLD && !GRP && !PARK && !FINISH && !CODES && NS == 2), "a ragged end of K: one walk, two stages");
    static_assert(!DUAL || KT != MIX, "DUAL instances take any K, or whole steps of it and a plain range");
    static_assert(!MIX || (DUAL && !FOLD && !GRP && !PARK && !FINISH && !CODES && (NS == 2 || MERGE)), "MIX: one walk, two stages");
    static_assert(!MERGE || MIX, "MERGE instances are MIX instances");
    // DUAL (DualScale's two ranges over the same K and the same weights): the tile's BM rows of LDS are BM / 2 rows of each
    // code tensor, the two halves of every wave's row blocks, so that a wave holds both sums of an output and a weight
    // tile is read once for both.  What two ranges in turn need a second register set for, these have as the second
    // half of their blocks, and each sum is scaled by its own range's scales at the end.
    // MIX (an input segment in front of a DualScale one: attention output | GELU'd MLP state): the plain range is walked
    // behind the two.  There the sums of both signs become one fp32 sum in output units, in the registers of the first, and
    // the second's start again from zero with the plain range, whose rows take the second half of the tile's: half the MFMAs
    // and fragment reads per step, two thirds of the DMA.  Three sums in two register sets: nothing is parked, no
    // third set, no ratio of scales, weights read once.  Bound by the matrix cores' rate under the power limit: 9216 x 3072 x
    // (3072 + 12288) int8 on 384 x 192 2.6 POP/s with both products (parked 2.1), e4m3 2.7 (rescaled in place 2.4).
    constexpr int OM = DUAL ? BM / 2 : BM;   // output rows of the tile
    constexpr int AR = MERGE ? BM / 2 : BM;  // rows of activation codes in LDS
    constexpr int NW = WGM * WGN, NT = NW * 64;
    constexpr int WM = BM / WGM, WN = BN / WGN;
    constexpr int TM = WM / 16, TN = WN / 16;
    constexpr int RPI = NT / 8;                                  // rows one pass of all threads covers
    constexpr int A_IT = (AR + RPI - 1) / RPI, B_IT = (BN + RPI - 1) / RPI;
    constexpr int A_TAIL = AR % RPI, B_TAIL = BN % RPI;          // rows of a last, partial pass (0: none)
    static_assert(A_TAIL % 8 == 0 && B_TAIL % 8 == 0 && WM % 16 == 0 && WN % 16 == 0, "tile does not divide over the waves");
    typedef typename AccT<FMT>::type acc_t;
    constexpr bool F8 = FMT == GEMM_F8;
    // Several ranges: int32 accumulators are folded into a second, fp32 set at the
    // end of each range.  fp32 accumulators (e4m3) need no second set: at a range
    // boundary they are rescaled from the finished range's scales to the next
    // one's (acc *= sx' sw' / (sx sw), one fp32 rounding), so the sum stays in
    // units of the current range and the epilogue divides by the last range's.
    //
    // GRP (int8): every K step of 128 is a group with its own de-quantisation
    // factor per output column (group-wise weight scales).  The step's int32
    // sums are multiplied by the factors and added to an fp32 set, which from
    // there on is treated like e4m3's fp32 accumulators: in units of the current
    // range, rescaled at range boundaries, scaled by 1/(sx sw) in the epilogue.
    // The group kernel runs the e4m3 schedule (whole-step fragments of 32 bytes,
    // refilled as the step lets go of them): both 64-byte K halves of an output
    // block are multiplied back to back into int32 temporaries, so no int32
    // accumulator set lives across steps.
    // LAG (one range): a column block's temporaries wait while the next block is multiplied, and
    // two of their values are converted and scaled behind every MFMA.  Bound by issue slots: an
    // int8 MFMA holds the matrix pipe for 16 clocks and takes two of the four VALU slots in them, the
    // four VALU instructions that belong to it the rest and more (25 to 27 clocks measured for an MFMA
    // with four, 17 with two; v_cvt_f32_i32 and a subtraction cost the same).  Left to itself the compiler gathers
    // a step's conversions at its end, behind the MFMAs of every wave, which two workgroups of 128 x 128
    // per CU hide and one of a big tile does not: 8192 x 10240 x 1280 on 256 x 256 in LAG order 155 us with the
    // int4 expansion, 128 x 128 165 to 167; 8192 x 1280 x 5120 on 192 x 256 69, 128 x 128 81 (256 x 128
    // 100 in the compiler's order, 95 in this one).  With several ranges the big tiles spill: 128 x 128, converted at once.
    static_assert(!GRP || (!F8 && NS == 2), "group factors: int8, two stages");
    // int8 tiles above 256 x 256 run the whole-step schedule too: one set of 32-byte fragments
    // instead of two sets of 16-byte ones leaves room for their accumulators
    constexpr bool WS = !F8 && !GRP && BM * BN > 256 * 256;
    constexpr bool S8 = F8 || GRP || WS;  // whole-step fragments
    //
    // PARK (int8, several ranges): no second register set at all.  When a range ends, its
    // int32 sums are scaled by the range's own 1 / (sx sw), i.e. taken to output units, and
    // added to this tile's fp32 slot of a workspace the caller lends; the accumulators
    // restart from zero.  The epilogue scales the last range's sums and adds the slot.
    // Each thread only ever reads back what it wrote itself.  This keeps the big tiles for
    // int8 with K segments or DualScale: a few hundred KB of traffic per tile and range
    // boundary against ~14 MB of operands.
    // Neither here nor in the second register set do a range's sums pass through another
    // range's scales: a side of a DualScale tensor that holds nothing may have the scale
    // limit / 0 = inf and adds exact zeros, where a ratio of the two scales would make
    // infinities and NaNs of the other side's sums.  For e4m3 that is SEP, taken where the
    // scales come from outside (segq_krange.own_sum): 2 x 2048 x 1536 x 3072 DualScale 61.9 us
    // rescaled in place, 62.2 us with the second set, and 256 x 256 tiles out of reach.
    static_assert(!PARK || (FOLD && !F8 && !GRP && FINISH), "parking: int8 with several ranges, finished in output units");
    static_assert(!WS || (!FOLD && !PARK), "int8 above 256 x 256: one range");
    static_assert(!SEP || (FOLD && F8 && !PARK && !FINISH), "SEP: e4m3 with several ranges");
    constexpr bool ACCF = FOLD && (!F8 || SEP) && !GRP && !PARK;
    constexpr bool HASF = ACCF || GRP;
    const acc_t acc_zero = {0, 0, 0, 0};
    // Split K (p.splits > 1): workgroup (tile, y) multiplies the y-th share of the K steps,
    // counted through the ranges, and writes an fp32 partial result that a second kernel
    // sums.  r_last is the range its last step lies in: the one whose units its
    // accumulators end up in (without a split: the last range).
    int r_last = p.nr - 1, r_begin = 0;  // (r_begin: the range its first step lies in)

    static_assert(NS >= 2 && (NS - 1) * (A_IT + B_IT) < 64, "vmcnt holds 6 bits");
    static_assert(!S8 || ((NS == 2 || MERGE) && TN >= 3), "the e4m3 schedule reads two weight fragments ahead in a two-stage ring");
    extern __shared__ __align__(16) uint8_t smem[];
    uint8_t* const As = smem;                  // [NS][AR][128]
    uint8_t* const Bs = smem + NS * AR * BK;   // [NS][BN][128]

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WGM, wn = wave / WGM;
    const int lrow = lane & 15, lgrp = lane >> 4;

    // Workgroups are dealt to the eight XCDs in turn, each with an L2 of its own.  Every XCD gets a
    // run of consecutive tiles (with a K split: of consecutive (share, tile) pairs), so that its
    // workgroups stream few distinct operand panels and its L2 serves most of their requests.
    int bid = blockIdx.x, zy = blockIdx.y;
    {
        const int nb = p.tiles_m * p.tiles_n;
        if (p.splits > 1) {
            const int total = nb * p.splits, lin = zy * nb + bid, q = total >> 3, r = total & 7, x = lin & 7;
            const int v = x * q + min(x, r) + (lin >> 3);
            zy = v / nb;
            bid = v - zy * nb;
        } else if ((nb & 7) == 0) {
            bid = (bid & 7) * (nb >> 3) + (bid >> 3);
        }
    }
    const int tile_id = bid;  // names this tile's room in the workspaces
    // Several ranges, no K split: the workgroups of XCD x walk the ranges starting from range
    // x mod nr (and wrap), so that at any K step only part of the chip is at a range boundary, where
    // int8 tiles store their sums to the workspace.  All workgroups of an XCD keep the same order:
    // they share operand panels through its L2.  The order of a tile's fp32 additions depends on
    // its XCD only, so a launch gives the same bits every time.  ph(j): the range walked j-th.
    const int r_off = (FOLD && p.rot) ? (int)(blockIdx.x & 7) % p.nr : 0;
    auto ph = [&](int j) { const int t = j + r_off; return t >= p.nr ? t - p.nr : t; };
    int tile_m, tile_n;
    {
        const int gsz = p.group_m * p.tiles_n;
        const int g = bid / gsz;
        const int first_m = g * p.group_m;
        const int rows_in_group = min(p.tiles_m - first_m, p.group_m);
        const int in_g = bid - g * gsz;
        tile_m = first_m + in_g % rows_in_group;
        tile_n = in_g / rows_in_group;
    }
    const int m0 = tile_m * OM, n0 = tile_n * BN;
    const int64_t z = zy;
    const uint8_t* const Ab = p.A + z * p.bsA;
    const uint8_t* const A2b = p.A2 ? p.A2 + z * p.bsA : nullptr;
    const uint8_t* const Bb = p.B + z * p.bsB;

    const int s_row = tid >> 3;
    const int s_lc = (tid & 7) ^ swz(s_row);
    uint32_t a_goff[A_IT], b_goff[B_IT];
#pragma unroll
    for (int i = 0; i < A_IT; ++i) {
        int row = s_row + i * RPI;
        if constexpr (DUAL && !MERGE) row = row / WM * (WM / 2) + row % (WM / 2);
        a_goff[i] = (uint32_t)min(m0 + row, p.M - 1) * (uint32_t)p.lda + s_lc * 16;
    }
#pragma unroll
    for (int i = 0; i < B_IT; ++i) b_goff[i] = (uint32_t)min(n0 + s_row + i * RPI, p.N - 1) * (uint32_t)p.ldb + s_lc * 16;
    const int w_lds = wave * 8 * BK;
    static_assert(!DUAL || ((MIX || RPI % WM == 0) && WM % 32 == 0), "a wave's eight rows of a pass come from one of the two tensors");
    const bool second = DUAL && (wave * 8) % WM >= WM / 2;
    uint32_t seconds = 0;  // MIX: the passes whose rows are of the second tensor
    if constexpr (MIX && !MERGE) {
#pragma unroll
        for (int i = 0; i < A_IT; ++i) seconds |= ((wave * 8 + i * RPI) % WM >= WM / 2 ? 1u : 0u) << i;
    }
    uint32_t wanted = MERGE ? ~0u : seconds | (((1u << B_IT) - 1u) << A_IT);  // MIX: the passes that a step of the plain range loads, activations then weights
    // KT: pieces of a row past the end of K.  They are loaded from the step's first piece instead, which is there (a weight
    // row that holds a NaN gives NaN either way), and what they became in the activations is cleared before it is read.
    const int k_tail = KT ? (p.r[0].k1 - p.r[0].k0) % BK : 0;
    const bool past_k = KT && k_tail != 0 && s_lc * 16 >= k_tail;
    uint32_t back = 0;  // what to go back by in the step that is loaded next
    auto clear_tail = [&](int buf) __attribute__((always_inline)) {
        if constexpr (KT) {
            if (past_k) {
#pragma unroll
                for (int i = 0; i < A_IT; ++i)
                    if (!(A_TAIL != 0 && i == A_IT - 1 && s_row >= A_TAIL))
                        *reinterpret_cast<uint4*>(As + buf * AR * BK + (s_row + i * RPI) * BK + (tid & 7) * 16) = make_uint4(0, 0, 0, 0);
            }
            __syncthreads();
        }
    };

    // a wave covers 8 rows of a pass, so whether it takes part in a partial last pass is wave-uniform
    const bool a_skip = A_TAIL != 0 && wave * 8 >= A_TAIL;
    const bool b_skip = B_TAIL != 0 && wave * 8 >= B_TAIL;
    auto dma1 = [&](const uint8_t* ap, const uint8_t* bp, int buf, int i, auto plain_c) {  // plain_c: a step of MIX's plain range
        if constexpr (MIX && decltype(plain_c)::value) {
            if (!((wanted >> i) & 1u)) return;
        }
        if (i < A_IT) {
            if (i == A_IT - 1 && a_skip) return;
            if constexpr (MIX && !MERGE && !decltype(plain_c)::value) ap += (seconds >> i) & 1u ? A2b - Ab : 0;
            load16_to_lds(ap + (KT ? a_goff[i] - back : a_goff[i]), As + buf * AR * BK + w_lds + i * RPI * BK);
        } else {
            if (i == A_IT + B_IT - 1 && b_skip) return;
            load16_to_lds(bp + (KT ? b_goff[i - A_IT] - back : b_goff[i - A_IT]), Bs + buf * BN * BK + w_lds + (i - A_IT) * RPI * BK);
        }
    };
    // "all but the newest nt tiles of this wave's DMA have landed, and all its LDS reads"
    auto wait_dma = [&](auto nt_c) {
        constexpr int nt = decltype(nt_c)::value;
        constexpr int full = A_IT + B_IT;
        if constexpr (nt == 0 || (A_TAIL == 0 && B_TAIL == 0)) {
            __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(nt * full));
        } else {
            const int miss = (a_skip ? 1 : 0) + (b_skip ? 1 : 0);
            if (miss == 0) __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(nt * full));
            else if (miss == 1) __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(nt * (full - 1)));
            else __builtin_amdgcn_s_waitcnt(waitcnt_vm_lgkm0(nt * (full - 2)));
        }
    };
    auto dma = [&](const uint8_t* ap, const uint8_t* bp, int buf, auto plain_c) {
#pragma unroll
        for (int i = 0; i < A_IT + B_IT; ++i) dma1(ap, bp, buf, i, plain_c);
    };

    acc_t acc[TN][TM];
    v4f accf[HASF ? TN : 1][HASF ? TM : 1];
#pragma unroll
    for (int a = 0; a < TN; ++a)
#pragma unroll
        for (int b = 0; b < TM; ++b) acc[a][b] = acc_zero;
    if constexpr (HASF) {
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = 0; b < TM; ++b) accf[a][b] = v4f{0.f, 0.f, 0.f, 0.f};
    }


    const int f_sw = swz(lrow);
    const int a_frag = (wm * (MERGE ? WM / 2 : WM) + lrow) * BK;
    const int b_frag = (wn * WN + lrow) * BK;
    // int8: two fragment sets, one per 64-byte K half of a step.  e4m3: one set of
    // 32-byte fragments (the 16 x 16 x 128 MFMA eats a whole step), whose registers
    // are refilled for the next step as the current one lets go of them.
    v4i fa[S8 ? 1 : 2][S8 ? 1 : TM], fb[S8 ? 1 : 2][S8 ? 1 : TN];
    v8i fa8[S8 ? TM : 1], fb8[S8 ? TN : 1];
    auto frag8 = [&](int buf, int i) {  // fragment i of the step in buffer buf: 0 .. TM-1 activations, then weights
      if constexpr (S8) {
        // Lane group g feeds K slot [32 g, 32 g + 32) of the MFMA with bytes [16 g, 16 g + 16) and
        // [64 + 16 g, 64 + 16 g + 16) of the step: activations and weights are permuted alike, so the
        // sum is the same, and each of the two reads has the int8 kernels' conflict-free pattern (the
        // four groups of a row read four neighbouring 16-byte pieces; reading pieces 2 g and 2 g + 1
        // instead costs a two-way bank conflict on every read).
        const int off0 = (lgrp ^ f_sw) << 4;
        const int off1 = ((4 + lgrp) ^ f_sw) << 4;
        // (MERGE: fragment i of the second half is read, as it stands)
        const uint8_t* src = (i < TM) ? As + buf * AR * BK + a_frag + (MERGE ? i - TM / 2 : i) * 16 * BK : Bs + buf * BN * BK + b_frag + (i - TM) * 16 * BK;
        const v4i lo = *reinterpret_cast<const v4i*>(src + off0);
        const v4i hi = *reinterpret_cast<const v4i*>(src + off1);
        const v8i f = v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        if (i < TM) fa8[i] = f;
        else fb8[i - TM] = f;
      }
    };

    // MERGE: dwords [d0, d1) of a fragment of codes of both signs -> those of the positive ones and of the negative ones, the
    // others zero: four VALU instructions per dword
    auto part_of = [](auto& pos, auto& neg, int d0, int d1) __attribute__((always_inline)) {
#pragma unroll
        for (int d = d0; d < d1; ++d) {
            const uint32_t v = (uint32_t)neg[d];
            const uint32_t mask = __builtin_amdgcn_perm(v, v << 8, 0x0B090A08u);  // every byte's sign, eight times
            pos[d] = (int)(v & ~mask);
            neg[d] = (int)(v & mask);
        }
    };
    auto part = [&](int i, int d0, int d1) __attribute__((always_inline)) {
        if constexpr (MERGE && S8) part_of(fa8[i], fa8[i + TM / 2], d0, d1);
    };
    auto part1 = [&](int h, int d) __attribute__((always_inline)) {  // dword d of set h's
        if constexpr (MERGE && !S8) part_of(fa[h][d / 4], fa[h][d / 4 + TM / 2], d % 4, d % 4 + 1);
    };

    // K half h of the tile in buffer buf -> fragment slot h, one 16-byte read at a
    // time: reads 0 .. TM-1 are the activation fragments, TM .. TM+TN-1 the weights
    auto frag1 = [&](int buf, int h, int i) {
        if constexpr (!S8) {
            const int off = ((h * 4 + lgrp) ^ f_sw) << 4;
            if (i < TM) fa[h][i] = *reinterpret_cast<const v4i*>(As + buf * AR * BK + a_frag + (MERGE ? i - TM / 2 : i) * 16 * BK + off);
            else fb[h][i - TM] = *reinterpret_cast<const v4i*>(Bs + buf * BN * BK + b_frag + (i - TM) * 16 * BK + off);
        }
    };
    auto frags = [&](int buf, int h) {
#pragma unroll
        for (int i = MERGE ? TM / 2 : 0; i < TM + TN; ++i) frag1(buf, h, i);
    };
    const int m_base = m0 + wm * WM + lrow;
    const int n_base = n0 + wn * WN + 4 * lgrp;
    v4f* const slot = PARK ? reinterpret_cast<v4f*>(p.park) + ((int64_t)zy * gridDim.x + tile_id) * (BM * BN / 4) + tid : nullptr;
    auto park = [&](int r) __attribute__((always_inline)) {
        if constexpr (PARK) {
            if (r < r_last) {
                const float* sx = p.r[ph(r)].sx;  // (one problem: parking serves no batch)
                const float* sw = p.r[ph(r)].sw;
                const int rs = p.r[ph(r)].sx_rs, cs = p.r[ph(r)].sw_cs;
                float rx[TM];
#pragma unroll
                for (int b = 0; b < TM; ++b) rx[b] = __builtin_amdgcn_rcpf(sx[(int64_t)min(m_base + b * 16, p.M - 1) * rs]);
#pragma unroll
                for (int a = 0; a < TN; ++a) {
                    v4f rw;
#pragma unroll
                    for (int v = 0; v < 4; ++v) rw[v] = __builtin_amdgcn_rcpf(sw[(int64_t)min(n_base + a * 16 + v, p.N - 1) * cs]);
                    v4f old[TM];
                    if (r > r_begin) {
#pragma unroll
                        for (int b = 0; b < TM; ++b) old[b] = slot[(a * TM + b) * NT];
                    }
#pragma unroll
                    for (int b = 0; b < TM; ++b) {
                        v4f t = __builtin_convertvector(acc[a][b], v4f) * rx[b] * rw;
                        if (r > r_begin) t += old[b];
                        slot[(a * TM + b) * NT] = t;
                        acc[a][b] = acc_zero;
                    }
                }
            }
        }
    };
    auto fold = [&](int r) __attribute__((always_inline)) {
        if constexpr (FOLD && !ACCF && (F8 || GRP)) {
            auto& facc = [&]() -> auto& { if constexpr (GRP) return accf; else return acc; }();
            if (r < r_last) {  // rescale to the next range's units
                const float* sx = p.r[ph(r)].sx + z * p.bsSx;
                const float* sw = p.r[ph(r)].sw + z * p.bsSw;
                const float* sx2 = p.r[ph(r + 1)].sx + z * p.bsSx;
                const float* sw2 = p.r[ph(r + 1)].sw + z * p.bsSw;
                const int rs = p.r[ph(r)].sx_rs, cs = p.r[ph(r)].sw_cs, rs2 = p.r[ph(r + 1)].sx_rs, cs2 = p.r[ph(r + 1)].sw_cs;
                float fx[TM];
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    const int64_t m = min(m_base + b * 16, p.M - 1);
                    fx[b] = sx2[m * rs2] * __builtin_amdgcn_rcpf(sx[m * rs]);
                }
#pragma unroll
                for (int a = 0; a < TN; ++a) {
                    v4f fw;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int64_t n = min(n_base + a * 16 + v, p.N - 1);
                        fw[v] = sw2[n * cs2] * __builtin_amdgcn_rcpf(sw[n * cs]);
                    }
#pragma unroll
                    for (int b = 0; b < TM; ++b) facc[a][b] = facc[a][b] * (fw * fx[b]);
                }
            }
        }
        if constexpr (ACCF) {
            const float* sx = p.r[ph(r)].sx + z * p.bsSx;
            const float* sw = p.r[ph(r)].sw + z * p.bsSw;
            const int rs = p.r[ph(r)].sx_rs, cs = p.r[ph(r)].sw_cs;
            float rx[TM];
#pragma unroll
            for (int b = 0; b < TM; ++b) rx[b] = recip<FMT>(sx[(int64_t)min(m_base + b * 16, p.M - 1) * rs]);
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                float rw[4];
#pragma unroll
                for (int v = 0; v < 4; ++v) rw[v] = recip<FMT>(sw[(int64_t)min(n_base + a * 16 + v, p.N - 1) * cs]);
#pragma unroll
                for (int b = 0; b < TM; ++b) {
#pragma unroll
                    for (int v = 0; v < 4; ++v) accf[a][b][v] += (float)acc[a][b][v] * rx[b] * rw[v];
                    acc[a][b] = acc_zero;
                }
            }
        }
    };

    // Two cursors walk the ranges: (lr, lk) is the tile loaded NS steps ahead,
    // (cr, ck) the tile being multiplied.  The end of the current range and the
    // source of its activations stay in registers, so the range table is read
    // only when a cursor crosses into the next range.
    int steps = 0;
    [[maybe_unused]] int n_dual = 0;  // MIX: how many of the steps are of the two ranges
    if constexpr (MIX) {}
    else if constexpr (KT) steps = (p.r[0].k1 - p.r[0].k0 + BK - 1) / BK;
    else
        for (int i = 0; i < p.nr; ++i) steps += (p.r[i].k1 - p.r[i].k0) / BK;
    int lr = 0, skip = 0;  // this workgroup's first step: `skip` steps into range lr
    if constexpr (MIX) {  // a step of the plain range counts half of one of the two
        const int d = (p.r[0].k1 - p.r[0].k0) / BK, all = 2 * d + (p.nr > 2 ? (p.r[2].k1 - p.r[2].k0) / BK : 0);
        auto step_at = [&](int c) { return c < 2 * d ? c >> 1 : c - d; };
        int first = 0;
        steps = all - d;
        if (p.splits > 1) {
            first = step_at((int)((int64_t)all * zy / p.splits));
            steps = step_at((int)((int64_t)all * (zy + 1) / p.splits)) - first;
        }
        n_dual = max(min(first + steps, d) - first, 0);
        lr = first < d ? 0 : 2;
        skip = first < d ? first : first - d;
        r_last = 2;
    } else if (p.splits > 1) {
        skip = (int)((int64_t)steps * zy / p.splits);
        steps = (int)((int64_t)steps * (zy + 1) / p.splits) - skip;
        while (lr + 1 < p.nr && skip >= (p.r[ph(lr)].k1 - p.r[ph(lr)].k0) / BK) {
            skip -= (p.r[ph(lr)].k1 - p.r[ph(lr)].k0) / BK;
            ++lr;
        }
        r_last = r_begin = lr;
        for (int left = skip + steps; r_last + 1 < p.nr && left > (p.r[ph(r_last)].k1 - p.r[ph(r_last)].k0) / BK; ++r_last)
            left -= (p.r[ph(r_last)].k1 - p.r[ph(r_last)].k0) / BK;
    }
    const int r_first = lr, k_first = p.r[ph(lr)].k0 + skip * BK;
    int lk = k_first, lk1 = p.r[ph(lr)].k1;
    const uint8_t* la = (MIX ? false : DUAL ? second : p.r[ph(lr)].a_sel == 1) ? A2b : Ab;
    [[maybe_unused]] const int k_plain = MIX && p.nr > 2 ? p.r[2].k0 : 0;
    if (KT && lk + BK > lk1) back = past_k ? s_lc * 16 : 0;
    auto advance_load = [&]() {
        lk += BK;
        if constexpr (KT) {
            if (lk + BK > lk1) back = past_k ? s_lc * 16 : 0;
            return;
        }
        if constexpr (MIX) {  // (past the last step nothing more is loaded)
            if (lk >= lk1) {
                lk = k_plain;
                lk1 = 0x7fffffff;
            }
            return;
        }
        if (lk >= lk1) {
            ++lr;
            const int rr = min(lr, p.nr - 1);  // past the last range nothing more is loaded
            lk = p.r[ph(rr)].k0;
            lk1 = (lr < p.nr) ? p.r[ph(rr)].k1 : 0x7fffffff;
            la = (p.r[ph(rr)].a_sel == 1) ? A2b : Ab;
        }
    };

    // The epilogue's vectors (1/sx per row, 1/sw and bias per column of this tile)
    // are fetched first of all, so that the wait for the first DMA covers them, and
    // parked in LDS behind the stages: the epilogue then starts without a round
    // trip to memory, and without the ~70 small loads per wave it would take there.
    // (DUAL: [1/sx | 1/sw | bias] of the first range, as the epilogue reads them, then [1/sx | 1/sw] of the second, MIX: and of
    // the third, zeros where this workgroup has no step of it)
    constexpr int EPI_FLOATS = MIX ? 3 * OM + 4 * BN : DUAL ? 2 * OM + 3 * BN : BM + 2 * BN, EPI_IT = (EPI_FLOATS + NT - 1) / NT;
    float* const epi = reinterpret_cast<float*>(smem + NS * (AR + BN) * BK);
    // group factors: a ring of four rows of BN floats behind the epilogue's vectors.  The row of
    // step s arrives with the step's operands and is read all through step s, at whose end the
    // row of step s + 2 is already on its way
    float* const grw = epi + EPI_FLOATS;
    int lslot = 0, cslot = 0;  // slots of the step being loaded / multiplied
    auto dma_g = [&]() {
        if constexpr (GRP) {
            if (wave < BN / 64) {
                const int n = min(n0 + wave * 64 + lane, p.N - 1);
                __builtin_amdgcn_global_load_lds((glb_ptr_t)(p.grw + (int64_t)(lk >> 7) * p.grw_gs + n),
                                                 (lds_ptr_t)(grw + lslot * BN + wave * 64), 4, 0, 0);
            }
            lslot = (lslot + 1) & 3;
        }
    };
    const int r_epi = ACCF || DUAL ? 0 : ph(r_last);  // the range (as the caller numbers them) whose units the accumulators end up in
    float epi_val[EPI_IT];
    const bool want_epi = p.out_dtype != SEGQ_ACC;  // raw accumulators come with no scales at all (null pointers)
#pragma unroll
    for (int i = 0; i < EPI_IT; ++i) {
        const int e = i * NT + tid;
        float v = 0.0f;
        if (!want_epi) {
        } else if (e < OM) {
            if constexpr (!ACCF) v = (p.r[r_epi].sx + z * p.bsSx)[(int64_t)min(m0 + e, p.M - 1) * p.r[r_epi].sx_rs];
        } else if (e < OM + BN) {
            if constexpr (!ACCF) v = (p.r[r_epi].sw + z * p.bsSw)[(int64_t)min(n0 + e - OM, p.N - 1) * p.r[r_epi].sw_cs];
        } else if (e < OM + 2 * BN) {
            if (p.bias) v = load_bias(p.bias, p.bias_dtype, min(n0 + e - OM - BN, p.N - 1));
        } else if (DUAL && e < 2 * OM + 2 * BN) {
            v = (p.r[1].sx + z * p.bsSx)[(int64_t)min(m0 + e - OM - 2 * BN, p.M - 1) * p.r[1].sx_rs];
        } else if (DUAL && e < 2 * OM + 3 * BN) {
            v = (p.r[1].sw + z * p.bsSw)[(int64_t)min(n0 + e - 2 * OM - 2 * BN, p.N - 1) * p.r[1].sw_cs];
        } else if (MIX && steps == n_dual) {
            v = __builtin_inff();
        } else if (MIX && e < 3 * OM + 3 * BN) {
            v = p.r[2].sx[(int64_t)min(m0 + e - 2 * OM - 3 * BN, p.M - 1) * p.r[2].sx_rs];
        } else if (MIX && e < EPI_FLOATS) {
            v = p.r[2].sw[(int64_t)min(n0 + e - 3 * OM - 3 * BN, p.N - 1) * p.r[2].sw_cs];
        }
        epi_val[i] = v;
    }

    // prologue: tiles 0 .. NS-1 on their way into buffers 0 .. NS-1; wait for tile 0
    int issued = 0;
#pragma unroll
    for (int t = 0; t < NS; ++t) {
        if (t < steps) {
            if (MIX && !MERGE && t >= n_dual) dma(la + lk, Bb + lk, t, std::true_type{});
            else dma(la + lk, Bb + lk, t, std::false_type{});
            dma_g();
            advance_load();
            ++issued;
        }
    }
    if (issued == NS && !GRP && !(MIX && !MERGE && n_dual < NS)) wait_dma(std::integral_constant<int, NS - 1>{});
    else wait_dma(std::integral_constant<int, 0>{});  // (with group factors and in plain steps the waves' DMA counts differ)
#pragma unroll
    for (int i = 0; i < EPI_IT; ++i) {
        const int e = i * NT + tid;
        if constexpr (KT || MIX) {  // (quotients, as exact as the general kernel's, which such launches had)
            if (e < EPI_FLOATS) epi[e] = (e < OM + BN || e >= OM + 2 * BN) ? 1.0f / epi_val[i] : epi_val[i];
        } else {
            if (e < EPI_FLOATS) epi[e] = (e < BM + BN && !ACCF) ? __builtin_amdgcn_rcpf(epi_val[i]) : epi_val[i];
        }
    }
    __syncthreads();
    if constexpr (KT) {
        if (steps == 1) clear_tail(0);
    }
    if constexpr (S8) {
#pragma unroll
        for (int i = MERGE ? TM / 2 : 0; i <= TM; ++i) frag8(0, i);  // activations and the first weight fragment
    } else {
        frags(0, 0);
        if (MERGE && n_dual > 0) {
#pragma unroll
            for (int d = 0; d < TM / 2 * 4; ++d) part1(0, d);
        }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the loop head must see them as landed on every path

    // One K step.  Fragment reads and DMA instructions are spread between the
    // MFMAs: a wave issues in order, and an LDS or DMA instruction that has to
    // queue holds up the MFMAs behind it, so a burst of them drains the matrix
    // pipe of the whole SIMD (both its waves are in the same phase).  Issued one
    // at a time they never queue.  DMA_ and MORE_ are compile-time so that the
    // steady-state loop body has no branches.
    int cr = r_first, ck = k_first, ck1 = p.r[ph(r_first)].k1;  // the tile being multiplied
    bool dirty = false;  // sums not yet folded into the second set (a split can end inside a range)
    int buf = 0;                                   // its buffer, s % NS
    constexpr int NDM = A_IT + B_IT;
    // Group factors: int32 sums of a column block and, in LAG order, of the one before it, whose factors are gf
    static_assert(!GRP || TN % 2 == 0, "group factors: two sets of temporaries in turn, also from one step to the next");
    constexpr bool LAG = GRP && !FOLD;
    v4i gt[2][GRP ? TM : 1];
    v4f gf = v4f{0.f, 0.f, 0.f, 0.f};
    if constexpr (GRP) {
#pragma unroll
        for (int b = 0; b < TM; ++b) gt[1][b] = acc_zero;
    }
    auto convert = [&](int a, int j) __attribute__((always_inline)) {  // piece j of 2 TM
        if constexpr (GRP) {
            const int b = j >> 1;
#pragma unroll
            for (int v = 2 * (j & 1); v < 2 * (j & 1) + 2; ++v) {
                float t = __builtin_fmaf((float)gt[a & 1][b][v], gf[v], accf[a][b][v]);
                if constexpr (LAG) asm volatile("" : "+v"(t));  // (keeps the conversion where it is written)
                accf[a][b][v] = t;
            }
        }
    };
    auto convert_block = [&](int a) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2 * TM; ++j) convert(a, j);
    };
    // Low-rank branch, one range: the first 32 columns of the tile's rows of T and L2T go into the stage that the last step but
    // one is done with, and land under that step; they are read behind the last one.
    // us, loaded there / this, int8: 4608 x 12288 x 3072 on 384 x 192 156 / 152, 4608 x 9216 122 / 120.5, 2304 x 12288 83 / 81,
    // 300 x 3072 x 1536 12.0 / 11.4.
    constexpr bool LRP = FINISH && !FOLD && !GRP && NS == 2;
    auto fetch_lr = [&](int buf) __attribute__((always_inline)) {
        if constexpr (LRP) {
            if (p.lr_rank > 0) {
                const int r4 = lane >> 2, c = (lane & 3) * 8;  // four 16-byte pieces a row
#pragma unroll
                for (int i = 0; i < (BM + 127) / 128; ++i) {
                    const int row = wave * 16 + i * 128;
                    if (row < BM) load16_to_lds(reinterpret_cast<const uint8_t*>(p.lr_t + (int64_t)min(m0 + row + r4, p.M - 1) * p.lr_ldt + c), As + buf * AR * BK + row * 64);
                }
#pragma unroll
                for (int i = 0; i < (BN + 127) / 128; ++i) {
                    const int row = wave * 16 + i * 128;
                    if (row < BN) load16_to_lds(reinterpret_cast<const uint8_t*>(p.lr_l2 + (int64_t)min(n0 + row + r4, p.N - 1) * p.lr_ldl + c), Bs + buf * BN * BK + row * 64);
                }
            }
        }
    };
    // e4m3 schedule of one step.  On entry the activation fragments and weight
    // fragment 0 are in registers.  Column block a reads weight fragment a + 2
    // (block 0 also fragment 1), so after block TN - 3 every read of this step is
    // issued; there the step has its barrier.  The last two blocks refill the
    // registers this step is done with: next weight fragment 0, then each
    // activation fragment right behind the last MFMA that reads it, with the DMA
    // of step s + 2 spread over the same MFMAs.
    // plain_c, dplain_c (MIX): this step, the one that it loads, is of the plain range: the second half of the row blocks only
    [[maybe_unused]] bool tail_left = false, next_dual = false;  // three stages: there is a step behind the next one; that one is of the pair
    auto step8 = [&](auto dma_c, auto more_c, auto plain_c, auto dplain_c) __attribute__((always_inline)) {
        constexpr bool DMA_ = decltype(dma_c)::value;
        constexpr bool MORE_ = decltype(more_c)::value;
        constexpr int B0 = decltype(plain_c)::value ? TM / 2 : 0;      // the first row block
        constexpr int NDM8 = A_IT + B_IT, TAIL = 2 * (TM - B0);  // DMA instructions over the tail's MFMAs
        // row blocks in the order of their MFMAs: MERGE has the negative codes' in front, so that the blocks that are read
        // for the next step, theirs, are free half a column block earlier
        auto nth = [](int j) __attribute__((always_inline)) { return MERGE && B0 == 0 ? (j + TM / 2) % TM : j; };
        constexpr int H = MERGE && B0 == 0 ? TM / 2 : 0;  // fragments to be parted, in column block 0
        const int nbuf = NS == 2 ? buf ^ 1 : buf + 1 == NS ? 0 : buf + 1;
        auto lo4 = [](const v8i& f) __attribute__((always_inline)) { return v4i{f[0], f[1], f[2], f[3]}; };
        auto hi4 = [](const v8i& f) __attribute__((always_inline)) { return v4i{f[4], f[5], f[6], f[7]}; };
        const float* const gsrc = grw + cslot * BN + wn * WN + 4 * lgrp;
#pragma unroll
        for (int a = 0; a < TN - 2; ++a) {
            if constexpr (GRP) {
                v4f g;
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    if (b == 0 && a == 0) frag8(buf, TM + 1);
                    if (b == (TM > 1 ? 1 : 0)) frag8(buf, TM + a + 2);
                    gt[a & 1][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo4(fb8[a]), lo4(fa8[b]), acc_zero, 0, 0, 0);
                    if constexpr (LAG) convert((a + TN - 1) % TN, b);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    gt[a & 1][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi4(fb8[a]), hi4(fa8[b]), gt[a & 1][b], 0, 0, 0);
                    if constexpr (LAG) convert((a + TN - 1) % TN, TM + b);
                    if (b == 0) g = *reinterpret_cast<const v4f*>(gsrc + a * 16);
                    __builtin_amdgcn_sched_barrier(0);
                }
                gf = g;
                if constexpr (!LAG) convert_block(a);
            } else if constexpr (WS) {
                // int8: the two 64-byte K halves of a block, TM MFMAs apart
#pragma unroll
                for (int j = B0; j < TM; ++j) {
                    const int b = nth(j);
                    if (j == B0 && a == 0) frag8(buf, TM + 1);
                    if (j == (TM > 1 ? B0 + 1 : 0)) frag8(buf, TM + a + 2);
                    if (a == 0 && H > 0) {  // low halves in front of their MFMAs, high ones among the positive codes'
                        if (j == 0) part(0, 0, 4);
                        if (j + 1 < H) part(j + 1, 0, 4);
                        else if (j + 1 > H) part(j - H, 4, 8);
                    }
                    if constexpr (!F8) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo4(fb8[a]), lo4(fa8[b]), acc[a][b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int j = B0; j < TM; ++j) {
                    const int b = nth(j);
                    if constexpr (!F8) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi4(fb8[a]), hi4(fa8[b]), acc[a][b], 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int j = B0; j < TM; ++j) {
                    const int b = nth(j);
                    if (j == B0 && a == 0) frag8(buf, TM + 1);
                    if (j == (TM > 1 ? B0 + 1 : 0)) frag8(buf, TM + a + 2);
                    if (a == 0 && H > 0) {
                        if (j == 0) part(0, 0, 8);
                        if (j + 1 < H) part(j + 1, 0, 8);
                    }
                    if constexpr (F8)
                        acc[a][b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb8[a], fa8[b], acc[a][b], 0, 0, 0, 0, 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (NS > 2 && (!decltype(dplain_c)::value || tail_left)) wait_dma(std::integral_constant<int, NS - 2>{});
        else wait_dma(std::integral_constant<int, 0>{});
        __syncthreads();
        if constexpr (KT && MORE_ && !DMA_) clear_tail(nbuf);  // (two stages: the next step is the last)
        if constexpr (LRP && MORE_ && !DMA_) fetch_lr(buf);
        const uint8_t* const ap = la + lk;
        const uint8_t* const bp = Bb + lk;
#pragma unroll
        for (int a = TN - 2; a < TN; ++a) {
            if constexpr (GRP) {
                v4f g;
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    gt[a & 1][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo4(fb8[a]), lo4(fa8[b]), acc_zero, 0, 0, 0);
                    if (LAG && !(a == TN - 1 && MORE_)) convert(a - 1, b);
                    if (b == TM - 1) g = *reinterpret_cast<const v4f*>(gsrc + a * 16);
                    const int j = (a - (TN - 2)) * TM + b;
                    if constexpr (DMA_) {
#pragma unroll
                        for (int i = j * NDM8 / TAIL; i < (j + 1) * NDM8 / TAIL; ++i) dma1(ap, bp, buf, i, dplain_c);
                        if (j == TAIL - 1) dma_g();
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int b = 0; b < TM; ++b) {
                    gt[a & 1][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi4(fb8[a]), hi4(fa8[b]), gt[a & 1][b], 0, 0, 0);
                    if (LAG && !(a == TN - 1 && MORE_)) convert(a - 1, TM + b);
                    if constexpr (MORE_) {
                        if (a == TN - 2 && b == 0) frag8(nbuf, TM);  // next weight fragment 0: free since block 0
                        if (a == TN - 1) frag8(nbuf, b);              // next activation fragment b: this was its last reader
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (LAG && a == TN - 1 && MORE_) {  // under the next step's first fragment reads
                    convert_block(a - 1);
                    __builtin_amdgcn_sched_barrier(0);
                }
                gf = g;
                if constexpr (!LAG) convert_block(a);
            } else if constexpr (WS) {
#pragma unroll
                for (int l = B0; l < TM; ++l) {
                    const int b = nth(l);
                    if constexpr (!F8) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(lo4(fb8[a]), lo4(fa8[b]), acc[a][b], 0, 0, 0);
                    const int j = (a - (TN - 2)) * (TM - B0) + l - B0;
                    if constexpr (DMA_) {
#pragma unroll
                        for (int i = j * NDM8 / TAIL; i < (j + 1) * NDM8 / TAIL; ++i) dma1(ap, bp, buf, i, dplain_c);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
#pragma unroll
                for (int l = B0; l < TM; ++l) {
                    const int b = nth(l);
                    if constexpr (!F8) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(hi4(fb8[a]), hi4(fa8[b]), acc[a][b], 0, 0, 0);
                    if constexpr (MORE_) {
                        if (a == TN - 2 && l == B0) frag8(nbuf, TM);  // next weight fragment 0: free since block 0
                        if (a == TN - 1 && (!MERGE || b >= TM / 2)) frag8(nbuf, b);              // next activation fragment b: this was its last reader
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int l = B0; l < TM; ++l) {
                    const int b = nth(l);
                    if constexpr (F8)
                        acc[a][b] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb8[a], fa8[b], acc[a][b], 0, 0, 0, 0, 0, 0);
                    const int j = (a - (TN - 2)) * (TM - B0) + l - B0;
                    if constexpr (DMA_) {
#pragma unroll
                        for (int i = j * NDM8 / TAIL; i < (j + 1) * NDM8 / TAIL; ++i) dma1(ap, bp, buf, i, dplain_c);
                    }
                    if constexpr (MORE_) {
                        if (a == TN - 2 && l == B0) frag8(nbuf, TM);  // next weight fragment 0: its registers were free since block 0
                        if (a == TN - 1 && (!MERGE || b >= TM / 2)) frag8(nbuf, b);              // next activation fragment b: this was its last reader
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        // A full LDS wait: the last activation fragments were read a few MFMAs ago
        // and this exposes part of their latency, but with reads still in flight
        // over the loop's back edge the compiler puts the same wait in front of the
        // next step's second MFMA, behind that step's first reads.
        __builtin_amdgcn_s_waitcnt(0xC07F);
        if constexpr (DMA_) advance_load();
        ck += BK;
        cslot = (cslot + 1) & 3;
        dirty = true;
        if (!KT && !MIX && ck >= ck1) {
            if constexpr (FOLD) fold(cr);
            dirty = false;
            ++cr;
            const int rr = min(cr, p.nr - 1);
            ck = p.r[ph(rr)].k0;
            ck1 = p.r[ph(rr)].k1;
        }
        buf = nbuf;
    };
    // Measurement hooks (off in the library that ships: `make variant`, see the Makefile): the int8 K loop
    // with its MFMAs, its fragment reads or its DMA compiled out, barriers and waits in place.  The
    // results are wrong; the durations say what each of the three costs alone and in pairs.
#ifdef SEGQ_ABLATE_MFMA
    constexpr bool abl_mfma = true;
#else
    constexpr bool abl_mfma = false;
#endif
#ifdef SEGQ_ABLATE_LDS
    constexpr bool abl_lds = true;
#else
    constexpr bool abl_lds = false;
#endif
#ifdef SEGQ_ABLATE_DMA
    constexpr bool abl_dma = true;
#else
    constexpr bool abl_dma = false;
#endif
    // (plain_c, dplain_c: as in step8)
    auto step_i8 = [&](auto dma_c, auto more_c, auto plain_c, auto dplain_c) __attribute__((always_inline)) {
        constexpr bool DMA_ = decltype(dma_c)::value;
        constexpr bool MORE_ = decltype(more_c)::value;
        constexpr int B0 = decltype(plain_c)::value ? TM / 2 : 0;           // the first row block
        constexpr int R0 = MERGE || decltype(plain_c)::value ? TM / 2 : 0;  // the first fragment that is read
        constexpr int H = MERGE && B0 == 0 ? TM / 2 : 0;                    // fragments to be parted
        constexpr int NM = (TM - B0) * TN, NR = TM + TN - R0;
        constexpr int RDE = (NM >= 2 * NR + 4) ? 2 : 1;
        constexpr int DME = (NM / NDM > 1) ? NM / NDM : 1;
        static_assert(S8 || (NR * RDE <= NM && NDM * DME <= NM), "more reads than MFMA slots");
        constexpr int P0 = NM - 4 * H;                                      // a dword per MFMA, the last of either half, behind its read
        const int nbuf = (buf + 1 == NS) ? 0 : buf + 1;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = B0; b < TM; ++b) {
                const int i = a * (TM - B0) + b - B0;
                if (i % RDE == 0 && i / RDE < NR && !abl_lds) frag1(buf, 1, R0 + i / RDE);
                if (H > 0 && i >= P0) part1(1, i - P0);
                if constexpr (!abl_mfma) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[0][a], fa[0][b], acc[a][b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        // Tile s+1 must have landed (the NS-2 tiles issued after it may still be in
        // flight) and this wave's reads of tile s must be done, before anyone reads
        // tile s+1 or overwrites the buffer of tile s.
        if (MIX && NS > 2 && decltype(dplain_c)::value && !tail_left) wait_dma(std::integral_constant<int, 0>{});
        else wait_dma(std::integral_constant<int, DMA_ ? NS - 2 : 0>{});
        __syncthreads();
        if constexpr (KT && MORE_ && !DMA_) clear_tail(nbuf);  // (two stages: the next step is the last)
        if constexpr (LRP && MORE_ && !DMA_) fetch_lr(buf);
        // tile s+NS goes where tile s was: both its halves are in registers
        const uint8_t* const ap = la + lk;
        const uint8_t* const bp = Bb + lk;
#pragma unroll
        for (int a = 0; a < TN; ++a)
#pragma unroll
            for (int b = B0; b < TM; ++b) {
                const int i = a * (TM - B0) + b - B0;
                if constexpr (DMA_) {
                    if (i % DME == DME - 1 && i / DME < NDM && !abl_dma) dma1(ap, bp, buf, i / DME, dplain_c);
                }
                if constexpr (MORE_) {
                    if (i % RDE == 0 && i / RDE < NR && !abl_lds) frag1(nbuf, 0, R0 + i / RDE);
                }
                if (H > 0 && i >= P0) {  // (of the next step, if that is one of the pair)
                    if (!decltype(dplain_c)::value || next_dual) part1(0, i - P0);
                }
                if constexpr (!abl_mfma) acc[a][b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fb[1][a], fa[1][b], acc[a][b], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        // The reads of the next tile's first half have had most of an MFMA group to
        // land.  Waiting for them here, explicitly, keeps the compiler from putting
        // a full LDS wait in front of the first MFMA at the loop head (it cannot
        // count reads across the back edge).
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0), vmcnt untouched
        if constexpr (DMA_) advance_load();
        ck += BK;
        dirty = true;
        if (!KT && !MIX && ck >= ck1) {  // the range is complete: fold it, move to the next one
            if constexpr (PARK) park(cr);
            else if constexpr (FOLD) fold(cr);
            dirty = false;
            ++cr;
            const int rr = min(cr, p.nr - 1);
            ck = p.r[ph(rr)].k0;
            ck1 = p.r[ph(rr)].k1;
        }
        buf = nbuf;
    };
    auto step = [&](auto dma_c, auto more_c) __attribute__((always_inline)) {
        if constexpr (S8) step8(dma_c, more_c, std::false_type{}, std::false_type{});
        else step_i8(dma_c, more_c, std::false_type{}, std::false_type{});
    };
    int s = 0;
    if constexpr (MIX) {
        constexpr std::true_type yes{};
        constexpr std::false_type no{};
        auto mstep = [&](auto plain_c, auto dplain_c) __attribute__((always_inline)) {
            if constexpr (S8) step8(yes, yes, plain_c, dplain_c);
            else step_i8(yes, yes, plain_c, dplain_c);
        };
        const int alike = MERGE ? min(n_dual - (S8 ? 0 : 1), steps - NS) : n_dual - NS;  // (plain steps are loaded like MERGE's others)
        for (; s < alike; ++s) mstep(no, no);
        // from here on a step loads a plain one or, behind the last, none (what it reads of that goes nowhere)
        for (; s < n_dual; ++s) {
            if (s + NS >= steps) wanted = 0;
            tail_left = s + 2 < steps;
            next_dual = s + 1 < n_dual;
            mstep(no, yes);
        }
        if (n_dual > 0) {  // the sums of both signs -> one, in output units
            const float* const rx2 = epi + OM + 2 * BN;
#pragma unroll
            for (int a = 0; a < TN; ++a) {
                const int n = wn * WN + a * 16 + 4 * lgrp;
                const v4f w = *reinterpret_cast<const v4f*>(epi + OM + n), w2 = *reinterpret_cast<const v4f*>(rx2 + OM + n);
#pragma unroll
                for (int b = 0; b < TM / 2; ++b) {
                    const int m = wm * (WM / 2) + b * 16 + lrow;
                    acc[a][b] = __builtin_bit_cast(acc_t, __builtin_convertvector(acc[a][b], v4f) * epi[m] * w +
                                                              __builtin_convertvector(acc[a][b + TM / 2], v4f) * rx2[m] * w2);
                    acc[a][b + TM / 2] = acc_zero;
                }
            }
        }
        for (; s < steps; ++s) {
            if (s + NS >= steps) wanted = 0;
            tail_left = s + 2 < steps;
            mstep(yes, yes);
        }
    }
    for (; s + NS < steps; ++s) step(std::true_type{}, std::true_type{});
    for (; s + 1 < steps; ++s) step(std::false_type{}, std::true_type{});
    if (s < steps) step(std::false_type{}, std::false_type{});
    if constexpr (LAG) convert_block(TN - 1);
    if constexpr (ACCF) {
        if (dirty) fold(cr);
    }
    if constexpr (FINISH) {
        // FINISH instances serve the launches that finish in output units (the others do not pay for
        // the registers of it): parked ranges, the low-rank branch and a tile split in two along K.  The sums are
        // scaled first (1 / (sx sw) of the range they are in units of, from the vectors parked in LDS) and what is
        // parked is added; then
        //  * a tile split in two along K: the two workgroups meet in the workspace (below);
        //  * low-rank branch (out += T L2): the product joins in fp32 on the matrix cores;
        // and the epilogue only adds the bias and the addend and rounds once.
        constexpr bool MEET = BM % 128 == 0 ? BN != 192 || BM == 256 : BN == 256;  // (tail_tile() of the dispatch: no K shares on the largest)
        v4f of[TN][TM];
        [[maybe_unused]] const bool parked = r_begin < r_last;
        // blocks whose loads are in flight at once (registers: the sums are still live).  What is parked comes back in two
        // halves: 256 x 256 tiles 600 x 15360 x 3072 143 -> 135 us a pass, 2100 274 -> 260, 9216 (288 x 192) 843 -> 834
        // against an instance without the finish; 351 rows in ten shares 75 -> 78
        constexpr int CH = PARK ? (TN * TM + 1) / 2 : 8;
#pragma unroll
        for (int c0 = 0; c0 < TN * TM; c0 += CH) {
            [[maybe_unused]] v4f old[CH];
            if constexpr (PARK) {
#pragma unroll
                for (int i = 0; i < CH; ++i)
                    if (c0 + i < TN * TM) old[i] = parked ? slot[(c0 + i) * NT] : v4f{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int i = 0; i < CH; ++i) {
                if (c0 + i < TN * TM) {
                    const int a = (c0 + i) / TM, b = (c0 + i) % TM;
                    v4f t;
                    if constexpr (HASF) t = accf[a][b];
                    else t = __builtin_convertvector(acc[a][b], v4f);
                    if constexpr (!ACCF) {
                        const v4f rw = *reinterpret_cast<const v4f*>(epi + BM + wn * WN + a * 16 + 4 * lgrp);
                        const float rx = epi[wm * WM + b * 16 + lrow];
                        if constexpr (PARK) t = t * rx * rw + old[i];
                        else t = t * (rw * rx);
                    }
                    of[a][b] = t;
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (MEET) {
            if (p.part && !meet_share<NT, CH>(p, of, tile_id, zy, tid, reinterpret_cast<int*>(epi))) return;
        }
        if (p.lr_rank > 0) {
            if constexpr (LRP) {
                const int lb = steps & 1;  // the stage of the last step but one
                lowrank_accumulate<true>(p, of, m0 + wm * WM, n0 + wn * WN, lane, steps > 1, As + lb * AR * BK + wm * WM * 64, Bs + lb * BN * BK + wn * WN * 64);
            } else {
                lowrank_accumulate<false>(p, of, m0 + wm * WM, n0 + wn * WN, lane);
            }
        }
        wide_epilogue<BM, BN, WGM, WGN, GEMM_F8, false, true>(p, of, of, smem, z, m0, n0, wave, lane, r_epi, epi);
        return;
    }
    if constexpr (MIX) {
        v4f of[TN][TM / 2];
        const float* const rx3 = epi + 2 * OM + 3 * BN;
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            const v4f w3 = *reinterpret_cast<const v4f*>(rx3 + OM + wn * WN + a * 16 + 4 * lgrp);
#pragma unroll
            for (int b = 0; b < TM / 2; ++b)
                of[a][b] = __builtin_bit_cast(v4f, acc[a][b]) +
                           __builtin_convertvector(acc[a][b + TM / 2], v4f) * rx3[wm * (WM / 2) + b * 16 + lrow] * w3;
        }
        if (p.part && !meet_share<NT, 8>(p, of, tile_id, zy, tid, reinterpret_cast<int*>(epi))) return;
        wide_epilogue<OM, BN, WGM, WGN, GEMM_F8, false, true>(p, of, of, smem, z, m0, n0, wave, lane, 0, epi);
    } else if constexpr (DUAL) {
        v4f of[TN][TM / 2];
        const float* const rx2 = epi + OM + 2 * BN;
#pragma unroll
        for (int a = 0; a < TN; ++a) {
            const int n = wn * WN + a * 16 + 4 * lgrp;
            const v4f w = *reinterpret_cast<const v4f*>(epi + OM + n), w2 = *reinterpret_cast<const v4f*>(rx2 + OM + n);
#pragma unroll
            for (int b = 0; b < TM / 2; ++b) {
                const int m = wm * (WM / 2) + b * 16 + lrow;
                of[a][b] = __builtin_convertvector(acc[a][b], v4f) * epi[m] * w + __builtin_convertvector(acc[a][b + TM / 2], v4f) * rx2[m] * w2;
            }
        }
        wide_epilogue<OM, BN, WGM, WGN, GEMM_F8, false, true>(p, of, of, smem, z, m0, n0, wave, lane, 0, epi);
    } else if constexpr (GRP) {
        v4f none[1][1];
        wide_epilogue<BM, BN, WGM, WGN, GEMM_F8, false, false>(p, accf, none, smem, z, m0, n0, wave, lane, r_epi, epi);
    } else if constexpr (CODES) {
        codes_epilogue<BM, BN, WGM, WGN, FMT>(p, acc, smem, m0, n0, wave, lane, epi);
    } else {
        wide_epilogue<BM, BN, WGM, WGN, FMT, false, ACCF>(p, acc, accf, smem, z, m0, n0, wave, lane, r_epi, epi);
    }
}

template <int BM, int BN, int WGM, int WGN, int FMT, bool B4, bool FOLD, bool ASEL>
int launch_wide_instance(const GemmParams& p, int64_t batch, hipStream_t st) {
    auto kern = gemm_wide_kernel<BM, BN, WGM, WGN, FMT, B4, FOLD, ASEL>;
    constexpr int lds = 2 * (BM + BN) * BK;
    if (p.dry) return SEGQ_OK;
    static unsigned long long attr_done = 0;
    if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds, &attr_done)) return rc;
    dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)batch);
    hipLaunchKernelGGL(kern, grid, dim3(WGM * WGN * 64), lds, st, p);
    return check_launch("segq_gemm");
}

// wide tile ids (after the generic ones): 256x256 | 256x128 | 128x256 | 128x128, eight waves each
template <int BM, int BN, int WGM, int WGN, int FMT, bool FOLD, int NS, bool GRP = false, bool PARK = false, bool FINISH = false,
          bool CODES = false, bool SEP = false, bool KT = false, bool DUAL = false, bool MIX = false,
          bool MERGE = false>
int launch_pipe_instance(const GemmParams& p, int64_t batch, hipStream_t st) {
    auto kern = gemm_pipe_kernel<BM, BN, WGM, WGN, FMT, FOLD, NS, GRP, PARK, FINISH, CODES, SEP, KT, DUAL, MIX, MERGE>;
    // the stages, the epilogue's vectors, and the ring of group factors
    constexpr int lds = NS * ((MERGE ? BM / 2 : BM) + BN) * BK + (MIX ? BM / 2 * 3 + 4 * BN : DUAL ? BM + 3 * BN : BM + 2 * BN) * 4 + (GRP ? 4 * BN * 4 : 0);
    if (p.dry) return SEGQ_OK;
    static unsigned long long attr_done = 0;
    if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds, &attr_done)) return rc;
    dim3 grid((unsigned)(p.tiles_m * p.tiles_n), (unsigned)batch);
    hipLaunchKernelGGL(kern, grid, dim3(WGM * WGN * 64), lds, st, p);
    return check_launch("segq_gemm");
}

// One walk of K with a ragged end: one range, or DualScale's two over the same run.
template <int FMT>
int launch_walk(const GemmParams& p, int cfg, int64_t batch, hipStream_t st) {
    constexpr int WM = FMT == GEMM_F8 ? 4 : 2, WN = FMT == GEMM_F8 ? 2 : 4;  // (e4m3 wants three or more column blocks per wave)
#define SEGQ_WALK(BM_, BN_, WGM_, WGN_, DUAL_) \
    return launch_pipe_instance<BM_, BN_, WGM_, WGN_, FMT, false, 2, false, false, false, false, false, true, DUAL_>(p, batch, st)
    switch (cfg) {
        case FIRST_KT_CFG: SEGQ_WALK(256, 256, 4, 2, false);
        case FIRST_KT_CFG + 1: SEGQ_WALK(256, 192, 4, 2, false);
        case FIRST_KT_CFG + 2: SEGQ_WALK(128, 128, WM, WN, false);
        case FIRST_DUAL_CFG: SEGQ_WALK(256, 192, 4, 2, true);
        case FIRST_DUAL_CFG + 1: SEGQ_WALK(128, 128, WM, WN, true);
    }
#undef SEGQ_WALK
    return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: no kernel for tile %d", cfg + 1);
}

// DualScale's two ranges in whole steps and a plain range or none behind them.  From one tensor of codes of both signs a stage is a
// third smaller, which leaves room for a third one.  us, three stages / two, e4m3: 9216 x 3072 x (3072 + 12288) on 128 x 192 600 / 630,
// 1024 rows in two shares 75 / 77; on 192 x 192, whose wave tiles load less per MFMA, 566 / 561; int8 level.  All three tiles have
// three: what that costs the largest lies within what runs of one card differ by.
template <int FMT>
int launch_mix(const GemmParams& p, int cfg, int64_t batch, hipStream_t st) {
#define SEGQ_MIX(BM_, BN_)                                                                                                                       \
    return p.r[0].a_sel ? launch_pipe_instance<BM_, BN_, 4, 2, FMT, false, 3, false, false, false, false, false, false, true, true, true>(p, batch, st) \
                        : launch_pipe_instance<BM_, BN_, 4, 2, FMT, false, 2, false, false, false, false, false, false, true, true>(p, batch, st)
    switch (cfg) {
        case FIRST_MIX_CFG: SEGQ_MIX(384, 192);
        case FIRST_MIX_CFG + 1: SEGQ_MIX(256, 256);
        case FIRST_MIX_CFG + 2: SEGQ_MIX(256, 192);
        // the three largest tiles of one range with the low-rank branch
        case FIRST_LR_CFG: return launch_pipe_instance<192, 288, 4, 2, FMT, false, 2, false, false, true>(p, batch, st);
        case FIRST_LR_CFG + 1: return launch_pipe_instance<288, 192, 2, 4, FMT, false, 2, false, false, true>(p, batch, st);
        case FIRST_LR_CFG + 2: return launch_pipe_instance<384, 192, 4, 2, FMT, false, 2, false, false, true>(p, batch, st);
    }
#undef SEGQ_MIX
    return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: no kernel for tile %d", cfg + 1);
}

template <int FMT, bool B4>
int launch_wide(const GemmParams& p, int wcfg, bool fold, bool asel, int64_t batch, hipStream_t st) {
    const bool tail = p.lr_rank > 0 || p.part;  // finishes in output units: the FINISH instances (tail_tile() says which exist)
    if constexpr (!B4 && FMT == GEMM_I8) {
        if (p.grw) {  // group-wise factors (the host has checked: plain codes, K ranges in whole steps)
            if (asel || tail) return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors need plain codes, and serve no low-rank branch");
            switch (wcfg) {
                case 0:
                    if (!fold) return launch_pipe_instance<256, 256, 4, 2, FMT, false, 2, true>(p, batch, st);
                    break;
                case 1:
                    return fold ? launch_pipe_instance<256, 128, 4, 2, FMT, true, 2, true>(p, batch, st)
                                : launch_pipe_instance<256, 128, 4, 2, FMT, false, 2, true>(p, batch, st);
                case 2:
                    return fold ? launch_pipe_instance<128, 256, 2, 4, FMT, true, 2, true>(p, batch, st)
                                : launch_pipe_instance<128, 256, 2, 4, FMT, false, 2, true>(p, batch, st);
                case 3:
                    return fold ? launch_pipe_instance<128, 128, 4, 2, FMT, true, 2, true>(p, batch, st)
                                : launch_pipe_instance<128, 128, 4, 2, FMT, false, 2, true>(p, batch, st);
                case 6:
                    if (!fold) return launch_pipe_instance<256, 192, 4, 2, FMT, false, 2, true>(p, batch, st);
                    break;
                case 7:
                    if (!fold) return launch_pipe_instance<192, 256, 2, 4, FMT, false, 2, true>(p, batch, st);
                    break;
            }
            return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: group factors run on the 256x128, 128x256 and 128x128 tiles of eight waves, and with one range on "
                                              "256x256, 256x192 and 192x256");
        }
    }
// a tile that exists with and without the tail / without only
#define SEGQ_PIPE2(BM_, BN_, WGM_, WGN_, FOLD_, PARK_)                                                               \
    return tail ? launch_pipe_instance<BM_, BN_, WGM_, WGN_, FMT, FOLD_, 2, false, PARK_, true>(p, batch, st)        \
                : launch_pipe_instance<BM_, BN_, WGM_, WGN_, FMT, FOLD_, 2, false, PARK_, false>(p, batch, st)
#define SEGQ_PIPE1(BM_, BN_, WGM_, WGN_, FOLD_, PARK_)                                                               \
    if (tail) break;                                                                                                 \
    return launch_pipe_instance<BM_, BN_, WGM_, WGN_, FMT, FOLD_, 2, false, PARK_, false>(p, batch, st)
#define SEGQ_PARK(BM_, BN_, WGM_, WGN_) return launch_pipe_instance<BM_, BN_, WGM_, WGN_, FMT, true, 2, false, true, true>(p, batch, st)
    if (p.oc) {  // the epilogue writes codes: instances of their own, so that the others carry no trace of it
        if constexpr (!B4) {
            if (!asel && !fold && !tail && !p.park) {
                switch (wcfg) {
                    case 0: return launch_pipe_instance<256, 256, 4, 2, FMT, false, 2, false, false, false, true>(p, batch, st);
                    case 3: return launch_pipe_instance<128, 128, (FMT == GEMM_F8 ? 4 : 2), (FMT == GEMM_F8 ? 2 : 4), FMT, false, 2, false, false, false, true>(p, batch, st);
                }
            }
        }
        return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: out_codes runs on tiles %d and %d with plain 8-bit codes on both sides and one range",
                    FIRST_WIDE_CFG + 1, FIRST_WIDE_CFG + 4);
    }
    if constexpr (!B4) {
        constexpr bool F8W = FMT == GEMM_F8;  // the e4m3 schedule wants three or more column blocks per wave
        if (!asel) {  // plain 8-bit operands, both straight to LDS: the software-pipelined kernel
            if (!fold) {
                switch (wcfg) {
                    case 0: SEGQ_PIPE2(256, 256, 4, 2, false, false);
                    case 1: SEGQ_PIPE2(256, 128, 4, 2, false, false);
                    case 2: SEGQ_PIPE1(128, 256, 2, 4, false, false);
                    case 3: SEGQ_PIPE2(128, 128, (F8W ? 4 : 2), (F8W ? 2 : 4), false, false);
                    case 4: SEGQ_PIPE1(192, 288, 4, 2, false, false);
                    case 5: SEGQ_PIPE1(288, 192, 2, 4, false, false);
                    case 6: SEGQ_PIPE2(256, 192, 4, 2, false, false);
                    case 7: SEGQ_PIPE2(192, 256, 2, 4, false, false);
                    case 8:  // four LDS stages: three K steps in flight per CU, for shapes that wait on HBM latency
                        if constexpr (!F8W) {
                            if (tail) break;
                            return launch_pipe_instance<128, 128, 2, 4, FMT, false, 4, false, false, false>(p, batch, st);
                        }
                        break;
                    case 9: SEGQ_PIPE1(384, 192, 4, 2, false, false);  // wave tiles of 96 x 96
                    case 10:  // 128 x 96, five LDS stages: few tokens, more workgroups with four K steps in flight each
                        if constexpr (!F8W) {
                            if (tail) break;
                            return launch_pipe_instance<128, 96, 4, 2, FMT, false, 5, false, false, false>(p, batch, st);
                        }
                        break;
                }
            } else if (p.park) {  // int8, several ranges, a workspace to park finished ranges in: every tile
                if constexpr (!F8W) {
                    switch (wcfg) {
                        case 0: SEGQ_PARK(256, 256, 4, 2);
                        case 1: SEGQ_PARK(256, 128, 4, 2);
                        case 2: if (tail) break; SEGQ_PARK(128, 256, 2, 4);
                        case 3: SEGQ_PARK(128, 128, 2, 4);
                        case 4: if (tail) break; SEGQ_PARK(192, 288, 4, 2);
                        case 5: if (tail) break; SEGQ_PARK(288, 192, 2, 4);
                        case 6: SEGQ_PARK(256, 192, 4, 2);
                        case 7: SEGQ_PARK(192, 256, 2, 4);
                    }
                }
            } else if constexpr (F8W) {
                if (p.sep) {  // independent sums without a workspace: a second register set
                    if (!tail) {
                        switch (wcfg) {
                            case 0: case 1: return launch_pipe_instance<256, 128, 4, 2, FMT, true, 2, false, false, false, false, F8W>(p, batch, st);
                            case 2: return launch_pipe_instance<128, 256, 2, 4, FMT, true, 2, false, false, false, false, F8W>(p, batch, st);
                            case 3: return launch_pipe_instance<128, 128, 4, 2, FMT, true, 2, false, false, false, false, F8W>(p, batch, st);
                        }
                    }
                } else {  // fp32 accumulators are rescaled in place: every tile serves several ranges
                    switch (wcfg) {
                        case 0: SEGQ_PIPE2(256, 256, 4, 2, true, false);
                        case 1: SEGQ_PIPE2(256, 128, 4, 2, true, false);
                        case 2: SEGQ_PIPE1(128, 256, 2, 4, true, false);
                        case 3: SEGQ_PIPE2(128, 128, 4, 2, true, false);
                        case 4: SEGQ_PIPE1(192, 288, 4, 2, true, false);
                        case 5: SEGQ_PIPE1(288, 192, 2, 4, true, false);
                        case 6: SEGQ_PIPE2(256, 192, 4, 2, true, false);
                        case 7: SEGQ_PIPE2(192, 256, 2, 4, true, false);
                        case 9: SEGQ_PIPE1(384, 192, 4, 2, true, false);
                    }
                }
            } else {
                switch (wcfg) {
                    case 0: case 1: SEGQ_PIPE2(256, 128, 4, 2, true, false);
                    case 2: SEGQ_PIPE1(128, 256, 2, 4, true, false);
                    case 3: SEGQ_PIPE2(128, 128, (F8W ? 4 : 2), (F8W ? 2 : 4), true, false);
                }
            }
        }
    }
#undef SEGQ_PIPE1
#undef SEGQ_PIPE2
#undef SEGQ_PARK
    if (tail)
        return fail(SEGQ_ERR_UNSUPPORTED, "segq_gemm: tile %d finishes neither a low-rank branch nor a two-way K split", wcfg + FIRST_WIDE_CFG + 1);
#define SEGQ_WIDE(BM_, BN_, WGM_, WGN_, FOLD_)                                                          \
    return asel ? launch_wide_instance<BM_, BN_, WGM_, WGN_, FMT, B4, FOLD_, true>(p, batch, st)       \
                : launch_wide_instance<BM_, BN_, WGM_, WGN_, FMT, B4, FOLD_, false>(p, batch, st)
    if (!fold) {
        switch (wcfg) {
            case 0: SEGQ_WIDE(256, 256, 4, 2, false);
            case 1: SEGQ_WIDE(256, 128, 4, 2, false);
            case 2: SEGQ_WIDE(128, 256, 2, 4, false);
            case 3: SEGQ_WIDE(128, 128, 2, 4, false);
        }
    } else {
        switch (wcfg) {  // a second accumulator set: halve the wave tile
            case 0: case 1: SEGQ_WIDE(256, 128, 4, 2, true);
            case 2: SEGQ_WIDE(128, 256, 2, 4, true);
            case 3: SEGQ_WIDE(128, 128, 2, 4, true);
        }
    }
#undef SEGQ_WIDE
    return fail(SEGQ_ERR_UNSUPPORTED,
                "segq_gemm: tile %d is not built for this launch (its code format, several ranges, a sign selection, a low-rank "
                "branch or a K split); tile 0 lets the library choose",
                FIRST_WIDE_CFG + wcfg + 1);
}

}  // namespace segq
