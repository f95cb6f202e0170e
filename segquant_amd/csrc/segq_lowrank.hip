// T = X L1 for a low-rank branch (the SVD optimiser's x (L1 / s)): many rows, a long contraction, 16 columns or more.
//
// Bound by what a compute unit takes in: 32 rows of 4608 x 3072 are 196 KB and L1 of rank 32, which every workgroup needs whole,
// another 196 KB out of the L2, at 50 to 60 KB/us.  Both go global -> LDS in whole 512-byte pieces of their rows, three or four
// stages of 256 of K in flight (fragments gathered straight from memory, 16 lines an instruction: 26 us at
// 4608 x 3072, rank 32).  The eight waves take the eight 32-wide steps of a stage, one each, and their sums meet in LDS.
#include "segq_common.h"

namespace segq {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));

// RB blocks of 16 rows, NB of 16 columns, NS stages
template <bool BF, int RB, int NB, int NS>
__global__ void __launch_bounds__(512) lowrank_rows_kernel(const uint16_t* x, int64_t ldx, const uint16_t* l1t, int64_t ldl, uint16_t* t, int64_t ldt,
                                                           int m, int k) {
    constexpr int W = 16 * NB, ROWS = 16 * (RB + NB), STAGE = ROWS * 512, LOADS = ROWS / 16;  // (a wave's per stage, two rows each)
    extern __shared__ __align__(16) uint8_t smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lrow = lane & 15, lgrp = lane >> 4;
    const int m0 = blockIdx.x * 16 * RB, n0 = blockIdx.y * W;
    // Rows 0 .. 16 RB - 1 of a stage are x's, the others l1t's.  A row's 16-byte piece p lies at p ^ (row & 7), so that the 16 rows
    // of a fragment read lie in all banks; the LDS side of a load is lane-linear, the global address is permuted.
    const uint8_t* src[LOADS];
    int piece[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
        const int row = (wave * LOADS + i) * 2 + (lane >> 5);
        piece[i] = (lane & 31) ^ (row & 7);
        src[i] = reinterpret_cast<const uint8_t*>(row < 16 * RB ? x + (int64_t)min(m0 + row, m - 1) * ldx : l1t + (int64_t)(n0 + row - 16 * RB) * ldl);
    }
    const int stages = (k + 255) / 256;
    auto fetch = [&](int s) __attribute__((always_inline)) {
        const int left = (k - s * 256) / 8;  // pieces of the row from here on (a multiple of eight)
        uint8_t* const dst = smem + s % NS * STAGE + wave * LOADS * 1024;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            const int p = piece[i] < left ? piece[i] : 0;  // (past the end: loaded, and not multiplied)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src[i] + s * 512 + p * 16),
                                             (__attribute__((address_space(3))) void*)(dst + i * 1024), 16, 0, 0);
        }
    };
    v4f acc[RB][NB];
#pragma unroll
    for (int b = 0; b < RB; ++b)
#pragma unroll
        for (int n = 0; n < NB; ++n) acc[b][n] = v4f{0.f, 0.f, 0.f, 0.f};
    for (int s = 0; s < NS && s < stages; ++s) fetch(s);
    const int off = ((wave * 4 + lgrp) ^ (lrow & 7)) * 16 + lrow * 512;
    constexpr int VM = (NS - 1) * LOADS;
    static_assert(VM < 64, "vmcnt holds 6 bits");
    for (int s = 0; s < stages; ++s) {
        if (s + NS <= stages) __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4 << 14) | 0x0F70);  // all but the NS - 1 stages behind it
        else __builtin_amdgcn_s_waitcnt(0x0F70);
        __syncthreads();
        const uint8_t* const st = smem + s % NS * STAGE + off;
        uint4 a[RB], b[NB];
#pragma unroll
        for (int i = 0; i < RB; ++i) a[i] = *reinterpret_cast<const uint4*>(st + i * 16 * 512);
#pragma unroll
        for (int n = 0; n < NB; ++n) b[n] = *reinterpret_cast<const uint4*>(st + (RB + n) * 16 * 512);
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
        __syncthreads();                     // everyone has read the stage: the next one may take its place
        if (s + NS < stages) fetch(s + NS);
        if (s * 256 + wave * 32 < k) {
#pragma unroll
            for (int i = 0; i < RB; ++i)
#pragma unroll
                for (int n = 0; n < NB; ++n) {
                    if constexpr (BF)
                        acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[i]), __builtin_bit_cast(bf16x8_t, b[n]), acc[i][n], 0, 0, 0);
                    else
                        acc[i][n] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a[i]), __builtin_bit_cast(f16x8_t, b[n]), acc[i][n], 0, 0, 0);
                }
        }
    }
    float* const part = reinterpret_cast<float*>(smem);  // (the last stage has been read, and nothing is on its way)
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int n = 0; n < NB; ++n)
#pragma unroll
            for (int v = 0; v < 4; ++v) part[(wave * 16 * RB + i * 16 + 4 * lgrp + v) * W + n * 16 + lrow] = acc[i][n][v];
    __syncthreads();
    for (int e = threadIdx.x; e < 16 * RB * W; e += 512) {
        float s = 0.0f;
#pragma unroll
        for (int w = 0; w < 8; ++w) s += part[w * 16 * RB * W + e];
        const int row = m0 + e / W;
        if (row < m) t[(int64_t)row * ldt + n0 + e % W] = (uint16_t)((BF ? pack2_bf16(s, 0.0f) : pack2_f16(s, 0.0f)) & 0xffffu);
    }
}

template <bool BF, int RB, int NB, int NS>
static int launch_lowrank(const uint16_t* x, int64_t ldx, const uint16_t* l1t, int64_t ldl, uint16_t* t, int64_t ldt, int m, int k, int r, hipStream_t st) {
    auto kern = lowrank_rows_kernel<BF, RB, NB, NS>;
    constexpr int stages = NS * 16 * (RB + NB) * 512, sums = 8 * 256 * RB * NB * 4, lds = stages > sums ? stages : sums;
    static unsigned long long attr_done = 0;
    if (const int rc = reserve_lds(reinterpret_cast<const void*>(kern), lds, &attr_done)) return rc;
    hipLaunchKernelGGL(kern, dim3((unsigned)((m + 16 * RB - 1) / (16 * RB)), (unsigned)(r / (16 * NB))), dim3(512), lds, st, x, ldx, l1t, ldl, t, ldt, m, k);
    return check_launch("segq_lowrank_rows");
}

// 32 rows a workgroup from where 16 would give a compute unit two workgroups, and L1 twice.
template <bool BF>
static int choose_lowrank(const uint16_t* x, int64_t ldx, const uint16_t* l1t, int64_t ldl, uint16_t* t, int64_t ldt, int m, int k, int r, hipStream_t st) {
    const bool two = m > 16 * device_cus();
    if (r % 64 == 0)
        return two ? launch_lowrank<BF, 2, 4, 3>(x, ldx, l1t, ldl, t, ldt, m, k, r, st) : launch_lowrank<BF, 1, 4, 3>(x, ldx, l1t, ldl, t, ldt, m, k, r, st);
    if (r % 32 == 0)
        return two ? launch_lowrank<BF, 2, 2, 4>(x, ldx, l1t, ldl, t, ldt, m, k, r, st) : launch_lowrank<BF, 1, 2, 4>(x, ldx, l1t, ldl, t, ldt, m, k, r, st);
    return two ? launch_lowrank<BF, 2, 1, 4>(x, ldx, l1t, ldl, t, ldt, m, k, r, st) : launch_lowrank<BF, 1, 1, 4>(x, ldx, l1t, ldl, t, ldt, m, k, r, st);
}

int lowrank_rows_impl(const void* x, int64_t ldx, const void* l1t, int64_t ldl, void* t, int64_t ldt, int64_t m, int64_t k, int64_t r, int32_t dtype,
                      hipStream_t st) {
    if (m < 0 || m > 0x7fffffff / 2 || k <= 0 || k > 0x7fffff00 || k % 64 || r <= 0 || r % 16 || r > 65536)
        return fail(SEGQ_ERR_ARG, "segq_lowrank_rows: m %lld, k %lld (a multiple of 64) or r %lld (a multiple of 16) out of range", (long long)m, (long long)k,
                    (long long)r);
    if (dtype != SEGQ_BF16 && dtype != SEGQ_F16) return fail(SEGQ_ERR_UNSUPPORTED, "segq_lowrank_rows: 16-bit dtypes only");
    if (m == 0) return SEGQ_OK;
    auto aligned = [](const void* q) { return q && reinterpret_cast<uintptr_t>(q) % 16 == 0; };
    if (!aligned(x) || !aligned(l1t) || !t || ldx % 8 || ldl % 8 || ldx < k || ldl < k || ldt < r)
        return fail(SEGQ_ERR_ARG, "segq_lowrank_rows: x and l1t need 16-byte aligned rows of at least k elements, t rows of at least r");
    const uint16_t *xs = static_cast<const uint16_t*>(x), *ls = static_cast<const uint16_t*>(l1t);
    uint16_t* ts = static_cast<uint16_t*>(t);
    return dtype == SEGQ_BF16 ? choose_lowrank<true>(xs, ldx, ls, ldl, ts, ldt, (int)m, (int)k, (int)r, st)
                              : choose_lowrank<false>(xs, ldx, ls, ldl, ts, ldt, (int)m, (int)k, (int)r, st);
}

}  // namespace segq
