// DualScale and a plain segment in one walk of K, int8 codes.
#include "segq_gemm_wide.h"

namespace segq {
int launch_mix_i8(const GemmParams& p, int cfg, int64_t batch, hipStream_t st) { return launch_mix<GEMM_I8>(p, cfg, batch, st); }
}  // namespace segq
