// DualScale and a plain segment in one walk of K, e4m3 codes.
#include "segq_gemm_wide.h"

namespace segq {
int launch_mix_f8(const GemmParams& p, int cfg, int64_t batch, hipStream_t st) { return launch_mix<GEMM_F8>(p, cfg, batch, st); }
}  // namespace segq
