// Blocked GEMM instances (one translation unit per weight format).
#include "fp4x_gemm.h"

namespace fp4x {
bool launch_gemm_bf16(const GemvLaunch& p, hipStream_t st) { return launch_gemm<FmtBF16>(p, st); }
bool gemm_few_rows(const GemvLaunch& p, int fmt) { return gemm_before_rows(p, fmt); }
bool gemm_few_tiles(const GemvLaunch& p) { return gemm_small(p); }
}  // namespace fp4x
