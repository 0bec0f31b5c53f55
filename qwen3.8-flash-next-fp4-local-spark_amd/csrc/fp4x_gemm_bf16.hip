// Blocked GEMM instances (one translation unit per weight format).
#include "fp4x_gemm.h"

namespace fp4x {
bool launch_gemm_bf16(const GemvLaunch& p, hipStream_t st) { return launch_gemm<FmtBF16>(p, st); }
bool gemm_few_rows(const GemvLaunch& p) { return gemm_before_rows(p); }
}  // namespace fp4x
