// Blocked GEMM instances (one translation unit per weight format).
#include "fp4x_gemm.h"

namespace fp4x {
bool launch_gemm_w8_f32(const GemvLaunch& p, hipStream_t st) { return launch_gemm<FmtW8<false>>(p, st); }
bool launch_gemm_w8_f16(const GemvLaunch& p, hipStream_t st) { return launch_gemm<FmtW8<true>>(p, st); }
}  // namespace fp4x
