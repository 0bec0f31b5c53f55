// Blocked GEMM instances (one translation unit per weight format).
#include "fp4x_gemm.h"

namespace fp4x {
bool launch_gemm_nv4(const GemvLaunch& p, hipStream_t st) { return launch_gemm<FmtNV4>(p, st); }
}  // namespace fp4x
