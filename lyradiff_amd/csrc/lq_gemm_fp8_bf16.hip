// FP8 GEMM kernels with bf16 outputs.
#include "lq_gemm_fp8_run.h"

namespace lq {

int run_fp8_bf16(const GemmParams& p, hipStream_t st) { return run_fp8_as<BF16Tag>(p, st); }

}  // namespace lq
