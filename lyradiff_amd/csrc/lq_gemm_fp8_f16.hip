// FP8 GEMM kernels with fp16 outputs.
#include "lq_gemm_fp8_run.h"

namespace lq {

int run_fp8_f16(const GemmParams& p, hipStream_t st) { return run_fp8_as<F16Tag>(p, st); }

}  // namespace lq
