// FP8 and INT8 GEMMs of few tiles with f16 outputs.
#include "lq_gemm_small.h"

namespace lq {

int run_small_fp8_f16(const GemmParams& p, int form, hipStream_t st) { return run_small_as<K_FP8, F16Tag>(p, form, st); }
int run_small_int8_f16(const GemmParams& p, int form, hipStream_t st) { return run_small_as<K_INT8, F16Tag>(p, form, st); }

}  // namespace lq
