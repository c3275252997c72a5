// Two FP8 GEMMs in one launch with bf16 outputs.
#include "lq_gemm_pair.h"

namespace lq {

int run_fp8_pair_bf16(const GemmPair& pair, int form, hipStream_t st) { return run_fp8_pair_as<BF16Tag>(pair, form, st); }

}  // namespace lq
