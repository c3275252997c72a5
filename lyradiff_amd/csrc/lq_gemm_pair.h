// Two FP8 GEMMs of one n and k in one launch, for one output type; each type is instantiated in a translation unit of its own
// (lq_gemm_pair_{f16,bf16}.hip).
#pragma once

#include "lq_gemm_core.h"

namespace lq {

template <typename OutTag> static int run_fp8_pair_as(const GemmPair& pair, int form, hipStream_t st) {
    switch (form) {
        case 0: return launch_gemm_pair<K_FP8, OutTag, 256, 256, 64, 2, 4, 3>(pair, st);
        case 2: return launch_gemm_pair<K_FP8, OutTag, 128, 128, 64, 2, 2, 3>(pair, st);
        case 3: return launch_gemm_pair<K_FP8, OutTag, 64, 64, 64, 2, 2, 3>(pair, st);
        case 4: return launch_gemm_pair<K_FP8, OutTag, 128, 256, 64, 2, 2, 3>(pair, st);
        case 6: return launch_gemm_pair<K_FP8, OutTag, 256, 256, 64, 2, 2, 4>(pair, st);
        case SMALL_32x32_K4: return launch_gemm_pair<K_FP8, OutTag, 32, 32, 64, 1, 1, 3, 4>(pair, st);
        case SMALL_32x64_K4: return launch_gemm_pair<K_FP8, OutTag, 32, 64, 64, 1, 2, 3, 4>(pair, st);
        case SMALL_64x128_K2: return launch_gemm_pair<K_FP8, OutTag, 64, 128, 64, 1, 2, 4, 2>(pair, st);
        case SMALL_128x128: return launch_gemm_pair<K_FP8, OutTag, 128, 128, 128, 2, 4, 4>(pair, st);
        case SMALL_192x128: return launch_gemm_pair<K_FP8, OutTag, 192, 128, 128, 2, 4, 3>(pair, st);
        default: set_error("gemm: unknown form %d for a pair", form); return LQ_ERR_ARG;
    }
}

}  // namespace lq
