// 8-bit GEMMs whose tiles leave most of the chip idle: the forms of GemmKernel whose wavefront groups share k out.
//
// What bounds them: a workgroup alone on a CU takes 0.17 us (64x64) to 0.3 us (128x256) per 64-byte k-tile whatever it computes --
// the barrier, the LDS round trip of the fragments and the matrix instructions follow each other -- and walks k by itself.  With
// k shared between two or four groups of wavefronts the chain is that much shorter and the CU has as many more chains to switch
// between; the partial sums meet in LDS (at most 128 KiB, about 1 us), not in memory.  Measured (us, FP8 to bf16, before -> now):
// 154x9216x3072 14.8 -> 9.9, 512x3072x3072 11.6 -> 8.8, 512x3072x12288 42 -> 29; INT8 1024x1280x1280 8.4 -> 6.5, 333x1280x5120 16 ->
// 10.  FP8 of few rows with no more than scales and bias goes to lq_gemm_rows.hip instead.
#pragma once

#include "lq_gemm_core.h"

namespace lq {

template <int KIND, typename OutTag> static int run_small_as(const GemmParams& p, int form, hipStream_t st) {
    switch (form) {
        case SMALL_32x32_K4: return launch_gemm<KIND, OutTag, 32, 32, 64, 1, 1, 3, 4>(p, st);
        case SMALL_32x64_K4: return launch_gemm<KIND, OutTag, 32, 64, 64, 1, 2, 3, 4>(p, st);
        case SMALL_64x128_K2: return launch_gemm<KIND, OutTag, 64, 128, 64, 1, 2, 4, 2>(p, st);
        case SMALL_128x128_K2: return launch_gemm<KIND, OutTag, 128, 128, 64, 2, 2, 3, 2>(p, st);
        default: set_error("gemm: unknown form %d", form); return LQ_ERR_ARG;
    }
}

}  // namespace lq
