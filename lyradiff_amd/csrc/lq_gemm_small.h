// 8-bit GEMMs of few tiles: the forms of GemmKernel whose wavefront groups share k out, and those whose eight wavefronts walk 128-byte k-tiles.
//
// What bounds them: a workgroup alone on a CU takes 0.17 us (64x64) to 0.3 us (128x256) per 64-byte k-tile whatever it computes --
// the barrier, the LDS round trip of the fragments, the transfers' issue and the matrix instructions follow each other -- and walks k by
// itself.  Two remedies:
//   * k shared between two or four groups of wavefronts (_K2, _K4), where tiles fill at most half of the chip: the chain is that much
//     shorter and the CU has as many more chains to switch between; the partial sums meet in LDS (at most 64 KiB), not in memory.
//   * k-tiles of 128 bytes and eight wavefronts, one workgroup per CU, where up to 256 tiles of 128x128 or of 192x128 make one round: half
//     the barriers, whole 128-byte lines of a row-major activation, a second wavefront on each SIMD beside the one that waits.  128x128
//     with k shared by two groups of four stood here before (us, then the general tiles / that / now, FP8: 333x9216x3072 16.5 / 14.7 /
//     12.9, 1024x3072x3072 15.9 / 14.6 / 12.6, 1024x3072x12288 52 / 43 / 38; INT8: 2048x1280x1280 8.8 / 8.8 / 7.9, 2048x1280x5120 26.5 /
//     22.6 / 19.4, 4096x640x2560 13.7 / 12.4 / 11.4).  192x128, general / now: FP8 512x9216x3072 20.3 / 16.7, 700x12288x3072 34.5 / 30.4 (two
//     rounds); INT8 8192x640x2560 21.2 / 17.1, 4096x1280x5120 33.4 / 29.6.  Three or four stages, four wavefronts of 64x64 in place of
//     eight of 64x32, level; 256x128 tiles 20.7 where 192x128 take 17.1.
// The second kind adds up k in one chain where k-shared groups add two or four: no other error against 64 bits in FP8 (2-norm, one chain and
// two alike: 333x9216x3072 bf16 1.6624e-3, 1024x3072x12288 f16 2.0735e-4, most of it the output's own rounding).
// More than one round of the second kind: for a row-major activation, with a residual, an activation function, gates or codes in the epilogue
// from k = 2560 up.  Two workgroups of four wavefronts per CU overlap one's epilogue with the other's walk, and k-panels take the cache
// lines' advantage away (us, four wavefronts / two rounds of these -- row-major, scales and bias: FP8 1024x9216x3072 37.9 / 32.7, x1152 18.4 /
// 17.4, INT8 1700x5120x5120 65 / 54; gated, FP8 900x9216x3072 40.4 / 37.4, x1152 20.7 / 23.4, k = 2048 0.93 to 1.04 times; INT8 with a
// residual x3072 43.1 / 39.6, x1152 21.3 / 23.5; k-panels, gated FP8 34.0 / 37.2, x1152 18.2 / 23.4, scales and bias 31.1 / 31.5, x1152 15.8 / 16.9).
// FP8 of few rows with no more than scales and bias goes to lq_gemm_rows.hip instead.
#pragma once

#include "lq_gemm_core.h"

namespace lq {

template <int KIND, typename OutTag> static int run_small_as(const GemmParams& p, int form, hipStream_t st) {
    switch (form) {
        case SMALL_32x32_K4: return launch_gemm<KIND, OutTag, 32, 32, 64, 1, 1, 3, 4>(p, st);
        case SMALL_32x64_K4: return launch_gemm<KIND, OutTag, 32, 64, 64, 1, 2, 3, 4>(p, st);
        case SMALL_64x128_K2: return launch_gemm<KIND, OutTag, 64, 128, 64, 1, 2, 4, 2>(p, st);
        case SMALL_128x128: return launch_gemm<KIND, OutTag, 128, 128, 128, 2, 4, 4>(p, st);
        case SMALL_192x128: return launch_gemm<KIND, OutTag, 192, 128, 128, 2, 4, 3>(p, st);
        default: set_error("gemm: unknown form %d", form); return LQ_ERR_ARG;
    }
}

}  // namespace lq
