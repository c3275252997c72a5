// Which tile form takes an 8-bit GEMM of few tiles (host code).
#include "lq_gemm_core.h"

namespace lq {

int few_tiles_form(int m, int m2, int n, int k, float* cost_out) {
    // Time of a launch by the number of workgroups each CU of 256 has to hold (us at k = 3072): up to 256 of them, up to 512, ...; more
    // than fit make whole rounds.  128x128 tiles share k from k = 2048 up: below, adding up two halves costs what the shorter walk
    // saves (us, one walk / shared, 128 to 256 tiles -- FP8 k = 1152: 7.0-7.7 / 7.6-8.7, 1792: 8.5-11.4 / 8.9-10.8, 2048: 9.2-12.5 /
    // 9.4-12.1, 2560: 10.6-15.3 / 10.5-14.3, 3072: 13.1-17.7 / 12.6-16.4; INT8 k = 1280: 8.7-10.0 / 8.5-9.9, 2048: 11.1-13.7 /
    // 10.4-12.7, 3072: 15.6-19.5 / 14.0-18.1).
    struct Cost { int form, bm, bn, per_round, groups; float us[4]; };
    static const Cost table[] = {{2, 128, 128, 512, 1, {16, 26}},
                                 {4, 128, 256, 512, 1, {21, 42}},
                                 {3, 64, 64, 1024, 1, {9.5f, 13, 19, 19}},
                                 {SMALL_128x128_K2, 128, 128, 256, 2, {14}},
                                 {SMALL_64x128_K2, 64, 128, 256, 2, {9}},
                                 {SMALL_32x64_K4, 32, 64, 512, 4, {6.2f, 10}},
                                 {SMALL_32x32_K4, 32, 32, 768, 4, {5, 7.5f, 11.5f}}};
    int best = 2;
    float least = 0.0f;
    for (const Cost& c : table) {
        if (k % (64 * c.groups) != 0 || (c.form == SMALL_128x128_K2 && k < 2048)) continue;
        const long tiles = (((long)m + c.bm - 1) / c.bm + ((long)m2 + c.bm - 1) / c.bm) * (((long)n + c.bn - 1) / c.bn), left = tiles % c.per_round;
        const float cost = (float)(tiles / c.per_round) * c.us[(c.per_round + 255) / 256 - 1] + (left == 0 ? 0.0f : c.us[(left - 1) / 256]);
        if (least == 0.0f || cost < least) { best = c.form; least = cost; }
    }
    if (cost_out != nullptr) *cost_out = least;
    return best;
}

bool fp8_rows_takes(const GemmParams& p);  // lq_gemm_rows.hip
int run_fp8_rows(const GemmParams& p, lq_dtype_t out_dtype, hipStream_t st);

int run_small(GemmKind kind, const GemmParams& p, lq_dtype_t out_dtype, int form, hipStream_t st) {
    // Few rows: one pass over the weights.  Up to 32 of them other epilogues, and rows of an activation that it does not take, have a
    // form that sums in the same order, so that a linear with and without one agrees to the bit.
    if (kind == K_FP8 && fp8_rows_takes(p)) return run_fp8_rows(p, out_dtype, st);
    if (kind == K_FP8 && p.m <= 32 && p.kb % 256 == 0 && form != SMALL_32x32_K4) form = SMALL_32x64_K4;
    if (out_dtype == LQ_BF16) return kind == K_FP8 ? run_small_fp8_bf16(p, form, st) : run_small_int8_bf16(p, form, st);
    return kind == K_FP8 ? run_small_fp8_f16(p, form, st) : run_small_int8_f16(p, form, st);
}

}  // namespace lq
