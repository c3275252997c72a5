// Which tile form takes an 8-bit GEMM of few tiles (host code).
#include "lq_gemm_core.h"

namespace lq {

static long tiles_of(int m, int m2, int n, int bm, int bn) {
    return (((long)m + bm - 1) / bm + ((long)m2 + bm - 1) / bm) * (((long)n + bn - 1) / bn);
}

// Short k: prologue and epilogue are most of the time, and only the forms of eight wavefronts and 128-byte k-tiles lead, by one round
// against the 1.25 or the half that 128x128 tiles of four wavefronts make (INT8, us, those / this: k = 640, 640 outputs, 4096 rows 6.7 / 6.3,
// 6000 7.6 / 7.0, 8192 9.5 / 8.4, 2048 rows, 80 tiles, 5.8 / 5.9; 1024x5120 11.1 / 10.0, 1500x1920 8.4 / 7.6; k = 768 1345x3040 11.7 / 9.9; k = 896
// 2048x1920 9.3 / 8.8; k = 1024 8192x640 13.2 / 11.6, 1024x5120 13.1 / 11.3).
int short_k_form(int m, int n, int k) {
    if (k < 640 || k % 128 != 0) return -1;
    const long t128 = tiles_of(m, 0, n, 128, 128);
    return t128 > 256 && tiles_of(m, 0, n, 192, 128) <= 256 ? SMALL_192x128 : t128 > 128 && t128 <= 256 ? SMALL_128x128 : -1;
}

int few_tiles_form(int m, int m2, int n, int k, bool rounds, float* cost_out) {
    // Time of a launch by the number of workgroups each CU of 256 has to hold (us at k = 3072): up to 256 of them, up to 512, ...; more
    // than fit make whole rounds.  k is a multiple of k_unit.
    struct Cost { int form, bm, bn, per_round, k_unit; float us[4]; };
    static const Cost table[] = {{2, 128, 128, 512, 64, {16, 26}},
                                 {4, 128, 256, 512, 64, {21, 42}},
                                 {3, 64, 64, 1024, 64, {9.5f, 13, 19, 19}},
                                 {SMALL_128x128, 128, 128, 256, 128, {12.6f}},
                                 {SMALL_192x128, 192, 128, 256, 128, {16.5f}},
                                 {SMALL_64x128_K2, 64, 128, 256, 128, {9}},
                                 {SMALL_32x64_K4, 32, 64, 512, 256, {6.2f, 10}},
                                 {SMALL_32x32_K4, 32, 32, 768, 256, {5, 7.5f, 11.5f}}};
    int best = 2;
    float least = 0.0f;
    for (const Cost& c : table) {
        if (k % c.k_unit != 0) continue;
        const long tiles = tiles_of(m, m2, n, c.bm, c.bn), left = tiles % c.per_round;
        if ((c.form == SMALL_128x128 || c.form == SMALL_192x128) && tiles > c.per_round && !rounds) continue;
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
