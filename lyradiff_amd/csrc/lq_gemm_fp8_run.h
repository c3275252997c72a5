// Tile configuration and launch of the FP8 GEMM for one output type; each type is instantiated in a translation unit of its own
// (lq_gemm_fp8_{f16,bf16,f32}.hip), so that they compile side by side.
#pragma once

#include "lq_gemm_core.h"

namespace lq {


template <typename OutTag> static constexpr lq_dtype_t out_enum() {
    return std::is_same<OutTag, F16Tag>::value ? LQ_F16 : std::is_same<OutTag, BF16Tag>::value ? LQ_BF16 : LQ_F32;
}

template <typename OutTag> static int run_fp8_as(GemmParams p, hipStream_t st) {
    constexpr bool out16 = out_enum<OutTag>() == LQ_F16 || out_enum<OutTag>() == LQ_BF16;
    const bool forced = tl_forced_tactic >= 0 || g_tactic_fp8 >= 0;
    const int requested = requested_tactic(g_tactic_fp8, LQ_W_FP8, p.m, p.n, p.k);
    int t = requested;
    // scales and bias, and at most the running maximum of the outputs (two instructions per four outputs)
    const bool plain_epilogue = p.gelu == 0 && p.out_scale == nullptr && p.C8 == nullptr && p.gate == nullptr &&
                                p.residual == nullptr && p.addend == nullptr;
    if (t < 0) {
        const long t256 = (long)((p.m + 255) / 256) * ((p.n + 255) / 256);
        const long t128 = (long)((p.m + 127) / 128) * ((p.n + 127) / 128);
        // 256x256 tiles, one wavefront per SIMD, when their last round on the 256 CUs is at least half full (measured on
        // the FLUX shapes at 4608 and 6912 rows, FP8 and INT8: ahead of the others by up to 10 % then, level or up to 4 %
        // behind otherwise); else 128x256 tiles, two workgroups per CU (finer tail, one workgroup's epilogue overlaps the
        // other's MFMA work)
        const long last256 = t256 % 256;
        t = t256 >= 192 ? ((last256 == 0 || last256 >= 128) ? 6 : 4) : (t128 >= 128 ? 2 : 3);  // 128x128 tiles from half a round up (4096x640x2560: 14.5 against 16.3 us with 64x64)
        if (p.k <= 1024 && t128 >= 192) t = 2;  // short K: prologue and epilogue dominate, smaller tiles overlap them better
        // More full 256x256 tiles than CUs and nothing but scales and bias in the epilogue: the persistent form
        // (4608x12288x3072: 134-140 us against 148 with 128x256 tiles, 6912x9216x3072: 156 against 161 with tactic 6)
        if (plain_epilogue && t256 > device_cu_count() && p.m % 256 == 0 && p.n % 256 == 0 && p.kb % 128 == 0 && p.k > 1024 &&
            out_enum<OutTag>() != LQ_F32)
            t = 7;
    }
    // Too few 256x256 tiles: the form whose rounds of workgroups cost least.  A forced or cached tactic stands.  k <= 1024: a
    // workgroup's ten or sixteen k-tiles leave nothing to share (1024x640x640: 4.7 us with 64x64 tiles, 4.9 with k shared).
    if (requested < 0 && out16 && p.k > 1024 && (long)((p.m + 255) / 256) * ((p.n + 255) / 256) < 192) {
        t = few_tiles_form(p.m, 0, p.n, p.k, p.a_panel == 0 && (plain_epilogue || p.k >= 2560));
        if (t >= SMALL_32x32_K4) return run_small(K_FP8, p, out_enum<OutTag>(), t, st);
    }
    // The 128-byte k-tile needs k % 128 == 0.  On k-panels, whose cache lines are whole in any k-tile, tactic 0 has the same bits and leads (4608x12288x3072 151 / 170 us, 4608x3072x12288 131 / 145).
    if (t == 1 && (p.kb % 128 != 0 || p.a_panel)) t = 0;
    // The per-shape cache is filled by timing the plain epilogue.  With one wavefront per SIMD nothing runs beside tactic 6's
    // epilogue: one that does more than scale and bias (activation, output maximum, codes, gate, residual) costs 13-18 us
    // per 256x256 tile there (transcendentals, or one exposed memory round trip per group of rows) and next to nothing with
    // two wavefronts per SIMD.  Measured at 4608 rows: 12288x3072 with GELU and the output maximum 209-214 us against
    // 153-160 us with tactic 4; 3072x12288 with gate and residual 139 us against 134 us with tactic 0, 3072x3072 55 against
    // 48 us.  A configuration forced by the caller is kept.
    if (t == 6 && !forced && p.out_max != nullptr) t = (long)((p.m + 255) / 256) * ((p.n + 255) / 256) > 256 ? 4 : 0;  // outside the persistent form the running maximum takes the activation epilogue
    if ((t == 6 || t == 7) && !forced && !plain_epilogue) t = (long)((p.m + 255) / 256) * ((p.n + 255) / 256) > 256 ? 4 : 0;
    if (t == 7) {  // the persistent form of tactic 6 where it applies, tactic 6 itself elsewhere
        const int rc = launch_persist_fp8(p, out_enum<OutTag>(), st);
        if (rc != 1) return rc;
        t = 6;
    }
    switch (t) {
        case 0: return launch_gemm<K_FP8, OutTag, 256, 256, 64, 2, 4, 3>(p, st);
        case 1: return launch_gemm<K_FP8, OutTag, 256, 256, 128, 2, 4, 2>(p, st);
        case 2: return launch_gemm<K_FP8, OutTag, 128, 128, 64, 2, 2, 3>(p, st);
        case 3: return launch_gemm<K_FP8, OutTag, 64, 64, 64, 2, 2, 3>(p, st);
        case 4: return launch_gemm<K_FP8, OutTag, 128, 256, 64, 2, 2, 3>(p, st);
        case 5: return launch_gemm<K_FP8, OutTag, 256, 128, 64, 2, 2, 3>(p, st);
        case 6: return launch_gemm<K_FP8, OutTag, 256, 256, 64, 2, 2, 4>(p, st);  // one wavefront per SIMD, 128x128 wavefront tiles
        default: set_error("lq_gemm_fp8: unknown tactic %d", t); return LQ_ERR_ARG;
    }
}

}  // namespace lq
