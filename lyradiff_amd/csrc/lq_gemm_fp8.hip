// FP8 e4m3 GEMM entry point (fp32 accumulation on v_mfma_f32_32x32x64_f8f6f4) with the fused
// per-tensor scale, bias, optional tanh-GELU and residual epilogue.  Reference contract:
// utils/cublasMMWrapper.cc:1104-1274 of lyraDiff (cuBLASLt FP8 matmul with A/B scale pointers and
// BIAS / GELU_BIAS epilogues).
#include "lq_gemm_core.h"

namespace lq {

int run_fp8_f16(const GemmParams& p, hipStream_t st);   // lq_gemm_fp8_{f16,bf16,f32}.hip
int run_fp8_bf16(const GemmParams& p, hipStream_t st);
int run_fp8_f32(const GemmParams& p, hipStream_t st);
int run_fp8_pair_f16(const GemmPair& pair, int form, hipStream_t st);  // lq_gemm_pair_{f16,bf16}.hip
int run_fp8_pair_bf16(const GemmPair& pair, int form, hipStream_t st);

}  // namespace lq

using namespace lq;

// LQ_OK: go on; 1: m == 0, nothing to do (pointers of empty tensors may be null); negative: error
static int fp8_check(const char* what, const void* C, const uint8_t* A, const uint8_t* B, const float* a_scale, const float* b_scale,
                     const void* bias, const void* residual, int m, int n, int k) {
    LQ_REQUIRE(m >= 0 && n > 0 && k > 0 && n % 32 == 0 && k % 64 == 0, LQ_ERR_SHAPE,
               "%s: need n %% 32 == 0 and k %% 64 == 0 (m=%d n=%d k=%d)", what, m, n, k);
    if (m == 0) return 1;
    LQ_REQUIRE(A && B && a_scale && b_scale, LQ_ERR_ARG, "%s: null pointer", what);
    LQ_REQUIRE(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0 &&
                   reinterpret_cast<uintptr_t>(C) % 16 == 0 && reinterpret_cast<uintptr_t>(bias) % 8 == 0 &&
                   reinterpret_cast<uintptr_t>(residual) % 16 == 0,
               LQ_ERR_ARG, "%s: A, B, C, residual must be 16-byte aligned, bias 8-byte aligned", what);
    return LQ_OK;
}

static int fp8_dispatch(const char* what, const GemmParams& p, lq_dtype_t out_dtype, lq_stream_t stream) {
    hipStream_t st = as_stream(stream);
    switch (out_dtype) {
        case LQ_F16: return run_fp8_f16(p, st);
        case LQ_BF16: return run_fp8_bf16(p, st);
        case LQ_F32: return run_fp8_f32(p, st);
        default: set_error("%s: unsupported output dtype %d", what, (int)out_dtype); return LQ_ERR_UNSUPPORTED;
    }
}

extern "C" int lq_gemm_fp8_ex(void* C, lq_dtype_t out_dtype, const uint8_t* A, const uint8_t* B_rows32,
                              const float* a_scale, const float* b_scale, const void* bias, int gelu,
                              const void* residual, float beta, int m, int n, int k, float* out_scale, uint8_t* C_fp8,
                              const float* C_fp8_scale, lq_stream_t stream) {
    int rc = fp8_check("lq_gemm_fp8", C, A, B_rows32, a_scale, b_scale, bias, residual, m, n, k);
    if (rc != LQ_OK) return rc > 0 ? LQ_OK : rc;
    LQ_REQUIRE(C || C_fp8, LQ_ERR_ARG, "lq_gemm_fp8: null pointer");
    LQ_REQUIRE((C_fp8 == nullptr) == (C_fp8_scale == nullptr), LQ_ERR_ARG, "lq_gemm_fp8: C_fp8 and C_fp8_scale go together");
    LQ_REQUIRE(reinterpret_cast<uintptr_t>(C_fp8) % 4 == 0, LQ_ERR_ARG, "lq_gemm_fp8: C_fp8 must be 4-byte aligned");
    LQ_REQUIRE(gelu >= 0 && gelu <= 2, LQ_ERR_ARG, "lq_gemm_fp8: gelu must be 0, 1 or 2");
    if (m == 0) return LQ_OK;
    GemmParams p = {};
    p.C = C; p.A = A; p.B = B_rows32; p.bias = bias; p.a_scale = a_scale; p.b_scale = b_scale;
    p.gelu = gelu; p.residual = (beta != 0.0f) ? residual : nullptr; p.beta = beta;
    p.out_scale = out_scale; p.C8 = C_fp8; p.c8_scale = C_fp8_scale; p.ldc8 = (size_t)n;
    p.m = m; p.n = n; p.k = k; p.kb = k;
    // with out_scale the 16-bit output exists to be cast once with that scale; a large one bypasses the cache on its way out
    p.stream_c = out_scale != nullptr && C != nullptr && (size_t)m * (size_t)n * (out_dtype == LQ_F32 ? 4 : 2) >= kStreamBytes;
    return fp8_dispatch("lq_gemm_fp8", p, out_dtype, stream);
}

extern "C" int lq_gemm_fp8_max(void* C, lq_dtype_t out_dtype, const uint8_t* A, const uint8_t* B_rows32, const float* a_scale,
                               const float* b_scale, const void* bias, int m, int n, int k, float* out_max, lq_stream_t stream) {
    int rc = fp8_check("lq_gemm_fp8_max", C, A, B_rows32, a_scale, b_scale, bias, nullptr, m, n, k);
    if (rc != LQ_OK) return rc > 0 ? LQ_OK : rc;
    LQ_REQUIRE(C && out_max, LQ_ERR_ARG, "lq_gemm_fp8_max: null pointer");
    GemmParams p = {};
    p.C = C; p.A = A; p.B = B_rows32; p.bias = bias; p.a_scale = a_scale; p.b_scale = b_scale;
    p.out_max = out_max; p.ldc8 = (size_t)n;
    p.m = m; p.n = n; p.k = k; p.kb = k;
    // the output exists to be read once by the activation + cast pass; a large one bypasses the cache on its way out (the
    // two-workgroups-per-CU kernels only: the persistent kernel's counted waits do not get along with such stores)
    p.stream_c = (size_t)m * (size_t)n * (out_dtype == LQ_F32 ? 4 : 2) >= kStreamBytes;
    return fp8_dispatch("lq_gemm_fp8_max", p, out_dtype, stream);
}

extern "C" int lq_gemm_fp8_panels(void* C, lq_dtype_t out_dtype, const uint8_t* A_panels, const uint8_t* B_rows32,
                                  const float* a_scale, const float* b_scale, const void* bias, int m, int n, int k,
                                  float* out_max, lq_stream_t stream) {
    int rc = fp8_check("lq_gemm_fp8_panels", C, A_panels, B_rows32, a_scale, b_scale, bias, nullptr, m, n, k);
    if (rc != LQ_OK) return rc > 0 ? LQ_OK : rc;
    LQ_REQUIRE(C, LQ_ERR_ARG, "lq_gemm_fp8_panels: null pointer");
    GemmParams p = {};
    p.C = C; p.A = A_panels; p.B = B_rows32; p.bias = bias; p.a_scale = a_scale; p.b_scale = b_scale;
    p.out_max = out_max; p.ldc8 = (size_t)n;
    p.m = m; p.n = n; p.k = k; p.kb = k;
    p.a_panel = 1;
    p.stream_c = out_max != nullptr && (size_t)m * (size_t)n * (out_dtype == LQ_F32 ? 4 : 2) >= kStreamBytes;  // as lq_gemm_fp8_max
    return fp8_dispatch("lq_gemm_fp8_panels", p, out_dtype, stream);
}

extern "C" int lq_gemm_fp8(void* C, lq_dtype_t out_dtype, const uint8_t* A, const uint8_t* B_rows32,
                           const float* a_scale, const float* b_scale, const void* bias, int gelu,
                           const void* residual, float beta, int m, int n, int k, lq_stream_t stream) {
    LQ_REQUIRE(C != nullptr || m == 0, LQ_ERR_ARG, "lq_gemm_fp8: null pointer");
    return lq_gemm_fp8_ex(C, out_dtype, A, B_rows32, a_scale, b_scale, bias, gelu, residual, beta, m, n, k, nullptr, nullptr,
                          nullptr, stream);
}

static int gemm_fp8_gated(void* C, lq_dtype_t out_dtype, const uint8_t* A, const uint8_t* B_rows32,
                                 const float* a_scale, const float* b_scale, const void* bias, const void* gate,
                                 size_t rows_per_gate, const void* residual, int m, int n, int k, int a_panel, lq_stream_t stream) {
    int rc = fp8_check("lq_gemm_fp8_gated", C, A, B_rows32, a_scale, b_scale, bias, residual, m, n, k);
    if (rc != LQ_OK) return rc > 0 ? LQ_OK : rc;
    LQ_REQUIRE(C && gate && residual, LQ_ERR_ARG, "lq_gemm_fp8_gated: null pointer");
    LQ_REQUIRE(rows_per_gate > 0, LQ_ERR_SHAPE, "lq_gemm_fp8_gated: rows_per_gate must be positive");
    LQ_REQUIRE(reinterpret_cast<uintptr_t>(gate) % 16 == 0, LQ_ERR_ARG, "lq_gemm_fp8_gated: gate must be 16-byte aligned");
    if (m == 0) return LQ_OK;
    GemmParams p = {};
    p.C = C; p.A = A; p.B = B_rows32; p.bias = bias; p.a_scale = a_scale; p.b_scale = b_scale;
    p.residual = residual; p.beta = 1.0f; p.gate = gate; p.gate_rows = rows_per_gate; p.ldc8 = (size_t)n;
    p.m = m; p.n = n; p.k = k; p.kb = k;
    p.a_panel = a_panel;
    return fp8_dispatch("lq_gemm_fp8_gated", p, out_dtype, stream);
}

extern "C" int lq_gemm_fp8_gated(void* C, lq_dtype_t out_dtype, const uint8_t* A, const uint8_t* B_rows32, const float* a_scale,
                                 const float* b_scale, const void* bias, const void* gate, size_t rows_per_gate, const void* residual,
                                 int m, int n, int k, lq_stream_t stream) {
    return gemm_fp8_gated(C, out_dtype, A, B_rows32, a_scale, b_scale, bias, gate, rows_per_gate, residual, m, n, k, 0, stream);
}

extern "C" int lq_gemm_fp8_gated_panels(void* C, lq_dtype_t out_dtype, const uint8_t* A_panels, const uint8_t* B_rows32,
                                        const float* a_scale, const float* b_scale, const void* bias, const void* gate,
                                        size_t rows_per_gate, const void* residual, int m, int n, int k, lq_stream_t stream) {
    return gemm_fp8_gated(C, out_dtype, A_panels, B_rows32, a_scale, b_scale, bias, gate, rows_per_gate, residual, m, n, k, 1, stream);
}

static int gemm_fp8_codes(uint8_t* C_fp8, size_t ldc, const float* C_fp8_scale, lq_dtype_t round_dtype,
                                 const uint8_t* A, const uint8_t* B_rows32, const float* a_scale, const float* b_scale,
                                 const void* bias, int gelu, int m, int n, int k, int panels, lq_stream_t stream) {
    LQ_REQUIRE(gelu >= 0 && gelu <= 2, LQ_ERR_ARG, "lq_gemm_fp8_codes: gelu must be 0, 1 or 2");
    LQ_REQUIRE(ldc >= (size_t)(n > 0 ? n : 0) && ldc % 4 == 0, LQ_ERR_SHAPE, "lq_gemm_fp8_codes: need ldc >= n and ldc %% 4 == 0 (ldc=%zu n=%d)", ldc, n);
    int rc = fp8_check("lq_gemm_fp8_codes", nullptr, A, B_rows32, a_scale, b_scale, bias, nullptr, m, n, k);
    if (rc != LQ_OK) return rc > 0 ? LQ_OK : rc;
    LQ_REQUIRE(C_fp8 && C_fp8_scale, LQ_ERR_ARG, "lq_gemm_fp8_codes: null pointer");
    LQ_REQUIRE(ldc >= (size_t)n && ldc % 4 == 0 && reinterpret_cast<uintptr_t>(C_fp8) % 4 == 0, LQ_ERR_SHAPE,
               "lq_gemm_fp8_codes: need ldc >= n, ldc %% 4 == 0 and a 4-byte aligned destination (ldc=%zu n=%d)", ldc, n);
    GemmParams p = {};
    p.A = A; p.B = B_rows32; p.bias = bias; p.a_scale = a_scale; p.b_scale = b_scale; p.gelu = gelu;
    p.C8 = C_fp8; p.c8_scale = C_fp8_scale; p.ldc8 = ldc;
    p.m = m; p.n = n; p.k = k; p.kb = k;
    p.a_panel = panels;   // both the activation read and the codes written, or neither
    p.c8_panel = panels;
    LQ_REQUIRE(!panels || n % 64 == 0, LQ_ERR_SHAPE, "lq_gemm_fp8_codes_panels: codes in k-panels need n %% 64 == 0 (n=%d)", n);
    return fp8_dispatch("lq_gemm_fp8_codes", p, round_dtype, stream);
}

extern "C" int lq_gemm_fp8_codes(uint8_t* C_fp8, size_t ldc, const float* C_fp8_scale, lq_dtype_t round_dtype, const uint8_t* A,
                                 const uint8_t* B_rows32, const float* a_scale, const float* b_scale, const void* bias, int gelu,
                                 int m, int n, int k, lq_stream_t stream) {
    return gemm_fp8_codes(C_fp8, ldc, C_fp8_scale, round_dtype, A, B_rows32, a_scale, b_scale, bias, gelu, m, n, k, 0, stream);
}

extern "C" int lq_gemm_fp8_codes_panels(uint8_t* C_fp8_panels, const float* C_fp8_scale, lq_dtype_t round_dtype,
                                        const uint8_t* A_panels, const uint8_t* B_rows32, const float* a_scale, const float* b_scale,
                                        const void* bias, int gelu, int m, int n, int k, lq_stream_t stream) {
    return gemm_fp8_codes(C_fp8_panels, (size_t)(n > 0 ? n : 0), C_fp8_scale, round_dtype, A_panels, B_rows32, a_scale, b_scale, bias, gelu,
                          m, n, k, 1, stream);
}

static long pair_tiles(int m, int m2, int n, int rows, int cols) {
    return (((long)m + rows - 1) / rows + ((long)m2 + rows - 1) / rows) * (((long)n + cols - 1) / cols);
}

// The form of one launch over m and m2 rows and its time (us at k = 3072), by the lines of run_fp8_as; persist: 256x256 tiles that are all
// full run in the persistent form there.  A round of 256 256x256 tiles or of 512 128x256 tiles takes 38, of the persistent form 35, and
// up to 256 128x256 tiles behind full rounds 18.
static int launch_form(int m, int m2, int n, int k, bool plain, bool persist, float* cost) {
    const long t256 = pair_tiles(m, m2, n, 256, 256), last256 = t256 % 256;
    // More than one round of eight wavefronts: the rule knows no layout here.  Pairs come as k-panels, where two rounds are level at long k with no
    // more than scales and bias and behind otherwise (600 + 512 rows 9216x3072, us, four wavefronts / two rounds: 44.7 / 41.8).
    if (t256 < 192) return few_tiles_form(m, m2, n, k, plain && k >= 2560, cost);
    *cost = (float)((t256 + 255) / 256) * (persist && t256 > 256 ? 35.0f : 38.0f);
    const bool wide = (last256 != 0 && last256 < 128) || (!plain && t256 > 256);
    if (!wide || (persist && t256 > 256)) return plain ? 6 : 0;
    const long t4 = pair_tiles(m, m2, n, 128, 256), left = t4 % 512;
    *cost = (float)(t4 / 512) * 38.0f + (left == 0 ? 0.0f : left <= 256 ? 18.0f : 38.0f);
    return 4;
}

// The form for both problems in one launch; -1: one after the other.  The second problem's tiles by themselves leave most of the chip idle
// for a whole walk over k; behind the first one's they cost nothing where its last round has room for them, and most of a round where it
// has not: the times of the rounds decide.  Measured (us, bf16, k-panels, two launches / one), 4096 + 512 rows: 9216x3072 121 / 114,
// 3072x3072 48 / 39, 12288x3072 with GELU to codes 161 / 153, 3072x12288 with gate 160 / 141; 6400 + 512: 176 / 160, 80 / 60, 244 / 236,
// 252 / 231; 400 + 100: 30 / 23, 16 / 10, 47 / 35, 47 / 31.  Two launches are ahead where the second only opens another round: 5120 + 512
// rows 3072x3072 51 / 57, 3072x12288 with gate 180 / 205; 8192 + 512 rows 3072x12288 277 / 297; 6144 + 64 rows 9216x3072 151 / 154 (the
// persistent form), 12288x3072 to codes 209 / 218; 4096 + 77 rows 12288x3072 147 / 153; 2500 + 200 rows 3072x12288 115 / 126.
static int pair_form(int m, int m2, int n, int k, bool plain) {
    if (m <= 32 || m2 <= 32) return -1;  // few rows have a kernel of their own
    for (int rows : {m, m2})
        if (requested_tactic(g_tactic_fp8, LQ_W_FP8, rows, n, k) >= 0) return -1;  // tactics stand
    if (k <= 1024) return pair_tiles(m, m2, n, 128, 128) >= 128 ? 2 : 3;
    float both, alone[2];
    const int form = launch_form(m, m2, n, k, plain, false, &both);
    for (int i = 0; i < 2; ++i) {
        const int rows = i ? m2 : m;
        launch_form(rows, 0, n, k, plain, plain && rows % 256 == 0 && n % 256 == 0 && k % 128 == 0, &alone[i]);
    }
    return both < alone[0] + alone[1] ? form : -1;
}

extern "C" int lq_gemm_fp8_pair_takes(int m, int m2, int n, int k, int plain) {
    return m > 0 && m2 > 0 && n > 0 && k > 0 && pair_form(m, m2, n, k, plain != 0) >= 0;
}

extern "C" int lq_gemm_fp8_pair(const lq_fp8_half_t* halves, lq_dtype_t dtype, int gelu, int panels, int n, int k, lq_stream_t stream) {
    LQ_REQUIRE(halves, LQ_ERR_ARG, "lq_gemm_fp8_pair: null pointer");
    LQ_REQUIRE(dtype == LQ_F16 || dtype == LQ_BF16, LQ_ERR_UNSUPPORTED, "lq_gemm_fp8_pair: dtype must be F16 or BF16");
    LQ_REQUIRE(gelu >= 0 && gelu <= 2, LQ_ERR_ARG, "lq_gemm_fp8_pair: gelu must be 0, 1 or 2");
    GemmPair pair = {};
    int problems = 0;
    for (int i = 0; i < 2; ++i) {
        const lq_fp8_half_t& h = halves[i];
        const int rc = fp8_check("lq_gemm_fp8_pair", h.C, h.A, h.B_rows32, h.a_scale, h.b_scale, h.bias, h.residual, h.m, n, k);
        if (rc < 0) return rc;
        if (rc > 0) continue;
        LQ_REQUIRE((h.C == nullptr) != (h.C_fp8 == nullptr), LQ_ERR_ARG, "lq_gemm_fp8_pair: one of C and C_fp8");
        LQ_REQUIRE((h.C_fp8 == nullptr) == (h.C_fp8_scale == nullptr), LQ_ERR_ARG, "lq_gemm_fp8_pair: C_fp8 and C_fp8_scale go together");
        LQ_REQUIRE(h.C_fp8 == nullptr || (reinterpret_cast<uintptr_t>(h.C_fp8) % 4 == 0 && (!panels || n % 64 == 0)), LQ_ERR_SHAPE,
                   "lq_gemm_fp8_pair: need a 4-byte aligned C_fp8, and n %% 64 == 0 for k-panels (n=%d)", n);
        LQ_REQUIRE((h.gate == nullptr) == (h.residual == nullptr) && (h.gate == nullptr || (h.C != nullptr && h.rows_per_gate > 0)), LQ_ERR_ARG,
                   "lq_gemm_fp8_pair: gate and residual go together, with C and a positive rows_per_gate");
        LQ_REQUIRE(reinterpret_cast<uintptr_t>(h.gate) % 16 == 0, LQ_ERR_ARG, "lq_gemm_fp8_pair: gate must be 16-byte aligned");
        LQ_REQUIRE(gelu == 0 || h.C_fp8 != nullptr, LQ_ERR_ARG, "lq_gemm_fp8_pair: the activation comes with C_fp8");
        GemmParams& p = pair.p[problems++];
        p.C = h.C; p.A = h.A; p.B = h.B_rows32; p.bias = h.bias; p.a_scale = h.a_scale; p.b_scale = h.b_scale; p.gelu = gelu;
        p.C8 = h.C_fp8; p.c8_scale = h.C_fp8_scale; p.ldc8 = (size_t)n;
        p.gate = h.gate; p.gate_rows = h.rows_per_gate; p.residual = h.residual; p.beta = 1.0f;
        p.m = h.m; p.n = n; p.k = k; p.kb = k;
        p.a_panel = panels != 0;
        p.c8_panel = panels != 0;
    }
    if (problems == 2) {
        const GemmParams &a = pair.p[0], &b = pair.p[1];
        LQ_REQUIRE((a.C8 == nullptr) == (b.C8 == nullptr) && (a.gate == nullptr) == (b.gate == nullptr), LQ_ERR_ARG,
                   "lq_gemm_fp8_pair: both halves need the same outputs");
        const int form = pair_form(a.m, b.m, n, k, a.gelu == 0 && a.C8 == nullptr && a.gate == nullptr);
        if (form >= 0) return dtype == LQ_BF16 ? run_fp8_pair_bf16(pair, form, as_stream(stream)) : run_fp8_pair_f16(pair, form, as_stream(stream));
    }
    for (int i = 0; i < problems; ++i) {
        const int rc = fp8_dispatch("lq_gemm_fp8_pair", pair.p[i], dtype, stream);
        if (rc != LQ_OK) return rc;
    }
    return LQ_OK;
}
