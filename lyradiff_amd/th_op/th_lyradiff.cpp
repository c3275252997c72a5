// torch custom classes `torch.classes.lyradiff.*` for the FLUX blocks, the way the reference's Python reaches them:
//     torch.classes.load_library(os.getenv("LYRA_LIB_PATH"))                      (lyradiff/__init__.py:4-5)
//     torch.classes.lyradiff.FluxTransformerBlockOp("bf16", 3072, 24, 128, 6, quant_level)
// Registered classes and methods follow src/lyradiff/th_op/pybind.cc:66-96 (FluxTransformerBlockOp,
// FluxSingleTransformerBlockOp, LyraDiffCommonContext; constructor arguments with the same names and defaults,
// initialize, forward, load_lora_by_name, clear_lora, reload_model_from_bin, reload_model_from_state_dict) and
// th_op/flux_transformer_block/FluxTransformerBlockOp.h:186-330,
// th_op/flux_single_transformer_block/FluxSingleTransformerBlockOp.h:184-290.
//
// Quant levels 1, 2 (FP8_W8A8, FP8_W8A8_FULL) and 7, 8 (INT4_W4A4, INT4_W4A4_FULL) are built, the levels whose blocks
// consist of quantized linears.  Every quantized linear, adaLN / gate / residual step, activation quantisation, the q/k
// RMSNorm, the rotary embedding and the softmax attention run on liblyraquant.so through its C ABI, and so does the 16-bit adaLN matmul of
// the non-FULL levels for the row counts that lq_linear16_rows_takes; PyTorch supplies device memory, the current stream and that matmul for
// other sizes and alignments.
// This file holds no device code and is compiled with the host compiler.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/custom_class.h>
#include <torch/script.h>

#include <cmath>
#include <cstdio>
#include <map>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "lyraquant.h"

namespace th = torch;

namespace torch_ext {

namespace {

lq_stream_t cur_stream() { return reinterpret_cast<lq_stream_t>(c10::hip::getCurrentHIPStream().stream()); }

lq_dtype_t lq_dt(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return LQ_F32;
        case at::kHalf: return LQ_F16;
        case at::kBFloat16: return LQ_BF16;
        default: TORCH_CHECK(false, "unsupported tensor dtype for the quantized-linear library");
    }
}

void* P(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
uint8_t* P8(const at::Tensor& t) { return static_cast<uint8_t*>(P(t)); }
const float* PF(const at::Tensor& t) { return static_cast<const float*>(P(t)); }

void ok(int rc, const char* what) { TORCH_CHECK(rc == LQ_OK, "[lyradiff Error][", what, "] ", lq_last_error()); }

at::TensorOptions on_gpu(at::ScalarType t) { return at::TensorOptions().dtype(t).device(at::kCUDA); }

// ---- where tensors come from: a state dict or the reference's raw .bin files ---------------------------------------
struct Source {
    virtual ~Source() = default;
    // `dtype` is the type the tensor is wanted in; 16-bit members of a .bin directory are stored in the model file type
    virtual at::Tensor get(const std::string& name, at::IntArrayRef shape, at::ScalarType dtype) const = 0;
};

struct DictSource : Source {
    th::Dict<std::string, th::Tensor> d;
    explicit DictSource(th::Dict<std::string, th::Tensor> dict) : d(std::move(dict)) {}
    at::Tensor get(const std::string& name, at::IntArrayRef shape, at::ScalarType dtype) const override {
        TORCH_CHECK(d.contains(name), "Cannot find a tensor of name ", name);  // TensorMap::at of the reference throws likewise
        at::Tensor t = d.at(name);
        int64_t want = 1;
        for (auto s : shape) want *= s;
        TORCH_CHECK(t.numel() == want && t.scalar_type() == dtype, name, ": got ", t.sizes(), " ", t.scalar_type(), ", expected ",
                    shape, " ", dtype);
        return t.reshape(shape).contiguous();
    }
};

// loadWeightFromBin (utils/memory_utils.cu:251-360): a headerless little-endian file of `model_file_type` elements,
// converted to the wanted type with round-to-nearest-even; scales, smoothing vectors and packed codes are always
// stored as fp32 / int8.
struct BinSource : Source {
    at::ScalarType file_type;
    explicit BinSource(const std::string& model_dtype) {
        if (model_dtype == "fp32") file_type = at::kFloat;
        else if (model_dtype == "fp16") file_type = at::kHalf;
        else if (model_dtype == "bf16") file_type = at::kBFloat16;
        else throw std::invalid_argument("wrong model_dtype");
    }
    at::Tensor get(const std::string& name, at::IntArrayRef shape, at::ScalarType dtype) const override {
        const bool sixteen = dtype == at::kHalf || dtype == at::kBFloat16;
        const at::ScalarType in_file = sixteen ? file_type : dtype;
        at::Tensor t = at::empty(shape, at::TensorOptions().dtype(in_file));
        const std::string path = name + ".bin";
        FILE* f = std::fopen(path.c_str(), "rb");
        TORCH_CHECK(f != nullptr, "[lyradiff Error] file ", path, " cannot be opened");
        const size_t bytes = (size_t)t.numel() * t.element_size();
        const size_t got = std::fread(t.data_ptr(), 1, bytes, f);
        const bool more = std::fgetc(f) != EOF;
        std::fclose(f);
        TORCH_CHECK(got == bytes && !more, "[lyradiff Error] file ", path, " does not hold ", t.numel(), " elements of ", in_file);
        return sixteen ? t.to(dtype) : t;
    }
};

// ---- the three kinds of linear ------------------------------------------------------------------------------------
// FP8 e4m3 per-tensor linear, quantised when loaded (MACROLoadFP8WeightFromBin / ...FromCache,
// utils/common_macro_def.h:66-92); the 16-bit host copy stays for LoRA merges (FP8LoraWeight, interface/IFLoraWeight.h:79-128).
struct FP8Linear {
    at::Tensor w_rows32, w_scale, in_scale, bias, master_h;
    int64_t n = 0, k = 0;

    void requantise(const at::Tensor& w16) {
        w_scale.zero_();
        ok(lq_fp8_amax_scale(static_cast<float*>(P(w_scale)), P(w16), lq_dt(w16.scalar_type()), (size_t)w16.numel(), cur_stream()),
           "lq_fp8_amax_scale");
        at::Tensor codes = at::empty({n, k}, on_gpu(at::kByte));
        ok(lq_fp8_scale_cast(P8(codes), P(w16), lq_dt(w16.scalar_type()), PF(w_scale), 1, (size_t)w16.numel(), cur_stream()),
           "lq_fp8_scale_cast");
        ok(lq_repack_rows32(P8(w_rows32), P8(codes), (size_t)n, (size_t)k, cur_stream()), "lq_repack_rows32");
    }
    void load(const Source& src, const std::string& key, int64_t d_out, int64_t d_in, at::ScalarType T) {
        n = d_out, k = d_in;
        master_h = src.get(key + ".weight", {n, k}, T).cpu().clone();
        in_scale = src.get(key + "_input_scale", {1}, at::kFloat).to(at::kCUDA);
        bias = src.get(key + ".bias", {n}, T).to(at::kCUDA);
        w_scale = at::zeros({1}, on_gpu(at::kFloat));
        w_rows32 = at::empty({n, k}, on_gpu(at::kByte));
        requantise(master_h.to(at::kCUDA));
    }
    void load_lora(const at::Tensor& delta, double alpha) {
        at::Tensor w16 = master_h.to(at::kCUDA);
        TORCH_CHECK(delta.numel() == w16.numel(), "lora_weights holds ", delta.numel(), " elements, the weight ", w16.numel());
        at::Tensor dl = delta.to(w16.options()).reshape(w16.sizes()).contiguous();
        ok(lq_load_lora(P(w16), P(dl), lq_dt(w16.scalar_type()), (size_t)w16.numel(), (float)alpha, cur_stream()), "lq_load_lora");
        requantise(w16);
    }
    void clear_lora() { requantise(master_h.to(at::kCUDA)); }

    // FP8 activations inside this file travel as k-panels [K/64][M][64] (lyraquant.h): the quantising kernels write them,
    // the GEMMs fetch them in whole cache lines; codes and outputs are those of the row-major calls.
    at::Tensor cast_input(const at::Tensor& x2) const {  // e4m3 codes of x [M, K] with the calibrated static scale, as k-panels
        at::Tensor q = at::empty({x2.size(1) / 64, x2.size(0), 64}, on_gpu(at::kByte));
        ok(lq_fp8_scale_cast_panels(P8(q), P(x2), lq_dt(x2.scalar_type()), PF(in_scale), 1, (size_t)x2.size(0), (size_t)x2.size(1),
                                    cur_stream()),
           "lq_fp8_scale_cast_panels");
        return q;
    }
    at::Tensor from_panels(const at::Tensor& q, int64_t m, at::ScalarType T) const {
        at::Tensor y = at::empty({m, n}, on_gpu(T));
        ok(lq_gemm_fp8_panels(P(y), lq_dt(T), P8(q), P8(w_rows32), PF(in_scale), PF(w_scale), P(bias), (int)m, (int)n, (int)k, nullptr,
                              cur_stream()),
           "lq_gemm_fp8_panels");
        return y;
    }
    at::Tensor from_panels_gated(const at::Tensor& q, int64_t m, const at::Tensor& gate, int64_t rows_per_gate,
                                 const at::Tensor& residual) const {
        at::Tensor y = at::empty({m, n}, residual.options());
        ok(lq_gemm_fp8_gated_panels(P(y), lq_dt(residual.scalar_type()), P8(q), P8(w_rows32), PF(in_scale), PF(w_scale), P(bias), P(gate),
                                    (size_t)rows_per_gate, P(residual), (int)m, (int)n, (int)k, cur_stream()),
           "lq_gemm_fp8_gated_panels");
        return y;
    }
};

// One half of an FP8 pair (lq_gemm_fp8_pair): the codes of its [m, K] input; the caller adds what the output is
lq_fp8_half_t half_of(const FP8Linear& l, const at::Tensor& q, int64_t m) {
    lq_fp8_half_t h = {};
    h.A = P8(q), h.B_rows32 = P8(l.w_rows32), h.a_scale = PF(l.in_scale), h.b_scale = PF(l.w_scale), h.bias = P(l.bias), h.m = (int)m;
    return h;
}
void gemm_pair(const lq_fp8_half_t& a, const lq_fp8_half_t& b, at::ScalarType T, int gelu, int panels, int64_t n, int64_t k) {
    const lq_fp8_half_t halves[2] = {a, b};
    ok(lq_gemm_fp8_pair(halves, lq_dt(T), gelu, panels, (int)n, (int)k, cur_stream()), "lq_gemm_fp8_pair");
}
// two linears of one shape on codes in k-panels, in one launch where that is faster, into ya and yb ([.., n])
void linear_pair(const FP8Linear& la, const at::Tensor& qa, const at::Tensor& ya, const FP8Linear& lb, const at::Tensor& qb, const at::Tensor& yb) {
    lq_fp8_half_t a = half_of(la, qa, qa.size(1)), b = half_of(lb, qb, qb.size(1));
    a.C = P(ya), b.C = P(yb);
    gemm_pair(a, b, ya.scalar_type(), 0, 1, la.n, la.k);
}
// the gated output projections behind the activations of both halves: gate [B, n], residual [B, S, n] -> [B, S, n]
std::vector<at::Tensor> gated_pair(const FP8Linear& la, const at::Tensor& qa, const at::Tensor& gate_a, const at::Tensor& res_a, const FP8Linear& lb,
                                   const at::Tensor& qb, const at::Tensor& gate_b, const at::Tensor& res_b, int panels) {
    at::Tensor ya = at::empty_like(res_a), yb = at::empty_like(res_b);
    lq_fp8_half_t a = half_of(la, qa, res_a.size(0) * res_a.size(1)), b = half_of(lb, qb, res_b.size(0) * res_b.size(1));
    a.C = P(ya), a.gate = P(gate_a), a.rows_per_gate = (size_t)res_a.size(1), a.residual = P(res_a);
    b.C = P(yb), b.gate = P(gate_b), b.rows_per_gate = (size_t)res_b.size(1), b.residual = P(res_b);
    gemm_pair(a, b, res_a.scalar_type(), 0, panels, la.n, la.k);
    return {ya, yb};
}

// W4A4 group-64 linear with its low-rank branch (W4A4GemmWeight.cc:65-83, W4A4Gemm.cc:113-169)
// Large problems run on one e4m3 byte per value, laid out from the packed weight in each call (lq_w4a4_weight_codes): same results, no
// widening in the GEMM.
struct W4A4Linear {
    at::Tensor w_rows32, w_scale, smooth, lora_up, lora_down, bias;
    int64_t n = 0, k = 0, rank = 32;

    void load(const Source& src, const std::string& prefix, int64_t d_out, int64_t d_in, bool has_bias, at::ScalarType T) {
        n = d_out, k = d_in;
        at::Tensor packed = src.get(prefix + "packed_weight", {n, k / 2}, at::kChar).to(at::kCUDA);
        w_rows32 = at::empty({n, k / 2}, on_gpu(at::kByte));
        ok(lq_repack_rows32(P8(w_rows32), P8(packed), (size_t)n, (size_t)(k / 2), cur_stream()), "lq_repack_rows32");
        w_scale = src.get(prefix + "weight_scale", {n, k / 64}, at::kFloat).to(at::kCUDA);
        smooth = src.get(prefix + "smooth", {k}, at::kFloat).to(at::kCUDA);
        lora_up = src.get(prefix + "lora_up", {n, rank}, T).to(at::kCUDA);
        lora_down = src.get(prefix + "lora_down", {rank, k}, T).to(at::kCUDA);
        if (has_bias) bias = src.get(prefix + "bias", {n}, T).to(at::kCUDA);
    }
    // quantise + low-rank down + GEMM with the epilogue options of lq_epilogue_t; returns the 16-bit output (undefined
    // when only codes are asked for), written to y if that is given
    at::Tensor run(const at::Tensor& x2, const lq_epilogue_t* epi, bool want_output, at::Tensor y = at::Tensor()) const {
        const int64_t m = x2.size(0);
        const at::ScalarType T = x2.scalar_type();
        at::Tensor act = at::empty({m, rank}, on_gpu(T));
        if (want_output && !y.defined()) y = at::empty({m, n}, on_gpu(T));
        if (lq_w4a4_prefers_codes((int)m, (int)n, (int)k)) {
            at::Tensor q = at::empty({m, k}, on_gpu(at::kByte)), s = at::empty({k / 64, m}, on_gpu(at::kFloat));
            at::Tensor w = at::empty({n, k}, on_gpu(at::kByte)), ws = at::empty({k / 64, n}, on_gpu(at::kFloat));
            ok(lq_w4a4_quantize_lora_down_codes(P8(q), static_cast<float*>(P(s)), P(act), lq_dt(T), P(x2), lq_dt(T), PF(smooth), P(lora_down),
                                                (int)m, (int)k, (int)rank, cur_stream()),
               "lq_w4a4_quantize_lora_down_codes");
            ok(lq_w4a4_weight_codes(P8(w), static_cast<float*>(P(ws)), P8(w_rows32), PF(w_scale), (int)n, (int)k, cur_stream()),
               "lq_w4a4_weight_codes");
            ok(lq_gemm_w4a4_codes(P(y), lq_dt(T), P8(q), P8(w), PF(s), PF(ws), P(bias), P(act), P(lora_up), lq_dt(T), (int)rank, (int)m, (int)n,
                                  (int)k, epi, cur_stream()),
               "lq_gemm_w4a4_codes");
            return y;
        }
        at::Tensor q = at::empty({m, k / 8}, on_gpu(at::kInt)), s = at::empty({m, k / 64}, on_gpu(at::kFloat));
        ok(lq_w4a4_quantize_lora_down(static_cast<uint32_t*>(P(q)), P(s), LQ_F32, P(act), lq_dt(T), P(x2), lq_dt(T), PF(smooth),
                                      P(lora_down), (int)m, (int)k, (int)rank, 64, cur_stream()),
           "lq_w4a4_quantize_lora_down");
        ok(lq_gemm_w4a4_ex(P(y), lq_dt(T), static_cast<const uint32_t*>(P(q)), P8(w_rows32), P(s), P(w_scale), LQ_F32, P(bias), P(act),
                           P(lora_up), lq_dt(T), (int)rank, (int)m, (int)n, (int)k, 64, epi, cur_stream()),
           "lq_gemm_w4a4_ex");
        return y;
    }
};

// adaLN linear: FP8 at the _FULL levels (AdaFP8LayerNormWeight.cc:36-92), a plain 16-bit linear otherwise (AdaLayerNormWeight)
struct AdaLinear {
    bool fp8 = false;
    FP8Linear q;
    at::Tensor weight, bias;
    void load(const Source& src, const std::string& prefix, int64_t dim, int64_t chunks, bool full, at::ScalarType T) {
        fp8 = full;
        if (full) { q.load(src, prefix + "linear", chunks * dim, dim, T); return; }
        weight = src.get(prefix + "linear.weight", {chunks * dim, dim}, T).to(at::kCUDA);
        bias = src.get(prefix + "linear.bias", {chunks * dim}, T).to(at::kCUDA);
    }
    // msa [chunks, B, D] from the (already SiLU'd) time embedding [B, D]  (AdaFP8LayerNorm.cc:100-175, invokeTranspose102)
    static at::Tensor chunked(const at::Tensor& flat, int64_t chunks, int64_t d) {
        const int64_t b = flat.size(0);
        return b > 1 ? flat.view({b, chunks, d}).transpose(0, 1).contiguous() : flat.view({chunks, 1, d});
    }
    static bool aligned(const at::Tensor& t, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(P(t)) % bytes == 0; }
    bool rows16() const { return aligned(weight, 16) && aligned(bias, 8); }  // a view into a larger buffer need not be: at::linear takes it
    at::Tensor msa(const at::Tensor& temb, int64_t chunks) const { return msa_of(temb, chunks, nullptr).first; }
    // with `other`, the adaLN linear of the other half of a double-stream block (same temb), both: in one launch where few rows let it
    std::pair<at::Tensor, at::Tensor> msa_of(const at::Tensor& temb, int64_t chunks, const AdaLinear* other) const {
        const int64_t b = temb.size(0), d = temb.size(1), n = chunks * d;
        const lq_dtype_t dt = lq_dt(temb.scalar_type());
        const bool rows = fp8 ? lq_linear_fp8_rows_takes((int)b, (int)n, (int)d) != 0
                              : lq_linear16_rows_takes((int)b, (int)n, (int)d) != 0 && aligned(temb, 16) && rows16() && (other == nullptr || other->rows16()) &&
                                    !(at::GradMode::is_enabled() && temb.requires_grad());
        at::Tensor y, y2;
        int rc = LQ_NOT_TAKEN;
        if (rows) y = at::empty({b, n}, temb.options());
        if (rows && other != nullptr) y2 = at::empty({b, n}, temb.options());
        if (rows && fp8)
            rc = lq_linear_fp8_rows(P(y), P(y2), P(temb), dt, P8(q.w_rows32), other ? P8(other->q.w_rows32) : nullptr, PF(q.in_scale),
                                    other ? PF(other->q.in_scale) : nullptr, PF(q.w_scale), other ? PF(other->q.w_scale) : nullptr, P(q.bias),
                                    other ? P(other->q.bias) : nullptr, (int)b, (int)n, (int)d, cur_stream());
        else if (rows)
            rc = lq_linear16_rows(P(y), P(y2), P(temb), P(weight), other ? P(other->weight) : nullptr, P(bias), other ? P(other->bias) : nullptr, dt,
                                  (int)b, (int)n, (int)d, cur_stream());
        if (rc < 0) ok(rc, "adaLN linear");
        if (rc == LQ_NOT_TAKEN) {
            if (other != nullptr) return {msa_of(temb, chunks, nullptr).first, other->msa_of(temb, chunks, nullptr).first};
            y = fp8 ? q.from_panels(q.cast_input(temb), b, temb.scalar_type()) : at::linear(temb, weight, bias);
        }
        return {chunked(y, chunks, d), other != nullptr ? chunked(y2, chunks, d) : at::Tensor()};
    }
};

// (1 + msa[1]) * LayerNorm(x) + msa[0] with the FP8 cast(s) of the consumers fused; x [B, S, D]
at::Tensor adaln_codes(const at::Tensor& x, const at::Tensor& msa, const at::Tensor& in_scale) {  // k-panels [D/64, B*S, 64]
    at::Tensor c = at::empty({x.size(2) / 64, x.size(0) * x.size(1), 64}, on_gpu(at::kByte));
    ok(lq_layernorm_mod_fp8_panels(P8(c), P(x), P(msa[1]), P(msa[0]), lq_dt(x.scalar_type()), PF(in_scale), (size_t)x.size(0),
                                   (size_t)x.size(1), (size_t)x.size(2), 1e-6f, cur_stream()),
       "lq_layernorm_mod_fp8_panels");
    return c;
}
at::Tensor adaln_16(const at::Tensor& x, const at::Tensor& msa) {
    at::Tensor y = at::empty_like(x);
    ok(lq_gate_residual_layernorm_mod(P(y), nullptr, nullptr, nullptr, P(x), P(msa[1]), P(msa[0]), lq_dt(x.scalar_type()),
                                      (size_t)x.size(0), (size_t)x.size(1), (size_t)x.size(2), 1e-6f, cur_stream()),
       "lq_gate_residual_layernorm_mod");
    return y;
}

// ---- between the QKV and the output projections ----------------------------------------------------------------------
// elements between the rotary tables of two batches: rope_emb is [B or 1, tokens, Dh / 2, 2, 2]
size_t rope_stride(const at::Tensor& rope, int64_t b, int64_t tokens, int64_t dh) {
    const int64_t per_batch = tokens * dh * 2;
    TORCH_CHECK(rope.numel() == per_batch || rope.numel() == b * per_batch, "rope_emb must be [B or 1, ", tokens, ", ", dh / 2, ", 2, 2]");
    return rope.numel() != per_batch ? (size_t)per_batch : 0;
}
// q/k RMSNorm + rotary embedding in place on qkv [B, S, 3D] whose first sc tokens are the text (invokeFusedRmsNormCatAndRope,
// kernels/rope/flux_apply_rope.cu:74-156)
void rotate(const at::Tensor& qkv, int64_t sc, const at::Tensor& norm_qk, const at::Tensor& norm_added_qk, const at::Tensor& rope, int64_t heads) {
    const int64_t b = qkv.size(0), s = qkv.size(1), dh = qkv.size(2) / 3 / heads;
    ok(lq_rmsnorm_rope_inplace(P(qkv), P(norm_qk), P(norm_added_qk), P(rope), rope_stride(rope, b, s, dh), lq_dt(qkv.scalar_type()), (int)b,
                               (int)s, (int)sc, (int)heads, (int)dh, 1e-6f, cur_stream()),
       "lq_rmsnorm_rope_inplace");
}
// the same with the concatenation [text, image] into a new tensor [B, Sc + S, 3D]
at::Tensor rotate_two(const at::Tensor& qkv, const at::Tensor& ctx_qkv, const at::Tensor& norm_qk, const at::Tensor& norm_added_qk,
                      const at::Tensor& rope, int64_t heads) {
    const int64_t b = qkv.size(0), s = qkv.size(1), sc = ctx_qkv.size(1), dh = qkv.size(2) / 3 / heads;
    at::Tensor cat = at::empty({b, sc + s, qkv.size(2)}, qkv.options());
    ok(lq_rmsnorm_rope(P(cat), P(qkv), P(ctx_qkv), P(norm_qk), P(norm_added_qk), P(rope), rope_stride(rope, b, sc + s, dh), lq_dt(qkv.scalar_type()),
                       (int)b, (int)s, (int)sc, (int)heads, (int)dh, 1e-6f, cur_stream()),
       "lq_rmsnorm_rope");
    return cat;
}
// softmax attention of cat [B, S, 3D] (q, k and v are strided parts of it); the caller adds the outputs
lq_attention_t attention_of(const at::Tensor& cat, int64_t heads) {
    const int64_t b = cat.size(0), s = cat.size(1), d = cat.size(2) / 3, dh = d / heads;  // dh is 64 or 128 here, the rotation takes no other
    const char* parts = static_cast<const char*>(P(cat));
    const size_t part = (size_t)d * cat.element_size();
    lq_attention_t a = {};
    a.q = parts, a.k = parts + part, a.v = parts + 2 * part;
    a.q_row = a.k_row = a.v_row = (size_t)(3 * d);
    a.q_batch = a.k_batch = a.v_batch = (size_t)(3 * d * s);
    a.dtype = lq_dt(cat.scalar_type()), a.batch = (int)b, a.seq_q = a.seq_k = (int)s, a.heads = (int)heads, a.head_dim = (int)dh;
    a.scale = 1.0f / std::sqrt((float)dh);
    return a;
}
at::Tensor attention_out(const at::Tensor& cat, int64_t heads) {  // [B, S, D]
    at::Tensor o = at::empty({cat.size(0), cat.size(1), cat.size(2) / 3}, cat.options());
    lq_attention_t a = attention_of(cat, heads);
    a.out = P(o);
    ok(lq_attention_ex(&a, cur_stream()), "lq_attention_ex");
    return o;
}
// the output as e4m3 codes in k-panels: the image's to `codes`, those of the first sc tokens to `ctx_codes`
void attention_codes(const at::Tensor& cat, int64_t heads, uint8_t* codes, const float* scale, int64_t sc = 0, uint8_t* ctx_codes = nullptr,
                     const float* ctx_scale = nullptr) {
    lq_attention_t a = attention_of(cat, heads);
    a.out_fp8 = codes, a.out_fp8_scale = scale, a.context = (int)sc, a.context_fp8 = ctx_codes, a.context_fp8_scale = ctx_scale;
    ok(lq_attention_ex(&a, cur_stream()), "lq_attention_ex");
}

// FluxAttnPostFP8Processor (FluxAttnPostFP8Processor.cc:93-240)
struct AttnPostFP8 {
    FP8Linear gelu_proj, ff_linear;
    void load(const Source& src, const std::string& prefix, int64_t dim, at::ScalarType T) {
        gelu_proj.load(src, prefix + "net.0.proj", 4 * dim, dim, T);
        ff_linear.load(src, prefix + "net.2", dim, 4 * dim, T);
    }
    // gate + residual + adaLN + cast: {codes for gelu_proj as k-panels, hidden}
    std::pair<at::Tensor, at::Tensor> gated_norm(const at::Tensor& x, const at::Tensor& attn, const at::Tensor& msa) const {
        const int64_t b = x.size(0), s = x.size(1), d = x.size(2);
        at::Tensor q1 = at::empty({d / 64, b * s, 64}, on_gpu(at::kByte)), hidden = at::empty_like(x);
        ok(lq_gate_residual_layernorm_mod_fp8_panels(P8(q1), P(hidden), P(attn), P(msa[2]), P(x), P(msa[4]), P(msa[3]), lq_dt(x.scalar_type()),
                                                     PF(gelu_proj.in_scale), (size_t)b, (size_t)s, (size_t)d, 1e-6f, cur_stream()),
           "lq_gate_residual_layernorm_mod_fp8_panels");
        return {q1, hidden};
    }
};
// FluxAttnPostFP8Processor::forward of the image and of the text half, their linears two to a launch
std::vector<at::Tensor> attn_post_pair(const AttnPostFP8& w, const at::Tensor& x, const at::Tensor& attn, const at::Tensor& msa,
                                       const AttnPostFP8& wc, const at::Tensor& c, const at::Tensor& cattn, const at::Tensor& cmsa) {
    const auto a = w.gated_norm(x, attn, msa), b = wc.gated_norm(c, cattn, cmsa);
    const int64_t ma = x.size(0) * x.size(1), mb = c.size(0) * c.size(1), f = w.gelu_proj.n;
    at::Tensor qa = at::empty({f / 64, ma, 64}, on_gpu(at::kByte)), qb = at::empty({f / 64, mb, 64}, on_gpu(at::kByte));
    lq_fp8_half_t ha = half_of(w.gelu_proj, a.first, ma), hb = half_of(wc.gelu_proj, b.first, mb);
    ha.C_fp8 = P8(qa), ha.C_fp8_scale = PF(w.ff_linear.in_scale);
    hb.C_fp8 = P8(qb), hb.C_fp8_scale = PF(wc.ff_linear.in_scale);
    gemm_pair(ha, hb, x.scalar_type(), 1, 1, f, w.gelu_proj.k);
    return gated_pair(w.ff_linear, qa, msa[5], a.second, wc.ff_linear, qb, cmsa[5], b.second, 1);
}

// FluxAttnPostInt4Processor (FluxAttnPostInt4Processor.cc:103-215)
struct AttnPostInt4 {
    W4A4Linear gelu_proj;
    FP8Linear ff_linear;
    void load(const Source& src, const std::string& prefix, int64_t dim, at::ScalarType T) {
        gelu_proj.load(src, prefix + "net.0.proj.", 4 * dim, dim, true, T);
        ff_linear.load(src, prefix + "net.2", dim, 4 * dim, T);
    }
    // everything up to ff_linear: {its input's codes [B*S, 4D], hidden}
    std::pair<at::Tensor, at::Tensor> activation(const at::Tensor& x, const at::Tensor& attn, const at::Tensor& msa) const {
        const int64_t b = x.size(0), s = x.size(1), d = x.size(2), m = b * s;
        at::Tensor norm = at::empty_like(x), hidden = at::empty_like(x);
        ok(lq_gate_residual_layernorm_mod(P(norm), P(hidden), P(attn), P(msa[2]), P(x), P(msa[4]), P(msa[3]), lq_dt(x.scalar_type()),
                                          (size_t)b, (size_t)s, (size_t)d, 1e-6f, cur_stream()),
           "lq_gate_residual_layernorm_mod");
        at::Tensor q2 = at::empty({m, 4 * d}, on_gpu(at::kByte));
        lq_epilogue_t epi = {2, nullptr, nullptr, 1, nullptr, P8(q2), (size_t)(4 * d), PF(ff_linear.in_scale)};
        gelu_proj.run(norm.view({m, d}), &epi, false);
        return {q2, hidden};
    }
};
// FluxAttnPostInt4Processor::forward of both halves, their FP8 output projections two to a launch
std::vector<at::Tensor> attn_post_pair(const AttnPostInt4& w, const at::Tensor& x, const at::Tensor& attn, const at::Tensor& msa,
                                       const AttnPostInt4& wc, const at::Tensor& c, const at::Tensor& cattn, const at::Tensor& cmsa) {
    const auto a = w.activation(x, attn, msa), b = wc.activation(c, cattn, cmsa);
    return gated_pair(w.ff_linear, a.first, msa[5], a.second, wc.ff_linear, b.first, cmsa[5], b.second, 0);
}

void check_input(const at::Tensor& t, const char* name, at::ScalarType T) {  // CHECK_TH_CUDA, CHECK_CONTIGUOUS, th_utils.h:14-33
    TORCH_CHECK(t.is_cuda(), name, " must be a CUDA tensor");
    TORCH_CHECK(t.is_contiguous(), name, " must be contiguous");
    TORCH_CHECK(t.scalar_type() == T, name, " dtype should be ", T);
}

struct BlockConfig {
    at::ScalarType T;
    int64_t dim, heads, head_dim, mlp_scale, level;
    bool int4, full;
    BlockConfig(const std::string& inference_dtype, int64_t embedding_dim, int64_t embedding_head_num, int64_t embedding_head_dim,
                int64_t mlp, int64_t quant_level)
        : dim(embedding_dim), heads(embedding_head_num), head_dim(embedding_head_dim), mlp_scale(mlp), level(quant_level) {
        if (inference_dtype == "fp16") T = at::kHalf;
        else if (inference_dtype == "bf16") T = at::kBFloat16;
        else TORCH_CHECK(false, "wrong inference_dtype");  // fp32 blocks hold no quantized linear in the reference either
        TORCH_CHECK(level == 1 || level == 2 || level == 7 || level == 8, "quant level ", level,
                    ": only the FP8 (1, 2) and INT4 (7, 8) blocks are built on this library");
        TORCH_CHECK(dim == heads * head_dim, "embedding_dim must equal embedding_head_num * embedding_head_dim");
        int4 = level >= 7;
        full = level == 2 || level == 8;
    }
};

std::string join(const std::vector<std::string>& parts) {
    std::string s;
    for (size_t i = 0; i < parts.size(); ++i) s += (i ? "." : "") + parts[i];
    return s;
}

}  // namespace

struct LyraDiffCommonContext : th::CustomClassHolder {
    // the reference creates its stream, cuBLAS handles and allocator here (th_op/lyradiff_common_context/
    // LyraDiffCommonContext.h); this library works on PyTorch's current stream and allocator and needs none of it
    LyraDiffCommonContext() = default;
};

// Double-stream block: FluxTransformerFP8Block.cc:159-262 / FluxTransformerInt4Block.cc:159-246
struct FluxTransformerBlockOp : th::CustomClassHolder {
    BlockConfig cfg;
    bool loaded = false;
    std::mutex lock;
    AdaLinear norm1, norm1_context;
    FP8Linear to_qkv, to_added_qkv, to_out, to_add_out;
    W4A4Linear to_qkv4, to_added_qkv4, to_out4, to_add_out4;
    AttnPostFP8 ff, ff_context;
    AttnPostInt4 ff4, ff_context4;
    at::Tensor norm_qk, norm_added_qk;

    FluxTransformerBlockOp(std::string inference_dtype, int64_t embedding_dim, int64_t embedding_head_num, int64_t embedding_head_dim,
                           int64_t mlp_scale, int64_t quant_level)
        : cfg(inference_dtype, embedding_dim, embedding_head_num, embedding_head_dim, mlp_scale, quant_level) {}

    void initialize(const c10::intrusive_ptr<LyraDiffCommonContext>&) {}

    void load(const Source& src, const std::string& p) {
        std::lock_guard<std::mutex> g(lock);
        const at::ScalarType T = cfg.T;
        const int64_t d = cfg.dim;
        norm1.load(src, p + "norm1.", d, 6, cfg.full, T);
        norm1_context.load(src, p + "norm1_context.", d, 6, cfg.full, T);
        if (cfg.int4) {
            to_qkv4.load(src, p + "attn.to_qkv.", 3 * d, d, true, T);
            to_added_qkv4.load(src, p + "attn.to_added_qkv.", 3 * d, d, true, T);
            to_out4.load(src, p + "attn.to_out.0.", d, d, true, T);
            to_add_out4.load(src, p + "attn.to_add_out.", d, d, true, T);
            ff4.load(src, p + "ff.", d, T);
            ff_context4.load(src, p + "ff_context.", d, T);
        } else {
            to_qkv.load(src, p + "attn.to_qkv", 3 * d, d, T);
            to_added_qkv.load(src, p + "attn.to_added_qkv", 3 * d, d, T);
            to_out.load(src, p + "attn.to_out.0", d, d, T);
            to_add_out.load(src, p + "attn.to_add_out", d, d, T);
            ff.load(src, p + "ff.", d, T);
            ff_context.load(src, p + "ff_context.", d, T);
        }
        auto nw = [&](const char* n) { return src.get(p + "attn." + n + ".weight", {cfg.head_dim}, T).to(at::kCUDA); };
        norm_qk = at::cat({nw("norm_q"), nw("norm_k")});
        norm_added_qk = at::cat({nw("norm_added_q"), nw("norm_added_k")});
        loaded = true;
    }
    void reload_model_from_state_dict(std::string prefix, th::Dict<std::string, th::Tensor> weights, std::string /*device*/) {
        load(DictSource(std::move(weights)), prefix);
    }
    void reload_model_from_bin(std::string model_path, std::string model_dtype) { load(BinSource(model_dtype), model_path); }

    std::map<std::string, FP8Linear*> lora_targets() {
        std::map<std::string, FP8Linear*> t = {{"attn.to_qkv", &to_qkv}, {"attn.to_added_qkv", &to_added_qkv},
                                               {"attn.to_out.0", &to_out}, {"attn.to_add_out", &to_add_out},
                                               {"ff.net.0.proj", &ff.gelu_proj}, {"ff.net.2", &ff.ff_linear},
                                               {"ff_context.net.0.proj", &ff_context.gelu_proj}, {"ff_context.net.2", &ff_context.ff_linear}};
        if (norm1.fp8) t["norm1.linear"] = &norm1.q, t["norm1_context.linear"] = &norm1_context.q;
        return t;
    }
    void load_lora_by_name(std::vector<std::string> lora_name, th::Tensor lora_weights, double lora_strength) {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        const std::string key = join(lora_name);
        // the reference's INT4 block weights register no LoRA targets (FluxTransformerInt4BlockWeight.cc:41-45)
        TORCH_CHECK(!cfg.int4, "no LoRA target named ", key, ": the INT4 blocks carry their low-rank branch in the checkpoint");
        auto t = lora_targets();
        auto it = t.find(key);
        TORCH_CHECK(it != t.end(), "no FP8 linear named ", key, " in this block");
        std::lock_guard<std::mutex> g(lock);
        it->second->load_lora(lora_weights, lora_strength);
    }
    void clear_lora() {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        if (cfg.int4) return;
        std::lock_guard<std::mutex> g(lock);
        for (auto& kv : lora_targets()) kv.second->clear_lora();
    }

    std::vector<th::Tensor> forward(th::Tensor hidden_states, th::Tensor encoder_hidden_states, th::Tensor rope_emb, th::Tensor temb_emb) {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        check_input(hidden_states, "hidden_states", cfg.T);
        check_input(encoder_hidden_states, "encoder_hidden_states", cfg.T);
        check_input(rope_emb, "rope_emb", cfg.T);
        check_input(temb_emb, "temb_emb", cfg.T);
        std::lock_guard<std::mutex> g(lock);
        const at::Tensor &x = hidden_states, &c = encoder_hidden_states;
        const int64_t b = x.size(0), s = x.size(1), sc = c.size(1), d = cfg.dim;
        at::Tensor temb = temb_emb.reshape({b, d});
        const auto both_msa = norm1.msa_of(temb, 6, &norm1_context);
        const at::Tensor &msa = both_msa.first, &cmsa = both_msa.second;
        // one batch: both halves' QKV side by side, text first, so that nothing has to be concatenated
        at::Tensor cat, qkv, cqkv;
        if (b == 1) {
            cat = at::empty({1, sc + s, 3 * d}, x.options());
            qkv = cat[0].slice(0, sc, sc + s), cqkv = cat[0].slice(0, 0, sc);
        } else {
            qkv = at::empty({b * s, 3 * d}, x.options()), cqkv = at::empty({b * sc, 3 * d}, x.options());
        }
        if (cfg.int4) {
            to_qkv4.run(adaln_16(x, msa).view({b * s, d}), nullptr, true, qkv);
            to_added_qkv4.run(adaln_16(c, cmsa).view({b * sc, d}), nullptr, true, cqkv);
        } else {
            linear_pair(to_qkv, adaln_codes(x, msa, to_qkv.in_scale), qkv, to_added_qkv, adaln_codes(c, cmsa, to_added_qkv.in_scale), cqkv);
        }
        if (b == 1) rotate(cat, sc, norm_qk, norm_added_qk, rope_emb, cfg.heads);
        else cat = rotate_two(qkv.view({b, s, 3 * d}), cqkv.view({b, sc, 3 * d}), norm_qk, norm_added_qk, rope_emb, cfg.heads);
        if (cfg.int4) {
            at::Tensor o = attention_out(cat, cfg.heads);
            at::Tensor attn = o.slice(1, sc, sc + s).contiguous().view({b * s, d}), cattn = o.slice(1, 0, sc).contiguous().view({b * sc, d});
            at::Tensor a_out = to_out4.run(attn, nullptr, true).view({b, s, d}), c_out = to_add_out4.run(cattn, nullptr, true).view({b, sc, d});
            return attn_post_pair(ff4, x, a_out, msa, ff_context4, c, c_out, cmsa);
        }
        at::Tensor q = at::empty({d / 64, b * s, 64}, on_gpu(at::kByte)), cq = at::empty({d / 64, b * sc, 64}, on_gpu(at::kByte));
        attention_codes(cat, cfg.heads, P8(q), PF(to_out.in_scale), sc, P8(cq), PF(to_add_out.in_scale));
        at::Tensor a_out = at::empty({b, s, d}, x.options()), c_out = at::empty({b, sc, d}, x.options());
        linear_pair(to_out, q, a_out, to_add_out, cq, c_out);
        return attn_post_pair(ff, x, a_out, msa, ff_context, c, c_out, cmsa);
    }
};

// Single-stream block: FluxSingleTransformerFP8Block.cc:163-291 / FluxSingleTransformerInt4Block.cc:178-316
struct FluxSingleTransformerBlockOp : th::CustomClassHolder {
    BlockConfig cfg;
    bool loaded = false;
    std::mutex lock;
    AdaLinear norm;
    FP8Linear to_qkv, proj_mlp, proj_out;
    W4A4Linear to_qkv4, proj_mlp4, proj_out_1, proj_out_2;
    at::Tensor norm_qk;

    FluxSingleTransformerBlockOp(std::string inference_dtype, int64_t embedding_dim, int64_t embedding_head_num,
                                 int64_t embedding_head_dim, int64_t mlp_scale, int64_t quant_level)
        : cfg(inference_dtype, embedding_dim, embedding_head_num, embedding_head_dim, mlp_scale, quant_level) {}

    void initialize(const c10::intrusive_ptr<LyraDiffCommonContext>&) {}

    void load(const Source& src, const std::string& p) {
        std::lock_guard<std::mutex> g(lock);
        const at::ScalarType T = cfg.T;
        const int64_t d = cfg.dim, f = cfg.mlp_scale * cfg.dim;
        norm.load(src, p + "norm.", d, 3, cfg.full, T);
        if (cfg.int4) {
            to_qkv4.load(src, p + "attn.to_qkv.", 3 * d, d, true, T);
            proj_mlp4.load(src, p + "proj_mlp.", f, d, true, T);
            proj_out_1.load(src, p + "proj_out.linears.0.", d, d, true, T);
            proj_out_2.load(src, p + "proj_out.linears.1.linear.", d, f, false, T);
        } else {
            to_qkv.load(src, p + "attn.to_qkv", 3 * d, d, T);
            proj_mlp.load(src, p + "proj_mlp", f, d, T);
            proj_out.load(src, p + "proj_out", d, d + f, T);
        }
        norm_qk = at::cat({src.get(p + "attn.norm_q.weight", {cfg.head_dim}, T).to(at::kCUDA),
                           src.get(p + "attn.norm_k.weight", {cfg.head_dim}, T).to(at::kCUDA)});
        loaded = true;
    }
    void reload_model_from_state_dict(std::string prefix, th::Dict<std::string, th::Tensor> weights, std::string /*device*/) {
        load(DictSource(std::move(weights)), prefix);
    }
    void reload_model_from_bin(std::string model_path, std::string model_dtype) { load(BinSource(model_dtype), model_path); }

    std::map<std::string, FP8Linear*> lora_targets() {
        std::map<std::string, FP8Linear*> t = {{"attn.to_qkv", &to_qkv}, {"proj_mlp", &proj_mlp}, {"proj_out", &proj_out}};
        if (norm.fp8) t["norm.linear"] = &norm.q;
        return t;
    }
    void load_lora_by_name(std::vector<std::string> lora_name, th::Tensor lora_weights, double lora_strength) {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        const std::string key = join(lora_name);
        TORCH_CHECK(!cfg.int4, "no LoRA target named ", key, ": the INT4 blocks carry their low-rank branch in the checkpoint");
        auto t = lora_targets();
        auto it = t.find(key);
        TORCH_CHECK(it != t.end(), "no FP8 linear named ", key, " in this block");
        std::lock_guard<std::mutex> g(lock);
        it->second->load_lora(lora_weights, lora_strength);
    }
    void clear_lora() {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        if (cfg.int4) return;
        std::lock_guard<std::mutex> g(lock);
        for (auto& kv : lora_targets()) kv.second->clear_lora();
    }

    th::Tensor forward(th::Tensor hidden_states, th::Tensor rope_emb, th::Tensor temb_emb) {
        TORCH_CHECK(loaded, "reload_model_from_state_dict has not been called");
        check_input(hidden_states, "hidden_states", cfg.T);
        check_input(rope_emb, "rope_emb", cfg.T);
        check_input(temb_emb, "temb_emb", cfg.T);
        std::lock_guard<std::mutex> g(lock);
        const at::Tensor& x = hidden_states;
        const int64_t b = x.size(0), s = x.size(1), d = cfg.dim, m = b * s, f = cfg.mlp_scale * d;
        const lq_dtype_t dt = lq_dt(cfg.T);
        at::Tensor msa = norm.msa(temb_emb.reshape({b, d}), 3);
        at::Tensor gate = msa[2].contiguous(), none;
        if (cfg.int4) {
            at::Tensor nh = adaln_16(x, msa).view({m, d});
            at::Tensor qkv = to_qkv4.run(nh, nullptr, true).view({b, s, 3 * d});
            rotate(qkv, 0, norm_qk, none, rope_emb, cfg.heads);
            at::Tensor attn = attention_out(qkv, cfg.heads).view({m, d});
            lq_epilogue_t gelu = {2, nullptr, nullptr, 1, nullptr, nullptr, 0, nullptr};
            at::Tensor mlp = proj_mlp4.run(nh, &gelu, true);
            at::Tensor h1 = proj_out_1.run(attn, nullptr, true);
            lq_epilogue_t tail = {0, P(h1), P(gate), (size_t)s, P(x), nullptr, 0, nullptr};
            return proj_out_2.run(mlp, &tail, true).view({b, s, d});
        }
        // one adaLN read yields the codes for to_qkv and for proj_mlp
        at::Tensor c_qkv = at::empty({d / 64, m, 64}, on_gpu(at::kByte)), c_mlp = at::empty({d / 64, m, 64}, on_gpu(at::kByte));
        ok(lq_layernorm_mod_fp8_dual_panels(P8(c_qkv), PF(to_qkv.in_scale), P8(c_mlp), PF(proj_mlp.in_scale), P(x), P(msa[1]), P(msa[0]),
                                            dt, (size_t)b, (size_t)s, (size_t)d, 1e-6f, cur_stream()),
           "lq_layernorm_mod_fp8_dual_panels");
        at::Tensor qkv = to_qkv.from_panels(c_qkv, m, cfg.T).view({b, s, 3 * d});
        rotate(qkv, 0, norm_qk, none, rope_emb, cfg.heads);
        // proj_out's input [attn | gelu(mlp)] as e4m3 codes in k-panels [(D + F)/64, M, 64]: a block of columns is a run of whole
        // panels, so the attention writes the first D/64 panels and the proj_mlp GEMM's epilogue the rest
        // (FluxSingleTransformerFP8Block.cc:216-253)
        at::Tensor q2 = at::empty({(d + f) / 64, m, 64}, on_gpu(at::kByte));
        attention_codes(qkv, cfg.heads, P8(q2), PF(proj_out.in_scale));
        ok(lq_gemm_fp8_codes_panels(P8(q2) + (size_t)(d / 64) * (size_t)m * 64, PF(proj_out.in_scale), dt, P8(c_mlp), P8(proj_mlp.w_rows32),
                                    PF(proj_mlp.in_scale), PF(proj_mlp.w_scale), P(proj_mlp.bias), 2, (int)m, (int)f, (int)d, cur_stream()),
           "lq_gemm_fp8_codes_panels");
        return proj_out.from_panels_gated(q2, m, gate, s, x.view({m, d})).view({b, s, d});
    }
};

}  // namespace torch_ext

// torch_ops.py registers its operators in the same namespace from Python, so this block is a fragment of it
TORCH_LIBRARY_FRAGMENT(lyradiff, m) {
    m.class_<torch_ext::LyraDiffCommonContext>("LyraDiffCommonContext").def(th::init<>());

    m.class_<torch_ext::FluxTransformerBlockOp>("FluxTransformerBlockOp")
        .def(th::init<std::string, int64_t, int64_t, int64_t, int64_t, int64_t>(), "",
             {th::arg("inference_dtype") = "bf16", th::arg("embedding_dim") = 3072, th::arg("embedding_head_num") = 24,
              th::arg("embedding_head_dim") = 128, th::arg("mlp_scale") = 6, th::arg("quant_level") = 0})
        .def("initialize", &torch_ext::FluxTransformerBlockOp::initialize)
        .def("forward", &torch_ext::FluxTransformerBlockOp::forward)
        .def("load_lora_by_name", &torch_ext::FluxTransformerBlockOp::load_lora_by_name)
        .def("clear_lora", &torch_ext::FluxTransformerBlockOp::clear_lora)
        .def("reload_model_from_bin", &torch_ext::FluxTransformerBlockOp::reload_model_from_bin)
        .def("reload_model_from_state_dict", &torch_ext::FluxTransformerBlockOp::reload_model_from_state_dict);

    m.class_<torch_ext::FluxSingleTransformerBlockOp>("FluxSingleTransformerBlockOp")
        .def(th::init<std::string, int64_t, int64_t, int64_t, int64_t, int64_t>(), "",
             {th::arg("inference_dtype") = "bf16", th::arg("embedding_dim") = 3072, th::arg("embedding_head_num") = 24,
              th::arg("embedding_head_dim") = 128, th::arg("mlp_scale") = 4, th::arg("quant_level") = 0})
        .def("initialize", &torch_ext::FluxSingleTransformerBlockOp::initialize)
        .def("forward", &torch_ext::FluxSingleTransformerBlockOp::forward)
        .def("load_lora_by_name", &torch_ext::FluxSingleTransformerBlockOp::load_lora_by_name)
        .def("clear_lora", &torch_ext::FluxSingleTransformerBlockOp::clear_lora)
        .def("reload_model_from_bin", &torch_ext::FluxSingleTransformerBlockOp::reload_model_from_bin)
        .def("reload_model_from_state_dict", &torch_ext::FluxSingleTransformerBlockOp::reload_model_from_state_dict);
}
