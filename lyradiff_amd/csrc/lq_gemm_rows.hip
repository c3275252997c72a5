// FP8 GEMM of at most 32 rows with scales and bias (the modulation linears of the FLUX blocks: one row, 57 MB of weights): a pass
// over the weights.
//
// What bounds it: the weights' way from memory.  The tiled forms bring them to LDS through a few stages per wavefront group, each
// with as many bytes of (repeated) activation rows, so that a workgroup has 16 KiB of weights on their way; here a wavefront
// requests both operands straight into registers -- a 32-row by 64-byte piece of the rows32 layout is two lane-linear kilobytes,
// already the matrix instruction's operand -- DEPTH k-tiles ahead, with neither a barrier nor an LDS round trip in the loop (it issues
// in 8 % of its cycles and waits in the others).  Measured (us, bf16, activation in k-panels, the tiled form -> this one; first
// weights from memory, 1.2 GB of them in turn, then one weight again and again, which the last-level cache keeps):
//   1x18432x3072 15.6 -> 12.1 (4.7 TB/s), 13.1 -> 10.2     1x9216x3072 9.4 -> 8.3, 5.6 -> 4.8     1x3072x3072 7.1 -> 4.8, 4.2 -> 3.4
//   1x3072x12288 17.7 -> 11.9, 12.2 -> 7.9     8x12288x3072 10.1 -> 8.8, 8.7 -> 6.7     24x9216x3072 9.7 -> 9.6, 5.8 -> 5.9
//   32x18432x3072 17.4 -> 14.9, 13.7 -> 11.2     32x9216x3072 9.9 -> 10.2, 5.9 -> 6.3     32x3072x12288 18.5 -> 17.1, 12.5 -> 10.8
// The order of the sums is that of the tiled forms with four k-groups (SMALL_32x32_K4, SMALL_32x64_K4): group g adds the k-tiles g,
// g + 4, ... and the four sums are added in group order, so every result has the same bits whichever form computes it.
#include "lq_gemm_core.h"

namespace lq {

//
// CAST: p.A is the 16-bit activation [m][k]; every workgroup makes the codes it needs by itself, in LDS, while its first weights are on
// their way (12 values per thread at 1 x 3072), in place of a launch of one workgroup in front of this one.  Same codes, same results.
// us from memory and cached, cast + this kernel / CAST: 1x18432x3072 15.6, 13.8 / 12.3, 10.3; 2x18432x3072 15.1, 13.5 / 13.0, 10.9;
// 1x3072x12288 16.1, 12.7 / 13.2, 10.1; below that the two calls cost 12.5 on the host: 4x9216x3072 9.0, 6.8, 1x9216x3072 7.9, 6.8.
template <typename OutTag, bool CAST> __device__ __forceinline__ void fp8_rows(const GemmParams& p, float4* part, char* x_codes) {
    constexpr int KW = 4, DEPTH = 6;  // x_codes: [m][kb + 16]
    const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
    const int kg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rounds = p.kb / (64 * KW);  // k-tiles of this group; kb is a multiple of 256
    // k-tile t of the 32 weight rows: 2 KiB at 2048 t, chunk c of row r at 512 c + 16 r; this lane takes the chunks lh and 2 + lh.
    const uint8_t* wb = p.B + (size_t)blockIdx.x * 32 * (size_t)p.kb + (size_t)kg * 2048 + lane * 16;
    const int row = min(lr, p.m - 1);  // the columns of the result past the last row are not stored
    const uint8_t* xb = CAST ? nullptr : p.a_panel ? p.A + ((size_t)kg * p.m + row) * 64 + lh * 16 : p.A + (size_t)row * p.kb + kg * 64 + lh * 16;
    const u32 xstep = (p.a_panel ? (u32)p.m * 64u : 64u) * KW;
    v4i w[DEPTH][2], x[DEPTH][2];
    auto load = [&](int d, int t) {
        const uint8_t* wp = wb + (size_t)t * (2048 * KW);
        const uint8_t* xp = xb + (size_t)t * xstep;
        w[d][0] = *reinterpret_cast<const v4i*>(wp);
        w[d][1] = *reinterpret_cast<const v4i*>(wp + 1024);
        if constexpr (!CAST) {
            x[d][0] = *reinterpret_cast<const v4i*>(xp);
            x[d][1] = *reinterpret_cast<const v4i*>(xp + 32);
        }
    };
    const char* xl = x_codes + row * (p.kb + 16) + kg * 64 + lh * 16;
    auto load_codes = [&](int d, int t) {
        if constexpr (CAST) {
            x[d][0] = *reinterpret_cast<const v4i*>(xl + t * (64 * KW));
            x[d][1] = *reinterpret_cast<const v4i*>(xl + t * (64 * KW) + 32);
        }
    };
    v16f acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    auto step = [&](int d, int t) {
        load_codes(d, t);
        const v8i a = __builtin_shufflevector(w[d][0], w[d][1], 0, 1, 2, 3, 4, 5, 6, 7);
        const v8i b = __builtin_shufflevector(x[d][0], x[d][1], 0, 1, 2, 3, 4, 5, 6, 7);
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 0, 0, 0, 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(d, min(d, rounds - 1));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (CAST) {
        const float inv = 1.0f / p.a_scale[0];
        const int per_row = p.kb / 8, chunks = p.m * per_row;  // 8 values each
        for (int c = threadIdx.x; c < chunks; c += 256) {
            float v[8];
            unpack8<OutTag>(*reinterpret_cast<const uint4*>(p.A + (size_t)c * 16), v);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] *= inv;
            const int r = c / per_row;
            *reinterpret_cast<uint2*>(x_codes + r * (p.kb + 16) + (c - r * per_row) * 8) =
                make_uint2(e4m3x4(v[0], v[1], v[2], v[3]), e4m3x4(v[4], v[5], v[6], v[7]));
        }
        __syncthreads();
    }
    int t = 0;
    for (; t + DEPTH < rounds; t += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            step(d, t + d);
            load(d, min(t + DEPTH + d, rounds - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (t + d < rounds) step(d, t + d);

    // a lane holds, of one row of C, four consecutive outputs per quad of registers; group g adds, scales and stores quad g
#pragma unroll
    for (int q = 0; q < 4; ++q) part[(kg * 4 + q) * 64 + lane] = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    const int n0 = (int)blockIdx.x * 32 + kg * 8 + lh * 4;
    const float alpha = p.a_scale[0] * p.b_scale[0];
    float bias[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (p.bias != nullptr) OutStore<OutTag>::load4(p.bias, (size_t)n0, bias);
    __syncthreads();
    float4 sum = part[kg * 64 + lane];
#pragma unroll
    for (int g = 1; g < KW; ++g) {
        const float4 v = part[(g * 4 + kg) * 64 + lane];
        sum.x += v.x; sum.y += v.y; sum.z += v.z; sum.w += v.w;
    }
    float y[4] = {sum.x * alpha, sum.y * alpha, sum.z * alpha, sum.w * alpha};
    if (p.bias != nullptr) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = y[e] + bias[e];
    }
    if (lr < p.m) OutStore<OutTag>::store4(p.C, (size_t)lr * p.n + n0, y);
}

template <typename OutTag> __global__ __launch_bounds__(256, 2) void fp8_rows_kernel(GemmParams p) {
    __shared__ float4 part[4 * 4 * 64];
    fp8_rows<OutTag, false>(p, part, nullptr);
}
// blockIdx.y: which of up to two linears of one shape on one input (the modulations of the two halves of a double-stream block)
template <typename OutTag> __global__ __launch_bounds__(256, 2) void fp8_rows_cast_kernel(GemmPair pair) {
    __shared__ float4 part[4 * 4 * 64];
    extern __shared__ __attribute__((aligned(16))) char x_codes[];
    fp8_rows<OutTag, true>(pair.p[blockIdx.y], part, x_codes);
}

// Rows whose codes every workgroup makes by itself: up to 12288 values.  Beyond, the n / 32 copies of that work cost what the launch in
// front saves (us from memory, two launches / one): 8x9216x3072 13.0 / 11.0, 2x3072x12288 15.0 / 15.7, 10x18432x3072 15.5 / 17.9.
constexpr int kCastRows = 8, kCastElems = 12288;

// Rows that are K bytes apart take a cache line each for the 64 bytes of a k-tile, which a workgroup of every 32 columns reads again;
// k-panels put them side by side.  From 17 such rows up that costs more than the tiles' LDS (us from memory / cached, tiled -> this): 16x9216x3072 9.5 -> 9.7 / 5.6 -> 6.7,
// 16x18432x3072 16.7 -> 13.8 / 13.4 -> 11.2, 16x3072x12288 17.9 -> 15.6 / 12.4 -> 11.7; 24x9216x3072 9.8 -> 10.8 / 5.9 -> 7.8,
// 32x12288x3072 10.4 -> 12.5 / 9.3 -> 9.4, 32x3072x12288 19.8 -> 21.0 / 12.7 -> 15.7.
bool fp8_rows_takes(const GemmParams& p) {
    return p.m <= (p.a_panel ? 32 : 16) && p.kb % 256 == 0 && p.C != nullptr && p.gelu == 0 && p.out_scale == nullptr && p.out_max == nullptr && p.C8 == nullptr &&
           p.gate == nullptr && p.residual == nullptr && p.addend == nullptr;
}

int run_fp8_rows(const GemmParams& p, lq_dtype_t out_dtype, hipStream_t st) {
    const dim3 grid((unsigned)(p.n / 32)), block(256);
    if (out_dtype == LQ_BF16) hipLaunchKernelGGL((fp8_rows_kernel<BF16Tag>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((fp8_rows_kernel<F16Tag>), grid, block, 0, st, p);
    return check_launch("fp8_rows");
}

}  // namespace lq

using namespace lq;

extern "C" int lq_linear_fp8_rows_takes(int m, int n, int k) {
    const bool few_tiles = ((long)m + 255) / 256 * (((long)n + 255) / 256) < 192;  // where run_fp8_as turns to the rows kernel
    return m >= 0 && m <= kCastRows && (long)m * k <= kCastElems && k > 1024 && k % 256 == 0 && few_tiles && requested_tactic(g_tactic_fp8, LQ_W_FP8, m, n, k) < 0;
}

extern "C" int lq_linear_fp8_rows(void* C, void* C2, const void* x, lq_dtype_t dtype, const uint8_t* B_rows32, const uint8_t* B2_rows32,
                                  const float* a_scale, const float* a_scale2, const float* b_scale, const float* b_scale2, const void* bias,
                                  const void* bias2, int m, int n, int k, lq_stream_t stream) {
    LQ_REQUIRE(dtype == LQ_F16 || dtype == LQ_BF16, LQ_ERR_UNSUPPORTED, "lq_linear_fp8_rows: dtype must be F16 or BF16");
    LQ_REQUIRE(m >= 0 && n > 0 && k > 0 && n % 32 == 0 && k % 64 == 0, LQ_ERR_SHAPE, "lq_linear_fp8_rows: need n %% 32 == 0 and k %% 64 == 0 (m=%d n=%d k=%d)",
               m, n, k);
    if (m == 0) return LQ_OK;
    const bool two = C2 != nullptr;
    LQ_REQUIRE(C && x && B_rows32 && a_scale && b_scale && (!two || (B2_rows32 && a_scale2 && b_scale2)), LQ_ERR_ARG, "lq_linear_fp8_rows: null pointer");
    if (!lq_linear_fp8_rows_takes(m, n, k) || reinterpret_cast<uintptr_t>(x) % 16 != 0) return LQ_NOT_TAKEN;
    LQ_REQUIRE((reinterpret_cast<uintptr_t>(B_rows32) | reinterpret_cast<uintptr_t>(C) | reinterpret_cast<uintptr_t>(B2_rows32) |
                reinterpret_cast<uintptr_t>(C2)) % 16 == 0 && (reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(bias2)) % 8 == 0,
               LQ_ERR_ARG, "lq_linear_fp8_rows: B and C must be 16-byte aligned, bias 8-byte aligned");
    GemmPair pair = {};
    for (int i = 0; i < (two ? 2 : 1); ++i) {
        GemmParams& p = pair.p[i];
        p.C = i ? C2 : C; p.A = static_cast<const uint8_t*>(x); p.B = i ? B2_rows32 : B_rows32; p.bias = i ? bias2 : bias;
        p.a_scale = i ? a_scale2 : a_scale; p.b_scale = i ? b_scale2 : b_scale;
        p.m = m; p.n = n; p.k = k; p.kb = k;
    }
    const dim3 grid((unsigned)(n / 32), two ? 2 : 1), block(256);
    const int lds = m * (k + 16);
    if (dtype == LQ_BF16) hipLaunchKernelGGL((fp8_rows_cast_kernel<BF16Tag>), grid, block, lds, as_stream(stream), pair);
    else hipLaunchKernelGGL((fp8_rows_cast_kernel<F16Tag>), grid, block, lds, as_stream(stream), pair);
    return check_launch("lq_linear_fp8_rows");
}
