// FP8 GEMM of at most 32 rows with scales and bias (the modulation linears of the FLUX blocks: one row, 57 MB of weights): a pass
// over the weights.
//
// What bounds it: the weights' way from memory.  The tiled forms bring them to LDS through a few stages per wavefront group, each
// with as many bytes of (repeated) activation rows, so that a workgroup has 16 KiB of weights on their way; here a wavefront
// requests both operands straight into registers -- a 32-row by 64-byte piece of the rows32 layout is two lane-linear kilobytes,
// already the matrix instruction's operand -- DEPTH k-tiles ahead, with neither a barrier nor an LDS round trip in the loop.
// Measured (us, bf16, replayed back to back, the tiled form -> this one): 1x18432x3072 13.9 -> 10.3 (5.5 TB/s), 1x9216x3072 6.2 -> 4.7,
// 1x3072x3072 4.8 -> 3.4, 1x3072x12288 12.8 -> 7.7, 8x12288x3072 9.4 -> 6.9, 32x18432x3072 15.1 -> 11.3, 32x9216x3072 6.6 -> 6.4.
// The order of the sums is that of the tiled forms with four k-groups (SMALL_32x32_K4, SMALL_32x64_K4): group g adds the k-tiles g,
// g + 4, ... and the four sums are added in group order, so every result has the same bits whichever form computes it.
#include "lq_gemm_core.h"

namespace lq {

template <typename OutTag> __global__ __launch_bounds__(256, 2) void fp8_rows_kernel(GemmParams p) {
    constexpr int KW = 4, DEPTH = 6;
    __shared__ float4 part[KW * 4 * 64];
    const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
    const int kg = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rounds = p.kb / (64 * KW);  // k-tiles of this group; kb is a multiple of 256
    // k-tile t of the 32 weight rows: 2 KiB at 2048 t, chunk c of row r at 512 c + 16 r; this lane takes the chunks lh and 2 + lh.
    const uint8_t* wb = p.B + (size_t)blockIdx.x * 32 * (size_t)p.kb + (size_t)kg * 2048 + lane * 16;
    const int row = min(lr, p.m - 1);  // the columns of the result past the last row are not stored
    const uint8_t* xb = p.a_panel ? p.A + ((size_t)kg * p.m + row) * 64 + lh * 16 : p.A + (size_t)row * p.kb + kg * 64 + lh * 16;
    const u32 xstep = (p.a_panel ? (u32)p.m * 64u : 64u) * KW;
    v4i w[DEPTH][2], x[DEPTH][2];
    auto load = [&](int d, int t) {
        const uint8_t* wp = wb + (size_t)t * (2048 * KW);
        const uint8_t* xp = xb + (size_t)t * xstep;
        w[d][0] = *reinterpret_cast<const v4i*>(wp);
        w[d][1] = *reinterpret_cast<const v4i*>(wp + 1024);
        x[d][0] = *reinterpret_cast<const v4i*>(xp);
        x[d][1] = *reinterpret_cast<const v4i*>(xp + 32);
    };
    v16f acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    auto step = [&](int d) {
        const v8i a = __builtin_shufflevector(w[d][0], w[d][1], 0, 1, 2, 3, 4, 5, 6, 7);
        const v8i b = __builtin_shufflevector(x[d][0], x[d][1], 0, 1, 2, 3, 4, 5, 6, 7);
        acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, b, acc, 0, 0, 0, 0, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(d, min(d, rounds - 1));
    __builtin_amdgcn_sched_barrier(0);
    int t = 0;
    for (; t + DEPTH < rounds; t += DEPTH) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) {
            step(d);
            load(d, min(t + DEPTH + d, rounds - 1));
            __builtin_amdgcn_sched_barrier(0);
        }
    }
#pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (t + d < rounds) step(d);

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

bool fp8_rows_takes(const GemmParams& p) {
    return p.m <= 32 && p.kb % 256 == 0 && p.C != nullptr && p.gelu == 0 && p.out_scale == nullptr && p.out_max == nullptr && p.C8 == nullptr &&
           p.gate == nullptr && p.residual == nullptr && p.addend == nullptr;
}

int run_fp8_rows(const GemmParams& p, lq_dtype_t out_dtype, hipStream_t st) {
    const dim3 grid((unsigned)(p.n / 32)), block(256);
    if (out_dtype == LQ_BF16) hipLaunchKernelGGL((fp8_rows_kernel<BF16Tag>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((fp8_rows_kernel<F16Tag>), grid, block, 0, st, p);
    return check_launch("fp8_rows");
}

}  // namespace lq
