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
