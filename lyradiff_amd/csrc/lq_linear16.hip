// 16-bit linears of few rows, y = x . W^T + bias with fp32 sums: the adaLN modulation of the FLUX blocks whose level keeps it in 16 bits
// (1 x 9216 x 3072 and 1 x 18432 x 3072: the weight's way from memory) and the key and value projections of SDXL's text states
// (154 x 640 x 2048, two of them: latency).  They are plain linears of the models (AdaLayerNorm.cc, BasicTransformerInt8Block.cc), one
// launch and 20 us or 2 x 10 us each in the vendor's library.
//
// One row (linear16_gemv_kernel): a stream of weights, each wavefront four rows of them, a kilobyte of a row per request, with
// three requests per row in flight; vector arithmetic, 64 partial sums per output added in one tree.  Two to four rows in that form are behind
// the other one (us from memory, this form / the other: 4x640x640 4.9 / 3.6, 4x9216x3072 17.1 / 16.0, 4x18432x3072 25.6 / 24.2).
// More rows (linear16_kernel): a workgroup of eight wavefronts owns 32 x 32 outputs and shares k out; wavefront g takes the 64-element pieces
// g, g + 8, ... of both operands.  Eight neighbouring lanes fetch one 128-byte line of a row (lanes that fetch 16 bytes of 32 rows each, the
// matrix operand's own order, make four times the requests: 154x1280x2048 twice: 23.6 us in that form, 9.6 now, the host's time for the call), and the piece reaches operand order through an LDS block
// of the wavefront's own: no barrier in the loop.  The eight partial sums meet in LDS and are added in wavefront order.
// us, library -> this: 1x9216x3072 21.6 -> 13.6 from memory (4.2 TB/s), 21.5 -> 11.4 cached; 1x18432x3072 66.8 -> 21.6 (5.2 TB/s);
// 2 x 154x640x2048 21 -> 9.6 (host time of the call)
#include "lq_common.h"

namespace lq {

struct Linear16Params {
    unsigned short* y[2];        // [m, n] of up to two linears with one input
    const unsigned short* w[2];  // [n, k]
    const unsigned short* bias[2];
    const unsigned short* x;     // [m, k]
    int m, n, k;
};

typedef __bf16 l16_bf8 __attribute__((ext_vector_type(8)));
typedef _Float16 l16_h8 __attribute__((ext_vector_type(8)));

constexpr int kGemvRows = 4;  // weight rows per wavefront

template <typename Tag> __global__ __launch_bounds__(256) void linear16_gemv_kernel(Linear16Params p) {
    constexpr int R = kGemvRows, U = 3;
    const int lane = threadIdx.x & 63, which = blockIdx.z;
    const int n0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + (threadIdx.x >> 6)) * R);
    if (n0 >= p.n) return;  // n is a multiple of R
    const unsigned short* w = p.w[which] + (size_t)n0 * p.k;
    float sum[R];
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] = 0.0f;
    for (int k0 = lane * 8; k0 < p.k; k0 += 512 * U) {
        uint4 wv[U][R], xv[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = k0 + 512 * u;
#pragma unroll
            for (int r = 0; r < R; ++r) wv[u][r] = at < p.k ? *reinterpret_cast<const uint4*>(w + (size_t)r * p.k + at) : make_uint4(0, 0, 0, 0);
            xv[u] = at < p.k ? *reinterpret_cast<const uint4*>(p.x + at) : make_uint4(0, 0, 0, 0);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float xf[8];
            unpack8<Tag>(xv[u], xf);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                float wf[8];
                unpack8<Tag>(wv[u][r], wf);
#pragma unroll
                for (int e = 0; e < 8; ++e) sum[r] = __builtin_fmaf(wf[e], xf[e], sum[r]);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r)
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) sum[r] += __shfl_xor(sum[r], off, 64);
    if (lane != 0) return;
    uint2 b = make_uint2(0, 0);
    const bool has_bias = p.bias[which] != nullptr;
    if (has_bias) b = *reinterpret_cast<const uint2*>(p.bias[which] + n0);
    const u32 bw[4] = {b.x & 0xFFFFu, b.x >> 16, b.y & 0xFFFFu, b.y >> 16};
    u32 o[4];
#pragma unroll
    for (int r = 0; r < R; ++r) o[r] = Elem<Tag>::store(has_bias ? sum[r] + Elem<Tag>::load(bw[r]) : sum[r]);
    *reinterpret_cast<uint2*>(p.y[which] + n0) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
}

template <typename Tag> __global__ __launch_bounds__(512, 2) void linear16_kernel(Linear16Params p) {
    constexpr int KW = 8, DEPTH = 2;
    __shared__ __attribute__((aligned(16))) char smem[KW * 8192];  // per wavefront: 32 rows x 128 bytes of w, then of x; later the partial sums
    const int lane = threadIdx.x & 63, lr = lane & 31, lh = lane >> 5;
    const int g = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int n0 = blockIdx.x * 32, m0 = blockIdx.y * 32, which = blockIdx.z;
    const int pieces = p.k / 64, mine = (pieces - g + KW - 1) / KW;  // of this wavefront (none when g >= pieces)
    // request i of a piece: rows 8 i + lane / 8, chunk lane % 8; rows past the last repeat it, their results are not stored
    const unsigned short* wp[4];
    const unsigned short* xp[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 8 * i + (lane >> 3), c = g * 64 + (lane & 7) * 8;
        wp[i] = p.w[which] + (size_t)min(n0 + r, p.n - 1) * p.k + c;
        xp[i] = p.x + (size_t)min(m0 + r, p.m - 1) * p.k + c;
    }
    char* block = smem + g * 8192;
    v4i w[DEPTH][4], x[DEPTH][4];
    auto load = [&](int d, int t) {
        const int at = min(t, mine - 1) * (64 * KW);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            w[d][i] = *reinterpret_cast<const v4i*>(wp[i] + at);
            x[d][i] = *reinterpret_cast<const v4i*>(xp[i] + at);
        }
    };
    v16f acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
    // chunk c of row r sits at slot c ^ (r & 7): eight lanes write a row's 128 bytes, the reads take one chunk of 32 rows, both over all banks
    auto step = [&](int d) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int r = 8 * i + (lane >> 3), at = r * 128 + (((lane & 7) ^ (r & 7)) << 4);
            *reinterpret_cast<v4i*>(block + at) = w[d][i];
            *reinterpret_cast<v4i*>(block + 4096 + at) = x[d][i];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // a wavefront's LDS accesses complete in order: this binds the compiler
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int at = lr * 128 + (((2 * s + lh) ^ (lr & 7)) << 4);
            const v4i a = *reinterpret_cast<const v4i*>(block + at), b = *reinterpret_cast<const v4i*>(block + 4096 + at);
            if constexpr (std::is_same<Tag, BF16Tag>::value)
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(l16_bf8, a), __builtin_bit_cast(l16_bf8, b), acc, 0, 0, 0);
            else
                acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(l16_h8, a), __builtin_bit_cast(l16_h8, b), acc, 0, 0, 0);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    if (mine > 0) {
#pragma unroll
        for (int d = 0; d < DEPTH; ++d) load(d, d);
        int t = 0;
        for (; t + DEPTH < mine; t += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; ++d) {
                step(d);
                load(d, t + DEPTH + d);
            }
        }
#pragma unroll
        for (int d = 0; d < DEPTH; ++d)
            if (t + d < mine) step(d);
    }
    __syncthreads();  // the sums below take the place of the blocks

    // a lane holds, of column m0 + lr of the result, four consecutive outputs per quad of registers
    float4* part = reinterpret_cast<float4*>(smem);
#pragma unroll
    for (int q = 0; q < 4; ++q) part[(g * 4 + q) * 64 + lane] = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
    __syncthreads();
    if (g >= 4) return;
    float y[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < KW; ++i) {
        const float4 v = part[(i * 4 + g) * 64 + lane];
        y[0] += v.x; y[1] += v.y; y[2] += v.z; y[3] += v.w;
    }
    const int row = m0 + lr, col = n0 + g * 8 + lh * 4;
    if (row >= p.m || col >= p.n) return;
    if (p.bias[which] != nullptr) {
        const uint2 b = *reinterpret_cast<const uint2*>(p.bias[which] + col);
        y[0] += Elem<Tag>::load(b.x & 0xFFFFu); y[1] += Elem<Tag>::load(b.x >> 16);
        y[2] += Elem<Tag>::load(b.y & 0xFFFFu); y[3] += Elem<Tag>::load(b.y >> 16);
    }
    *reinterpret_cast<uint2*>(p.y[which] + (size_t)row * p.n + col) =
        make_uint2(Elem<Tag>::store(y[0]) | (Elem<Tag>::store(y[1]) << 16), Elem<Tag>::store(y[2]) | (Elem<Tag>::store(y[3]) << 16));
}

}  // namespace lq

using namespace lq;

// Every 32 rows stream the weight again, and a workgroup's eight wavefronts share one k: large weights are the library's from 17 rows up, and
// long sums, too, where its split of k has more workgroups (us from memory, library / this): 16x9216x3072 20.5 / 17.1, 32x 17.3 / 19.6,
// 128x 25.0 / 36.2; 16x18432x3072 63.9 / 25.7, 32x 29.7 / 29.1, 64x 33.9 / 39.3; 128x10240x1280 17.2 / 17.6; 16x4096x4096 15.8 / 13.2, 32x
// 13.7 / 14.3.  Smaller weights: 256x5120x1280 18.7 / 15.0, 256x3840x1280 13.9 / 12.0, 256x1280x1280 7.2 / 6.9, 256x640x640 6.3 / 4.1,
// 154x1280x2048 twice 20.4 / 9.7.  16x1280x5120 10.1 / 14.5, 8x3072x12288 19.1 / 27.0.  One row: 640x640 6.4 / 3.2, 18432x3072 67 / 22, 3072x12288
// 20.3 / 19.9, 3072x15360 22.8 / 23.7.
extern "C" int lq_linear16_rows_takes(int m, int n, int k) {
    if (m <= 0 || n <= 0 || k <= 0 || n % 4 != 0 || k % 64 != 0) return 0;
    return (m == 1 && k <= 12288) || (m <= 256 && k <= 4096 && (m <= 16 || (long)n * k <= (1L << 23)));
}

extern "C" int lq_linear16_rows(void* y, void* y2, const void* x, const void* w, const void* w2, const void* bias, const void* bias2,
                                lq_dtype_t dtype, int m, int n, int k, lq_stream_t stream) {
    LQ_REQUIRE(dtype == LQ_F16 || dtype == LQ_BF16, LQ_ERR_UNSUPPORTED, "lq_linear16_rows: dtype must be F16 or BF16");
    LQ_REQUIRE(m >= 0 && n > 0 && k > 0 && n % 4 == 0 && k % 64 == 0, LQ_ERR_SHAPE, "lq_linear16_rows: need n %% 4 == 0 and k %% 64 == 0 (m=%d n=%d k=%d)", m,
               n, k);
    if (m == 0) return LQ_OK;
    LQ_REQUIRE(y && x && w && (y2 == nullptr) == (w2 == nullptr) && (y2 != nullptr || bias2 == nullptr), LQ_ERR_ARG, "lq_linear16_rows: null pointer");
    LQ_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(w2)) % 16 == 0 &&
                   (reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(y2) | reinterpret_cast<uintptr_t>(bias) | reinterpret_cast<uintptr_t>(bias2)) % 8 == 0,
               LQ_ERR_ARG, "lq_linear16_rows: x and w must be 16-byte aligned, y and bias 8-byte aligned");
    const long m_tiles = ((long)m + 31) / 32, n_tiles = ((long)n + 31) / 32;
    LQ_REQUIRE(m_tiles <= 65535, LQ_ERR_SHAPE, "lq_linear16_rows: too many rows (%d)", m);
    auto us = [](const void* v) { return static_cast<const unsigned short*>(v); };
    Linear16Params p = {{static_cast<unsigned short*>(y), static_cast<unsigned short*>(y2)}, {us(w), us(w2)}, {us(bias), us(bias2)}, us(x), m, n, k};
    const unsigned both = y2 != nullptr ? 2 : 1;
    hipStream_t st = as_stream(stream);
    if (m == 1) {
        const dim3 grid((unsigned)((n / kGemvRows + 3) / 4), 1, both), block(256);
        if (dtype == LQ_BF16) hipLaunchKernelGGL((linear16_gemv_kernel<BF16Tag>), grid, block, 0, st, p);
        else hipLaunchKernelGGL((linear16_gemv_kernel<F16Tag>), grid, block, 0, st, p);
        return check_launch("lq_linear16_rows");
    }
    const dim3 grid((unsigned)n_tiles, (unsigned)m_tiles, both), block(512);
    if (dtype == LQ_BF16) hipLaunchKernelGGL((linear16_kernel<BF16Tag>), grid, block, 0, st, p);
    else hipLaunchKernelGGL((linear16_kernel<F16Tag>), grid, block, 0, st, p);
    return check_launch("lq_linear16_rows");
}
