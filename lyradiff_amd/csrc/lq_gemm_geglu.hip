// INT8 up projection of a GEGLU feed-forward with the activation and the next linear's static INT8 codes in its epilogue:
// out[m, c] = q( pre[c] * T( h * gate(g) ) ), h = T(T(y[m, c]) + bias[c]), g = T(T(y[m, inner + c]) + bias[inner + c]),
// y = A . B^T * alpha: lq_gemm_int8 (static scale, no bias) followed by lq_geglu_int8, the same bits, without the [m, 2 * inner] tensor
// between them.  It stands where lyraDiff's BasicTransformerInt8Block calls the GEMM and invokeInt8FusedBiasGeglu
// (layers/basic_transformer/BasicTransformerInt8Block.cc:440-490, kernels/ffn_int8/ffn_kernels_int8.cu:102-147).
//
// What bounds it: with k of 640 or 1280 the plain GEMM is short of work per output: of 41 us at 8192 x 5120 x 640 half is writing
// 84 MB, and the GEGLU pass behind it reads them again (27 us).  Here an output costs some 25 vector instructions instead, about
// as many cycles as its matrix instructions at k = 640.
//   * A wavefront's two 32-column blocks are a value block and the gate block of the same outputs: h and g meet in a lane's registers.
//   * The gate factor comes from the table of lq_quant_int8.hip (60 KB for fp16), which leaves room for one workgroup per CU: eight
//     wavefronts that stay, two per SIMD, and walk over the tiles; the transfers run on across the tiles, NST k-tiles ahead.
//   * Four codes per register quad, two half-wave exchanges per 32 x 32 block, 16 bytes per lane to memory: no LDS on the way out.
#include "lq_gemm_core.h"
#include "lq_gate_table.h"

namespace lq {

struct GegluParams {
    int8_t* out;
    const uint8_t *a, *b;  // codes [m, k] and weights of 2 * inner rows in rows32 layout
    const float *alpha_col, *alpha_row;
    const void* bias;       // T [2 * inner] or null
    const float* pre;       // [inner] or null
    const float* out_scale;
    const unsigned short* table;
    int m, inner, k, tiles_m, tiles_n;
};

template <typename Tag, int MT> struct GegluGemm {
    static constexpr int NW = 8, BM = 4 * 32 * MT, BN = 64, BKB = 64, NST = 4;  // BN outputs: as many value and as many gate rows of B
    static constexpr int A_B = BM * BKB, STAGE_B = A_B + 2 * BN * BKB, PER = MT + 1;
    static constexpr u32 LO = GateTable<Tag>::LO, COUNT = GateTable<Tag>::COUNT;
    static constexpr int ENTRIES_B = 2 * COUNT * 2, TABLE_B = (ENTRIES_B + 1023) / 1024 * 1024;
    // of a tile's columns: alpha of the value rows and of the gate rows, pre (fp32), bias of both (T): a KiB each tile
    static constexpr int PAR_B = 1024, P_GATE = 256, P_PRE = 512, P_BIAS = 768;
    static constexpr int SMEM_BYTES = TABLE_B + NST * STAGE_B + 2 * PAR_B;
    static_assert(ENTRIES_B % 16 == 0 && SMEM_BYTES <= 160 * 1024, "LDS plan");

    static __device__ __forceinline__ void barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

    // codes of eight outputs from their accumulators; params: values of the eight columns
    static __device__ __forceinline__ void outputs(const int* hv, const int* gv, const float* av, const float* ag, const float* pre, const u32* bv,
                                                   const u32* bg, const unsigned short* gate, float s, float r, bool slow, u32* words) {
        float t[8];
        if constexpr (std::is_same<Tag, F16Tag>::value) {
            // sums and products of two fp16 numbers rounded once are what fp32 arithmetic and a second rounding give (24 >= 2 * 11 + 2 bits)
            f16x2_t h[4], g[4], gel[4];
            u32 far = 0;  // largest distance from the table's first entry, both signs, in either half
            typedef unsigned short us2 __attribute__((ext_vector_type(2)));
            us2 worst = {0, 0};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float h0 = (float)hv[2 * i] * av[2 * i], h1 = (float)hv[2 * i + 1] * av[2 * i + 1];
                float g0 = (float)gv[2 * i] * ag[2 * i], g1 = (float)gv[2 * i + 1] * ag[2 * i + 1];
                asm volatile("" : "+v"(h0), "+v"(h1), "+v"(g0), "+v"(g1));  // rounded to fp32 before the conversion
                h[i] = __builtin_bit_cast(f16x2_t, pack2_f16(h0, h1)) + __builtin_bit_cast(f16x2_t, bv[i]);
                g[i] = __builtin_bit_cast(f16x2_t, pack2_f16(g0, g1)) + __builtin_bit_cast(f16x2_t, bg[i]);
                const u32 bits = __builtin_bit_cast(u32, g[i]);
                const us2 off = __builtin_bit_cast(us2, bits & 0x7FFF7FFFu) - (us2){(unsigned short)LO, (unsigned short)LO};
                worst = __builtin_elementwise_max(worst, off);
                const us2 sign = __builtin_bit_cast(us2, (__builtin_bit_cast(u32, __builtin_bit_cast(us2, bits) >> 15)) * COUNT);
                const u32 at = __builtin_bit_cast(u32, __builtin_elementwise_min(off, (us2){(unsigned short)(COUNT - 1), (unsigned short)(COUNT - 1)}) + sign);
                const unsigned short lo = gate[at & 0xFFFFu], hi = gate[at >> 16];
                gel[i] = __builtin_bit_cast(f16x2_t, (u32)lo | ((u32)hi << 16));
            }
            far = worst[0] > worst[1] ? worst[0] : worst[1];
            if (__builtin_expect(far >= COUNT, 0)) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const u32 bits = (__builtin_bit_cast(u32, g[i]) >> (16 * e)) & 0xFFFFu;
                        if ((bits & 0x7FFFu) - LO >= COUNT) gel[i][e] = (_Float16)gate_outside_table<Tag>((float)g[i][e]);
                    }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const f16x2_t p = h[i] * gel[i];
                t[2 * i] = (float)p[0] * pre[2 * i];
                t[2 * i + 1] = (float)p[1] * pre[2 * i + 1];
            }
        } else {
            float gel[8], h[8];
            u32 gb[8], far = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float h0 = (float)hv[2 * i] * av[2 * i], h1 = (float)hv[2 * i + 1] * av[2 * i + 1];
                float g0 = (float)gv[2 * i] * ag[2 * i], g1 = (float)gv[2 * i + 1] * ag[2 * i + 1];
                round_through2<Tag>(h0, h1);
                round_through2<Tag>(g0, g1);
                h0 += __uint_as_float(bv[i] << 16);
                h1 += __uint_as_float(bv[i] & 0xFFFF0000u);
                round_through2<Tag>(h0, h1);
                h[2 * i] = h0;
                h[2 * i + 1] = h1;
                g0 += __uint_as_float(bg[i] << 16);
                g1 += __uint_as_float(bg[i] & 0xFFFF0000u);
                asm volatile("" : "+v"(g0), "+v"(g1));
                const u32 w = pack2_bf16(g0, g1);
                gb[2 * i] = w & 0xFFFFu;
                gb[2 * i + 1] = w >> 16;
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32 off = (gb[i] & 0x7FFFu) - LO;
                far = max(far, off);
                gel[i] = Elem<Tag>::load(gate[min(off, COUNT - 1) + (gb[i] >> 15) * COUNT]);
            }
            if (__builtin_expect(far >= COUNT, 0)) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if ((gb[i] & 0x7FFFu) - LO >= COUNT) gel[i] = gate_outside_table<Tag>(Elem<Tag>::load(gb[i]));
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float p0 = h[2 * i] * gel[2 * i], p1 = h[2 * i + 1] * gel[2 * i + 1];
                round_through2<Tag>(p0, p1);
                t[2 * i] = p0 * pre[2 * i];
                t[2 * i + 1] = p1 * pre[2 * i + 1];
            }
        }
        int q[8];
        quant8<-128, 127>(t, s, r, slow, q);
        words[0] = pack4_s8(q[0], q[1], q[2], q[3]);
        words[1] = pack4_s8(q[4], q[5], q[6], q[7]);
    }

    static __device__ __forceinline__ void run(const GegluParams& p, char* smem) {
        const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave >> 1, wn = wave & 1;
        const u32 smem_base = (u32)(uintptr_t)(__attribute__((address_space(3))) char*)smem;
        const int total = p.tiles_m * p.tiles_n, ktiles = p.k / BKB;
        const size_t block_stride = (size_t)(p.k / 16) * 512;
        char* const stages = smem + TABLE_B;
        char* const params = stages + NST * STAGE_B;

        // ---- transfers: steps (tile, k-tile) in the order in which they are used, `it` is the next one to request ----
        struct {
            const uint8_t *a, *b;
            u32 a_voff[MT];
            int tile, kt, stage, parity;
        } it;
        it.tile = (int)blockIdx.x;
        it.kt = it.stage = it.parity = 0;
        const int b_block = wave >> 1, b_half = wave & 1;  // LDS block order: value and gate block of the wavefronts wn = 0, then wn = 1
        auto request_tile = [&] {
            int tm, tn;
            tile_coords<(MT == 2 ? 4 : 8)>(it.tile, p.tiles_m, p.tiles_n, tm, tn);
            const int m0 = tm * BM, c0 = tn * BN, row_last = p.m - 1 - m0;
            it.a = p.a + (size_t)m0 * p.k;
            it.b = p.b + (size_t)(c0 / 32 + (b_block >> 1) + (b_block & 1) * (p.inner / 32)) * block_stride + b_half * 1024;
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int slot = (wave * MT + i) * 64 + lane, row = slot / 4, c = (slot % 4) ^ chunk_swizzle<4>(row);
                it.a_voff[i] = (u32)min(row, row_last) * (u32)p.k + c * 16;
            }
            const u32 dst = smem_base + TABLE_B + NST * STAGE_B + it.parity * PAR_B;
            if (wave < 2) dma4(p.alpha_col + c0 + (wave ? p.inner : 0), lane * 4, dst + wave * P_GATE);
            else if (wave == 2) { if (p.pre != nullptr) dma4(p.pre + c0, lane * 4, dst + P_PRE); }
            else if (wave == 3) { if (p.bias != nullptr) dma4(static_cast<const unsigned short*>(p.bias) + c0, (lane & 31) * 4 + (lane >> 5) * (u32)p.inner * 2, dst + P_BIAS); }
        };
        auto request_step = [&] {
            if (it.kt == 0) request_tile();
            const u32 sa = smem_base + TABLE_B + it.stage * STAGE_B;
#pragma unroll
            for (int i = 0; i < MT; ++i) dma16(it.a + it.kt * BKB, it.a_voff[i], sa + (wave * MT + i) * 1024);
            dma16(it.b + (size_t)it.kt * 2048, lane * 16, sa + A_B + wave * 1024);
            it.stage = it.stage + 1 == NST ? 0 : it.stage + 1;
            if (++it.kt == ktiles) {  // past the last tile: that tile again, into places nobody reads any more
                it.kt = 0;
                it.parity ^= 1;
                if (it.tile + (int)gridDim.x < total) it.tile += (int)gridDim.x;
            }
        };
#pragma unroll
        for (int s = 0; s < NST; ++s) request_step();
        for (int c = wave; c < TABLE_B / 1024; c += NW) dma16(p.table, min(c * 1024 + lane * 16, ENTRIES_B - 16), smem_base + c * 1024);
        if (tid < 128) {  // absent vectors, in both places of the parameters: a factor of 1, a sum with -0
            char* par = params + (tid >> 6) * PAR_B;
            if (p.pre == nullptr) reinterpret_cast<float*>(par + P_PRE)[tid & 63] = 1.0f;
            if (p.bias == nullptr) reinterpret_cast<u32*>(par + P_BIAS)[tid & 63] = 0x80008000u;
        }

        const float arow = p.alpha_row[0], s = p.out_scale[0], r = 1.0f / s;
        const bool slow = recip_unsafe(s, r);
        const int xrow = wm * (32 * MT) + lr, xsw = chunk_swizzle<4>(xrow);
        const int w_off = A_B + wn * 4096 + lane * 16;
        v4i wf[2][2], xf[2][MT];  // operands of k-step 0 and 1 of a k-tile
        auto load_w = [&](const char* st, int ks, int j) { wf[ks][j] = *reinterpret_cast<const v4i*>(st + w_off + j * 2048 + ks * 1024); };
        auto load_x = [&](const char* st, int ks, int i) { xf[ks][i] = *reinterpret_cast<const v4i*>(st + (xrow + i * 32) * BKB + (((2 * ks + lh) ^ xsw) << 4)); };
        v16i acc[MT][2];
        // the matrix instructions of k-step ks beside the operand reads of the step behind it
        auto half_step = [&](int ks, const char* next) {
#pragma unroll
            for (int x = 0; x < 2 * MT; ++x) {
                if (x == 0) { load_x(next, ks ^ 1, 0); load_w(next, ks ^ 1, 0); }
                else if (x == 1) load_w(next, ks ^ 1, 1);
                else if (x == 2 && MT == 2) load_x(next, ks ^ 1, 1);
                acc[x >> 1][x & 1] = __builtin_amdgcn_mfma_i32_32x32x32_i8(wf[ks][x & 1], xf[ks][x >> 1], acc[x >> 1][x & 1], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        wait_vmcnt<0>();
        barrier();
        load_x(stages, 0, 0);
        load_w(stages, 0, 0);
        load_w(stages, 0, 1);
        if constexpr (MT == 2) load_x(stages, 0, 1);
        int stage = 0, parity = 0;
        for (int tile = (int)blockIdx.x; tile < total; tile += (int)gridDim.x, parity ^= 1) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int v = 0; v < 16; ++v) acc[i][j][v] = 0;
            for (int kt = 0; kt < ktiles; ++kt) {
                half_step(0, stages + stage * STAGE_B);
                stage = stage + 1 == NST ? 0 : stage + 1;
                // this wavefront's share of the next k-tile; what else was requested behind it (columns' values, stores) only adds to the count
                wait_vmcnt<PER*(NST - 2)>();
                barrier();        // the next k-tile is complete, and everybody has read this one
                request_step();   // into the place of this one
                __builtin_amdgcn_sched_barrier(0);
                half_step(1, stages + stage * STAGE_B);
            }
            // ---- epilogue: lane: row lr of a block, columns q4 * 8 + lh * 4 + (0..3) ----
            int tm, tn;
            tile_coords<(MT == 2 ? 4 : 8)>(tile, p.tiles_m, p.tiles_n, tm, tn);
            const char* par = params + parity * PAR_B;
            u32 words[MT][4];
#pragma unroll
            for (int qq = 0; qq < 2; ++qq) {
                float av[8], ag[8], pre[8];
                u32 bv[4], bg[4];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int c = wn * 32 + (2 * qq + u) * 8 + lh * 4;
                    const float4 v = *reinterpret_cast<const float4*>(par + c * 4), g = *reinterpret_cast<const float4*>(par + P_GATE + c * 4);
                    const float4 f = *reinterpret_cast<const float4*>(par + P_PRE + c * 4);
                    const uint2 x = *reinterpret_cast<const uint2*>(par + P_BIAS + c * 2), y = *reinterpret_cast<const uint2*>(par + P_BIAS + 128 + c * 2);
                    av[4 * u] = v.x * arow; av[4 * u + 1] = v.y * arow; av[4 * u + 2] = v.z * arow; av[4 * u + 3] = v.w * arow;
                    ag[4 * u] = g.x * arow; ag[4 * u + 1] = g.y * arow; ag[4 * u + 2] = g.z * arow; ag[4 * u + 3] = g.w * arow;
                    pre[4 * u] = f.x; pre[4 * u + 1] = f.y; pre[4 * u + 2] = f.z; pre[4 * u + 3] = f.w;
                    bv[2 * u] = x.x; bv[2 * u + 1] = x.y; bg[2 * u] = y.x; bg[2 * u + 1] = y.y;
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    int hv[8], gv[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) { hv[e] = acc[i][0][qq * 8 + e]; gv[e] = acc[i][1][qq * 8 + e]; }
                    outputs(hv, gv, av, ag, pre, bv, bg, reinterpret_cast<const unsigned short*>(smem), s, r, slow, &words[i][2 * qq]);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const int row = tm * BM + wm * (32 * MT) + i * 32 + lr;
                const auto x = __builtin_amdgcn_permlane32_swap(words[i][0], words[i][2], false, false);  // columns 0..7 | 16..23
                const auto y = __builtin_amdgcn_permlane32_swap(words[i][1], words[i][3], false, false);  // columns 8..15 | 24..31
                if (row < p.m) *reinterpret_cast<uint4*>(p.out + (size_t)row * p.inner + tn * BN + wn * 32 + lh * 16) = make_uint4(x[0], x[1], y[0], y[1]);
            }
        }
        wait_vmcnt<0>();
    }
};

template <typename Tag, int MT> __global__ __launch_bounds__(512, 2) void gemm_geglu_kernel(GegluParams p) {
    extern __shared__ __attribute__((aligned(16))) char lq_smem[];
    GegluGemm<Tag, MT>::run(p, lq_smem);
}

template <typename Tag, int MT> static int launch_geglu_gemm(GegluParams p, hipStream_t st) {
    using G = GegluGemm<Tag, MT>;
    p.tiles_m = (p.m + G::BM - 1) / G::BM;
    p.tiles_n = p.inner / G::BN;
    const int total = p.tiles_m * p.tiles_n, cus = device_cu_count();
    static bool attr_done = false;
    return launch_with_lds(gemm_geglu_kernel<Tag, MT>, p, (unsigned)(total < cus ? total : cus), 512u, G::SMEM_BYTES, attr_done, st);
}

template <typename Tag> static int geglu_gemm_typed(GegluParams p, hipStream_t st) {
    if (int rc = gate_table_on_device(std::is_same<Tag, F16Tag>::value, st, &p.table); rc != LQ_OK) return rc;
    // 256 rows per tile as soon as they make a tile for most CUs
    const long big = (long)((p.m + 255) / 256) * (p.inner / 64);
    return big * 4 >= 3L * device_cu_count() ? launch_geglu_gemm<Tag, 2>(p, st) : launch_geglu_gemm<Tag, 1>(p, st);
}

}  // namespace lq

using namespace lq;

extern "C" int lq_gemm_int8_geglu_takes(int m, int inner, int k) {
    return m >= 0 && inner > 0 && inner % 64 == 0 && inner < (1 << 29) && k >= 256 && k % 64 == 0 &&
           requested_tactic(g_tactic_int8, LQ_W_INT8, m, 2 * inner, k) < 0;  // tactics stand
}

extern "C" int lq_gemm_int8_geglu(int8_t* out, const int8_t* A, const int8_t* B_rows32, const float* alpha_col, const float* alpha_row, const void* bias,
                                  lq_dtype_t dtype, const float* pre_quant_scale, const float* input_quant_scale, int m, int inner, int k,
                                  lq_stream_t stream) {
    LQ_REQUIRE(out && A && B_rows32 && alpha_col && alpha_row && input_quant_scale, LQ_ERR_ARG, "lq_gemm_int8_geglu: null pointer");
    LQ_REQUIRE(dtype == LQ_F16 || dtype == LQ_BF16, LQ_ERR_UNSUPPORTED, "lq_gemm_int8_geglu: the rounded values in between must be F16 or BF16");
    LQ_REQUIRE(m >= 0 && inner > 0 && inner % 64 == 0 && k >= 256 && k % 64 == 0, LQ_ERR_SHAPE,
               "lq_gemm_int8_geglu: need inner %% 64 == 0, k %% 64 == 0 and k >= 256 (m=%d inner=%d k=%d)", m, inner, k);
    // a lane's offset inside a tile's rows, and the tile count, are 32 bits
    LQ_REQUIRE((long long)k * 256 < 0x7fffffffLL && ((long long)m + 127) / 128 * (inner / 64) < 0x3fffffffLL && inner < (1 << 29), LQ_ERR_SHAPE,
               "lq_gemm_int8_geglu: problem too large (m=%d inner=%d k=%d)", m, inner, k);
    LQ_REQUIRE((reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(B_rows32) | reinterpret_cast<uintptr_t>(out)) % 16 == 0 &&
                   (reinterpret_cast<uintptr_t>(alpha_col) | reinterpret_cast<uintptr_t>(pre_quant_scale) | reinterpret_cast<uintptr_t>(bias)) % 4 == 0,
               LQ_ERR_ARG, "lq_gemm_int8_geglu: A, B and out must be 16-byte aligned, scales and bias 4-byte");
    if (m == 0) return LQ_OK;
    GegluParams p = {};
    p.out = out; p.a = reinterpret_cast<const uint8_t*>(A); p.b = reinterpret_cast<const uint8_t*>(B_rows32);
    p.alpha_col = alpha_col; p.alpha_row = alpha_row; p.bias = bias; p.pre = pre_quant_scale; p.out_scale = input_quant_scale;
    p.m = m; p.inner = inner; p.k = k;
    return dtype == LQ_F16 ? geglu_gemm_typed<F16Tag>(p, as_stream(stream)) : geglu_gemm_typed<BF16Tag>(p, as_stream(stream));
}
