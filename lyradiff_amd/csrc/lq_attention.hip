// Softmax attention of the transformer blocks (no mask, no dropout): O = softmax(scale * Q K^T) V per batch and head, 16-bit
// operands, fp32 scores, probabilities, maxima, sums and accumulators; for the second product alone the probabilities are rounded to
// T.  It stands where lyraDiff's attention processors call their flash attention
// (layers/flux_attention_processor/FluxAttentionFP8Processor.cc:246-291, layers/basic_transformer/BasicTransformerInt8Block.cc:
// 330-420), between the q/k normalisation + rotary kernel and the output projection.
//
// What bounds it: per 64 keys a wavefront of 32 queries issues 32 matrix instructions (head dimension 128, 1024 cycles) and
// about 200 vector instructions, and a wavefront alone issues one instruction every 5-6 cycles (measured: a matrix instruction
// and 5 vector ones fit 34 cycles, 8 need 47), so the two kinds of work have to come from different wavefronts of a SIMD, and
// on real data the power limit sets the clock (1.88 GHz at 1.0 PFLOP/s against 2.39 GHz on zeros).
//   * Scores are computed transposed, S^T = K Q^T (keys are the rows of the 32x32 result): a lane then holds 16 keys of ONE
//     query per 32x32 block, so the row maximum and sum are per-lane arithmetic plus one exchange between the two half-waves,
//     and the probabilities already are the second product's operand (O^T = V^T P^T) when the sum over keys runs in the
//     order in which the lanes hold them.  V^T comes from row-major V tiles through the transposing LDS read.
//   * K and V tiles of 64 keys travel global -> LDS without registers; the 16-byte chunks of a row are XOR-swizzled on the
//     way so that both kinds of read are conflict free.
//   * Two forms.  NW == 8 (head dimension 128, enough queries to fill the chip): the wavefronts 0-3 and 4-7, one of each per
//     SIMD, alternate between a matrix phase (PV of a tile, QK of the next) and a vector phase (softmax), kept half a tile
//     apart by the workgroup barriers; left to themselves two wavefronts of a SIMD drift into step and both pipes idle half the
//     time.  NW == 4: two or more workgroups per CU run freely, one barrier per tile; a head dimension of 64 leaves registers
//     for three wavefronts per SIMD, which cover for each other without phases.
//   * Vector instructions are counted: beside a matrix wavefront that keeps its pipe full each takes 6.7 cycles (5.0 alone), an exponential
//     11.8 (9.0), so the row maximum is v_maximum3 (fmaxf quietens its operands first), m * c is formed when m changes, and V lies below K in
//     LDS, where its reads need no address arithmetic beyond their offsets: 243 vector instructions per tile of 64 keys, 270 without these.
// Measured (settled, random operands, bf16; in parentheses before the last paragraph's changes, same run, then the library attention):
// 24 heads of 128, 4608 tokens 257 us = 1.0 PFLOP/s (264; 506), 6912 tokens 576 us (596; 908), 1600 tokens 44.7 us (45.9; 135), 1000 tokens
// 23.7 us (24.2); 2 x 10 heads of 64, 4096 tokens 122.7 us (125.5; 190).  NW == 4 at 24 x 4608 tokens of 128: 299 us; NW == 8 at 64: 147 us.
// Error against 64 bits, 2-norm, standard normal operands, 24 heads of 128: bf16 2.22e-3 at 1000 tokens, 2.27e-3 at 4608 (the library
// attention too), 2.29e-3 at 6912; f16 2.7e-4 to 2.9e-4.  The row sum is that of the fp32 probabilities, which takes as long as one of the rounded ones.
// What was measured and is not here (4608 tokens, beside 257 us): a rescaled output only where the maximum grew by more than 2^8, 239 us, but a
// fifth more error, since the largest probabilities are then rounded; softmax and matrix instructions mixed in one wavefront's stream, 286.
#include "lq_common.h"

namespace lq {

int device_cu_count();  // lq_gemm_persist.hip

struct AttnParams {
    const unsigned short *q, *k, *v;
    unsigned short* out;                // [batch, sq, heads, DH]
    size_t q_row, k_row, v_row;         // elements between two tokens
    size_t q_batch, k_batch, v_batch;   // elements between two batches; heads are DH elements apart
    int batch, heads, sq, sk;
    int q_blocks;                       // ceil(sq / (32 * NW))
    float scale_log2;                   // softmax scale * log2(e)
    int context;                        // leading tokens of a batch that have codes of their own (text tokens)
    // codes in place of `out`: e4m3 as k-panels [heads * DH / 64][rows][64], the context's rows into a tensor of their own; or int8 rows
    uint8_t *fp8, *fp8_context;
    const float *fp8_scale, *fp8_context_scale;
    int8_t* int8;
    const float *int8_pre, *int8_scale;
};

typedef __bf16 attn_bf8 __attribute__((ext_vector_type(8)));
typedef _Float16 attn_h8 __attribute__((ext_vector_type(8)));
typedef short attn_s4 __attribute__((ext_vector_type(4)));
typedef short attn_s8 __attribute__((ext_vector_type(8)));

template <typename Tag> __device__ __forceinline__ v16f attn_mfma(attn_s8 a, attn_s8 b, v16f c) {
    if constexpr (std::is_same<Tag, BF16Tag>::value)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(attn_bf8, a), __builtin_bit_cast(attn_bf8, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(attn_h8, a), __builtin_bit_cast(attn_h8, b), c, 0, 0, 0);
}
template <typename Tag> __device__ __forceinline__ u32 attn_pack(float a, float b) {
    if constexpr (std::is_same<Tag, BF16Tag>::value) return pack2_bf16(a, b);
    else return pack2_f16(a, b);
}
// v_maximum3.  NaN where an operand is one: a row with such a score is NaN throughout, whatever its maximum.
__device__ __forceinline__ float attn_max(float a, float b, float c) {
    return __builtin_elementwise_maximum(__builtin_elementwise_maximum(a, b), c);
}
// 16 bytes per lane from global memory to LDS byte address lds_addr + 16 * lane, awaited with attn_wait_vmcnt
__device__ __forceinline__ void attn_dma16(const void* gbase, u32 voff, u32 lds_addr) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr), "v"(voff), "s"(gbase) : "memory");
}
template <int N> __device__ __forceinline__ void attn_wait_vmcnt() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// the two values a lane and its partner in the other half-wave hold
__device__ __forceinline__ void attn_halves(float x, float& lo, float& hi) {
    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    lo = __uint_as_float(sw[0]);
    hi = __uint_as_float(sw[1]);
}

template <typename Tag, int DH, int NW>
__global__ __launch_bounds__(NW * 64, 2) void attention_kernel(AttnParams p) {
    extern __shared__ __attribute__((aligned(16))) char lq_smem[];
    constexpr bool PHASES = NW == 8;
    constexpr int NSTAGE = PHASES ? 4 : 2;     // tiles of K and of V in LDS
    constexpr int KT = 64;                     // keys per tile
    constexpr int ROWB = DH * 2, CH = DH / 8;  // bytes and 16-byte chunks of a row
    constexpr int TILE_B = KT * ROWB;
    constexpr int DMA = TILE_B / 1024 / NW;    // transfers per wavefront for a tile of K or V
    constexpr int RPD = 1024 / ROWB;           // rows per transfer
    constexpr int KSTEPS = DH / 16, DB = DH / 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = PHASES ? wave >> 2 : 0;
    const int lr = lane & 31, lh = lane >> 5;
    // workgroups of one XCD (ids congruent mod 8) take consecutive blocks of queries of the same heads, so that an XCD's L2
    // holds the K and V of the few heads it works on
    const int per_xcd = (int)gridDim.x / 8;
    int pid = blockIdx.x;
    if (pid < per_xcd * 8) pid = (pid & 7) * per_xcd + (pid >> 3);
    const int bh = pid / p.q_blocks;
    const int head = bh % p.heads, b = bh / p.heads;
    const int q0 = (pid % p.q_blocks) * (32 * NW) + wave * 32;
    const int ntiles = (p.sk + KT - 1) / KT;
    const u32 smem_base = (u32)(uintptr_t)(__attribute__((address_space(3))) char*)lq_smem;

    // ---- K and V tiles -> LDS: row r of a tile at r * ROWB, its chunk c at c ^ f(r).  K reads take one chunk column of 32
    // rows, 16 lanes at a time: f spreads 16 rows over the 256 bytes of a bank cycle.  The transposing V read takes 64 bytes of
    // four consecutive rows: f moves those rows to different quarters.  The swizzle is applied on the global side.
    const unsigned short* k_base = p.k + (size_t)b * p.k_batch + (size_t)head * DH;
    const unsigned short* v_base = p.v + (size_t)b * p.v_batch + (size_t)head * DH;
    const u32 k_pitch = (u32)p.k_row * 2, v_pitch = (u32)p.v_row * 2;
    const int d_row = lane / CH, d_ch = lane % CH;
    u32 ck[DMA], cv[DMA];
#pragma unroll
    for (int i = 0; i < DMA; ++i) {
        const int r = (wave * DMA + i) * RPD + d_row;
        ck[i] = (d_ch ^ (CH == 16 ? (r & 15) : ((r >> 1) & 7))) * 16;
        cv[i] = (d_ch ^ (CH == 16 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2))) * 16;
    }
    auto k_tile = [&](int t) { return (NSTAGE + t % NSTAGE) * TILE_B; };
    auto v_tile = [&](int t) { return (t % NSTAGE) * TILE_B; };
    // tiles and rows past the end repeat the last ones: the number of transfers in flight stays a compile-time constant
    auto src_row = [&](int t, int i) { return (u32)min(min(t, ntiles - 1) * KT + (wave * DMA + i) * RPD + d_row, p.sk - 1); };
    auto issue_k = [&](int t, int i) {
        attn_dma16(k_base, __umul24(src_row(t, i), k_pitch) + ck[i], smem_base + k_tile(t) + (wave * DMA + i) * 1024);
    };
    auto issue_v = [&](int t, int i) {
        attn_dma16(v_base, __umul24(src_row(t, i), v_pitch) + cv[i], smem_base + v_tile(t) + (wave * DMA + i) * 1024);
    };

    // The rows of V past the last key, cleared by the wavefront that fetched them, after its wait and ahead of the barrier that hands
    // the tile over: their probability is 0, which does not undo an infinity of the row they repeat.  (Of K they are masked.)
    auto clear_v = [&](int t) {
        if (t != ntiles - 1 || (t + 1) * KT <= p.sk) return;
        int left = p.sk - t * KT;
        asm volatile("" : "+s"(left));  // keeps the comparisons, of use in one tile, out of the registers of the loop
#pragma unroll
        for (int i = 0; i < DMA; ++i)
            if ((wave * DMA + i) * RPD + d_row >= left)
                *reinterpret_cast<uint4*>(lq_smem + v_tile(t) + (wave * DMA + i) * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    };

    // ---- operands: queries in registers for the whole kernel (lane: one row, chunks 2 * ks + lh)
    attn_s8 qf[KSTEPS];
    {
        const unsigned short* qp = p.q + (size_t)b * p.q_batch + (size_t)min(q0 + lr, p.sq - 1) * p.q_row + (size_t)head * DH + lh * 8;
#pragma unroll
        for (int ks = 0; ks < KSTEPS; ++ks) qf[ks] = *reinterpret_cast<const attn_s8*>(qp + ks * 16);
    }
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks) asm volatile("" : "+v"(qf[ks]));  // the loads are waited for here, not inside the loop
    if constexpr (PHASES) {
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int i = 0; i < DMA; ++i) { issue_k(t, i); issue_v(t, i); }
    } else {
#pragma unroll
        for (int i = 0; i < DMA; ++i) issue_k(0, i);
#pragma unroll
        for (int i = 0; i < DMA; ++i) { issue_k(1, i); issue_v(0, i); }
    }
    u32 k_off[KSTEPS], v_off[DB];
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ++ks)
        k_off[ks] = lr * ROWB + (((2 * ks + lh) ^ (CH == 16 ? (lr & 15) : ((lr >> 1) & 7))) << 4);
    {   // 16 lanes read a 4-row x 16-column block, lane i the four elements at row i / 4, and receive column i of it
        const int i = lane & 15, r = i >> 2;
#pragma unroll
        for (int d = 0; d < DB; ++d) {
            const int ch = d * 4 + ((lane >> 4) & 1) * 2 + ((i & 3) >> 1);
            v_off[d] = (4 * lh + r) * ROWB + ((ch ^ (CH == 16 ? (r << 2) : ((r >> 1) << 2))) << 4) + (i & 1) * 8;
        }
    }

    v16f o[DB], s[2];
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = 0.0f;
    // The maximum starts at the lowest finite float: a tile whose scores are all -inf then adds nothing, where a start at -inf
    // would make (-inf) - (-inf) of it.
    float m_run = -__FLT_MAX__, l_run[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const float c = p.scale_log2;
    float mc = fmaxf(m_run * c, -__FLT_MAX__);
    // Probabilities of a tile, in fp32 and, two keys per word, in T: words 4 * kk .. 4 * kk + 3 are the operand of PV step kk.  The row
    // sum takes the former, beside the matrix instructions (SUM_LATE); at a head dimension of 64 the 32 registers would cost the third
    // wavefront per SIMD, and the sum is formed with the exponentials.
    constexpr bool SUM_LATE = DH == 128;
    float e[32];
    u32 pw[16];

    // ---- the matrix instructions of one tile: PV (4 blocks of 16 keys x DB blocks of 32 columns), then QK of the next tile
    // (2 blocks of 32 keys x KSTEPS); the operand of step n is read RING steps ahead
    constexpr int NPV = 4 * DB, NQK = 2 * KSTEPS, STEPS = NPV + NQK;
    constexpr int RING = 8;
    static_assert(NPV >= RING && NPV == NQK, "tile plan");
    attn_s8 fr[RING];
    typedef __attribute__((address_space(3))) attn_s4* lds_s4;
    auto load_k = [&](int t, int j) { return *reinterpret_cast<const attn_s8*>(lq_smem + k_tile(t) + k_off[j % KSTEPS] + (j / KSTEPS) * 32 * ROWB); };
    auto load_v = [&](int t, int i) {
        const char* vp = lq_smem + v_tile(t) + v_off[i % DB] + (i / DB) * 16 * ROWB;
        const attn_s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(vp));
        const attn_s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4)(vp + 8 * ROWB));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    auto load_step = [&](int t, int n) { return n < NPV ? load_v(t, n) : load_k(t + 1, n - NPV); };
    auto qk_step = [&](attn_s8 kf, int j) {
        const int kb = j / KSTEPS, ks = j % KSTEPS;
        if (ks == 0) {
#pragma unroll
            for (int e = 0; e < 16; ++e) s[kb][e] = 0.0f;
        }
        s[kb] = attn_mfma<Tag>(kf, qf[ks], s[kb]);
    };
    auto pv_step = [&](attn_s8 vf, int i) {
        const int kk = i / DB;
        const attn_s8 pf = __builtin_bit_cast(attn_s8, v4i{(int)pw[4 * kk], (int)pw[4 * kk + 1], (int)pw[4 * kk + 2], (int)pw[4 * kk + 3]});
        o[i % DB] = attn_mfma<Tag>(vf, pf, o[i % DB]);
    };
    // The running maximum is the true one (no slack): the largest probability of a row is then exactly 1 and carries no
    // rounding error of its own, which keeps the result as close to the fp32 evaluation as a softmax over whole rows.
    auto softmax = [&](int t) {
        if ((t + 1) * KT > p.sk) {  // keys past the end, in the last tile
            const int left = p.sk - t * KT - 4 * lh;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (kb * 32 + 8 * (i >> 2) + (i & 3) >= left) s[kb][i] = -__builtin_inff();
        }
        // four independent chains, here and below: nobody else fills the latency of a dependent vector instruction
        float mq[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) mq[e] = attn_max(s[0][e], s[1][e], s[0][4 + e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) mq[e] = attn_max(mq[e], s[1][4 + e], s[0][8 + e]);
#pragma unroll
        for (int e = 0; e < 4; ++e) mq[e] = attn_max(mq[e], s[1][8 + e], s[0][12 + e]);
        mq[0] = attn_max(mq[0], mq[1], s[1][12]);
        mq[2] = attn_max(mq[2], mq[3], s[1][13]);
        float lo, hi;
        attn_halves(attn_max(mq[0], mq[2], __builtin_elementwise_maximum(s[1][14], s[1][15])), lo, hi);
        const float mx = __builtin_elementwise_maximum(lo, hi);
        if (__any(mx > m_run)) {
            const float m_new = mx > m_run ? mx : m_run;
            const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c);
            m_run = m_new;
            mc = fmaxf(m_run * c, -__FLT_MAX__);  // finite too: c > 1 would make -inf of the start, and NaN of a score of -inf
#pragma unroll
            for (int i = 0; i < 4; ++i) l_run[i] *= alpha;
#pragma unroll
            for (int d = 0; d < DB; ++d)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[d][i] *= alpha;
        }
#pragma unroll
        for (int i = 0; i < 32; ++i) e[i] = __builtin_fmaf(s[i >> 4][i & 15], c, -mc);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 8; ++i) e[i] = __builtin_amdgcn_exp2f(e[i]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (g < 3) {
                    e[8 * g + 8 + 2 * i] = __builtin_amdgcn_exp2f(e[8 * g + 8 + 2 * i]);
                    e[8 * g + 9 + 2 * i] = __builtin_amdgcn_exp2f(e[8 * g + 9 + 2 * i]);
                }
                if constexpr (!SUM_LATE) { l_run[i] += e[8 * g + 2 * i]; l_run[i] += e[8 * g + 2 * i + 1]; }
                pw[4 * g + i] = attn_pack<Tag>(e[8 * g + 2 * i], e[8 * g + 2 * i + 1]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        // all of it happens here: left alone, the compiler moves the exponentials next to the matrix instructions that use them
#pragma unroll
        for (int i = 0; i < 16; ++i) asm volatile("" : "+v"(pw[i]));
#pragma unroll
        for (int i = 0; i < (SUM_LATE ? 32 : 0); ++i) asm volatile("" : "+v"(e[i]));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto barrier = [&] {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };

    // ---- tile 0's scores.  PHASES: phase 2t is group 0's matrix phase of tile t (QK of t, PV of t - 1) and group 1's vector
    // phase of tile t - 1; in phase 2t + 1 they have changed places.  A tile is read from phase 2t to 2t + 3 and its place is
    // taken again by tile t + 4, whose transfers start in phase 2t + 4 at the earliest; every wavefront has waited for its share
    // of tile t ahead of the barrier that opens phase 2t.
    attn_wait_vmcnt<2 * DMA>();
    if constexpr (PHASES) clear_v(0);
    barrier();
    if constexpr (PHASES) {
        if (grp == 1) barrier();
#pragma unroll
        for (int i = 0; i < DMA; ++i) { issue_k(2, i); issue_v(2, i); }
    }
#pragma unroll
    for (int j = 0; j < NQK; ++j) qk_step(load_k(0, j), j);

    // The QK part of the last iteration works on a repeated tile and is not used: one loop body keeps the accumulators in place.
    for (int t = 0; t < ntiles; ++t) {
        if constexpr (PHASES) {
            if (grp == 1) {
                attn_wait_vmcnt<2 * DMA>();  // this wavefront's share of tile t + 1
                clear_v(t + 1);
            }
            barrier();
            softmax(t);
#pragma unroll
            for (int n = 0; n < RING; ++n) fr[n] = load_step(t, n);
            if (grp == 0) {
                attn_wait_vmcnt<2 * DMA>();
                clear_v(t + 1);
            }
            barrier();
            __builtin_amdgcn_s_setprio(1);
        } else {
            // K of tile t + 1 and V of tile t have landed, and everybody is done with K of tile t and V of tile t - 1
            attn_wait_vmcnt<0>();
            clear_v(t);
            barrier();
#pragma unroll
            for (int i = 0; i < DMA; ++i) { issue_k(t + 2, i); issue_v(t + 1, i); }
            softmax(t);
#pragma unroll
            for (int n = 0; n < RING; ++n) fr[n] = load_step(t, n);
        }
#pragma unroll
        for (int n = 0; n < STEPS; ++n) {
            if (n < NPV) pv_step(fr[n % RING], n);
            else qk_step(fr[n % RING], n - NPV);
            if (n + RING < STEPS) fr[n % RING] = load_step(t, n + RING);
            if (n >= NPV) {
#pragma unroll
                for (int u = 0; u < 16 / NQK; ++u) {
                    const int x = (n - NPV) * (16 / NQK) + u;
                    if constexpr (SUM_LATE) { l_run[x % 4] += e[2 * x]; l_run[x % 4] += e[2 * x + 1]; }
                }
            }
            if constexpr (PHASES) {  // tile t + 3, spread over the phase: a burst would stall the wavefront on the memory queue
                if (n % 4 == 2 && n / 4 < DMA) issue_k(t + 3, n / 4);
                if (n % 4 == 2 && n / 4 >= DMA && n / 4 < 2 * DMA) issue_v(t + 3, n / 4 - DMA);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (PHASES) __builtin_amdgcn_s_setprio(0);
    }
    if (PHASES && grp == 0) barrier();
    attn_wait_vmcnt<0>();
    __syncthreads();  // nobody reads or fills the tiles any more

    // ---- O^T / sum -> rows of T through a wavefront-private strip, 16 bytes per lane on the way out
    float lo, hi;
    attn_halves((l_run[0] + l_run[1]) + (l_run[2] + l_run[3]), lo, hi);
    const float inv = 1.0f / (lo + hi);
    constexpr int PITCH = ROWB + 16;
    char* strip = lq_smem + wave * (32 * PITCH);
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4)
            *reinterpret_cast<uint2*>(strip + lr * PITCH + (d * 32 + 8 * q4 + 4 * lh) * 2) =
                make_uint2(attn_pack<Tag>(o[d][4 * q4] * inv, o[d][4 * q4 + 1] * inv), attn_pack<Tag>(o[d][4 * q4 + 2] * inv, o[d][4 * q4 + 3] * inv));
    const size_t o_row = (size_t)p.heads * DH;
    // a row of the strip is the output rounded to T; codes are made from that, as the casts behind the attention make them
    auto strip_row = [&](int r) { return *reinterpret_cast<const uint4*>(strip + r * PITCH + d_ch * 16); };
    if (p.fp8 != nullptr) {
        const float inv_rest = 1.0f / p.fp8_scale[0], inv_ctx = p.context > 0 ? 1.0f / p.fp8_context_scale[0] : 0.0f;
        const size_t panel = (size_t)head * (DH / 64) + d_ch / 8;
#pragma unroll
        for (int i = 0; i < 32 / RPD; ++i) {
            const int r = i * RPD + d_row, token = q0 + r;
            const bool ctx = token < p.context;
            const float f = ctx ? inv_ctx : inv_rest;
            const int rows = ctx ? p.context : p.sq - p.context;
            float y[8];
            unpack8<Tag>(strip_row(r), y);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] *= f;
            uint8_t* dst = (ctx ? p.fp8_context : p.fp8) + (panel * ((size_t)p.batch * rows) + (size_t)b * rows + (ctx ? token : token - p.context)) * 64 + (d_ch % 8) * 8;
            if (token < p.sq) *reinterpret_cast<uint2*>(dst) = make_uint2(e4m3x4(y[0], y[1], y[2], y[3]), e4m3x4(y[4], y[5], y[6], y[7]));
        }
        return;
    }
    if (p.int8 != nullptr) {
        const float sc = p.int8_scale[0], rcp = fast_recip(sc);
        const bool slow = scale_out_of_range(sc);
        float pre[8];
        const float* pp = p.int8_pre + (size_t)head * DH + d_ch * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) pre[e] = p.int8_pre != nullptr ? pp[e] : 1.0f;
        int8_t* dst = p.int8 + (size_t)b * p.sq * o_row + (size_t)head * DH + d_ch * 8;
#pragma unroll
        for (int i = 0; i < 32 / RPD; ++i) {
            const int r = i * RPD + d_row;
            float y[8];
            unpack8<Tag>(strip_row(r), y);
#pragma unroll
            for (int e = 0; e < 8; ++e) y[e] = y[e] * pre[e];
            int q[8];
            quant8<-128, 127>(y, sc, rcp, slow, q);
            if (q0 + r < p.sq)
                *reinterpret_cast<uint2*>(dst + (size_t)(q0 + r) * o_row) = make_uint2(pack4_s8(q[0], q[1], q[2], q[3]), pack4_s8(q[4], q[5], q[6], q[7]));
        }
        return;
    }
    unsigned short* op = p.out + (size_t)b * p.sq * o_row + (size_t)head * DH;
#pragma unroll
    for (int i = 0; i < 32 / RPD; ++i) {
        const int r = i * RPD + d_row;
        if (q0 + r < p.sq) *reinterpret_cast<uint4*>(op + (size_t)(q0 + r) * o_row + d_ch * 8) = strip_row(r);
    }
}

template <typename Tag, int DH, int NW> static int launch_attention(AttnParams p, hipStream_t st) {
    constexpr int lds = 2 * (NW == 8 ? 4 : 2) * 64 * DH * 2;
    static_assert(NW * 32 * (DH * 2 + 16) <= lds, "the output strips take the place of the tiles");
    p.q_blocks = (p.sq + 32 * NW - 1) / (32 * NW);
    auto kern = attention_kernel<Tag, DH, NW>;
    static bool attr_done = false;  // raising the dynamic LDS limit is idempotent; races are benign
    if (!attr_done && lds > 48 * 1024) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        if (e != hipSuccess) {
            set_error("lq_attention: cannot raise LDS limit to %d bytes: %s", lds, hipGetErrorString(e));
            return LQ_ERR_HIP;
        }
        attr_done = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)(p.q_blocks * p.batch * p.heads)), dim3(NW * 64), lds, st, p);
    return check_launch("lq_attention");
}

template <typename Tag> static int attention_typed(const AttnParams& p, int head_dim, hipStream_t st) {
    if (head_dim == 64) return launch_attention<Tag, 64, 4>(p, st);
    // Blocks of 128 queries, one workgroup per CU or fewer: spread over the chip.  From there on the phased form with 256
    // queries per workgroup (24 heads, us, NW == 4 / NW == 8: 1000 tokens 27.6 / 34.8, 1200 tokens 32.8 / 40.5, 1365 tokens 50.6 / 45.5, 1600 tokens
    // 57.3 / 51.0, 4608 tokens 310 / 273, 6912 tokens 677 / 597).
    const long long small = (long long)p.batch * p.heads * ((p.sq + 127) / 128);
    return small <= device_cu_count() ? launch_attention<Tag, 128, 4>(p, st) : launch_attention<Tag, 128, 8>(p, st);
}

}  // namespace lq

using namespace lq;

static int attention_entry(const char* what, const lq_attention_t& a, lq_stream_t stream) {
    LQ_REQUIRE(a.dtype == LQ_F16 || a.dtype == LQ_BF16, LQ_ERR_UNSUPPORTED, "%s: tensors must be F16 or BF16", what);
    LQ_REQUIRE(a.batch >= 0 && a.heads > 0 && a.seq_q >= 0 && a.seq_k > 0 && (a.head_dim == 64 || a.head_dim == 128), LQ_ERR_SHAPE,
               "%s: need head_dim 64 or 128 and at least one key (batch=%d heads=%d seq_q=%d seq_k=%d head_dim=%d)", what, a.batch, a.heads,
               a.seq_q, a.seq_k, a.head_dim);
    LQ_REQUIRE(a.scale > 0.0f, LQ_ERR_ARG, "%s: the softmax scale must be positive", what);  // the largest score is taken before scaling
    LQ_REQUIRE(a.context >= 0 && a.context <= a.seq_q, LQ_ERR_SHAPE, "%s: context=%d of %d queries", what, a.context, a.seq_q);
    if (a.batch == 0 || a.seq_q == 0) return LQ_OK;
    const int outputs = (a.out != nullptr) + (a.out_fp8 != nullptr || a.context_fp8 != nullptr) + (a.out_int8 != nullptr);
    LQ_REQUIRE(outputs == 1 && a.q && a.k && a.v, LQ_ERR_ARG, "%s: null pointer", what);
    const uintptr_t bits = reinterpret_cast<uintptr_t>(a.out) | reinterpret_cast<uintptr_t>(a.q) | reinterpret_cast<uintptr_t>(a.k) |
                           reinterpret_cast<uintptr_t>(a.v) | ((a.q_row | a.k_row | a.v_row | a.q_batch | a.k_batch | a.v_batch) * 2);
    LQ_REQUIRE(bits % 16 == 0, LQ_ERR_ARG, "%s: tensors and their row and batch strides must be multiples of 16 bytes", what);
    const size_t width = (size_t)a.heads * a.head_dim, longest = a.k_row > a.v_row ? a.k_row : a.v_row;
    LQ_REQUIRE(a.q_row >= width && a.k_row >= width && a.v_row >= width, LQ_ERR_SHAPE, "%s: a row stride is shorter than heads * head_dim", what);
    // a lane's offset inside one batch of K or V is 32 bits, a product of two 24-bit numbers
    LQ_REQUIRE(longest < ((size_t)1 << 23) && a.seq_k < (1 << 24) && (size_t)a.seq_k * longest < ((size_t)1 << 31) &&
                   (long long)a.batch * a.heads * ((a.seq_q + 127) / 128) <= 0x7fffffffLL,
               LQ_ERR_SHAPE, "%s: tensors too large (seq_k=%d, row stride %zu)", what, a.seq_k, longest);
    if (a.out_fp8 != nullptr || a.context_fp8 != nullptr) {
        LQ_REQUIRE((a.context == a.seq_q || (a.out_fp8 && a.out_fp8_scale)) && (a.context == 0 || (a.context_fp8 && a.context_fp8_scale)), LQ_ERR_ARG,
                   "%s: codes need a destination and a scale for each part of the tokens", what);
        LQ_REQUIRE((reinterpret_cast<uintptr_t>(a.out_fp8) | reinterpret_cast<uintptr_t>(a.context_fp8)) % 8 == 0, LQ_ERR_ARG,
                   "%s: codes must be 8-byte aligned", what);
    }
    LQ_REQUIRE(a.out_int8 == nullptr || (a.int8_scale != nullptr && reinterpret_cast<uintptr_t>(a.out_int8) % 8 == 0), LQ_ERR_ARG,
               "%s: int8 codes need a scale and 8-byte alignment", what);
    auto us = [](const void* x) { return static_cast<const unsigned short*>(x); };
    AttnParams p{};
    p.q = us(a.q); p.k = us(a.k); p.v = us(a.v);
    p.out = static_cast<unsigned short*>(a.out);
    p.q_row = a.q_row; p.k_row = a.k_row; p.v_row = a.v_row;
    p.q_batch = a.q_batch; p.k_batch = a.k_batch; p.v_batch = a.v_batch;
    p.batch = a.batch; p.heads = a.heads; p.sq = a.seq_q; p.sk = a.seq_k;
    p.scale_log2 = a.scale * 1.4426950408889634f;
    p.context = a.context;
    // the kernel looks at fp8 to know that codes are wanted; tokens of a part that is empty never come up
    p.fp8 = a.out_fp8 != nullptr ? a.out_fp8 : a.context_fp8;
    p.fp8_context = a.context_fp8;
    p.fp8_scale = a.out_fp8_scale != nullptr ? a.out_fp8_scale : a.context_fp8_scale; p.fp8_context_scale = a.context_fp8_scale;
    p.int8 = a.out_int8; p.int8_pre = a.int8_pre; p.int8_scale = a.int8_scale;
    return a.dtype == LQ_BF16 ? attention_typed<BF16Tag>(p, a.head_dim, as_stream(stream)) : attention_typed<F16Tag>(p, a.head_dim, as_stream(stream));
}

extern "C" int lq_attention(void* out, const void* q, size_t q_row, size_t q_batch, const void* k, size_t k_row, size_t k_batch, const void* v,
                            size_t v_row, size_t v_batch, lq_dtype_t dtype, int batch, int seq_q, int seq_k, int heads, int head_dim,
                            float scale, lq_stream_t stream) {
    lq_attention_t a = {};
    a.out = out; a.q = q; a.q_row = q_row; a.q_batch = q_batch; a.k = k; a.k_row = k_row; a.k_batch = k_batch; a.v = v; a.v_row = v_row; a.v_batch = v_batch;
    a.dtype = dtype; a.batch = batch; a.seq_q = seq_q; a.seq_k = seq_k; a.heads = heads; a.head_dim = head_dim; a.scale = scale;
    return attention_entry("lq_attention", a, stream);
}

extern "C" int lq_attention_ex(const lq_attention_t* a, lq_stream_t stream) {
    LQ_REQUIRE(a, LQ_ERR_ARG, "lq_attention_ex: null pointer");
    return attention_entry("lq_attention_ex", *a, stream);
}
