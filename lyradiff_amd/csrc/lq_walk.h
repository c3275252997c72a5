// Rows of 512 * NF + 64 * TAIL 16-bit values (640, 768, 1152, 1280 columns) that a wavefront holds as a whole: a lane has eight columns of each
// pass of 512 and TAIL of the rest, where passes of eight per lane alone would leave most lanes of the last one without any.
#pragma once

#include "lq_common.h"

namespace lq {

// int8 codes of N values, two or four to the last word; CLAMP false: s is the values' own largest over 127 (quant_pack_unclamped)
template <int N, bool CLAMP> __device__ __forceinline__ void walk_quant_s8(const float* t, float s, float r, bool slow, u32* words) {
    if constexpr (!CLAMP) quant_pack_unclamped<N>(t, s, r, slow, words);
    else {
        float rq[N];
        quant8_round<127, N>(t, s, r, slow, rq);
        int q[(N + 3) / 4 * 4] = {};
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int v = cvt_i32_sat(rq[i]);
            q[i] = v < -128 ? -128 : (v > 127 ? 127 : v);
        }
#pragma unroll
        for (int i = 0; i < N; i += 4) words[i / 4] = pack4_s8(q[i], q[i + 1], q[i + 2], q[i + 3]);
    }
}

template <typename Tag, int NF, int TAIL> struct WalkRow {
    static_assert(TAIL == 2 || TAIL == 4, "a lane's share of the rest is four or eight bytes");
    static constexpr int E = 8 * NF + TAIL, DIM = 64 * E;  // values per lane and per row
    uint4 full[NF];
    u32 tail[TAIL / 2];

    __device__ __forceinline__ void load(const void* base, size_t row, int lane) {
        const unsigned short* p = static_cast<const unsigned short*>(base) + row * DIM;
#pragma unroll
        for (int i = 0; i < NF; ++i) full[i] = *reinterpret_cast<const uint4*>(p + i * 512 + lane * 8);
        if constexpr (TAIL == 2) tail[0] = *reinterpret_cast<const u32*>(p + NF * 512 + lane * 2);
        else {
            const uint2 v = *reinterpret_cast<const uint2*>(p + NF * 512 + lane * 4);
            tail[0] = v.x; tail[1] = v.y;
        }
    }
    __device__ __forceinline__ void unpack(float* o) const {
#pragma unroll
        for (int i = 0; i < NF; ++i) unpack8<Tag>(full[i], o + 8 * i);
#pragma unroll
        for (int i = 0; i < TAIL / 2; ++i) {
            o[8 * NF + 2 * i] = Elem<Tag>::load(tail[i] & 0xFFFFu);
            o[8 * NF + 2 * i + 1] = Elem<Tag>::load(tail[i] >> 16);
        }
    }
    __device__ __forceinline__ void words(u32* w) const {  // two values each
#pragma unroll
        for (int i = 0; i < NF; ++i) w[4 * i] = full[i].x, w[4 * i + 1] = full[i].y, w[4 * i + 2] = full[i].z, w[4 * i + 3] = full[i].w;
#pragma unroll
        for (int i = 0; i < TAIL / 2; ++i) w[4 * NF + i] = tail[i];
    }
    static __device__ __forceinline__ void store_words(void* base, size_t row, int lane, const u32* w) {
        unsigned short* o = static_cast<unsigned short*>(base) + row * DIM;
#pragma unroll
        for (int i = 0; i < NF; ++i) *reinterpret_cast<uint4*>(o + i * 512 + lane * 8) = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
        if constexpr (TAIL == 2) *reinterpret_cast<u32*>(o + NF * 512 + lane * 2) = w[4 * NF];
        else *reinterpret_cast<uint2*>(o + NF * 512 + lane * 4) = make_uint2(w[4 * NF], w[4 * NF + 1]);
    }
    // the lane's share of a vector of floats, or ones where there is none
    static __device__ __forceinline__ void load_f32(const float* v, int lane, float* o) {
#pragma unroll
        for (int i = 0; i < E; ++i) o[i] = 1.0f;
        if (v == nullptr) return;
#pragma unroll
        for (int i = 0; i < 8 * NF; i += 4) {
            const float4 f = *reinterpret_cast<const float4*>(v + (i / 8) * 512 + lane * 8 + i % 8);
            o[i] = f.x; o[i + 1] = f.y; o[i + 2] = f.z; o[i + 3] = f.w;
        }
#pragma unroll
        for (int i = 0; i < TAIL; i += 2) {
            const float2 f = *reinterpret_cast<const float2*>(v + NF * 512 + lane * TAIL + i);
            o[8 * NF + i] = f.x; o[8 * NF + i + 1] = f.y;
        }
    }
    template <bool CLAMP> static __device__ __forceinline__ void store_codes(void* base, size_t row, int lane, const float* t, float s, float r, bool slow) {
        uint8_t* o = static_cast<uint8_t*>(base) + row * DIM;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
            u32 w[2];
            walk_quant_s8<8, CLAMP>(t + 8 * i, s, r, slow, w);
            *reinterpret_cast<uint2*>(o + i * 512 + lane * 8) = make_uint2(w[0], w[1]);
        }
        u32 w;
        walk_quant_s8<TAIL, CLAMP>(t + 8 * NF, s, r, slow, &w);
        if constexpr (TAIL == 2) *reinterpret_cast<unsigned short*>(o + NF * 512 + lane * 2) = (unsigned short)w;
        else *reinterpret_cast<u32*>(o + NF * 512 + lane * 4) = w;
    }
};

}  // namespace lq
