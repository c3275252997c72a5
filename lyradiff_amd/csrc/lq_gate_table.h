// The GEGLU gate factor as a function of the 16-bit gate value: what lq_quant_int8.hip, which holds the formula and the table in device
// memory, shares with the kernels that look it up.
#pragma once

#include "lq_common.h"

namespace lq {

// magnitudes with an entry (bit patterns LO .. LO + COUNT - 1), entries of the positive values, then of the negative ones
template <typename Tag> struct GateTable;
template <> struct GateTable<F16Tag> { static constexpr u32 LO = 0x0C00u, COUNT = 0x4800u - 0x0C00u; };   // 2^-12 .. 8
template <> struct GateTable<BF16Tag> { static constexpr u32 LO = 0x3980u, COUNT = 0x4100u - 0x3980u; };

// the factor of a value without an entry, rounded to T: below the table the inner factor is 0.5, beyond it 0 or 1
template <typename Tag> __device__ __forceinline__ float gate_outside_table(float g) {
    const float c = fabsf(g) < 1.0f ? 0.5f : (g < 0.0f ? 0.0f : 1.0f);
    return round_through<Tag>(g * c);
}

// The table of the current device, built before the stream's next kernel (lq_quant_int8.hip).
int gate_table_on_device(bool f16, hipStream_t st, const unsigned short** table);

}  // namespace lq
