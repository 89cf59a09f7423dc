// Float weights in registers: 8 weights of one row, loaded as 16-byte pieces and widened exactly to
// f32 (F16 through the hardware conversion, BF16 as the high half of an f32).
#pragma once

#include "kernels.h"

#include <hip/hip_fp16.h>

namespace sgk {

// 16 bytes of weights, non-temporal (read once per product, as in the quantized matvec)
typedef unsigned int u32x4_nt __attribute__((ext_vector_type(4)));
__device__ __forceinline__ uint4 ld16_nt(const uint8_t * p) {
    const u32x4_nt v = __builtin_nontemporal_load(reinterpret_cast<const u32x4_nt *>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// 16 bytes of weights (4 F32 or 8 F16 / BF16) as f32
template <int WT>
__device__ __forceinline__ void widen16(uint4 q, float * o) {
    const uint32_t w[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if constexpr (WT == F32) {
            o[i] = __uint_as_float(w[i]);
        } else if constexpr (WT == F16) {
            o[2 * i] = __half2float(__ushort_as_half((unsigned short) (w[i] & 0xFFFFu)));
            o[2 * i + 1] = __half2float(__ushort_as_half((unsigned short) (w[i] >> 16)));
        } else {
            o[2 * i] = __uint_as_float(w[i] << 16);
            o[2 * i + 1] = __uint_as_float(w[i] & 0xFFFF0000u);
        }
    }
}

// 8 consecutive weights of one row as f32 (p 16-byte aligned)
template <int WT> struct WLoad {
    uint4 q;
    __device__ void load(const uint8_t * p) { q = ld16_nt(p); }
    __device__ void to_f32(float * o) const { widen16<WT>(q, o); }
};
template <> struct WLoad<F32> {
    uint4 u, v;
    __device__ void load(const uint8_t * p) {
        u = ld16_nt(p);
        v = ld16_nt(p + 16);
    }
    __device__ void to_f32(float * o) const {
        widen16<F32>(u, o);
        widen16<F32>(v, o + 4);
    }
};

} // namespace sgk
