// Scaling of activation rows to fp16, shared by the kernels that lay activations out for the tile kernels (tile_gemm.hpp).
#pragma once
#include "common.hpp"

namespace mfq {

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Largest magnitudes of the even and of the odd values: bits of either type order like their values, one packed maximum per pair.
__device__ __forceinline__ u16x2_t pair_top(u16x2_t top, u32x4_t v) {
#pragma unroll
    for (int t = 0; t < 4; ++t) top = __builtin_elementwise_max(top, __builtin_bit_cast(u16x2_t, v[t] & 0x7fff7fffu));
    return top;
}
// larger of the magnitudes in `top` (bits of either type order like their values) and of a chunk's finite values
template <int XF16>
__device__ __forceinline__ uint32_t finite_top(uint32_t top, u32x4_t v) {
    constexpr uint32_t kInf = XF16 ? 0x7c00u : 0x7f80u;
    for (int t = 0; t < 4; ++t) {
        const uint32_t a = v[t] & 0x7fffu, b = (v[t] >> 16) & 0x7fffu;
        if (a < kInf) top = max(top, a);
        if (b < kInf) top = max(top, b);
    }
    return top;
}
// exponent e of a row: its largest magnitude is f * 2^e, f in [0.5, 1); the row is scaled by 2^(9 - e)
template <int XF16>
__device__ __forceinline__ int row_exp(uint32_t top) {
    const float amax = x_to_f32<XF16>(static_cast<uint16_t>(top));
    int e = 0;
    if (amax > 0.f) frexpf(amax, &e);
    return max(e, kMinRowExp);
}
// fp16 scales of a tensor's neurons, ng of each, and where the power of two of each neuron goes (none with blocks = 0).
struct RowScales {
    const uint16_t *scales;
    int ng, out, blocks;
    float *rowscale;
};
// 2^(e - 8), e = exponent of a neuron's largest |scale| (in [2^(e-1), 2^e)), so that codes of eight bits times scales divided by it
// stay at 2^15 and below.  A wave per neuron; a NaN or infinite scale does not set the range.
__device__ __forceinline__ void row_scale(const RowScales &rs, int row, int lane) {
    const uint16_t *sc = rs.scales + static_cast<int64_t>(row) * rs.ng;
    uint32_t top = 0;  // magnitudes of finite halves order like their bits
    for (int g0 = lane; g0 < rs.ng; g0 += 512) {
        uint32_t v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = g0 + 64 * i < rs.ng ? sc[g0 + 64 * i] & 0x7fffu : 0u;
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (v[i] < 0x7c00u) top = max(top, v[i]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) top = max(top, static_cast<uint32_t>(__shfl_xor(static_cast<int>(top), o, 64)));
    int e = 0;
    if (top > 0) frexpf(f16_to_f32(static_cast<uint16_t>(top)), &e);
    if (lane == 0) rs.rowscale[row] = ldexpf(1.f, e - 8);
}
// Eight values times inv, a power of two: exact unless the result is subnormal in fp16, i.e. below the row's maximum by 2^22 and
// more, and then rounded to nearest even.
template <int XF16>
__device__ __forceinline__ u32x4_t scaled_f16(u32x4_t v, float inv) {
    u32x4_t h;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        float lo, hi;
        if constexpr (XF16) {
            lo = f16_to_f32(v[t] & 0xffffu);
            hi = f16_to_f32(v[t] >> 16);
        } else {
            lo = __uint_as_float(v[t] << 16);
            hi = __uint_as_float(v[t] & 0xffff0000u);
        }
        h[t] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo * inv, hi * inv}, half2_t));  // v_cvt_pk_f16_f32
    }
    return h;
}

}  // namespace mfq
