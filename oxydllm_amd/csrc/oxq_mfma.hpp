// Matrix-core operand helpers shared by the tile kernels: the bit-exact
// T((q - z) * s) dequantisation of a pair of weights and the
// v_mfma_f32_16x16x32_{f16,bf16} wrappers.
#pragma once

#include "oxq_device.hpp"

namespace oxq {

template <typename TT> struct MfmaOps;

template <> struct MfmaOps<F16Traits> {
    // exact (bias+q) - (bias+z), then one correctly rounded multiply
    __device__ static __forceinline__ uint32_t dequant_pair(uint32_t p, uint32_t negzb, uint32_t s) {
        const half2_t d = __builtin_bit_cast(half2_t, p) + __builtin_bit_cast(half2_t, negzb);
        return __builtin_bit_cast(uint32_t, d * __builtin_bit_cast(half2_t, s));
    }
    __device__ static __forceinline__ uint32_t splat(float v) {
        const uint16_t h = F16Traits::from_f32(v);
        return (uint32_t)h | ((uint32_t)h << 16);
    }
    __device__ static __forceinline__ float4_t mfma(const uint32_t a[4], const uint32_t b[4], float4_t c) {
        u32x4_t av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, av),
                                                      __builtin_bit_cast(half8_t, bv), c, 0, 0, 0);
    }
};

template <> struct MfmaOps<BF16Traits> {
    __device__ static __forceinline__ uint32_t dequant_pair(uint32_t p, uint32_t negzb, uint32_t s) {
        // widen (exact), subtract (exact), multiply (exact in f32), round once to bf16
        const float lo = (__builtin_bit_cast(float, p << 16) + __builtin_bit_cast(float, negzb << 16)) *
                         __builtin_bit_cast(float, s << 16);
        const float hi = (__builtin_bit_cast(float, p & 0xFFFF0000u) +
                          __builtin_bit_cast(float, negzb & 0xFFFF0000u)) *
                         __builtin_bit_cast(float, s & 0xFFFF0000u);
        return (uint32_t)BF16Traits::from_f32(lo) | ((uint32_t)BF16Traits::from_f32(hi) << 16);
    }
    __device__ static __forceinline__ uint32_t splat(float v) {
        const uint16_t h = BF16Traits::from_f32(v);
        return (uint32_t)h | ((uint32_t)h << 16);
    }
    __device__ static __forceinline__ float4_t mfma(const uint32_t a[4], const uint32_t b[4], float4_t c) {
        u32x4_t av = {a[0], a[1], a[2], a[3]}, bv = {b[0], b[1], b[2], b[3]};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av),
                                                       __builtin_bit_cast(bf16x8_t, bv), c, 0, 0, 0);
    }
};

// An accumulator tile holds four rows of one column a lane; stored like that a store instruction writes 2 bytes a lane in pieces of
// 32.  These turn the 4 x 4 of a quad of lanes: lane q gets columns 0 .. 3 of row q, one 8 (16) byte store.
__device__ __forceinline__ uint32_t quad_xor(uint32_t v, std::integral_constant<int, 1>) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, false);  // quad_perm 1 0 3 2
}
__device__ __forceinline__ uint32_t quad_xor(uint32_t v, std::integral_constant<int, 2>) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, false);  // quad_perm 2 3 0 1
}
// rows 0, 1 and 2, 3 as pairs of 16 bits
__device__ __forceinline__ uint2 quad_turn16(uint32_t r01, uint32_t r23, int lane) {
    constexpr std::integral_constant<int, 1> by1{};
    constexpr std::integral_constant<int, 2> by2{};
    const uint32_t sel = (lane & 1) ? 0x03020706u : 0x05040100u;  // of the even lane's column, then the odd one's
    const uint32_t a = perm_b32(quad_xor(r01, by1), r01, sel), b = perm_b32(quad_xor(r23, by1), r23, sel);  // rows q & 1, 2 + (q & 1)
    const uint32_t got = quad_xor((lane & 2) ? a : b, by2);
    return (lane & 2) ? uint2{got, b} : uint2{a, got};
}
__device__ __forceinline__ float4_t quad_turn32(float4_t v, int lane) {
    constexpr std::integral_constant<int, 1> by1{};
    constexpr std::integral_constant<int, 2> by2{};
    const bool odd = lane & 1, high = lane & 2;
    uint32_t e[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float x = v[i];
        e[i] = __builtin_bit_cast(uint32_t, x);
    }
    uint32_t p[2][2];  // columns q & 2, (q & 2) + 1 of rows q & 1 and 2 + (q & 1)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const uint32_t mine = odd ? e[2 * h + 1] : e[2 * h], got = quad_xor(odd ? e[2 * h] : e[2 * h + 1], by1);
        p[h][0] = odd ? got : mine, p[h][1] = odd ? mine : got;
    }
    float4_t o;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const uint32_t got = quad_xor(high ? p[0][c] : p[1][c], by2);
        o[c] = __builtin_bit_cast(float, high ? got : p[0][c]), o[2 + c] = __builtin_bit_cast(float, high ? p[1][c] : got);
    }
    return o;
}

}  // namespace oxq
