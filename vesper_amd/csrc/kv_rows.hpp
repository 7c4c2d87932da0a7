// Device helpers for the rows that enter the cache: loads of eight elements, the rotary embedding and the roundings, shared by the
// append kernels and the one-launch token step.
#pragma once

#include "vsp_common.hpp"

namespace vsp {

// apply_rotary_emb (src/nn/functional.cpp:445-494) on N consecutive elements of a row, N a multiple of 4: pairs (2i, 2i+1), every
// product and sum rounded on its own as the reference's separate elementwise ops do.  t: the elements' {cos, sin} pairs, two
// per 16-byte load.
template <int N>
__device__ inline void rope_pairs(float (&x)[N], const float4* t) {
#pragma clang fp contract(off)  // no fused multiply-add: the products are rounded before the sum
#pragma unroll
    for (int j = 0; j < N / 4; ++j) {
        const float4 cs = t[j];
        {
            const float x0 = x[4 * j], x1 = x[4 * j + 1];
            const float t1 = x0 * cs.x, t2 = x1 * cs.y, t3 = x0 * cs.y, t4 = x1 * cs.x;
            x[4 * j] = t1 - t2;
            x[4 * j + 1] = t3 + t4;
        }
        {
            const float x0 = x[4 * j + 2], x1 = x[4 * j + 3];
            const float t1 = x0 * cs.z, t2 = x1 * cs.w, t3 = x0 * cs.w, t4 = x1 * cs.z;
            x[4 * j + 2] = t1 - t2;
            x[4 * j + 3] = t3 + t4;
        }
    }
}

template <typename SrcT>
__device__ inline void load8(const SrcT* p, float (&x)[8]) {
    if constexpr (sizeof(SrcT) == 2) {
        const uint4 w = *(const uint4*)p;
        const uint32_t ww[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            x[2 * j] = __builtin_bit_cast(float, ww[j] << 16);
            x[2 * j + 1] = __builtin_bit_cast(float, ww[j] & 0xffff0000u);
        }
    } else {
        const float4 lo = *(const float4*)p, hi = *(const float4*)(p + 4);
        x[0] = lo.x, x[1] = lo.y, x[2] = lo.z, x[3] = lo.w, x[4] = hi.x, x[5] = hi.y, x[6] = hi.z, x[7] = hi.w;
    }
}
// two fp32 -> packed bf16 pair with the reference's rounding (f32_to_bf16_bits): both words are rounded in place and one
// byte permute picks their high halves
__device__ inline uint32_t round_pack_bf16x2(float lo, float hi) {
    uint32_t a = __builtin_bit_cast(uint32_t, lo), b = __builtin_bit_cast(uint32_t, hi);
    a += 0x7FFFu + ((a >> 16) & 1u);
    b += 0x7FFFu + ((b >> 16) & 1u);
    return __builtin_amdgcn_perm(b, a, 0x07060302u);
}
__device__ inline uint4 pack8_bf16(const float (&x)[8]) {
    return uint4{round_pack_bf16x2(x[0], x[1]), round_pack_bf16x2(x[2], x[3]), round_pack_bf16x2(x[4], x[5]), round_pack_bf16x2(x[6], x[7])};
}

// eight bf16 elements with their pairs cs[0..1], rotated and rounded
__device__ inline uint4 rope8_bf16(uint4 w, const float4* cs) {
    float x[8];
    load8<uint16_t>((const uint16_t*)&w, x);
    rope_pairs<8>(x, cs);
    return pack8_bf16(x);
}

// ggml's block_q8_0, identical to vsp_q8_0_quantize_row: d = amax / 127 and 1 / d (fp32 divisions), q = roundf(x / d) (half away from zero)
struct q8_scale {
    uint16_t bits;  // d as fp16
    float inverse;
};
__device__ inline q8_scale q8_block_scale(float amax) {
    const float d = __fdiv_rn(amax, 127.0f);
    return q8_scale{__builtin_bit_cast(uint16_t, (_Float16)d), d != 0.0f ? __fdiv_rn(1.0f, d) : 0.0f};
}
__device__ inline int8_t q8_round(float x, float inverse) { return (int8_t)(int)roundf(__fmul_rn(x, inverse)); }
__device__ inline uint32_t q8_pack4(const float* x, float inverse) {
    uint32_t w = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) w |= (uint32_t)(uint8_t)q8_round(x[j], inverse) << (8 * j);
    return w;
}

}  // namespace vsp
