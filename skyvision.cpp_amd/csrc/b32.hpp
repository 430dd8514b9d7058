// b32.hpp - 8 consecutive values of a 32-value block as the operand of a
// 32-value type's product: ggml's Q8_0 (quantize_row_q8_0_ref: d = amax / 127
// as fp16, q = roundf(x / d)) by the four lanes 4 k .. 4 k + 3 that hold the
// block, or the fp16 rounding that F16 tables take.
#pragma once

#include "common.hpp"
#include "wave_ops.hpp"

namespace mimoe {

__device__ __forceinline__ uint4 b32_f16x8(const float (&v)[8]) {
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) h[j] = f32_to_fp16_bits(v[2 * j]) | (f32_to_fp16_bits(v[2 * j + 1]) << 16);
    return make_uint4(h[0], h[1], h[2], h[3]);
}

// the lane's 8 codes and the block's fp16 scale (bits)
__device__ __forceinline__ void b32_q8_codes(const float (&v)[8], int (&q)[8], uint32_t &dh) {
    float amax = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) amax = fmaxf(amax, fabsf(v[j]));
    amax = fmaxf(amax, dpp_f<0xB1>(amax));   // the other lanes of the four
    amax = fmaxf(amax, dpp_f<0x4E>(amax));
    const float d = amax / 127.0f;
    const float id = d != 0.0f ? 1.0f / d : 0.0f;
    dh = f32_to_fp16_bits(d);
#pragma unroll
    for (int j = 0; j < 8; ++j) q[j] = (int)roundf(v[j] * id);
}

// the same as fp16(d q)
__device__ __forceinline__ uint4 b32_q8x8(const float (&v)[8]) {
    int q[8];
    uint32_t dh;
    b32_q8_codes(v, q, dh);
    const float d = fp16_bits_to_f32(dh);
    uint32_t h[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        half2_t p;
        p[0] = (_Float16)(d * (float)q[2 * j]);
        p[1] = (_Float16)(d * (float)q[2 * j + 1]);
        h[j] = __builtin_bit_cast(uint32_t, p);
    }
    return make_uint4(h[0], h[1], h[2], h[3]);
}

}  // namespace mimoe
