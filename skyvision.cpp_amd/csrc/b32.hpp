// b32.hpp - 8 consecutive values of a 32-value block as the operand of a
// 32-value type's product: ggml's Q8_0 (quantize_row_q8_0_ref: d = amax / 127
// as fp16, q = roundf(x / d)) by the four lanes 4 k .. 4 k + 3 that hold the
// block, or the fp16 rounding that F16 tables take.
#pragma once

#include "common.hpp"
#include "launch.hpp"
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

// the lane's 8 codes to q8 and (lead: the first lane of the four) the block's
// word {fp16 d, sum of its 32 codes << 16} to ds
__device__ __forceinline__ void b32_store_codes(const float (&v)[8], int8_t *q8, uint32_t *ds, bool lead) {
    int q[8];
    uint32_t dh;
    b32_q8_codes(v, q, dh);
    uint32_t c[2] = {0u, 0u};
#pragma unroll
    for (int j = 0; j < 8; ++j) c[j >> 2] |= (uint32_t)(q[j] & 0xff) << (8 * (j & 3));
    int sum = __builtin_amdgcn_sdot4(0x01010101, (int)c[0], __builtin_amdgcn_sdot4(0x01010101, (int)c[1], 0, false), false);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xf, 0xf, true);
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x4E, 0xf, 0xf, true);
    *(uint2 *)q8 = make_uint2(c[0], c[1]);
    if (lead) *ds = dh | (uint32_t)sum << 16;
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

// values 8 c .. 8 c + 7 of row r (at x, K values) as o asks
template <bool VEC>
__device__ __forceinline__ void b32_prep8(const float *row, int64_t r, int64_t c, int64_t K, const B32Prep &o) {
    float v[8];
    if (8 * c < K) {
        const float *x = row + 8 * c;
        if constexpr (VEC) {
            const float4 a = *(const float4 *)x, b = *(const float4 *)(x + 4);
            v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
        } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] = x[j];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = 0.f;
    }
    if (o.mode == B32_PREP_CODES) b32_store_codes(v, o.q8 + r * K + 8 * c, o.ds + r * (K / 32) + c / 4, (c & 3) == 0);
    else *(uint4 *)(o.xh + r * o.ldo + 8 * c) = o.mode == B32_PREP_F16 ? b32_f16x8(v) : b32_q8x8(v);
}

}  // namespace mimoe
