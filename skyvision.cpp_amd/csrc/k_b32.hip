// k_b32.hip - expert tables in the 32-value block formats (Q4_0, Q5_0, Q8_0)
// and in F16: the types the reference's converters write by default (Q8_0:
// convert/convert_hf_to_gguf.py:55-57, convert/convert_qwen3omni.py:60-61,135;
// Q5_0: convert/convert_nemotronomni.py:113-114; F16 / Q4_0:
// convert/convert_diffusiongemma.py:62).
//
// ggml-cpu semantics (ggml_mul_mat_id with these tables): the activation rows
// are converted to the weight type's vec_dot_type first, Q8_0 (32-value blocks,
// d = amax / 127 stored as fp16) for Q4_0 / Q5_0 / Q8_0 and fp16 (round to
// nearest even) for F16; each block then contributes an exact integer dot
// times the two fp16 scales, F16 rows exact fp16 x fp16 products.
//
//  * quantizers of weight rows (mi_quantize; ggml quantize_row_*_ref),
//  * the activation pass: Q8_0 codes + fp16 scales (GEMV), fp16(d q) or fp16(x)
//    rows (GEMM, and F16's GEMV),
//  * the grouped GEMV (decode): 8 lanes per weight row, each lane one 32-value
//    block per 256 values, integer dots on v_dot4_i32_i8 / fp16 pairs on
//    v_dot2_f32_f16.
// The grouped GEMM (prefill) is k_gb.hip.
//
// Block layouts (ggml block_q4_0 / q5_0 / q8_0, no padding, so blocks start
// at any even byte):
//   Q4_0 18 B: d f16 | qs[16]            value j < 16: low nibble of qs[j], 16 + j: high; x = d (q - 8)
//   Q5_0 22 B: d f16 | qh u32 | qs[16]   5th bit of value j: bit j of qh;                 x = d (q - 16)
//   Q8_0 34 B: d f16 | qs[32] i8                                                          x = d q
#include "act.hpp"
#include "b32.hpp"
#include "common.hpp"
#include "launch.hpp"

namespace mimoe {

template <int WT> struct B32Fmt;
template <> struct B32Fmt<2> { static constexpr int BYTES = 18, WORDS = 5, OFF = 8; };    // Q4_0
template <> struct B32Fmt<6> { static constexpr int BYTES = 22, WORDS = 6, OFF = 16; };   // Q5_0
template <> struct B32Fmt<8> { static constexpr int BYTES = 34, WORDS = 9, OFF = 0; };    // Q8_0

// ------------------------------------------------------------------ block loads
// The WORDS aligned dwords that intersect the block at p (an even address; a
// block spans WORDS dwords at either alignment).  Every dword read holds at
// least one byte of the block, so no read leaves the table's pages.
template <int WT>
__device__ inline void b32_words(const uint8_t *p, uint32_t (&w)[B32Fmt<WT>::WORDS], uint32_t &mis) {
    const uintptr_t a = (uintptr_t)p;
    mis = (uint32_t)(a & 2u);
    const uint32_t *q = (const uint32_t *)(a - mis);
#pragma unroll
    for (int i = 0; i < B32Fmt<WT>::WORDS; ++i) w[i] = q[i];
}
// the 4 block bytes from byte offset OFF (even): bytes [mis + OFF, ...) of
// the words (compile-time word indices keep the words in registers)
template <int OFF, int N>
__device__ inline uint32_t b32_dword(const uint32_t (&w)[N], uint32_t mis) {
    constexpr int k = OFF >> 2;   // OFF % 4 is 0 or 2
    if constexpr ((OFF & 2) == 0) return mis ? __builtin_amdgcn_alignbyte(w[k + 1], w[k], 2) : w[k];
    else return mis ? w[k + 1] : __builtin_amdgcn_alignbyte(w[k + 1], w[k], 2);
}
__device__ inline float b32_d(uint32_t w0, uint32_t mis) {
    return fp16_bits_to_f32(mis ? (w0 >> 16) : (w0 & 0xffffu));
}

// signed codes of values 4i .. 4i + 3 of the block as bytes, i < 8 (Q8_0:
// the codes; Q4_0 / Q5_0: the unsigned codes q, the offset is applied by the
// caller through the block's activation sum)
template <int WT, int I>
__device__ inline uint32_t b32_codes4(const uint32_t (&w)[B32Fmt<WT>::WORDS], uint32_t mis) {
    if constexpr (WT == 8) {
        return b32_dword<2 + 4 * I>(w, mis);
    } else {
        constexpr int QS = WT == 2 ? 2 : 6;
        const uint32_t qs = b32_dword<QS + 4 * (I & 3)>(w, mis);
        uint32_t v = I < 4 ? (qs & 0x0F0F0F0Fu) : ((qs >> 4) & 0x0F0F0F0Fu);
        if constexpr (WT == 6) {
            const uint32_t qh = b32_dword<2>(w, mis);
            const uint32_t b = (qh >> (4 * I)) & 0xFu;   // 5th bits of values 4I .. 4I + 3
            v |= ((b & 1u) << 4) | ((b & 2u) << 11) | ((b & 4u) << 18) | ((b & 8u) << 25);
        }
        return v;
    }
}
template <int WT, int I = 0>
__device__ inline void b32_codes_all(const uint32_t (&w)[B32Fmt<WT>::WORDS], uint32_t mis, uint32_t (&c)[8]) {
    c[I] = b32_codes4<WT, I>(w, mis);
    if constexpr (I < 7) b32_codes_all<WT, I + 1>(w, mis, c);
}

// ------------------------------------------------------------------ quantizers
// One thread per 32-value block, the oracle's statement order (the scale and
// codes bit for bit; fp16 by integer rounding, independent of denormal mode).
template <int WT>
__global__ void __launch_bounds__(256) k_quantize_b32(const float *src, uint8_t *dst, int64_t nblocks) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nblocks) return;
    const float *x = src + i * 32;
    if constexpr (WT == 1) {
        uint32_t *o = (uint32_t *)(dst + i * 64);
#pragma unroll
        for (int j = 0; j < 16; ++j) o[j] = f32_to_fp16_bits(x[2 * j]) | (f32_to_fp16_bits(x[2 * j + 1]) << 16);
        return;
    }
    uint8_t *y = dst + i * B32Fmt<WT == 1 ? 8 : WT>::BYTES;
    if constexpr (WT == 8) {
        float amax = 0.0f;
        for (int j = 0; j < 32; ++j) amax = fmaxf(amax, fabsf(x[j]));
        const float d = amax / 127.0f;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const uint32_t dh = f32_to_fp16_bits(d);
        y[0] = (uint8_t)dh;
        y[1] = (uint8_t)(dh >> 8);
        for (int j = 0; j < 32; ++j) y[2 + j] = (uint8_t)(int8_t)roundf(x[j] * id);
    } else {
        constexpr float NEG = WT == 2 ? -8.0f : -16.0f;
        constexpr float ADD = WT == 2 ? 8.5f : 16.5f;
        constexpr int TOP = WT == 2 ? 15 : 31;
        float amax = 0.0f, mx = 0.0f;
        for (int j = 0; j < 32; ++j) {
            const float v = x[j];
            if (amax < fabsf(v)) {
                amax = fabsf(v);
                mx = v;
            }
        }
        const float d = mx / NEG;
        const float id = d != 0.0f ? 1.0f / d : 0.0f;
        const uint32_t dh = f32_to_fp16_bits(d);
        y[0] = (uint8_t)dh;
        y[1] = (uint8_t)(dh >> 8);
        uint32_t qh = 0;
        uint8_t *qs = y + (WT == 2 ? 2 : 6);
        for (int j = 0; j < 16; ++j) {
            const float x0 = x[j] * id, x1 = x[16 + j] * id;
            const int8_t t0 = (int8_t)(x0 + ADD), t1 = (int8_t)(x1 + ADD);
            const uint32_t c0 = (uint32_t)(uint8_t)(t0 < TOP ? t0 : TOP);
            const uint32_t c1 = (uint32_t)(uint8_t)(t1 < TOP ? t1 : TOP);
            qs[j] = (uint8_t)((c0 & 0x0Fu) | ((c1 & 0x0Fu) << 4));
            qh |= ((c0 & 0x10u) >> 4) << j;
            qh |= ((c1 & 0x10u) >> 4) << (j + 16);
        }
        if constexpr (WT == 6)
            for (int b = 0; b < 4; ++b) y[2 + b] = (uint8_t)(qh >> (8 * b));
    }
}

int launch_quantize_b32(int type, const float *src, void *dst, int64_t nblocks, hipStream_t st) {
    if (nblocks <= 0) return 0;
    const dim3 grid((unsigned)((nblocks + 255) / 256));
    uint8_t *o = (uint8_t *)dst;
    switch (type) {
    case 1: hipLaunchKernelGGL(k_quantize_b32<1>, grid, dim3(256), 0, st, src, o, nblocks); break;
    case 2: hipLaunchKernelGGL(k_quantize_b32<2>, grid, dim3(256), 0, st, src, o, nblocks); break;
    case 6: hipLaunchKernelGGL(k_quantize_b32<6>, grid, dim3(256), 0, st, src, o, nblocks); break;
    case 8: hipLaunchKernelGGL(k_quantize_b32<8>, grid, dim3(256), 0, st, src, o, nblocks); break;
    default: return -3;
    }
    return hip_check_launch();
}

// ------------------------------------------------------------------ activations
// Rows of K values (K % 32 == 0, row r at src + r * ld) into the operand form
// of a consumer weight type (B32Prep): Q8_0 codes [r][K] and fp16 scales
// [r][K/32] (GEMV of Q4_0 / Q5_0 / Q8_0), fp16(d q) rows [r][ldo] (their GEMM),
// or fp16(x) rows [r][ldo] (F16, both paths); the Q8_0 scale and codes are the
// oracle's bit for bit.  Memory-bound; 8 values per thread, four threads per
// block (16-byte loads and stores; 600 rows of 2048: 5.0 us,
// one value per lane 8.5).
// VEC: 16-byte aligned rows.
template <bool VEC>
__global__ void __launch_bounds__(256) k_prep_b32(const float *src, int64_t ld, int64_t nrows, int64_t K, B32Prep o) {
    const int64_t w = o.mode == B32_PREP_CODES ? K : o.ldo, nch = w / 8;   // 8-value chunks per row (a multiple of 4)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrows * nch) return;   // the four threads of a block leave together
    const int64_t r = i / nch, c = i - r * nch;
    float v[8];
    if (8 * c < K) {
        const float *x = src + r * ld + 8 * c;
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
    if (o.pre_act == 4) {   // ggml_sqr(ggml_relu(u)) before the quantization
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = relu_sqr(v[j]);
    }
    if (o.mode == B32_PREP_CODES) {
        int q[8];
        uint32_t dh;
        b32_q8_codes(v, q, dh);
        uint32_t lo = 0, hi = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            lo |= (uint32_t)(q[j] & 0xff) << (8 * j);
            hi |= (uint32_t)(q[4 + j] & 0xff) << (8 * j);
        }
        *(uint2 *)(o.q8 + r * K + 8 * c) = make_uint2(lo, hi);
        if ((c & 3) == 0) o.dh[r * (K / 32) + c / 4] = (uint16_t)dh;
    } else {
        *(uint4 *)(o.xh + r * o.ldo + 8 * c) = o.mode == B32_PREP_F16 ? b32_f16x8(v) : b32_q8x8(v);
    }
}

int launch_prep_b32(const float *src, int64_t ld, int64_t nrows, int64_t K, const B32Prep &o, hipStream_t st) {
    if (nrows <= 0) return 0;
    if (K % 32) return -6;
    if (o.mode != B32_PREP_CODES && (o.ldo < K || o.ldo % 32)) return -6;
    const int64_t threads = nrows * ((o.mode == B32_PREP_CODES ? K : o.ldo) / 8);
    const dim3 grid((unsigned)((threads + 255) / 256));
    const bool vec = ld % 4 == 0 && (uintptr_t)src % 16 == 0;
    if (vec) hipLaunchKernelGGL(k_prep_b32<true>, grid, dim3(256), 0, st, src, ld, nrows, K, o);
    else hipLaunchKernelGGL(k_prep_b32<false>, grid, dim3(256), 0, st, src, ld, nrows, K, o);
    return hip_check_launch();
}

// ------------------------------------------------------------------ GEMV
// dot of one 32-value block (this lane's) with the activation row's block
template <int WT>
__device__ inline float b32_block_dot(const uint8_t *wblk, const int8_t *xq, float dx) {
    uint32_t w[B32Fmt<WT>::WORDS], mis;
    b32_words<WT>(wblk, w, mis);
    const uint4 xa = *(const uint4 *)xq, xb = *(const uint4 *)(xq + 16);
    const uint32_t xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
    uint32_t cw[8];
    b32_codes_all<WT>(w, mis, cw);
    int isum = 0, xsum = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        isum = __builtin_amdgcn_sdot4((int)cw[i], (int)xv[i], isum, false);
        if constexpr (WT != 8) xsum = __builtin_amdgcn_sdot4(0x01010101, (int)xv[i], xsum, false);
    }
    const float dw = b32_d(w[0], mis);
    // the expression orders of ggml_vec_dot_q{4,5,8}_0_q8_0
    if constexpr (WT == 8) return (float)isum * (dw * dx);
    else if constexpr (WT == 6) return (dw * dx) * (float)(isum - 16 * xsum);
    else return (float)(isum - 8 * xsum) * dw * dx;
}

__device__ inline float f16_block_dot(const uint8_t *wblk, const _Float16 *xh) {
    float acc = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const uint4 wv = *(const uint4 *)(wblk + 16 * c);
        const uint4 xv = *(const uint4 *)(xh + 8 * c);
        const uint32_t wa[4] = {wv.x, wv.y, wv.z, wv.w}, xa[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
        for (int i = 0; i < 4; ++i)
            acc = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, wa[i]), __builtin_bit_cast(half2_t, xa[i]),
                                         acc, false);
    }
    return acc;
}

// Grid (column blocks, active experts), 4 waves of 8 row groups x 8 lanes; a
// row group owns one weight row (GLU: groups 0-3 the gate rows, 4-7 the
// matching up rows), lane sl takes blocks sl, sl + 8, ... of it for every
// token of the expert (the row's bytes come from HBM once, from the caches
// for the later tokens).
template <int WT>
__global__ void __launch_bounds__(256) k_gemv_b32(B32Args g) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int rs = lane >> 3, sl = lane & 7;
    const int j = blockIdx.y;
    if (j >= *g.n_active) return;
    const int e = g.active_e[j];
    const int cnt = g.counts[e], off = g.offsets[e];
    const bool glu = g.glu != 0;
    const int64_t col0 = ((int64_t)blockIdx.x * 4 + wave) * (glu ? 4 : 8);
    int64_t col = col0 + (glu ? (rs & 3) : rs);
    const bool col_ok = col < g.ncols;
    if (!col_ok) col = 0;
    const ExpertMat *M = &g.a;
    int64_t wrow = col;
    if (glu && rs >= 4) {
        if (g.fused) wrow = g.I + col;
        else M = &g.b;
    }
    const uint8_t *rowp = M->data + (int64_t)e * M->mat_bytes + wrow * M->row_bytes;
    const int64_t Kin = M->K, nbr = Kin / 32;
    for (int m = 0; m < cnt; ++m) {
        const int p = g.perm[off + m];
        const int64_t arow = g.ne11 == 1 ? p / g.K : p;
        float acc = 0.f;
        for (int64_t b = sl; b < nbr; b += 8) {
            if constexpr (WT == 1) {
                acc += f16_block_dot(rowp + 64 * b, g.xh + arow * Kin + 32 * b);
            } else {
                const float dx = fp16_bits_to_f32(g.dh[arow * nbr + b]);
                acc += b32_block_dot<WT>(rowp + (int64_t)B32Fmt<WT>::BYTES * b, g.q8 + arow * Kin + 32 * b, dx);
            }
        }
        acc += __shfl_xor(acc, 1, 64);
        acc += __shfl_xor(acc, 2, 64);
        acc += __shfl_xor(acc, 4, 64);
        if (glu) {
            const float other = __shfl(acc, lane + 32 < 64 ? lane + 32 : lane, 64);
            if (rs < 4 && sl == 0 && col_ok) g.y[(int64_t)p * g.ldy + col] = act_pair(g.act, acc, other);
        } else {
            if (sl == 0 && col_ok) g.y[(int64_t)p * g.ldy + col] = acc;
        }
    }
}

// ------------------------------------------------------------------ launch
int launch_gemv_b32(const B32Args &g, hipStream_t st) {
    if (g.max_active <= 0) return 0;
    if (g.a.K % 32) return -6;
    const int64_t per_block = (g.glu ? 4 : 8) * 4;
    const dim3 grid((unsigned)((g.ncols + per_block - 1) / per_block), (unsigned)g.max_active);
    switch (g.a.type) {
    case 1: hipLaunchKernelGGL(k_gemv_b32<1>, grid, dim3(256), 0, st, g); break;
    case 2: hipLaunchKernelGGL(k_gemv_b32<2>, grid, dim3(256), 0, st, g); break;
    case 6: hipLaunchKernelGGL(k_gemv_b32<6>, grid, dim3(256), 0, st, g); break;
    case 8: hipLaunchKernelGGL(k_gemv_b32<8>, grid, dim3(256), 0, st, g); break;
    default: return -3;
    }
    return hip_check_launch();
}

}  // namespace mimoe
