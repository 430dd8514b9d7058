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
//  * the activation pass: Q8_0 codes + scale words (GEMV), fp16(d q) or fp16(x)
//    rows (GEMM, and F16's GEMV),
//  * the grouped GEMV (decode): 8 lanes per weight row, each lane one 32-value
//    block per 256 values, integer dots on v_dot4_i32_i8 / fp16 pairs on
//    v_dot2_f32_f16, the next product's activation pass in its epilogue.
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
template <> struct B32Fmt<2> { static constexpr int BYTES = 18, WORDS = 5; };   // Q4_0
template <> struct B32Fmt<6> { static constexpr int BYTES = 22, WORDS = 6; };   // Q5_0
template <> struct B32Fmt<8> { static constexpr int BYTES = 34, WORDS = 9; };   // Q8_0

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
// of a consumer weight type (B32Prep): Q8_0 codes [r][K] and scale words
// [r][K/32] (GEMV of Q4_0 / Q5_0 / Q8_0), fp16(d q) rows [r][ldo] (their GEMM),
// or fp16(x) rows [r][ldo] (F16, both paths); the Q8_0 scale and codes are the
// oracle's bit for bit.  Memory-bound; 8 values per thread, four threads per
// block (16-byte loads and stores; 600 rows of 2048: 5.0 us,
// one value per lane 8.5).
// Where the router's launch reads the same rows it writes them instead
// (k_route.hip).
// VEC: 16-byte aligned rows.
template <bool VEC>
__global__ void __launch_bounds__(256) k_prep_b32(const float *src, int64_t ld, int64_t nrows, int64_t K, B32Prep o) {
    const int64_t w = o.mode == B32_PREP_CODES ? K : o.ldo, nch = w / 8;   // 8-value chunks per row (a multiple of 4)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nrows * nch) return;   // the four threads of a block leave together
    const int64_t r = i / nch;
    b32_prep8<VEC>(src + r * ld, r, i - r * nch, K, o);
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
// One block (32 values) of a weight row in registers (blocks start at any even byte)
template <int WT> struct GvBlk { uint32_t w[B32Fmt<WT>::WORDS]; };
template <> struct GvBlk<1> { uint4 v[4]; };

// the WORDS dwords from the dword at or below the block's first byte: each
// holds at least one byte of the block, so no read leaves the table's pages
template <int WT>
__device__ __forceinline__ void gv_load(const uint8_t *p, GvBlk<WT> &o) {
    if constexpr (WT == 1) {
#pragma unroll
        for (int c = 0; c < 4; ++c) o.v[c] = *(const uint4 *)(p + 16 * c);
    } else {
        const uint8_t *q = p - ((uintptr_t)p & 2u);
        __builtin_memcpy(o.w, __builtin_assume_aligned(q, 4), 4 * B32Fmt<WT>::WORDS);
    }
}

// the block's codes, 4 to a dword in value order (Q4_0 / Q5_0: unsigned; F16: the values), and its scale;
// mis: 2 where the block starts in the middle of a dword, else 0
template <int WT>
__device__ __forceinline__ float gv_codes(const GvBlk<WT> &o, uint32_t mis, uint32_t (&c)[8]) {
    constexpr int NW = B32Fmt<WT>::WORDS;
    // bytes 2 + 4 i .. of the block: from word i (mis 0) or i + 1
    auto after = [&](int i) __attribute__((always_inline)) {
        const uint32_t hi = i + 1 < NW ? o.w[i + 1] : 0u;
        return mis ? hi : __builtin_amdgcn_alignbyte(hi, o.w[i], 2);
    };
    const float d = fp16_bits_to_f32(mis ? o.w[0] >> 16 : o.w[0] & 0xffffu);
    if constexpr (WT == 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) c[i] = after(i);
    } else {
        constexpr int O = WT == 6 ? 1 : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t q = after(i + O);
            c[i] = q & 0x0F0F0F0Fu;
            c[4 + i] = (q >> 4) & 0x0F0F0F0Fu;
        }
        if constexpr (WT == 6) {
            const uint32_t qh = after(0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                // fifth bits of 4 values, bit j to bit 8 j (four copies 7 bits apart, no carry), then to bit 4
                const uint32_t b = (qh >> (4 * i)) & 0xFu;
                c[i] |= (__umul24(b, 0x204081u) & 0x01010101u) << 4;
            }
        }
    }
    return d;
}

// LDS of a pass: the activation blocks of up to GV_NT tokens, GV_KS values of
// each (quant: codes, then {fp16 scale, sum of the codes} words; F16: values)
constexpr int GV_NT = 4, GV_KS = 4096, GV_WAVES = 8;
template <int WT> constexpr int gv_row() { return WT == 1 ? 2 * GV_KS : GV_KS + GV_KS / 8; }

// acc[n] += the lane's blocks sl, sl + 8, ... of its weight row times tokens
// n0 .. n0 + NT - 1 (rows s_p[n0 + n], clamped to the last), block by block
template <int WT, int NT>
__device__ __forceinline__ void gv_pass(const B32Side &s, int kdiv, const uint8_t *rowp, const int *s_p, int n0, int cnt,
                                        uint8_t *xs, float (&acc)[GV_NT], int sl, int tid) {
    constexpr int U = WT != 1 && NT == 1 ? 4 : 2;   // blocks in flight per lane
    constexpr int BB = WT == 1 ? 64 : B32Fmt<WT == 1 ? 8 : WT>::BYTES, ROW = gv_row<WT>();
    const int K = (int)s.a.K, nbr = K / 32;
#pragma unroll
    for (int n = 0; n < GV_NT; ++n) acc[n] = 0.f;
    for (int k0 = 0; k0 < nbr; k0 += GV_KS / 32) {
        const int nb = nbr - k0 < GV_KS / 32 ? nbr - k0 : GV_KS / 32;
        GvBlk<WT> w[U];
        auto load = [&](int b) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int bb = b + 8 * u < nb ? b + 8 * u : 0;   // (block 0 again: not used)
                gv_load<WT>(rowp + (int64_t)BB * (k0 + bb), w[u]);
            }
        };
        load(sl);
        if (k0 || n0) __syncthreads();   // (the activations before are read)
#pragma unroll
        for (int n = 0; n < NT; ++n) {
            const int p = s_p[n0 + n < cnt ? n0 + n : cnt - 1];
            const int64_t r = kdiv > 1 ? p / kdiv : p;
            uint8_t *o = xs + n * ROW;
            if constexpr (WT == 1) {
                const uint8_t *src = (const uint8_t *)(s.xh + r * K + 32 * k0);
                for (int i = tid; i < 4 * nb; i += 64 * GV_WAVES) *(uint4 *)(o + 16 * i) = *(const uint4 *)(src + 16 * i);
            } else {
                const uint8_t *src = (const uint8_t *)(s.q8 + r * K + 32 * k0);
                for (int i = tid; i < 2 * nb; i += 64 * GV_WAVES) *(uint4 *)(o + 16 * i) = *(const uint4 *)(src + 16 * i);
                const uint32_t *sd = s.ds + r * nbr + k0;
                for (int i = tid; i < nb; i += 64 * GV_WAVES) *(uint32_t *)(o + GV_KS + 4 * i) = sd[i];
            }
        }
        __syncthreads();
        for (int b0 = sl; b0 < nb; b0 += 8 * U) {
            if (b0 != sl) load(b0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int b = b0 + 8 * u;
                if (b >= nb) break;
                if constexpr (WT == 1) {
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        float d = 0.f;
#pragma unroll
                        for (int c = 0; c < 4; ++c) {
                            const uint4 xv = *(const uint4 *)(xs + (n * ROW + 64 * b + 16 * c));
                            const uint32_t wa[4] = {w[u].v[c].x, w[u].v[c].y, w[u].v[c].z, w[u].v[c].w};
                            const uint32_t xa[4] = {xv.x, xv.y, xv.z, xv.w};
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                d = __builtin_amdgcn_fdot2(__builtin_bit_cast(half2_t, wa[i]), __builtin_bit_cast(half2_t, xa[i]),
                                                           d, false);
                        }
                        acc[n] += d;
                    }
                } else {
                    uint32_t c[8];
                    const float dw = gv_codes<WT>(w[u], (uint32_t)(uintptr_t)(rowp + (int64_t)BB * (k0 + b)) & 2u, c);
#pragma unroll
                    for (int n = 0; n < NT; ++n) {
                        const uint4 xa = *(const uint4 *)(xs + (n * ROW + 32 * b)), xb = *(const uint4 *)(xs + (n * ROW + 32 * b + 16));
                        const uint32_t ds = *(const uint32_t *)(xs + (n * ROW + GV_KS + 4 * b));
                        const uint32_t xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
                        int isum = 0;
#pragma unroll
                        for (int i = 0; i < 8; ++i) isum = __builtin_amdgcn_sdot4((int)c[i], (int)xv[i], isum, false);
                        const float dx = fp16_bits_to_f32(ds & 0xffffu);
                        const int xsum = (int)ds >> 16;
                        // the expression orders of ggml_vec_dot_q{4,5,8}_0_q8_0
                        if constexpr (WT == 8) acc[n] += (float)isum * (dw * dx);
                        else if constexpr (WT == 6) acc[n] += (dw * dx) * (float)(isum - 16 * xsum);
                        else acc[n] += (float)(isum - 8 * xsum) * dw * dx;
                    }
                }
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        acc[n] += __shfl_xor(acc[n], 1, 64);
        acc[n] += __shfl_xor(acc[n], 2, 64);
        acc[n] += __shfl_xor(acc[n], 4, 64);
    }
}

// A work-group (8 waves) owns 64 weight rows of one active expert (GLU: 32
// gate rows and the matching up rows), a wave 8 row groups x 8 lanes (GLU:
// groups 0-3 gate, 4-7 up); lane sl takes blocks sl, sl + 8, ... of its row.
// The expert's tokens run four to a pass through LDS, a weight block decoded
// once for the four.
//
// The gate/up form writes the down product's operand itself (a GLU
// work-group's 32 columns are one Q8_0 block of each row), the bits of
// launch_prep_b32 on the fp32 values.  With g.ids the expert list comes from
// the ids: work-group row j belongs to slot j, and leaves unless the slot is
// its expert's first (and its id one of the n_expert).  SH: the shared expert's work-groups come first.
//
// What bounds it: the load path (a block is 2 - 3 loads of at most 16 bytes
// at dword-aligned addresses; the same bytes at their own, 2-byte aligned
// addresses: qwen3omni Q8_0 T = 5 gate/up 36.7 against 31.2 us, down 24.5
// against 19.8) and the work-groups in flight (four blocks ahead with one
// token in the pass, two with more: at 125 registers 16 waves per CU; eight
// ahead spills, 24 - 32 waves per CU with two tokens a pass are slower for
// many rows).  Against the form before (each lane reading its blocks dword by
// dword and the activations from the caches for every token anew, the GLU
// rows quantized by a launch of their own, a dispatch launch, the shared
// expert as a layer of its own), layer us: moondream3 Q8_0 T = 1 47.6 -> 37,
// Q4_0 T = 5 72 -> 62; qwen3omni Q8_0 T = 5 / 16 78.5 / 150 -> 71 / 131 (69
// with x's codes from the router's launch), Q5_0 T = 12 127 -> 101; nemotronomni Q5_0 T = 1 / 4 / 16 109 / 177 / 302 ->
// 47 / 80 / 176; diffusiongemma F16 T = 4 / 16 104 / 273 -> 95 / 203.
enum { GV_STORE = 0, GV_GLU = 1, GV_RELU_SQR = 2 };
template <int WT, int EPI, bool SH>
__global__ void __launch_bounds__(64 * GV_WAVES) __attribute__((amdgpu_waves_per_eu(4))) k_gemv_b32(B32Args g) {
    __shared__ __attribute__((aligned(16))) uint8_t xs[GV_NT * gv_row<WT>()];
    __shared__ float s_v[GV_NT][64];
    __shared__ int s_p[GV_SD_IDS];
    __shared__ int s_cnt[GV_WAVES];
    constexpr bool GLU = EPI == GV_GLU;
    constexpr int COLS = GLU ? 32 : 64;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int rs = lane >> 3, sl = lane & 7;
    const bool shared = SH && (int)blockIdx.x < g.sh_wgs;
    const B32Side s = shared ? g.sh : (const B32Side &)g;
    int e = 0, cnt, cb;
    const int32_t *perm = nullptr;   // the rows (null: in s_p)
    if (shared) {
        cb = blockIdx.x;
        cnt = (int)g.sh_rows;
    } else {
        const unsigned lin = blockIdx.x - (SH ? g.sh_wgs : 0), j = lin / (unsigned)g.ncb;
        cb = (int)(lin - j * (unsigned)g.ncb);
        if (g.ids) {
            const int id = tid < g.rows ? g.ids[tid] : -1;
            e = g.ids[j];
            // (before any address is formed from it; past here no thread
            // without a slot matches e)
            if ((unsigned)e >= (unsigned)g.n_expert) {
                if (g.bad_total && cb == 0 && tid == 0) atomicAdd(g.bad_total, 1);
                return;
            }
            const uint64_t m = __ballot(id == e);
            if (lane == 0) s_cnt[wave] = __popcll(m);
            __syncthreads();
            int before = 0, total = 0;
#pragma unroll
            for (int i = 0; i < GV_WAVES; ++i) {
                if (i < wave) before += s_cnt[i];
                total += s_cnt[i];
            }
            if (id == e) s_p[before + __popcll(m & ((1ull << lane) - 1))] = tid;
            __syncthreads();
            if (s_p[0] != (int)j) return;
            cnt = total;
        } else {
            if ((int)j >= *g.n_active) return;
            e = g.active_e[j];
            cnt = g.counts[e];
            perm = g.perm + g.offsets[e];
        }
    }
    const int64_t col = (int64_t)cb * COLS + wave * (COLS / GV_WAVES) + (GLU ? (rs & 3) : rs);
    const bool col_ok = col < s.ncols;
    int64_t wrow = col_ok ? col : 0;
    const uint8_t *rowp = s.a.data + (int64_t)e * s.a.mat_bytes;
    int64_t rb = s.a.row_bytes;
    if (GLU && rs >= 4) {
        if (s.fused) {
            wrow += s.I;
        } else {
            rowp = s.b.data + (int64_t)e * s.b.mat_bytes;
            rb = s.b.row_bytes;
        }
    }
    rowp += wrow * rb;
    const int kdiv = g.ne11 == 1 && !shared ? g.K : 1;
    for (int q0 = 0; q0 < cnt; q0 += GV_SD_IDS) {   // (rows that fit s_p)
        const int qn = cnt - q0 < GV_SD_IDS ? cnt - q0 : GV_SD_IDS;
        if (shared || perm) {
            if (q0) __syncthreads();
            for (int i = tid; i < qn; i += 64 * GV_WAVES) s_p[i] = shared ? q0 + i : perm[q0 + i];
            __syncthreads();
        }
        for (int n0 = 0; n0 < qn; n0 += GV_NT) {
            const int nt = qn - n0 < GV_NT ? qn - n0 : GV_NT;
            float acc[GV_NT];
            if (nt == 1) gv_pass<WT, 1>(s, kdiv, rowp, s_p, n0, qn, xs, acc, sl, tid);
            else if (nt == 2) gv_pass<WT, 2>(s, kdiv, rowp, s_p, n0, qn, xs, acc, sl, tid);
            else gv_pass<WT, GV_NT>(s, kdiv, rowp, s_p, n0, qn, xs, acc, sl, tid);
            if constexpr (EPI == GV_STORE) {
#pragma unroll
                for (int n = 0; n < GV_NT; ++n) {
                    if (n >= nt || sl != 0 || !col_ok) continue;
                    const int p = s_p[n0 + n];
                    s.y[(int64_t)p * s.ldy + col] = shared && g.sh_w ? acc[n] * g.sh_w[p] : acc[n];
                }
            } else {
#pragma unroll
                for (int n = 0; n < GV_NT; ++n) {
                    if (n >= nt) continue;
                    const float other = GLU ? __shfl(acc[n], (lane + 32) & 63, 64) : 0.f;
                    if (sl == 0 && (!GLU || rs < 4))
                        s_v[n][wave * (COLS / GV_WAVES) + rs] = GLU ? act_pair(g.act, acc[n], other) : relu_sqr(acc[n]);
                }
                __syncthreads();
                const int n = tid / (COLS / 8), c8 = tid % (COLS / 8);   // 8 values per thread, four threads per block
                const int64_t c0 = (int64_t)cb * COLS + 8 * c8;
                if (n < nt && c0 < s.ncols) {
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i) v[i] = s_v[n][8 * c8 + i];
                    const int64_t p = s_p[n0 + n];
                    if (g.next_f16) *(uint4 *)(s.oxh + p * s.ncols + c0) = b32_f16x8(v);
                    else b32_store_codes(v, s.oq8 + p * s.ncols + c0, s.ods + p * (s.ncols / 32) + c0 / 32, (c8 & 3) == 0);
                }
                // (s_v is written again after the barrier in front of the next pass's products)
            }
        }
    }
}

// ------------------------------------------------------------------ launch
template <int WT, int EPI>
static int gv_launch(const B32Args &a, hipStream_t st) {
    B32Args g = a;
    constexpr int COLS = EPI == GV_GLU ? 32 : 64;
    g.ncb = (int)((g.ncols + COLS - 1) / COLS);
    g.sh_wgs = g.sh_rows > 0 ? (int)((g.sh.ncols + COLS - 1) / COLS) : 0;
    const int64_t wgs = g.sh_wgs + (int64_t)g.ncb * (g.ids ? g.rows : g.max_active);
    if (wgs > 0x7fffffff) return -6;
    const dim3 grid((unsigned)wgs), block(64 * GV_WAVES);
    if (g.sh_wgs) hipLaunchKernelGGL((k_gemv_b32<WT, EPI, true>), grid, block, 0, st, g);
    else hipLaunchKernelGGL((k_gemv_b32<WT, EPI, false>), grid, block, 0, st, g);
    return hip_check_launch();
}

int launch_gemv_b32(const B32Args &g, hipStream_t st) {
    if (g.max_active <= 0) return 0;
    if (g.a.K % 32 || g.a.K > 0x7fffffff) return -6;
    if (g.ids && (g.rows > GV_SD_IDS || g.n_expert <= 0)) return -6;
    if ((g.glu || g.relu_sqr) && g.ncols % 32) return -6;
    if (g.sh_rows > 0 && (g.sh.a.type != g.a.type || g.sh.a.K % 32 || ((g.glu || g.relu_sqr) && g.sh.ncols % 32))) return -6;
#define GV_TYPE(T)                                                \
    case T:                                                       \
        if (g.glu) return gv_launch<T, GV_GLU>(g, st);            \
        if (g.relu_sqr) return gv_launch<T, GV_RELU_SQR>(g, st);  \
        return gv_launch<T, GV_STORE>(g, st);
    switch (g.a.type) {
        GV_TYPE(1)
        GV_TYPE(2)
        GV_TYPE(6)
        GV_TYPE(8)
    default: return -3;
    }
#undef GV_TYPE
}

}  // namespace mimoe
