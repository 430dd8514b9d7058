// k_gb.hip - grouped MFMA GEMM of the 32-value block formats (Q4_0, Q5_0,
// Q8_0) and F16 expert tables: gate/up with the GLU (or relu^2) and the next
// product's activation operand in the epilogue, and the plain product.
//
// A work-group of NW waves owns a balanced tile of at most BM dispatched rows
// of one expert and 64 NW weight rows: each wave two column tiles of 32 (GLU:
// the gate rows and the matching up rows of its 32 act columns) against the
// tile's row tiles of 32 on v_mfma_f32_32x32x16_f16, so each activation
// operand read from LDS feeds two MFMAs and each dequantized weight operand
// one per row tile.
//
// The K loop runs over groups of 64 values = two blocks.  Lane half h of the
// MFMA takes block h of the group: step s multiplies values 8 s .. 8 s + 7 of
// both blocks, so a lane needs one whole block of its weight row per group
// (one scale) and the activations stay in their natural order (K chunk 4 h +
// s).
//
// Both operands reach LDS by buffer loads that write LDS directly:
//  * weights, KG groups (a stage) at a time into a buffer of the wave's own:
//    each row's run of the stage as 16-byte pieces from the dword at or below
//    its first byte (blocks start at any even byte, and rows may be
//    misaligned), 80 - 280 bytes of a row at a time.  The lanes take their
//    blocks out into registers (v_alignbyte by the block's misalignment),
//    which frees the buffer for the next stage's loads while this one is
//    computed.
//  * activations, KG / 2 groups at a time, double buffered: 128 bytes per row
//    and group, piece c of row r in slot c ^ (r & 7); rows past the tile read
//    out of range (no memory traffic).
// Dequantization (in registers) and the LDS reads of the next step sit
// between the MFMAs of a step.
//
// What bounds it (timing-only copies without the loads, or without the
// arithmetic): the weight stream, by the length of its runs - Q5_0 rows (K
// 2688) in runs of 44, 88 and 176 bytes: 152, 121 and 105 us for 439 MB, as
// contiguous memory 88 - and beside it the dequantization (Q5_0 104 us alone,
// 142 with the stream); F16 gate/up streams at 5.5 TB/s (1.02 GB in 186 us).
// Against the form before (weights loaded by each lane for itself, dword by
// dword, 192-row tiles), kernel times under the profiler: Q8_0 moondream3 T =
// 600 gate/up 268 -> 104 us, down 127 -> 66 us, and the GLU rows' pass (13.7
// us) is in the epilogue; diffusiongemma F16 T = 256 257 -> 186 and 135 -> 107
// us; nemotronomni Q5_0 T = 200 up 333 -> 134 us (165 with the shared expert
// in it).
#include "act.hpp"
#include "b32.hpp"
#include "common.hpp"
#include "launch.hpp"
#include "wave_ops.hpp"

namespace mimoe {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void_t;
typedef __amdgpu_buffer_rsrc_t rsrc_t;

// BB: bytes of a block; G: of a 64-value group
template <int WT> struct GBFmt;
template <> struct GBFmt<1> { static constexpr int BB = 64, G = 128; };
template <> struct GBFmt<2> { static constexpr int BB = 18, G = 36; };
template <> struct GBFmt<6> { static constexpr int BB = 22, G = 44; };
template <> struct GBFmt<8> { static constexpr int BB = 34, G = 68; };
// 16-byte pieces of a row that hold KG groups from the dword at or below the
// first (quant: an odd number, so that the rows of a column tile start on 16
// different banks), and the loads of a column tile's 32 rows
template <int WT, int KG> constexpr int gb_pieces() {
    return WT == 1 ? 8 * KG : ((GBFmt<WT>::G * KG + 2 + 15) / 16) | 1;
}
template <int WT, int KG> constexpr int gb_loads() { return (gb_pieces<WT, KG>() + 1) / 2; }
template <int WT, int KG> constexpr int gb_wtile() { return 1024 * gb_loads<WT, KG>(); }   // bytes of a column tile

enum { GB_STORE = 0, GB_GLU = 1, GB_RELU_SQR = 2 };

constexpr uint32_t GB_FAR = 0xF8000000u;   // an offset past xh (at most GB_MAX_X bytes), far from wrapping

__device__ inline rsrc_t gb_rsrc(const void *p, uint32_t nbytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)nbytes, 0x00020000);
}

// at most N vector-memory loads of this wave outstanding and no LDS access, then the barrier
template <int N>
__device__ __forceinline__ void gb_sync() {
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4));
    asm volatile("s_barrier" ::: "memory");
}

// the weight loads of one column tile (32 rows) of the wave
template <int WT, int KG> struct GBW {
    static constexpr int PC = gb_pieces<WT, KG>(), NLD = gb_loads<WT, KG>();
    rsrc_t r;
    uint32_t off[NLD];   // byte offset at stage 0 of load j's piece of this lane
    // where the lane finds its block of group 0 in the weight buffer (quant:
    // its codes' first dword and its scale; F16: its row), and the byte shift
    // of the codes into place
    uint32_t at, dat, sh;

    // stage st's loads to dst
    __device__ __forceinline__ void issue(uint8_t *dst, int st) const {
        rsrc_t res = r;   // the builtin takes no const-qualified resource
#pragma unroll
        for (int j = 0; j < NLD; ++j)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(res, (lds_void_t *)(dst + 1024 * j), 16, (int)off[j],
                                                     GBFmt<WT>::G * KG * st, 0, 0);
    }
};

// rows n0 .. n0 + 31 of the matrix at mat (N rows of K values, rb bytes apart;
// rows past N read zeros), staged at byte base of the weight buffer
template <int WT, int KG>
__device__ __forceinline__ GBW<WT, KG> gb_wdesc(const uint8_t *mat, int64_t n0, int64_t N, int64_t rb, int64_t K, int lane,
                                                uint32_t base) {
    using F = GBFmt<WT>;
    GBW<WT, KG> d;
    constexpr int PC = GBW<WT, KG>::PC;
    const uint32_t l32 = (uint32_t)lane & 31u, h = (uint32_t)lane >> 5;
    const uint32_t row = base + l32 * (16u * PC);
    const int64_t left = N - n0;
    const uint8_t *p = mat + (left > 0 ? n0 : 0) * rb;
    const uint32_t mis = WT == 1 ? 0u : (uint32_t)((uintptr_t)p & 3u);
    const int64_t rows = left < 32 ? left : 32;
    const uint32_t bytes = left > 0 ? (uint32_t)(mis + (rows - 1) * rb + K / 32 * F::BB + 3) & ~3u : 0u;
    d.r = gb_rsrc(p - mis, bytes);
#pragma unroll
    for (int j = 0; j < GBW<WT, KG>::NLD; ++j) {
        const uint32_t q = 64u * (uint32_t)j + (uint32_t)lane, r = q / PC, k = q - r * PC;
        if constexpr (WT == 1) d.off[j] = r * (uint32_t)rb + 16u * (k ^ (r & 7u));
        else d.off[j] = r < 32 ? ((mis + r * (uint32_t)rb) & ~3u) + 16u * k : 0x80000000u;   // (past the resource)
    }
    if constexpr (WT == 1) {
        d.at = row;
        d.dat = d.sh = 0;
    } else {
        const uint32_t b = ((mis + l32 * (uint32_t)rb) & 3u) + h * F::BB;   // the block's first byte in the row's pieces
        d.dat = row + b;
        d.at = row + ((b + 2u) & ~3u);
        d.sh = (b + 2u) & 3u;
    }
    return d;
}

// the lane's block of one group in registers (zero: a zero block)
template <int WT> struct GBRaw { uint32_t q[WT == 8 ? 8 : 4], qh; half2_t d2; };
template <> struct GBRaw<1> { u32x4 v[4]; };

template <int WT, int KG>
__device__ __forceinline__ void gb_read(const GBW<WT, KG> &d, const uint8_t *w, int g, int lane, bool zero, GBRaw<WT> &o) {
    using F = GBFmt<WT>;
    if constexpr (WT == 1) {
        const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const u32x4 v = *(const u32x4 *)(w + (d.at + 16u * (uint32_t)(8 * g + ((4 * h + s) ^ (l32 & 7)))));
            o.v[s] = zero ? u32x4{0u, 0u, 0u, 0u} : v;
        }
    } else {
        constexpr int NW = WT == 8 ? 8 : WT == 6 ? 5 : 4;
        uint32_t v[NW + 1];
#pragma unroll
        for (int i = 0; i <= NW; ++i) v[i] = *(const uint32_t *)(w + (d.at + (uint32_t)(F::G * g + 4 * i)));
        uint16_t db = *(const uint16_t *)(w + (d.dat + (uint32_t)(F::G * g)));
        if (zero) db = 0;
        const _Float16 dh = __builtin_bit_cast(_Float16, db);
        o.d2 = half2_t{dh, dh};
        constexpr int O = WT == 6 ? 1 : 0;   // Q5_0: the fifth bits first
        if constexpr (WT == 6) o.qh = __builtin_amdgcn_alignbyte(v[1], v[0], d.sh);
#pragma unroll
        for (int i = 0; i < NW - O; ++i) o.q[i] = __builtin_amdgcn_alignbyte(v[i + O + 1], v[i + O], d.sh);
    }
}

// 4 unsigned byte codes -> (code - off) * d: bytes into fp16 1024 + code
// (exact), minus 1024 + off (exact), times d (one rounding)
__device__ __forceinline__ void gb_bytes(uint32_t x, float off, half2_t d2, uint32_t &lo, uint32_t &hi) {
    const _Float16 c = (_Float16)(1024.0f + off);
    const half2_t cc = {c, c};
    const half2_t a = (__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, x, 0x04010400u)) - cc) * d2;
    const half2_t b = (__builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, x, 0x04030402u)) - cc) * d2;
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, b);
}

// weight operand of step s: values 8 s .. 8 s + 7 of the lane's block
template <int WT, int S>
__device__ __forceinline__ half8_t gb_operand(const GBRaw<WT> &r) {
    if constexpr (WT == 1) {
        return __builtin_bit_cast(half8_t, r.v[S]);
    } else {
        uint32_t c[2];
        if constexpr (WT == 8) {
            c[0] = r.q[2 * S] ^ 0x80808080u;   // signed -> q + 128
            c[1] = r.q[2 * S + 1] ^ 0x80808080u;
        } else {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const uint32_t qs = r.q[2 * (S & 1) + i];   // values 0-15: low nibbles, 16-31: high
                c[i] = (S < 2 ? qs : qs >> 4) & 0x0F0F0F0Fu;
                if constexpr (WT == 6) {
                    // fifth bits of 4 values, bit j to bit 8 j (four copies 7 bits apart, no carry), then to bit 4
                    const uint32_t b = (r.qh >> (8 * S + 4 * i)) & 0xFu;
                    c[i] |= (__umul24(b, 0x204081u) & 0x01010101u) << 4;
                }
            }
        }
        constexpr float off = WT == 8 ? 128.0f : WT == 6 ? 16.0f : 8.0f;
        u32x4 o;
        uint32_t lo, hi;
        gb_bytes(c[0], off, r.d2, lo, hi);
        o[0] = lo; o[1] = hi;
        gb_bytes(c[1], off, r.d2, lo, hi);
        o[2] = lo; o[3] = hi;
        return __builtin_bit_cast(half8_t, o);
    }
}

// step s of a group: NRT x 2 MFMAs on the activation operands a and the weight
// operands b, between them next() - the operands of the step after (VALU and
// LDS reads), spread over the MFMAs
template <int NRT, int NA, int NV, typename Next>
__device__ __forceinline__ void gb_step(const half8_t (&a)[NRT], const half8_t (&b)[2], f32x16 (&acc)[NA][2], Next &&next) {
    constexpr int PER = (NV + 2 * NRT - 1) / (2 * NRT);
#pragma unroll
    for (int rt = 0; rt < NRT; ++rt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) acc[rt][ct] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a[rt], b[ct], acc[rt][ct], 0, 0, 0);
    next();
#pragma unroll
    for (int k = 0; k < NRT; ++k) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);       // an MFMA
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);     // an LDS read
        __builtin_amdgcn_sched_group_barrier(0x2, PER, 0);     // VALU
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
}

template <int WT>
__device__ __forceinline__ half8_t gb_operand_s(const GBRaw<WT> &r, int s) {
    return s == 0 ? gb_operand<WT, 0>(r) : s == 1 ? gb_operand<WT, 1>(r) : s == 2 ? gb_operand<WT, 2>(r) : gb_operand<WT, 3>(r);
}

// The K loop for NRT row tiles.  A stage is KG groups of weights and two
// halves of KA = KG / 2 groups of activations; stage 0's weight loads are out
// already.  Per stage:
//   wait for the weights and the first half's activations; take the lanes'
//   weight blocks out of the (wave's own, single) weight buffer into
//   registers; put out the second half's activations and the next stage's
//   weights, over that buffer; compute the first half;
//   wait for the second half (the weight loads, put out after it, stay in
//   flight); put out the next stage's first half; compute the second.
template <int WT, int NRT, int NA, int NW, int BM, int KG>
__device__ __forceinline__ void gb_kloop(rsrc_t rx, const uint32_t *aoff, const GBW<WT, KG> (&wd)[2], int64_t K, int wave,
                                         int lane, int wbase, _Float16 *a0, _Float16 *a1, uint8_t *ws,
                                         f32x16 (&acc)[NA][2]) {
    constexpr int KA = KG / 2;
    constexpr int NAL = 4 * NRT / NW;   // activation loads per wave and group (8 rows each)
    static_assert(4 * NRT % NW == 0, "whole loads per wave");
    constexpr int NV = WT == 1 ? 2 : WT == 6 ? 44 : 32;   // VALU instructions of a step's two weight operands
    const int nk = (int)((K + 63) / 64), nst = (nk + KG - 1) / KG;
    const bool odd = (K & 63) != 0;
    const int l32 = lane & 31, h = lane >> 5;
    auto issue_a = [&](int kb, _Float16 *a) __attribute__((always_inline)) {
#pragma unroll
        for (int g = 0; g < KA; ++g)
#pragma unroll
            for (int j = 0; j < NAL; ++j)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, (lds_void_t *)(a + (64 * BM * g + 512 * (wave + NW * j))), 16,
                                                         (int)aoff[j], 128 * (kb + g), 0, 0);
    };
#pragma unroll
    for (int rt = 0; rt < NA; ++rt)
#pragma unroll
        for (int ct = 0; ct < 2; ++ct)
#pragma unroll
            for (int i = 0; i < 16; ++i) acc[rt][ct][i] = 0.f;
    issue_a(0, a0);
    // the groups g0 .. g0 + KA - 1 of a stage, activations in A
    auto half = [&](const GBRaw<WT> (&raw)[KG][2], int g0, const _Float16 *A, int n) __attribute__((always_inline)) {
        const char *ab = (const char *)A + 128 * l32;
        half8_t a[2][NRT], b[2][2];
        auto operands = [&](int q) __attribute__((always_inline)) {   // of step q of the half
#pragma unroll
            for (int rt = 0; rt < NRT; ++rt)
                a[q & 1][rt] = *(const half8_t *)(ab + (128 * BM * (q >> 2) + 4096 * rt) + 16 * ((4 * h + (q & 3)) ^ (l32 & 7)));
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) b[q & 1][ct] = gb_operand_s<WT>(raw[g0 + (q >> 2)][ct], q & 3);
        };
        operands(0);
#pragma unroll
        for (int q = 0; q < 4 * KA; ++q) {
            if ((q & 3) == 0 && q > 0 && (q >> 2) >= n) break;
            gb_step<NRT, NA, NV>(a[q & 1], b[q & 1], acc, [&]() __attribute__((always_inline)) {
                if (q + 1 < 4 * KA) operands(q + 1);
            });
        }
    };
    // full: the stage's groups and the next stage exist
    auto stage = [&](int st, bool full) __attribute__((always_inline)) {
        const int kb = KG * st;
        gb_sync<0>();
        GBRaw<WT> raw[KG][2];
#pragma unroll
        for (int g = 0; g < KG; ++g) {
            // K % 64 = 32: the last group's second block is past the row
            const bool zero = !full && odd && kb + g == nk - 1 && (lane >> 5) != 0;
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) gb_read<WT, KG>(wd[ct], ws, g, lane, zero, raw[g][ct]);
        }
        __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the blocks are in registers
        const bool second = full || kb + KA < nk, next = full || st + 1 < nst;
        if (second) issue_a(kb + KA, a1);
        // The counted wait in front of the second half (2 NLD loads may stay
        // out) holds only if these activation loads go out before all of the
        // weight loads: no pass of the compiler may exchange them (the two go
        // to different LDS arrays, so nothing else orders them).
        asm volatile("" ::: "memory");
        if (next) {
#pragma unroll
            for (int ct = 0; ct < 2; ++ct) wd[ct].issue(ws + (wbase + ct * gb_wtile<WT, KG>()), st + 1);
        }
        half(raw, 0, a0, full ? KA : nk - kb);
        if (second) {
            if (next) gb_sync<2 * GBW<WT, KG>::NLD>();
            else gb_sync<0>();
            if (next) issue_a(kb + KG, a0);
            half(raw, KA, a1, full ? KA : nk - kb - KA);
        }
    };
    int st = 0;
    for (; st + 2 <= nst; ++st) stage(st, true);
    stage(st, false);
}

// The next product's operand of 32 columns n .. n + 31 (one Q8_0 block) of the
// tile's rows, from values v(i) of MFMA layout rows 32 rt + 8 (i / 4) + 4 h +
// i % 4, column lane % 32: 16 rows at a time through 2 KB of the wave's own
// LDS (its weight buffer) into rows, four lanes per row; the arithmetic and
// bits of launch_prep_b32 on the fp32 values.
template <typename V>
__device__ __forceinline__ void gb_next_rows(const GBSide &g, int next_f16, float *lds, int rt, int mrows, int64_t n, int lane,
                                             const int *s_p, V &&v) {
    const int l32 = lane & 31, h = lane >> 5;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
#pragma unroll
        for (int i = 0; i < 8; ++i) lds[(8 * (i >> 2) + 4 * h + (i & 3)) * 32 + l32] = v(8 * half + i);
        wave_lds_sync();
        const float4_t a = *(const float4_t *)(lds + 8 * lane), b = *(const float4_t *)(lds + 8 * lane + 4);
        wave_lds_sync();   // (rewritten next)
        const float x[8] = {a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};
        const uint4 o = next_f16 ? b32_f16x8(x) : b32_q8x8(x);
        const int m = 32 * rt + 16 * half + (lane >> 2);
        if (m < mrows) *(uint4 *)(g.xo + (int64_t)s_p[m] * g.ldo + n + 8 * (lane & 3)) = o;
    }
}

template <int ACT, int NA>
__device__ __forceinline__ void gb_glu_out(const GBSide &g, int next_f16, const f32x16 (&acc)[NA][2], int nrt, int mrows, int64_t n0,
                                           int lane, const int *s_p, float *lds) {
    const bool in = n0 < g.ncols;   // (the padding columns of an odd block count: zeros)
#pragma unroll
    for (int rt = 0; rt < NA; ++rt)
        if (rt < nrt)
            gb_next_rows(g, next_f16, lds, rt, mrows, n0, lane, s_p, [&](int i) __attribute__((always_inline)) {
                return in ? act_pair(ACT, acc[rt][0][i], acc[rt][1][i]) : 0.f;
            });
}

// SH: the shared expert's rows are in this launch (GBArgs::sh; a form of its
// own, the selection in front of the first loads costs 1 - 2 us per layer)
template <int WT, int EPI, int BM, int NW, int KG, bool SH>
__global__ void __launch_bounds__(64 * NW) __attribute__((amdgpu_waves_per_eu(2))) k_gb(GBArgs g) {
#ifdef __HIP_DEVICE_COMPILE__   // (the host pass needs the stub alone, and rejects the builtins' second instantiation)
    constexpr int NA = BM / 32;
    constexpr int WTILE = gb_wtile<WT, KG>(), WREG = 2 * WTILE;   // a column tile's and a wave's weight bytes
    __shared__ __attribute__((aligned(128))) _Float16 As0[BM * 64 * (KG / 2)];
    __shared__ __attribute__((aligned(128))) _Float16 As1[BM * 64 * (KG / 2)];
    __shared__ __attribute__((aligned(128))) uint8_t Ws[NW * WREG];
    // The shared expert's work-groups first: on XCD x the column tiles c % 8
    // = x, the row tiles of each one after another (its weights from that
    // XCD's L2).  Then work-group 8 q + x on XCD x: the x-th eighth of the
    // tiles in expert order, one after another, column tile q % nct (the
    // column tiles of one row tile share that XCD's L2 for the activations,
    // the row tiles of one expert for the weights).
    const bool shared = SH && (int)blockIdx.x < g.sh_wgs;
    const GBSide s = shared ? g.sh : (const GBSide &)g;
    int e = 0, start, mrows, ctile;
    if (shared) {
        const int qq = blockIdx.x >> 3, cq = qq / g.sh_tiles;
        ctile = 8 * cq + ((int)blockIdx.x & 7);
        if (ctile >= s.nct) return;
        start = BM * (qq - cq * g.sh_tiles);
        mrows = (int)g.sh_rows - start;
        if (mrows > BM) mrows = BM;
    } else {
        const int lin = blockIdx.x - (SH ? g.sh_wgs : 0), qq = lin >> 3, nt = *g.n_tiles, per = (nt + 7) >> 3;
        const int kk = qq / s.nct, tile = (lin & 7) * per + kk;
        ctile = qq - kk * s.nct;
        if (kk >= per || tile >= nt) return;
        e = g.tile_e[tile];
        start = g.tile_start[tile];
        mrows = g.tile_rows[tile];
    }
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int nrt = (mrows + 31) >> 5;
    constexpr bool GLU = EPI == GB_GLU;
    const int64_t K = s.a.K;
    const int64_t n0 = (int64_t)ctile * (GLU ? 32 * NW : 64 * NW) + (GLU ? 32 : 64) * wave;
    const uint8_t *ma = s.a.data + (int64_t)e * s.a.mat_bytes;
    const int wbase = wave * WREG;
    const uint32_t b0 = (uint32_t)wbase, b1 = b0 + (uint32_t)WTILE;
    GBW<WT, KG> wd[2];
    wd[0] = gb_wdesc<WT, KG>(ma, n0, s.a.N, s.a.row_bytes, K, lane, b0);
    if (!GLU) wd[1] = gb_wdesc<WT, KG>(ma, n0 + 32, s.a.N, s.a.row_bytes, K, lane, b1);
    else if (s.fused) wd[1] = gb_wdesc<WT, KG>(ma, s.I + n0, s.a.N, s.a.row_bytes, K, lane, b1);
    else wd[1] = gb_wdesc<WT, KG>(s.b.data + (int64_t)e * s.b.mat_bytes, n0, s.b.N, s.b.row_bytes, K, lane, b1);
    // the tile's rows: the slot indices first (their loads ahead of the
    // weights', which stay in flight), as activation offsets of this lane's
    // loads and, for the epilogue, one per thread
    constexpr int NAL = BM / (8 * NW);
    static_assert(BM <= 64 * NW, "a row per thread");
    int prow[NAL];
#pragma unroll
    for (int j = 0; j < NAL; ++j) {
        const int r = 8 * (wave + NW * j) + (lane >> 3);
        prow[j] = r < mrows ? (shared ? start + r : g.perm[start + r]) : -1;
    }
    const int my_p = tid < mrows ? (shared ? start + tid : g.perm[start + tid]) : -1;
    asm volatile("" ::: "memory");   // (keeps the order)
#pragma unroll
    for (int ct = 0; ct < 2; ++ct) wd[ct].issue(Ws + (wbase + ct * WTILE), 0);
    uint32_t aoff[NAL];
#pragma unroll
    for (int j = 0; j < NAL; ++j)
        aoff[j] = prow[j] < 0 ? GB_FAR
                              : (uint32_t)(g.ne11 == 1 && !shared ? prow[j] / g.K : prow[j]) * (2u * (uint32_t)s.ldx) +
                                    16u * (uint32_t)((lane & 7) ^ (lane >> 3));
    const rsrc_t rx = gb_rsrc(s.xh, s.xbytes);
    f32x16 acc[NA][2];
#define GB_LOOP(N) gb_kloop<WT, N, NA, NW, BM, KG>(rx, aoff, wd, K, wave, lane, wbase, As0, As1, Ws, acc)
    if constexpr (NA == 1) GB_LOOP(1);
    else {
        if (nrt == 1) GB_LOOP(1);
        else if (nrt == 2) GB_LOOP(2);
        else if (nrt == 3) GB_LOOP(3);
        else GB_LOOP(4);
    }
#undef GB_LOOP
    // the rows' slot indices to LDS, in the first activation buffer once no
    // wave reads it
    int *s_p = (int *)As0;
    lds_barrier();
    if (tid < BM) s_p[tid] = my_p;
    lds_barrier();
    const int l32 = lane & 31, h = lane >> 5;
    if constexpr (EPI == GB_GLU) {
        if (n0 >= s.ldo) return;
        float *lds = (float *)(Ws + wbase);   // (no load is in flight and no other wave reads it)
        switch (g.act) {
        case 0: gb_glu_out<0, NA>(s, g.next_f16, acc, nrt, mrows, n0, lane, s_p, lds); break;
        case 1: gb_glu_out<1, NA>(s, g.next_f16, acc, nrt, mrows, n0, lane, s_p, lds); break;
        case 2: gb_glu_out<2, NA>(s, g.next_f16, acc, nrt, mrows, n0, lane, s_p, lds); break;
        default: gb_glu_out<3, NA>(s, g.next_f16, acc, nrt, mrows, n0, lane, s_p, lds); break;
        }
    } else {
#pragma unroll
        for (int ct = 0; ct < 2; ++ct) {
            const int64_t n = n0 + 32 * ct;
#pragma unroll
            for (int rt = 0; rt < NA; ++rt) {
                if (rt >= nrt) continue;
                if constexpr (EPI == GB_RELU_SQR) {
                    if (n < s.ldo)
                        gb_next_rows(s, g.next_f16, (float *)(Ws + wbase), rt, mrows, n, lane, s_p, [&](int i) __attribute__((always_inline)) {
                            return n < s.ncols ? relu_sqr(acc[rt][ct][i]) : 0.f;
                        });
                } else {
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const int m = 32 * rt + 8 * (i >> 2) + 4 * h + (i & 3);
                        if (m < mrows && n + l32 < s.ncols) {
                            const float v = acc[rt][ct][i];
                            s.y[(int64_t)s_p[m] * s.ldy + n + l32] = shared && g.sh_w ? v * g.sh_w[s_p[m]] : v;
                        }
                    }
                }
            }
        }
    }
#endif
}

// Plain product of F16 tables in tiles of at most GF_BM = 192 rows, for
// mul_mat_id (the rule and its times: gf_tiles in api.cpp): 128 weight rows
// per work-group, 32 per wave, each lane loading its own 16 bytes per step
// (F16 needs no unpacking, so little is won by staging it), the next group
// while the current one is computed; activations through 2 x 24 KB of LDS.
// Three work-groups fit a CU, so one's start and stores run beside another's
// K loop, which decides for a short K and many rows (k_gb with F16 has LDS for
// one), and an expert of 129 - 192 rows is one tile.  The operands and their
// order, and so the bits, are k_gb's.  K 1024, N 2048, E 64, 8000 rows: 130 us
// in 128-row tiles of k_gb, 98 here (the call; 268 MB of weights).
__global__ void __launch_bounds__(256) k_gf(GBArgs g) {
    __shared__ __attribute__((aligned(16))) _Float16 As[2][GF_BM * 64];
    __shared__ int s_row[GF_BM], s_p[GF_BM];   // activation and output row of each tile row (past the tile: row 0)
    const int tile = blockIdx.y;
    if (tile >= *g.n_tiles) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l32 = lane & 31, h = lane >> 5;
    const int e = g.tile_e[tile], start = g.tile_start[tile], mrows = g.tile_rows[tile];
    const int nrt = (mrows + 31) >> 5;
    const int64_t col = (int64_t)blockIdx.x * 128 + 32 * wave + l32, K = g.a.K;
    const bool col_ok = col < g.ncols;
    // (a column past the matrix: row 0, not stored)
    const uint8_t *row = g.a.data + (int64_t)e * g.a.mat_bytes + (col_ok ? col : 0) * g.a.row_bytes;
    if (tid < GF_BM) {
        const int p = tid < mrows ? g.perm[start + tid] : -1;
        s_p[tid] = p;
        s_row[tid] = p < 0 ? 0 : (g.ne11 == 1 ? p / g.K : p);
    }
    __syncthreads();
    // 16-byte piece q = tid + 256 i of a group: tile row q / 8, K chunk q % 8, in slot chunk ^ (row & 7)
    constexpr int NC = GF_BM * 8 / 256;
    uint4 areg[NC];
    auto load_a = [&](int kb) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int q = tid + 256 * i, r = q >> 3, c = q & 7;
            areg[i] = r < 32 * nrt ? *(const uint4 *)(g.xh + (int64_t)s_row[r] * g.ldx + 64 * (int64_t)kb + 8 * c)
                                   : make_uint4(0, 0, 0, 0);
        }
    };
    auto store_a = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < NC; ++i) {
            const int q = tid + 256 * i, r = q >> 3, c = q & 7;
            *(uint4 *)(&As[buf][(r * 8 + (c ^ (r & 7))) * 8]) = areg[i];
        }
    };
    // steps 0 - 3 of a group: values 8 s .. 8 s + 7 of block h (K % 64 = 32: zeros past the row)
    auto load_w = [&](int kb, uint4 (&w)[4]) __attribute__((always_inline)) {
        const int64_t k = 64 * (int64_t)kb + 32 * h;
#pragma unroll
        for (int s = 0; s < 4; ++s) w[s] = k < K ? *(const uint4 *)(row + 2 * (k + 8 * s)) : make_uint4(0, 0, 0, 0);
    };
    f32x16 acc[GF_BM / 32];
#pragma unroll
    for (int t = 0; t < GF_BM / 32; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][i] = 0.f;
    const int nk = (int)((K + 63) / 64);
    uint4 cur[4], nxt[4];
    load_a(0);
    load_w(0, cur);
    store_a(0);
    __syncthreads();
    for (int kb = 0; kb < nk; ++kb) {
        const bool more = kb + 1 < nk;
        if (more) {
            load_a(kb + 1);
            load_w(kb + 1, nxt);
        }
        const _Float16 *A = As[kb & 1];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const half8_t b = __builtin_bit_cast(half8_t, cur[s]);
#pragma unroll
            for (int t = 0; t < GF_BM / 32; ++t)
                if (t < nrt) {
                    const int r = 32 * t + l32;
                    const half8_t a = *(const half8_t *)(&A[(r * 8 + ((4 * h + s) ^ (r & 7))) * 8]);
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, acc[t], 0, 0, 0);
                }
        }
        if (more) {
            store_a((kb + 1) & 1);
#pragma unroll
            for (int s = 0; s < 4; ++s) cur[s] = nxt[s];
        }
        __syncthreads();
    }
    if (!col_ok) return;
#pragma unroll
    for (int t = 0; t < GF_BM / 32; ++t)
        if (t < nrt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int m = 32 * t + 8 * (i >> 2) + 4 * h + (i & 3);
                if (m < mrows) g.y[(int64_t)s_p[m] * g.ldy + col] = acc[t][i];
            }
}

// ------------------------------------------------------------------ launch
template <int WT, int EPI>
static int gb_launch(const GBArgs &a, hipStream_t st) {
    GBArgs g = a;
    // 32-row tiles, waves per work-group and groups per stage (layer us, same
    // box, 2 waves x 2 groups / 4 x 2 / 4 x 4 / 2 x 4): qwen3omni widths, T =
    // 100: Q8_0 206 / 201 / 227 / 216, Q5_0 175 / 172 / 165 / 174, Q4_0 150 /
    // 148 / 146 / 150; moondream3 T = 64: Q8_0 140 / 149 / 160 / 157, F16 207
    // / 201 / 214 / 212; diffusiongemma F16 T = 256 342 / 329 / 349 / 343;
    // nemotronomni Q5_0 T = 200 491 / 497 / 483 / 473.
    constexpr int NS = WT == 1 ? 4 : 2, KS = WT == 1 || WT == 8 ? 2 : 4;
    const int nw = g.bm == GB_BM_LARGE ? 4 : NS;
    const int per = EPI == GB_GLU ? 32 * nw : 64 * nw;
    auto column_tiles = [&](const GBSide &s) {   // (with the padding columns)
        return (int)(((EPI == GB_STORE ? s.ncols : s.ldo) + per - 1) / per);
    };
    g.nct = column_tiles(g);
    int64_t wgs = 8 * (int64_t)g.nct * ((g.max_tiles + 7) / 8);
    g.sh_wgs = g.sh_tiles = 0;
    if (g.sh_rows > 0) {
        g.sh.nct = column_tiles(g.sh);
        g.sh_tiles = (int)((g.sh_rows + g.bm - 1) / g.bm);
        const int64_t sw = 8 * (int64_t)((g.sh.nct + 7) / 8) * g.sh_tiles;
        if (sw > 0x7fffffff) return -6;
        g.sh_wgs = (int)sw;
        wgs += sw;
    }
    if (wgs > 0x7fffffff) return -6;
    const dim3 grid((unsigned)wgs), block((unsigned)(64 * nw));
    if (g.sh_wgs) {
        if (g.bm == GB_BM_LARGE) hipLaunchKernelGGL((k_gb<WT, EPI, GB_BM_LARGE, 4, 2, true>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((k_gb<WT, EPI, GB_BM_SMALL, NS, KS, true>), grid, block, 0, st, g);
    } else {
        if (g.bm == GB_BM_LARGE) hipLaunchKernelGGL((k_gb<WT, EPI, GB_BM_LARGE, 4, 2, false>), grid, block, 0, st, g);
        else hipLaunchKernelGGL((k_gb<WT, EPI, GB_BM_SMALL, NS, KS, false>), grid, block, 0, st, g);
    }
    return hip_check_launch();
}

static bool gb_side_ok(const GBArgs &g, const GBSide &s) {
    if (s.a.K % 32 || s.ldx % 64 || (uintptr_t)s.xh % 16) return false;
    if (s.xrows <= 0 || s.xrows * s.ldx * 2 > GB_MAX_X) return false;
    if (s.a.row_bytes > GB_MAX_ROW_BYTES || (g.glu && !s.fused && s.b.row_bytes > GB_MAX_ROW_BYTES)) return false;
    return !((g.glu || g.relu_sqr) && (s.ncols % 32 || s.ldo % 64 || !s.xo));
}

int launch_gb(const GBArgs &g, hipStream_t st) {
    if (g.max_tiles <= 0) return 0;
    if (g.bm == GF_BM) {
        if (g.a.type != 1 || g.glu || g.relu_sqr || g.sh_rows > 0 || !gb_side_ok(g, g)) return -6;
        const int64_t nct = (g.ncols + 127) / 128;
        if (nct > 0x7fffffff || g.max_tiles > 65535) return -6;
        hipLaunchKernelGGL(k_gf, dim3((unsigned)nct, (unsigned)g.max_tiles), dim3(256), 0, st, g);
        return hip_check_launch();
    }
    if (g.bm != GB_BM_SMALL && g.bm != GB_BM_LARGE) return -6;
    if (!gb_side_ok(g, g)) return -6;
    if (g.sh_rows > 0 && (!gb_side_ok(g, g.sh) || g.sh.a.type != g.a.type || g.sh_rows > g.sh.xrows)) return -6;
    GBArgs a = g;
    a.xbytes = (uint32_t)(g.xrows * g.ldx * 2);
    a.sh.xbytes = (uint32_t)(g.sh.xrows * g.sh.ldx * 2);
#define GB_TYPE(T)                                              \
    case T:                                                     \
        if (g.glu) return gb_launch<T, GB_GLU>(a, st);          \
        if (g.relu_sqr) return gb_launch<T, GB_RELU_SQR>(a, st); \
        return gb_launch<T, GB_STORE>(a, st);
    switch (g.a.type) {
        GB_TYPE(1)
        GB_TYPE(2)
        GB_TYPE(6)
        GB_TYPE(8)
    default: return -3;
    }
#undef GB_TYPE
}

}  // namespace mimoe
