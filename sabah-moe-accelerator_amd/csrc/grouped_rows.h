// Group-major expert rows for any row count and any k: the matrix product of
// an expert's rows with the (token, slot) pairs routed to it, for every 256-element
// or 32-element format below, with int8 MFMA.  It runs MUL_MAT_ID over
// many tokens (MMID), a layer's gate/up + SwiGLU (NM = 2) and its down rows.
//
// Work split: an item is up to 16 PT pairs of one expert (k_group_pairs
// writes the list); grid = (row tiles, items), 256 threads.  A wave owns 16
// rows, or G = 2 groups of 16 (of one matrix, or the same rows of gate and up), over
// the whole of k, 256 elements per step: the step's weight bytes (coalesced
// 16-byte chunks) and the pairs' q8 chunks are loaded into registers while the step
// before is computed, stored to LDS, and each wave decodes its rows' chunk once into
// MFMA operands for all of the item's 16-pair tiles.  A row's fp32 sum is kept
// in the lane and grows in block order, so the results are the token-major
// kernels', bit for bit, in every format.
//
// What bounds it: decoding.  A 512-token IQ3_XXS / IQ4_NL layer (top-10 of 512,
// 2560 / 640; 1.1 GB of weights), medians of 150 traced calls: gate/up 257 us (2.50 TB/s; VALU busy
// 67 %, LDS 62 %, most of it codebook look-ups), down 229 us (2.06 TB/s; VALU 63 %, LDS 30 %), two to
// three waves per SIMD, and 30 us of grouping, quantisation and combine; the layer 515 us against
// 4,680 token-major.  A Q4_K / Q6_K layer at 1,999 tokens, top-8 of 128 (125 pairs per
// expert): 437 us against 777 with the fixed-shape kernels.
#pragma once
#include "prefill_kernels.h"

namespace sabah {

constexpr int kRowsTile = 64;                 // rows per workgroup and matrix: four waves of 16

// bytes of a row's 256 elements, and the 16-byte chunks that hold them at any even
// address, made odd: rows 16 * odd bytes apart start on different LDS banks
__host__ __device__ constexpr int step_bytes(int qt) { return 256 / block_elems(qt) * block_bytes(qt); }
__host__ __device__ constexpr int step_chunks(int qt) { return ((14 + step_bytes(qt) + 15) / 16) | 1; }

// formats paired with 32-element q8_0 blocks: one fp32 term per 32 elements and a
// last step that may be partial
__host__ __device__ constexpr bool step_q8_0(int qt) { return act_type(qt) == QT_Q8_0; }
__host__ __device__ constexpr bool grouped_rows_type(int qt) {
    return qt == QT_Q8_0 || qt == QT_Q4_K || qt == QT_Q5_K || qt == QT_Q6_K || qt == QT_IQ3_S || qt == QT_IQ3_XXS ||
           qt == QT_IQ4_NL || qt == QT_IQ4_XS;
}

// the order of the activations' bytes (mfma_chunk_store)
__host__ __device__ constexpr int rows_act_order(int qt) { return qt == QT_IQ4_NL || qt == QT_IQ4_XS ? 2 : 1; }

// reads at any even LDS address
struct __attribute__((packed, aligned(2))) LdsU32x {
    uint32_t v;
};
struct __attribute__((packed, aligned(2))) LdsU64x {
    uint64_t v;
};
__device__ inline uint32_t lds_u32x(const uint8_t* p) { return reinterpret_cast<const LdsU32x*>(p)->v; }
__device__ inline uint64_t lds_u64x(const uint8_t* p) { return reinterpret_cast<const LdsU64x*>(p)->v; }
// the same through the dwords that hold them and a byte shift, for the formats whose
// fields start between dwords
__device__ inline uint32_t lds_u32f(const uint8_t* p) {
    const uint32_t sh = (uint32_t)reinterpret_cast<uintptr_t>(p) & 3u;
    const uint32_t* d = reinterpret_cast<const uint32_t*>(p - sh);
    return __builtin_amdgcn_alignbyte(d[1], d[0], sh);
}
__device__ inline uint64_t lds_u64f(const uint8_t* p) {
    const uint32_t sh = (uint32_t)reinterpret_cast<uintptr_t>(p) & 3u;
    const uint32_t* d = reinterpret_cast<const uint32_t*>(p - sh);
    const uint32_t d0 = d[0], d1 = d[1], d2 = d[2];
    return (uint64_t)__builtin_amdgcn_alignbyte(d2, d1, sh) << 32 | __builtin_amdgcn_alignbyte(d1, d0, sh);
}
__device__ inline uint32_t lds_u16(const uint8_t* p) { return *reinterpret_cast<const uint16_t*>(p); }
// the sums so far are formed here (fewer matrix results live at a time)
template <typename V>
__device__ inline void pin4(V (&v)[4]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(v[i]));
}
__device__ inline long op_of(uint32_t lo, uint32_t hi) { return (long)((uint64_t)hi << 32 | lo); }

typedef _Float16 v4f16 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));
__device__ inline u16x2 as_u16x2(uint32_t v) { return __builtin_bit_cast(u16x2, v); }
template <typename V>
__device__ inline uint32_t as_word(V v) { return __builtin_bit_cast(uint32_t, v); }

// 256 elements of the lane's row decoded into MFMA B operands (B[s]: lane
// quarter q's eight elements 32 s + 8 q .. + 7, or of mfma_chunk_store's order 2) with the scales of its
// sub-blocks.  ns: 32-element blocks of the row left (q8_0 formats): the scale
// of a block past the row is 0, and so is its term (its activations are zeros).
template <int QT>
struct RowOps {
    long B[8];
    uint32_t sc[4];               // packed integer scales (Q8_0, IQ4_NL: none)
    float d[step_q8_0(QT) ? 8 : 2];
    v4f16 mn;                     // Q4_K, Q5_K: the mins of 16-element groups 4 q .. 4 q + 3
};

template <int QT>
__device__ inline void row_ops(const uint8_t* unit, const uint8_t* tabs, int q, int ns, RowOps<QT>& O) {
    if constexpr (QT == QT_IQ3_S) {
        Iq3sBlockOps I;
        iq3s_block_ops(unit, tabs, q, I);
#pragma unroll
        for (int s = 0; s < 8; ++s) O.B[s] = I.B[s];
        O.sc[0] = I.ls[0];
        O.sc[1] = I.ls[1];
        O.d[0] = h2f(I.d);
    } else if constexpr (QT == QT_IQ3_XXS) {
        uint32_t sc[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t aux = lds_u32f(unit + 66 + 4 * s), q2 = lds_u16(unit + 2 + 8 * s + 2 * q);
            const uint32_t s7 = (aux >> (7 * q)) & 127u;
            const uint32_t sg = s7 | ((uint32_t)(__builtin_popcount(s7) & 1) << 7);
            O.B[s] = op_of(lds_u32(tabs, kLdsGrid + 4u * ((q2 & 0xFFu) | ((sg & 15u) << 8))),
                           lds_u32(tabs, kLdsGrid + 4u * ((q2 >> 8) | ((sg >> 4) << 8))));
            sc[s] = 2u * (aux >> 28) + 1u;
        }
        O.sc[0] = sc[0] | sc[2] << 8 | sc[4] << 16 | sc[6] << 24;
        O.sc[1] = sc[1] | sc[3] << 8 | sc[5] << 16 | sc[7] << 24;
        O.d[0] = h2f(lds_u16(unit));
    } else if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
        const uint32_t dd = lds_u32x(unit), s0 = lds_u32x(unit + 4), s1 = lds_u32x(unit + 8), s2 = lds_u32x(unit + 12);
        // get_scale_min_k4 on whole words: items 0..3, then 4..7
        O.sc[0] = s0 & 0x3F3F3F3Fu;
        O.sc[1] = (s2 & 0x0F0F0F0Fu) | ((s0 >> 2) & 0x30303030u);
        const uint32_t m0 = s1 & 0x3F3F3F3Fu, m1 = ((s2 >> 4) & 0x0F0F0F0Fu) | ((s1 >> 2) & 0x30303030u);
        const uint32_t mw = (q & 2 ? m1 : m0) >> (16 * (q & 1));
        const _Float16 ma = (_Float16)(unsigned short)(mw & 0xFFu), mb = (_Float16)(unsigned short)((mw >> 8) & 0xFFu);
        O.mn = v4f16{ma, ma, mb, mb};
        O.d[0] = h2f(dd);
        O.d[1] = h2f(dd >> 16);
        const uint64_t qh = QT == QT_Q5_K ? lds_u64x(unit + 16 + 8 * q) : 0;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
            const uint64_t w = lds_u64x(unit + (QT == QT_Q5_K ? 48 : 16) + 32 * p + 8 * q);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                uint64_t v = (w >> (4 * u)) & 0x0F0F0F0F0F0F0F0Full;
                if constexpr (QT == QT_Q5_K) v |= ((qh >> (2 * p + u)) & 0x0101010101010101ull) << 4;
                O.B[2 * p + u] = (long)v;
            }
        }
    } else if constexpr (QT == QT_Q6_K) {
#pragma unroll
        for (int i = 0; i < 4; ++i) O.sc[i] = lds_u32f(unit + 192 + 4 * i);
        O.d[0] = h2f(lds_u16(unit + 208));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint64_t l0 = lds_u64f(unit + 64 * h + 8 * q), l1 = lds_u64f(unit + 64 * h + 32 + 8 * q);
            const uint64_t hb = lds_u64f(unit + 128 + 32 * h + 8 * q);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const uint64_t lo = (t & 1 ? l1 : l0) >> (4 * (t >> 1)), hi = hb >> (2 * t);
                const uint64_t v = (lo & 0x0F0F0F0F0F0F0F0Full) | ((hi & 0x0303030303030303ull) << 4);
                // q - 32 per byte, q < 64: q + 96 stays in its byte, and flipping bit 7 takes 128 off
                const uint32_t a = ((uint32_t)v + 0x60606060u) ^ 0x80808080u;
                const uint32_t b = ((uint32_t)(v >> 32) + 0x60606060u) ^ 0x80808080u;
                O.B[4 * h + t] = op_of(a, b);
            }
        }
    } else if constexpr (QT == QT_Q8_0) {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            O.B[s] = (long)lds_u64f(unit + 34 * s + 2 + 8 * q);
            O.d[s] = s < ns ? h2f(lds_u16(unit + 34 * s)) : 0.0f;
        }
    } else if constexpr (QT == QT_IQ4_NL) {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t n = lds_u32f(unit + 18 * s + 2 + 4 * q);
            O.B[s] = op_of(iq4_levels(n & 0x0F0F0F0Fu), iq4_levels((n >> 4) & 0x0F0F0F0Fu));
            O.d[s] = s < ns ? h2f(lds_u16(unit + 18 * s)) : 0.0f;
        }
    } else {
        static_assert(QT == QT_IQ4_XS, "a grouped_rows_type");
        const uint32_t dh = lds_u32x(unit), sl = lds_u32x(unit + 4), sh = dh >> 16;
        O.d[0] = h2f(dh);
        O.sc[0] = O.sc[1] = 0;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t n = lds_u32x(unit + 8 + 16 * s + 4 * q);
            O.B[s] = op_of(iq4_levels(n & 0x0F0F0F0Fu), iq4_levels((n >> 4) & 0x0F0F0F0Fu));
            O.sc[s >> 2] |= (((sl >> (4 * s)) & 15u) | (((sh >> (2 * s)) & 3u) << 4)) << (8 * (s & 3));
        }
    }
}

// two int16 -> two fp16 (exact up to 2,048)
__device__ inline uint32_t half2_of(uint32_t v) {
    typedef _Float16 v2f16 __attribute__((ext_vector_type(2)));
    return as_word(v2f16{(_Float16)(short)(v & 0xFFFFu), (_Float16)(short)(v >> 16)});
}
// sum mn_j bs_j over a step's sixteen 16-element groups on fp16 MFMA: exact (the
// mins are below 64, the sums at most 2,032, every partial sum an integer below 2^24)
__device__ inline v4f32 min_sums(const v4f16& mn, const v4f16& bs) {
    return __builtin_amdgcn_mfma_f32_16x16x16f16(bs, mn, v4f32{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
}

// acc[i] (the lane's row, pair 4 q + i of a tile) += the step's term(s), the
// unit dot's integers and fp32 steps in its order.  dx: the tile's activation
// scales (dx[4 q + i]; q8_0: a row of them per 32 elements, dx_stride apart);
// bs: Q4_K, Q5_K: the 16-element sums 4 q .. 4 q + 3 of pair r.
template <int QT>
__device__ inline void step_term(const RowOps<QT>& O, const long (&X)[8], const float* dx, int dx_stride,
                                 const v4f16& bs, int q, float (&acc)[4]) {
    const v4i32 z = {0, 0, 0, 0};
    if constexpr (step_q8_0(QT)) {
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(X[s], O.B[s], z, 0, 0, 0);
            const float4 dx4 = *reinterpret_cast<const float4*>(dx + s * dx_stride + 4 * q);
            const float dxv[4] = {dx4.x, dx4.y, dx4.z, dx4.w};
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn((float)d[i], __fmul_rn(O.d[s], dxv[i])));
            if (s & 1) pin4(acc);
        }
    } else {
        const float4 dx4 = *reinterpret_cast<const float4*>(dx + 4 * q);
        const float dxv[4] = {dx4.x, dx4.y, dx4.z, dx4.w};
        if constexpr (QT == QT_IQ4_XS) {
            float t[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) t[i] = __fmul_rn(O.d[0], dxv[i]);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(X[s], O.B[s], z, 0, 0, 0);
                const float ls = (float)((int)((O.sc[s >> 2] >> (8 * (s & 3))) & 0xFFu) - 32);
#pragma unroll
                for (int i = 0; i < 4; ++i) acc[i] = __fadd_rn(acc[i], __fmul_rn(__fmul_rn(t[i], ls), (float)d[i]));
                if (s & 1) pin4(acc);
            }
            return;
        }
        int isum[4] = {0, 0, 0, 0};
        if constexpr (QT == QT_Q6_K) {
            // a scale per 16 elements: two products per sub-block, the other half's weights zero
            const long first = q < 2 ? -1L : 0L;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const v4i32 da = __builtin_amdgcn_mfma_i32_16x16x32_i8(X[s], O.B[s] & first, z, 0, 0, 0);
                const v4i32 db = __builtin_amdgcn_mfma_i32_16x16x32_i8(X[s], O.B[s] & ~first, z, 0, 0, 0);
                const int sa = (int)(int8_t)(O.sc[s >> 1] >> (16 * (s & 1))), sb = (int)(int8_t)(O.sc[s >> 1] >> (16 * (s & 1) + 8));
#pragma unroll
                for (int i = 0; i < 4; ++i) isum[i] += __mul24(sa, da[i]) + __mul24(sb, db[i]);   // |da| <= 16 * 32 * 127
                if (s & 1) pin4(isum);
            }
        } else {
            constexpr bool K = QT == QT_Q4_K || QT == QT_Q5_K;
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                const v4i32 d = __builtin_amdgcn_mfma_i32_16x16x32_i8(X[s], O.B[s], z, 0, 0, 0);
                const int ls = (int)(K ? (O.sc[s >> 2] >> (8 * (s & 3))) & 0xFFu : (O.sc[s & 1] >> (8 * (s >> 1))) & 0xFFu);
#pragma unroll
                for (int i = 0; i < 4; ++i) isum[i] += __mul24(ls, d[i]);   // |d| <= 32 * 62 * 127
                if (s == 3) pin4(isum);
            }
        }
        if constexpr (QT == QT_Q4_K || QT == QT_Q5_K) {
            const v4f32 ms = min_sums(O.mn, bs);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                acc[i] = __fadd_rn(acc[i], __fsub_rn(__fmul_rn(__fmul_rn(O.d[0], dxv[i]), (float)isum[i]),
                                                     __fmul_rn(__fmul_rn(O.d[1], dxv[i]), ms[i])));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float c = __fmul_rn(__fmul_rn(O.d[0], dxv[i]), (float)isum[i]);
                if constexpr (QT == QT_IQ3_XXS) c = __fmul_rn(c, 0.25f);
                acc[i] = __fadd_rn(acc[i], c);
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Four-tile items of Q4_K and Q6_K: the integer scale folded into the weights
// once, as two int8 operands: scale * q = (hi << SHIFT) + lo.  A step's block sum is
// then two chains of v_mfma_i32_16x16x64_i8 (64 elements each, the lane's 16
// bytes of a row's chunk as they lie) that accumulate in the matrix unit, with no
// multiply-add per 32 elements; the sums are the same exact integers.
//   Q4_K: q <= 15, sc = 8 a + b: hi = q a, lo = q b, both <= 105 (SHIFT 3);
//   Q6_K: p = sc (q - 32), |p| <= 4,096: hi = p >> 7 (-32 .. 32), lo = p & 127 (SHIFT 7).
// ---------------------------------------------------------------------------
template <int QT>
struct FoldOps {
    v4i32 hi[4], lo[4];
    float d[2];
    v4f16 mn;
};
template <int QT>
__device__ inline void fold_ops(const uint8_t* unit, int q, FoldOps<QT>& F) {
    if constexpr (QT == QT_Q4_K) {
        RowOps<QT> O;
        row_ops<QT>(unit, nullptr, q, 8, O);
        F.d[0] = O.d[0];
        F.d[1] = O.d[1];
        F.mn = O.mn;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            const uint32_t sc = (O.sc[s >> 2] >> (8 * (s & 3))) & 0xFFu;
            const unsigned short b = (unsigned short)(sc & 7u), a = (unsigned short)(sc >> 3);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const u16x2 w = as_u16x2((uint32_t)((uint64_t)O.B[s] >> (32 * u)));   // bytes <= 15: no carry into the next
                F.hi[s >> 1][2 * (s & 1) + u] = (int)as_word(w * u16x2{a, a});
                F.lo[s >> 1][2 * (s & 1) + u] = (int)as_word(w * u16x2{b, b});
            }
        }
    } else {
        static_assert(QT == QT_Q6_K, "folded formats: Q4_K, Q6_K");
        F.d[0] = h2f(lds_u16(unit + 208));
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint64_t l0 = lds_u64f(unit + 64 * h + 8 * q), l1 = lds_u64f(unit + 64 * h + 32 + 8 * q);
            const uint64_t hb = lds_u64f(unit + 128 + 32 * h + 8 * q), sw = lds_u64f(unit + 192 + 8 * h);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const int s = 4 * h + t;
                const uint64_t lo = (t & 1 ? l1 : l0) >> (4 * (t >> 1)), hi = hb >> (2 * t);
                const uint64_t v = (lo & 0x0F0F0F0F0F0F0F0Full) | ((hi & 0x0303030303030303ull) << 4);
                // the lane's elements lie in half q / 2 of the item: scale byte 2 t + q / 2
                const int sc = (int)(int8_t)((uint32_t)(sw >> (32 * (t >> 1))) >> (16 * (t & 1) + 8 * (q >> 1)));
                const unsigned short m16 = (unsigned short)sc, c16 = (unsigned short)(-32 * sc);
                const u16x2 m = {m16, m16}, c = {c16, c16};
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const uint32_t w = (uint32_t)(v >> (32 * u));
                    const u16x2 pe = as_u16x2(w & 0x00FF00FFu) * m + c, po = as_u16x2((w >> 8) & 0x00FF00FFu) * m + c;
                    const uint32_t he = as_word(__builtin_bit_cast(i16x2, pe) >> 7), ho = as_word(__builtin_bit_cast(i16x2, po) >> 7);
                    F.hi[s >> 1][2 * (s & 1) + u] = (int)__builtin_amdgcn_perm(ho, he, 0x06020400u);
                    F.lo[s >> 1][2 * (s & 1) + u] = (int)((as_word(pe) & 0x007F007Fu) | (as_word(po) & 0x007F007Fu) << 8);
                }
            }
        }
    }
}
template <int QT>
__device__ inline void fold_term(const FoldOps<QT>& F, const v4i32 (&X)[4], const float* dx, const v4f16& bs, int q,
                                 float (&acc)[4]) {
    v4i32 H = {0, 0, 0, 0}, L = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        H = __builtin_amdgcn_mfma_i32_16x16x64_i8(X[t], F.hi[t], H, 0, 0, 0);
        L = __builtin_amdgcn_mfma_i32_16x16x64_i8(X[t], F.lo[t], L, 0, 0, 0);
    }
    const float4 dx4 = *reinterpret_cast<const float4*>(dx + 4 * q);
    const float dxv[4] = {dx4.x, dx4.y, dx4.z, dx4.w};
    v4f32 ms = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (QT == QT_Q4_K) ms = min_sums(F.mn, bs);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int isum = H[i] * (QT == QT_Q4_K ? 8 : 128) + L[i];
        float c = __fmul_rn(__fmul_rn(F.d[0], dxv[i]), (float)isum);
        if constexpr (QT == QT_Q4_K) c = __fsub_rn(c, __fmul_rn(__fmul_rn(F.d[1], dxv[i]), ms[i]));
        acc[i] = __fadd_rn(acc[i], c);
    }
}

struct GroupedRowsArgs {
    const uint8_t *w0, *w1;       // bank bases [n_experts][rows][row bytes] (w1: up)
    size_t expert_stride;
    const int4* items;            // (expert, first position, pairs, 0); *n_items of them
    const int* n_items;
    const int* pair_of;           // pair at each position (MMID, or x_div > 0)
    int x_div;                    // input row of position p: pair_of[p] / x_div, or p itself (0)
    const uint8_t* xq;            // q8 rows in MFMA operand order, xq_stride bytes apart
    int xq_stride;
    int rows, k;
    float* out;                   // [position][rows]
    float* dst;                   // MMID: dst[t][s] rows
    size_t dst_nb1, dst_nb2;
    int n_ids;
};

// what becomes of the sums: out[position][row]; MUL_MAT_ID's dst[t][s][row]; or
// h = silu(gate) * up, the wave's two row groups being the same rows of two matrices
enum : int { kRowsOut = 0, kRowsMmid = 1, kRowsSwiglu = 2 };

template <int QT, int G, int PT, int MODE>
__global__ __launch_bounds__(kThreads, 2) void k_grouped_rows(GroupedRowsArgs a) {
    static_assert(MODE != kRowsSwiglu || G == 2, "gate and up");
    constexpr bool MMID = MODE == kRowsMmid, SWIGLU = MODE == kRowsSwiglu;
    constexpr int NT = kThreads, CB = step_bytes(QT), CPR = step_chunks(QT);
    constexpr int NLM = (kRowsTile * CPR + NT - 1) / NT, NL = G * NLM, TP = 16 * PT;   // loads per row group and in all
    constexpr bool Q80 = step_q8_0(QT), BS = QT == QT_Q4_K || QT == QT_Q5_K;
    constexpr bool FOLD = PT == 4 && (QT == QT_Q4_K || QT == QT_Q6_K);
    // a row's address mod 16 is the same at every step
    constexpr bool FIXED = CB % 16 == 0;
    typedef __attribute__((address_space(1))) const u32x4 g_u32x4;
    __shared__ __align__(16) uint8_t tabs[table_bytes(QT) ? table_bytes(QT) : 16];
    __shared__ __align__(16) uint8_t raw[NL * NT * 16 + 16];   // 16: dwords read past a field's end
    __shared__ __align__(16) uint8_t xs[TP * kActChunkStride];
    __shared__ __align__(16) float sdx[(Q80 ? 8 : 1) * TP];
    __shared__ __align__(16) uint32_t sbs[BS ? TP * 8 : 4];  // 16 fp16 sums per pair
    __shared__ size_t sdst[MMID ? TP : 1];                   // byte offset of each pair's dst row
    const int4 it = a.items[blockIdx.y];
    if ((int)blockIdx.y >= *a.n_items) return;               // uniform: the list is shorter than its bound
    const int e = it.x, g0 = it.y, cnt = it.z, nt = (cnt + 15) >> 4;
    const int tid = (int)threadIdx.x, wave = tid >> 6, lane = tid & 63, r = lane & 15, q = lane >> 4;
    const int row0 = (int)blockIdx.x * (SWIGLU ? kRowsTile : G * kRowsTile);
    const int rb = (int)row_bytes(QT, a.k), nch = (a.k + 255) >> 8;
    const uint8_t* base[G];       // of each row group's matrix
    base[0] = a.w0 + (size_t)e * a.expert_stride;
    if constexpr (G == 2) base[1] = SWIGLU ? a.w1 + (size_t)e * a.expert_stride : base[0];
    // row i of the workgroup's group m (rows past the matrix repeat its last)
    auto row_of = [&](int m, int i) { return min(row0 + (SWIGLU ? 0 : kRowsTile * m) + i, a.rows - 1); };

    TableRegs<QT, NT> tr = load_tables<QT, NT>(tid);
    // the thread's i-th 16-byte chunk of a matrix's step: chunk c % CPR of staged row c / CPR,
    // as an offset from base; len: the step's bytes (chunks past the row's end repeat its last)
    auto load_off = [&](int m, int i, int s, int len) {
        const int c = min(tid + NT * i, kRowsTile * CPR - 1), rw = c / CPR;
        const uint32_t o = (uint32_t)row_of(m, rw) * (uint32_t)rb + (uint32_t)(s * CB);
        const uint32_t lead = ((uint32_t)reinterpret_cast<uintptr_t>(base[m]) + o) & 15u;
        return o - lead + 16u * (uint32_t)min(c - rw * CPR, (int)(lead + (uint32_t)len - 1u) >> 4);
    };
    uint32_t wf[NL];              // FIXED: load_off at step 0, + 16 (never negative); else the row's offset
    int wj[FIXED ? 1 : NLM];
#pragma unroll
    for (int i = 0; i < NL; ++i) {
        if constexpr (FIXED) {
            wf[i] = load_off(i / NLM, i % NLM, 0, CB) + 16u;
        } else {
            const int c = min(tid + NT * (i % NLM), kRowsTile * CPR - 1), rw = c / CPR;
            if (i < NLM) wj[FIXED ? 0 : i] = c - rw * CPR;
            wf[i] = (uint32_t)row_of(i / NLM, rw) * (uint32_t)rb;
        }
    }
    u32x4 wd[NL];
    auto load_w = [&](int s) {
        if constexpr (!FIXED) {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                const uint32_t o = wf[i] + (uint32_t)(s * CB);
                const uint32_t lead = ((uint32_t)reinterpret_cast<uintptr_t>(base[i / NLM]) + o) & 15u;
                const int j = min(wj[FIXED ? 0 : i % NLM], (int)(lead + (uint32_t)CB - 1u) >> 4);
                wd[i] = *(g_u32x4*)(base[i / NLM] - 16 + (o + 16u - lead + 16u * (uint32_t)j));
            }
        } else if (!Q80 || rb - s * CB >= CB) {
#pragma unroll
            for (int i = 0; i < NL; ++i) wd[i] = *(g_u32x4*)(base[i / NLM] + (size_t)s * CB - 16 + wf[i]);
        } else {
#pragma unroll
            for (int i = 0; i < NL; ++i)
                wd[i] = *(g_u32x4*)(base[i / NLM] - 16 + (load_off(i / NLM, i % NLM, s, rb - s * CB) + 16u));
        }
    };
    load_w(0);
    // sixteen threads per pair: 16 bytes of its chunk each, and its scales and sums
    const ActLayout XL(a.k, Q80 ? QT_Q8_0 : QT_Q8_K);
    const int xp = tid >> 4, xk = tid & 15;
    uint32_t xo[PT];
#pragma unroll
    for (int p = 0; p < PT; ++p) {
        const int pos = g0 + min(16 * p + xp, cnt - 1);
        xo[p] = (uint32_t)(a.x_div ? a.pair_of[pos] / a.x_div : pos) * (uint32_t)a.xq_stride;
    }
    if (MMID && tid < TP) {
        const int pr = a.pair_of[g0 + min(tid, cnt - 1)];
        sdst[tid] = (size_t)(pr / a.n_ids) * a.dst_nb2 + (size_t)(pr % a.n_ids) * a.dst_nb1;
    }
    u32x4 xd[PT];
    float xdx[PT];
    uint32_t xbs[PT];
    // every tile's loads are issued (tiles past the item re-read its last pair): under a
    // condition the registers they fill end up in scratch memory
    auto load_xs = [&](int s) {
        const uint8_t *xc = a.xq + s * kActChunkStride, *xd0 = a.xq + XL.off_d + (Q80 ? 32 : 4) * s;
        const uint8_t* xb = a.xq + XL.off_bsum + 32 * s;
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            xd[p] = *reinterpret_cast<const u32x4*>(xc + (xo[p] + 16u * (uint32_t)xk));
            xdx[p] = *reinterpret_cast<const float*>(xd0 + (xo[p] + (Q80 ? 4u * (uint32_t)(xk & 7) : 0u)));
            if constexpr (BS) xbs[p] = *reinterpret_cast<const uint32_t*>(xb + (xo[p] + 4u * (uint32_t)(xk & 7)));
        }
    };
    load_xs(0);
    store_tables<QT, NT>(tabs, tr, tid);

    float acc[G][PT][4];
#pragma unroll
    for (int m = 0; m < G; ++m)
#pragma unroll
        for (int p = 0; p < PT; ++p)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[m][p][i] = 0.0f;
    uint32_t my_row[G];
#pragma unroll
    for (int m = 0; m < G; ++m) my_row[m] = (uint32_t)row_of(m, 16 * wave + r) * (uint32_t)rb;
    const uint8_t* const xl = xs + r * kActChunkStride + 16 * q;
    // the lane's staged row of group m at step s
    auto unit_of = [&](int m, int s) {
        const uint32_t lead = ((uint32_t)reinterpret_cast<uintptr_t>(base[m]) + my_row[m] + (uint32_t)(s * CB)) & 15u;
        return raw + NLM * NT * 16 * m + (16 * wave + r) * (16 * CPR) + lead;
    };
    auto read_x = [&](int p, long (&X)[8]) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const u32x4 v = *reinterpret_cast<const u32x4*>(xl + 16 * p * kActChunkStride + 64 * t);
            X[2 * t] = op_of(v.x, v.y);
            X[2 * t + 1] = op_of(v.z, v.w);
        }
    };
#pragma unroll 1
    for (int s = 0; s < nch; ++s) {
        if (s) __syncthreads();                              // the step before is computed
#pragma unroll
        for (int i = 0; i < NL; ++i) *reinterpret_cast<u32x4*>(raw + 16 * (tid + NT * i)) = wd[i];
#pragma unroll
        for (int p = 0; p < PT; ++p) {
            if (p >= nt) continue;
            *reinterpret_cast<u32x4*>(xs + (16 * p + xp) * kActChunkStride + 16 * xk) = xd[p];
            if (Q80 ? xk < 8 : xk == 0) sdx[(Q80 ? TP * xk : 0) + 16 * p + xp] = xdx[p];
            if (BS && xk < 8)
                sbs[8 * (16 * p + xp) + xk] = half2_of(xbs[p]);
        }
        __syncthreads();
        if (s + 1 < nch) {
            load_w(s + 1);
            load_xs(s + 1);
        }
        if constexpr (FOLD) {
            // one group at a time: its operands take 32 registers
#pragma unroll
            for (int m = 0; m < G; ++m) {
                FoldOps<QT> F;
                fold_ops<QT>(unit_of(m, s), q, F);
#pragma unroll
                for (int p = 0; p < PT; ++p) {
                    if (p >= nt) continue;
                    v4i32 X[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) X[t] = *reinterpret_cast<const v4i32*>(xl + 16 * p * kActChunkStride + 64 * t);
                    v4f16 bs = {0, 0, 0, 0};
                    if constexpr (BS) bs = *reinterpret_cast<const v4f16*>(sbs + 8 * (16 * p + r) + 2 * q);
                    fold_term<QT>(F, X, sdx + 16 * p, bs, q, acc[m][p]);
                }
            }
        } else {
            const int ns = Q80 ? (a.k - 256 * s) >> 5 : 8;
            long X[8];
            read_x(0, X);
            RowOps<QT> O[G];
#pragma unroll
            for (int m = 0; m < G; ++m) {
                row_ops<QT>(unit_of(m, s), tabs, q, ns, O[m]);
            }
#pragma unroll
            for (int p = 0; p < PT; ++p) {
                if (p >= nt) continue;
                if (p) read_x(p, X);
                v4f16 bs = {0, 0, 0, 0};
                if constexpr (BS) bs = *reinterpret_cast<const v4f16*>(sbs + 8 * (16 * p + r) + 2 * q);
#pragma unroll
                for (int m = 0; m < G; ++m) step_term<QT>(O[m], X, sdx + 16 * p, TP, bs, q, acc[m][p]);
            }
        }
    }
#pragma unroll
    for (int m = 0; m < (SWIGLU ? 1 : G); ++m) {
        const int row = row0 + kRowsTile * m + 16 * wave + r;
        if (row >= a.rows) break;
        float* const out = MMID ? nullptr : a.out + (size_t)(g0 + 4 * q) * a.rows + row;
#pragma unroll
        for (int p = 0; p < PT; ++p) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int j = 16 * p + 4 * q + i;
                if (j >= cnt) continue;
                float v = acc[m][p][i];
                if constexpr (SWIGLU) v = __fmul_rn(silu_f32(v), acc[G - 1][p][i]);
                if constexpr (MMID) *reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.dst) + sdst[j] + 4 * (size_t)row) = v;
                else out[(size_t)(16 * p + i) * a.rows] = v;
            }
        }
    }
}

}  // namespace sabah
