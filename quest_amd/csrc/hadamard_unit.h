// One wave's share of the fused activation kernel -- up to 32 blocks of 128 of a row, or of several short ones -- in the register layout that
// hadamard_mfma.hip describes at its top.  Shared by that kernel and by gemm_decode_fused.hip and gemm_e2m3_fused.hip, which quantise a few
// tokens inside the GEMM's workgroups: one sequence of operations, so that both give the same bits.
#pragma once
#include "common.h"

namespace quest {
namespace hq {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));

typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef _Float16 v2h __attribute__((ext_vector_type(2)));

// acc + lo(w)^2 + hi(w)^2 for a dword of two 16-bit floats (squares of 16-bit floats are exact in fp32)
template <int DT>
__device__ __forceinline__ float dot2_self(uint32_t w, float acc) {
    if constexpr (DT == QUEST_DTYPE_BF16)
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2bf, w), __builtin_bit_cast(v2bf, w), acc, false);
    else
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, w), __builtin_bit_cast(v2h, w), acc, false);
}

template <int DT>
__device__ __forceinline__ v16f mfma_h(const v4i &a, const v4i &b, const v16f &c) {
    if constexpr (DT == QUEST_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Sum over the G lanes (G a power of two, aligned) of each half-wave that hold one row, and over the two half-waves.
template <int G>
__device__ __forceinline__ float lanes_sum_f(float v) {
    if constexpr (G >= 2) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));
    if constexpr (G >= 4) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));
    if constexpr (G >= 8) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x141, 0xF, 0xF, true));
    if constexpr (G >= 16) v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));
    if constexpr (G >= 32) v += lane_xor_f<16>(v);
    return v;
}
template <int G>
__device__ __forceinline__ float group_sum_f(float v) {
    v = lanes_sum_f<G>(v);
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int G>
__device__ __forceinline__ int group_sum_i(int v) {
    if constexpr (G >= 2) v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, true);
    if constexpr (G >= 4) v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, true);
    if constexpr (G >= 8) v += __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, true);
    if constexpr (G >= 16) v += __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, true);
    if constexpr (G >= 32) v += lane_xor_i<16>(v);
    const auto r = __builtin_amdgcn_permlane32_swap((unsigned)v, (unsigned)v, false, false);
    return (int)r[0] + (int)r[1];
}

// ---- Rows that are not whole 128s, without the transform: the sum of squares in one order, whether the row is quantised here (ragged_sum: the row, or the
// wave's 32 blocks of it where several waves share one, in every lane of the row) or by the row kernel for packed codes (ordered_sum in rowops.hip), so
// that its scale does not depend on that.  A chunk of eight elements is a chain of four dot products; the sixteen chunks of a block and the 32 blocks of a
// wave are balanced trees, the chunks paired by bits 1, 3, 2 and 0 of their number (two of a lane's eight, then the half-waves).  bq[s] is chunk 2 s + h;
// blocks past the row's end are zeros, which change no sum.
template <int DT>
__device__ __forceinline__ float chunk_sum(uint32_t x, uint32_t y, uint32_t z, uint32_t w) {
    return dot2_self<DT>(w, dot2_self<DT>(z, dot2_self<DT>(y, dot2_self<DT>(x, 0.f))));
}
// the tree over the sixteen lanes that hold a block's chunks
__device__ __forceinline__ float chunks_tree(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xF, 0xF, true));        // lane xor 2
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xF, 0xF, true));       // xor 8: row_ror:8
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xF, 0xF, true));       // row_ror:4, which is xor 4 by now
    return v + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xF, 0xF, true));  // xor 1
}
// the tree over the G lanes that hold a row's (a wave's) blocks
template <int G>
__device__ __forceinline__ float blocks_tree(float v) {
    v = lanes_sum_f<(G < 16 ? G : 16)>(v);
    if constexpr (G >= 32) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
        v = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    }
    return v;
}
// The row is spread (see below) on the way, chunk by chunk as the loads arrive: left to the compiler that comes after the scale, 0.1 us of a short launch.
__device__ __forceinline__ void spread_chunk(uint32_t (&yb)[4][8], const v4u (&bq)[8], int s);
template <int DT, int G>
__device__ __forceinline__ float ragged_sum(uint32_t (&yb)[4][8], const v4u (&bq)[8]) {
    float c[8];
#pragma unroll
    for (int s = 0; s < 8; s++) {
        c[s] = chunk_sum<DT>(bq[s][0], bq[s][1], bq[s][2], bq[s][3]);
        spread_chunk(yb, bq, s);
        __builtin_amdgcn_sched_barrier(0);
    }
    const float v = ((c[0] + c[1]) + (c[4] + c[5])) + ((c[2] + c[3]) + (c[6] + c[7]));
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return blocks_tree<G>(__uint_as_float(r[0]) + __uint_as_float(r[1]));
}

// ---- the four A fragments: +-entry with sign (-1)^(popcount(n & 7 & j) + n3 h) [* (-1)^n4] [* -1]; lane (n, h)
__device__ __forceinline__ void signed_entries(v4i (&hv)[2][2], int n, int h, uint32_t entry_bits) {
    const uint32_t lane_flip = ((n >> 3) & 1) & h;
    uint32_t base[4];
#pragma unroll
    for (int d = 0; d < 4; d++) {
        uint32_t w = 0;
#pragma unroll
        for (int e = 0; e < 2; e++) {
            const int j = 2 * d + e;
            const uint32_t neg = (__builtin_popcount(n & 7 & j) & 1) ^ lane_flip;
            w |= (entry_bits ^ (neg << 15)) << (16 * e);
        }
        base[d] = w;
    }
    const uint32_t s0_flip = ((n >> 4) & 1) ? 0x80008000u : 0u;
#pragma unroll
    for (int d = 0; d < 4; d++) {
        hv[0][0][d] = (int)base[d];
        hv[0][1][d] = (int)(base[d] ^ 0x80008000u);
        hv[1][0][d] = (int)(base[d] ^ s0_flip);
        hv[1][1][d] = (int)(base[d] ^ s0_flip ^ 0x80008000u);
    }
}

// ---- No transform: the loaded chunks are the outputs already and only have to change lanes: lane (n, h) loaded the chunks whose k has bit 3 equal to h
// and the code below wants those whose bit 2 is h, so the two half-waves trade half of every chunk (nothing is multiplied: NaN and Inf stay where they are).
// yb[mt][q * 2 + pair]: outputs 32 mt + 8 q + 4 h + {0,1} / {2,3} of block n.
__device__ __forceinline__ void spread_chunk(uint32_t (&yb)[4][8], const v4u (&bq)[8], int s) {
#pragma unroll
    for (int p = 0; p < 2; p++) {
        // outputs 16 s + 8 (q & 1) + 4 h + 2 p + {0, 1}: pair 2 h + p of the chunk held by the half-wave q & 1
        const auto sw = __builtin_amdgcn_permlane32_swap(bq[s][p], bq[s][2 + p], false, false);
#pragma unroll
        for (int qo = 0; qo < 2; qo++) yb[s >> 1][(2 * (s & 1) + qo) * 2 + p] = sw[qo];
    }
}

// ---- Hadamard: 8 k-steps x 4 row tiles; then round to the dtype (the transform's output exists only in dtype) and sum the
// squares.  yb as above.  entry_bits == 0: no transform.
template <int DT>
__device__ __forceinline__ float transform(uint32_t (&yb)[4][8], const v4u (&bq)[8], const v4i (&hv)[2][2], uint32_t entry_bits) {
    float sumsq = 0.f;
    if (entry_bits == 0) {                      // uniform
#pragma unroll
        for (int s = 0; s < 8; s++) spread_chunk(yb, bq, s);
#pragma unroll
        for (int s = 0; s < 8; s++)
#pragma unroll
            for (int p = 0; p < 2; p++)
#pragma unroll
                for (int qo = 0; qo < 2; qo++) sumsq = dot2_self<DT>(yb[s >> 1][(2 * (s & 1) + qo) * 2 + p], sumsq);
    } else {
        v16f acc[4];
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[mt][r] = 0.f;
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const v4i b = __builtin_bit_cast(v4i, bq[s]);
#pragma unroll
            for (int mt = 0; mt < 4; mt++) {
                const int neg = ((mt & 1) & ((s >> 1) & 1)) ^ (((mt >> 1) & 1) & ((s >> 2) & 1));
                acc[mt] = mfma_h<DT>(hv[s & 1][neg], b, acc[mt]);
            }
        }
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int p = 0; p < 2; p++) {
                    const uint32_t w = pack2_rne<DT>(acc[mt][q * 4 + 2 * p], acc[mt][q * 4 + 2 * p + 1]);
                    yb[mt][q * 2 + p] = w;
                    sumsq = dot2_self<DT>(w, sumsq);            // both squares straight from the packed pair
                }
    }
    return sumsq;
}

// ---- codes.  Outputs 8 Q + 4 h + {0..3} (Q = 4 mt + q) give one half-word c3 c2 c1 c0 of two's-complement nibbles.
// Scales in the quantiser's fast range (everything but degenerate rows) take the clamp-free form: the code
// arrives in the top nibble of an integer and is shifted into the half-word by one v_alignbit per code.
// Lane (n, 0) ends with dwords 0..7 of the block's 64 packed bytes, lane (n, 1) with dwords 8..15: dword D is the
// half-word Q = D of lane (n, 0) below that of lane (n, 1).  v_permlane32_swap hands the lower lane both half-words
// t and the upper lane both half-words t + 8.  in_range: whether the lane's row is one whose scale counts.
template <int DT>
__device__ __forceinline__ void nibbles(uint32_t (&dw)[8], const uint32_t (&yb)[4][8], uint32_t s16, bool in_range) {
    const float sf = to_f32<DT>(s16);
    uint32_t hw[16];
    if (__builtin_expect(__builtin_amdgcn_ballot_w64(in_range && !quant_fast_ok(sf)) == 0, 1)) {
        // (falls through: behind the code for degenerate rows it is a jump over 600 instructions; bf16 [8192, 4096] 17.1 us and 16.1, [16384, 2816] 24.1 and 22.9, fp16
        // the same to 1 %, as the tiles' two forms in hadamard_mfma.hip would be)
        const float inv28 = quant_inv28(sf);
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t w0 = yb[mt][q * 2], w1 = yb[mt][q * 2 + 1];
                uint32_t g = (uint32_t)quant_top_nibble_half<DT, 1>(w1, inv28) >> 28;
                g = push_top_nibble(g, quant_top_nibble_half<DT, 0>(w1, inv28));
                g = push_top_nibble(g, quant_top_nibble_half<DT, 1>(w0, inv28));
                hw[mt * 4 + q] = push_top_nibble(g, quant_top_nibble_half<DT, 0>(w0, inv28));
            }
    } else {
        const float inv = quant_inv(sf);
#pragma unroll
        for (int mt = 0; mt < 4; mt++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const uint32_t w0 = yb[mt][q * 2], w1 = yb[mt][q * 2 + 1];
                const uint32_t c0 = (uint32_t)quant_code_inv_i(lo_f32<DT>(w0), inv) & 15u;
                const uint32_t c1 = (uint32_t)quant_code_inv_i(hi_f32<DT>(w0), inv) & 15u;
                const uint32_t c2 = (uint32_t)quant_code_inv_i(lo_f32<DT>(w1), inv) & 15u;
                const uint32_t c3 = (uint32_t)quant_code_inv_i(hi_f32<DT>(w1), inv) & 15u;
                hw[mt * 4 + q] = (((c3 * 16 + c2) * 16 + c1) * 16) + c0;
            }
    }
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const auto sw = __builtin_amdgcn_permlane32_swap(hw[t], hw[t + 8], false, false);
        dw[t] = sw[0] | (sw[1] << 16);
    }
}

// ---- RMSNorm in front of the transform: dtype(dtype(f32(x) * rsqrt(mean(x^2) + eps)) * w), ss_row the sum of the row's squares
template <int DT>
__device__ __forceinline__ void normalise(v4u (&bq)[8], const v4u (&wq)[8], float ss_row, int K, float eps) {
    const float mean_sq = __fmul_rn(ss_row, __fdiv_rn(1.0f, (float)K));
    const float r = __frsqrt_rn(__fadd_rn(mean_sq, eps));
#pragma unroll
    for (int s = 0; s < 8; s++)
#pragma unroll
        for (int d = 0; d < 4; d++) {
            const uint32_t y = pack2_rounded_products<DT>(__fmul_rn(lo_f32<DT>(bq[s][d]), r), __fmul_rn(hi_f32<DT>(bq[s][d]), r));
            bq[s][d] = pack2_rounded_products<DT>(__fmul_rn(lo_f32<DT>(y), lo_f32<DT>(wq[s][d])),
                                                  __fmul_rn(hi_f32<DT>(y), hi_f32<DT>(wq[s][d])));
        }
}

// ---- codes as E2M3: lane (n, h)'s 24 bytes of half g of the block's k-step h, inv = quant_inv of the row's scale.  FAST: the scale is in the
// quantiser's fast range.
typedef _Float16 v32h __attribute__((ext_vector_type(32)));
typedef unsigned v6u __attribute__((ext_vector_type(6)));
typedef unsigned v16u __attribute__((ext_vector_type(16)));
template <int DT, bool FAST>
__device__ __forceinline__ v6u e2m3_group(const uint32_t (&yb)[4][8], int g, float inv) {
    v16u hp;                                    // dword d = 4 q + 2 h' + p: outputs 8 q + 4 h' + 2 p + {0, 1} of the group
#pragma unroll
    for (int j = 0; j < 8; j++) {               // j = 2 q + p
        const auto sw = __builtin_amdgcn_permlane32_swap(yb[g][j], yb[g + 2][j], false, false);
#pragma unroll
        for (int hh = 0; hh < 2; hh++) {
            float f0, f1;
            if constexpr (FAST) {
                f0 = quant_floor_half<DT, 0>(sw[hh], inv);
                f1 = quant_floor_half<DT, 1>(sw[hh], inv);
            } else {
                f0 = quant_code_inv(lo_f32<DT>(sw[hh]), inv);
                f1 = quant_code_inv(hi_f32<DT>(sw[hh]), inv);
            }
            // to fp16 (round towards zero saturates at +-65504 instead of overflowing), then + 1/2
            const v2h c = __builtin_bit_cast(v2h, __builtin_amdgcn_cvt_pkrtz(f0, f1)) + v2h{(_Float16)0.5f, (_Float16)0.5f};
            hp[4 * (j >> 1) + 2 * hh + (j & 1)] = __builtin_bit_cast(unsigned, c);
        }
    }
    return __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(__builtin_bit_cast(v32h, hp), 1.0f);
}

}  // namespace hq

// Whether `v` survives a round trip through the 16-bit dtype, and its bits there.
inline bool representable16(float v, int dtype, uint32_t *bits) {
    uint32_t u;
    __builtin_memcpy(&u, &v, 4);
    if (dtype == QUEST_DTYPE_BF16) {
        if (u & 0xFFFFu) return false;
        *bits = u >> 16;
        return true;
    }
    const _Float16 hf = (_Float16)v;
    if ((float)hf != v) return false;
    uint16_t b;
    __builtin_memcpy(&b, &hf, 2);
    *bits = b;
    return true;
}

}  // namespace quest
