// Row-wise kernels of the W4A4 linear path for gfx950: the Gaussian-clip scale, the INT4
// quantiser with nibble packing and row sums, the scale epilogue on an int32 matrix, the
// block-128 Walsh-Hadamard transform, and the single-pass fusion of Hadamard + scale +
// quantise + pack that the linear layer uses.  All are HBM-bound: every row is read once with
// 16-byte loads per lane and kept in registers until its outputs are written.
//
// Reference statements of the same arithmetic (file:line under gemm-quest/ of the reference):
//   scale      quest/quantize_kernel.cu:38-94,   benchmarks/utils.py:193-209
//   quantise   quest/quantize_kernel.cu:120-229, benchmarks/utils.py:334-365
//   epilogue   quest/quantize_kernel.cu:264-306, benchmarks/utils.py:535-545
//   Hadamard   benchmarks/utils.py:17,38-39,89-90
#include "hadamard_unit.h"

namespace quest {

// ---------------------------------------------------------------------------------------------
// Walsh-Hadamard butterflies on one 16-byte chunk per lane.  A 128-element block is spread over
// 16 consecutive lanes x 8 registers: distances 1, 2, 4 are inside the lane, 8, 16, 32, 64 are
// lane xor 1, 2, 4, 8.  Each butterfly is (a, b) -> (a + b, a - b) with `a` the element at the
// lower index, so the result is the same bit pattern as the textbook in-place loop.
// ---------------------------------------------------------------------------------------------
// One stage across lanes for the chunk's eight values: v <- v + sign * v[partner], one DPP multiply-add each (sign = -1 on the
// upper lane of a pair, whose difference so comes out negated: b - a for a - b; the caller turns it back once for all
// stages).  sign * v is exact, so every value is the textbook sum or difference, rounded once.  The leading s_nop covers
// the two wait states a DPP read needs after the write of its register, which the compiler does not track through asm.
#define QUEST_FWHT_STAGE(CTRL)                                                                                                    \
    asm("s_nop 1\n\t"                                                                                                             \
        "v_fmac_f32_dpp %0, %0, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %1, %1, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %2, %2, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %3, %3, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %4, %4, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %5, %5, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %6, %6, %8 " CTRL " row_mask:0xf bank_mask:0xf\n\t"                                                       \
        "v_fmac_f32_dpp %7, %7, %8 " CTRL " row_mask:0xf bank_mask:0xf"                                                           \
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]), "+v"(v[7])                          \
        : "v"(sign))

// Which of the 16 chunks of its block a lane works on: chunk lane % 16 with its two low bits flipped on the lanes whose bit 2
// is set.  The chunk at distance 4 is then eight lanes' mirror image (row_half_mirror), a DPP move like the other distances,
// where lane xor 4 would be a trip through the LDS crossbar.
__device__ __forceinline__ int fwht_chunk_of(int i) { return i ^ ((i & 4) != 0 ? 3 : 0); }

// The unscaled transform of a block whose lanes hold the chunks above, with `factor` as what the results have yet to be
// multiplied by: had_scale, negated on the lanes whose values the stages left negated (scaled() below).
__device__ __forceinline__ void fwht128_chunk(float (&v)[8], int lane, float had_scale, float &factor) {
#pragma unroll
    for (int h = 1; h < 8; h <<= 1) {
#pragma unroll
        for (int j = 0; j < 8; j++) {
            if ((j & h) == 0) {
                float a = v[j], b = v[j + h];
                v[j] = a + b;
                v[j + h] = a - b;
            }
        }
    }
    const int c = fwht_chunk_of(lane);
    float sign = (c & 1) ? -1.f : 1.f;
    QUEST_FWHT_STAGE("quad_perm:[1,0,3,2]");
    sign = (c & 2) ? -1.f : 1.f;
    QUEST_FWHT_STAGE("quad_perm:[2,3,0,1]");
    sign = (c & 4) ? -1.f : 1.f;
    QUEST_FWHT_STAGE("row_half_mirror");
    sign = (c & 8) ? -1.f : 1.f;
    QUEST_FWHT_STAGE("row_ror:8");
    factor = (__builtin_popcount(c & 15) & 1) ? -had_scale : had_scale;
}

// A product that turns no zero negative: a difference of equals is +0 in the textbook order, whatever lane it was taken on.
__device__ __forceinline__ float scaled(float v, float factor) { return __builtin_fmaf(v, factor, 0.f); }

template <int DT>
__device__ __forceinline__ void unpack8(const uint4 &raw, float (&v)[8]) {
    v[0] = lo_f32<DT>(raw.x); v[1] = hi_f32<DT>(raw.x);
    v[2] = lo_f32<DT>(raw.y); v[3] = hi_f32<DT>(raw.y);
    v[4] = lo_f32<DT>(raw.z); v[5] = hi_f32<DT>(raw.z);
    v[6] = lo_f32<DT>(raw.w); v[7] = hi_f32<DT>(raw.w);
}

template <int DT>
__device__ __forceinline__ uint4 pack8(const float (&v)[8]) {
    uint4 r;
    r.x = pack2_from_f32<DT>(v[0], v[1]);
    r.y = pack2_from_f32<DT>(v[2], v[3]);
    r.z = pack2_from_f32<DT>(v[4], v[5]);
    r.w = pack2_from_f32<DT>(v[6], v[7]);
    return r;
}

// eight codes (as floats in [-8, 7]) -> one dword, element 0 in the lowest nibble
__device__ __forceinline__ uint32_t pack_nibbles8(const float (&q)[8], int &sum) {
    uint32_t w = 0;
#pragma unroll
    for (int e = 0; e < 8; e++) {
        int c = (int)q[e];
        sum += c;
        w |= ((uint32_t)c & 0xFu) << (4 * e);
    }
    return w;
}

// The sum of squares of a row without the transform from its chunks' sums, in the order of the kernels that quantise such a row inside its tile or GEMM
// (ragged_sum in hadamard_unit.h).  Thread t holds chunks t, t + BLOCK, ...: sixteen lanes a block.
// slots: N * BLOCK / 16, one for every block
template <int BLOCK, int N>
__device__ __forceinline__ float ordered_sum(const float (&part)[N], int nchunks, float *slots) {
    const int lane = threadIdx.x & 63;
    float block[N];
#pragma unroll
    for (int i = 0; i < N; i++) block[i] = hq::chunks_tree(part[i]);
    if ((lane & 15) == 0) {
#pragma unroll
        for (int i = 0; i < N; i++) slots[(i * BLOCK + (int)threadIdx.x) >> 4] = block[i];
    }
    __syncthreads();
    constexpr int kBlocks = N * BLOCK / 16;
    if constexpr (kBlocks == 16) return hq::blocks_tree<16>(slots[lane & 15]);
    float total = 0.f;
#pragma unroll
    for (int b = 0; b < kBlocks; b += 64) {
        if (kBlocks > 128 && b * 16 >= nchunks) break;              // uniform
        const float v = hq::blocks_tree<32>(slots[b + (lane & (kBlocks - 1))]);
        total += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 0));
        if constexpr (kBlocks > 32) total += __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 32));
    }
    return total;
}

// ---------------------------------------------------------------------------------------------
// Fused Hadamard + scale + quantise + pack: one workgroup per row, NCHUNK 16-byte chunks per
// thread, the row lives in registers between its single read and its writes.
// Vector instructions bound it, not memory: at about 34 per element it took 36.5 us for bf16 [11008, 4096] (113 MB, 3.1 TB/s);
// with the DPP multiply-add stages, the clamp-free quantiser and the dot-product row sum it is about 16.
// FP32 (QUEST_QUANT_FROM_FP32): scale and codes come from the transform's fp32 output and the unrounded scale -- the
// arithmetic of the reference's evaluation-side fake quantiser (src/eval_hswag.py:201-214), which never holds the
// rotated tensor in 16 bits -- instead of from the dtype-rounded tensor the inference path materialises.
// PLAIN: no transform (had_scale == 0), in 16 bits; such rows can end anywhere and are summed in an order of their own.  Kernels of their own, for in one
// kernel the transform pays for them ([11008, 4096] packed: 26.6 us alone, 27.2 with the other's code beside it) and they for its registers: [16384, 30016]
// in 333 us with 113, 217 with 60.
// ---------------------------------------------------------------------------------------------
// Most waves on a SIMD: plain rows of more than 8192 elements have room for eight, which is slower: bf16 [16384, 10976] 84 us, with four 78.
constexpr int plain_waves(int nchunk) { return nchunk > 4 ? 4 : 8; }
template <int DT, int NCHUNK, int BLOCK, bool FP32, bool PLAIN>
__global__ void __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(1, PLAIN ? plain_waves(NCHUNK) : 8)))
hadamard_quantize_kernel(const uint16_t *__restrict__ x, uint16_t *__restrict__ scale,
                         uint32_t *__restrict__ packed, int32_t *__restrict__ row_sum,
                         uint16_t *__restrict__ x_had, int K, float had_scale, int scale_rule, int sum_bias) {
    static_assert(!(FP32 && PLAIN));
    __shared__ float slots_f[PLAIN ? NCHUNK * (BLOCK / 16) : BLOCK / 64];
    __shared__ int slots_i[BLOCK / 64];
    const int row = blockIdx.x;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int nchunks = K >> 3;
    const bool had = !PLAIN && had_scale != 0.f;
    const int chunk0 = had ? fwht_chunk_of(tid) : tid;         // blocks of 16 chunks: a row holds whole ones
    const uint4 *xr = reinterpret_cast<const uint4 *>(x + (size_t)row * K);
    const bool absmax = scale_rule == QUEST_SCALE_ABSMAX;

    uint4 raw[NCHUNK];
#pragma unroll
    for (int i = 0; i < NCHUNK; i++) {
        const int c = i * BLOCK + chunk0;
        raw[i] = (c < nchunks) ? xr[c] : make_uint4(0, 0, 0, 0);
    }

    float y[FP32 ? NCHUNK : 1][8];
    float sumsq = 0.f, amax = 0.f, part[PLAIN ? NCHUNK : 1];
    if constexpr (PLAIN) {
#pragma unroll
        for (int i = 0; i < NCHUNK; i++) part[i] = hq::chunk_sum<DT>(raw[i].x, raw[i].y, raw[i].z, raw[i].w);
        if (absmax) {                           // uniform
#pragma unroll
            for (int i = 0; i < NCHUNK; i++) {
                float v[8];
                unpack8<DT>(raw[i], v);
                sumsq += part[i];               // (whether there is a NaN)
#pragma unroll
                for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
            }
        }
    } else {
#pragma unroll
        for (int i = 0; i < NCHUNK; i++) {
            float (&v)[8] = y[FP32 ? i : 0];
            unpack8<DT>(raw[i], v);
            if (had) {
                float factor;
                fwht128_chunk(v, lane, had_scale, factor);
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = scaled(v[e], factor);
                raw[i] = make_uint4(pack2_rounded_products<DT>(v[0], v[1]), pack2_rounded_products<DT>(v[2], v[3]),
                                    pack2_rounded_products<DT>(v[4], v[5]), pack2_rounded_products<DT>(v[6], v[7]));
                if (!FP32) unpack8<DT>(raw[i], v);  // the transform's output exists only in dtype
            }
            // the squares of 16-bit floats are exact in fp32: the multiply-add rounds as multiply and add would (the fp32
            // transform's squares are not, and stay separate)
#pragma unroll
            for (int e = 0; e < 8; e++) sumsq = FP32 ? sumsq + v[e] * v[e] : __builtin_fmaf(v[e], v[e], sumsq);
            if (absmax) {                       // uniform
#pragma unroll
                for (int e = 0; e < 8; e++) amax = fmaxf(amax, fabsf(v[e]));
            }
        }
    }
    if (x_had != nullptr) {
        uint4 *hr = reinterpret_cast<uint4 *>(x_had + (size_t)row * K);
#pragma unroll
        for (int i = 0; i < NCHUNK; i++) {
            const int c = i * BLOCK + chunk0;
            if (c < nchunks) hr[c] = raw[i];
        }
    }

    // QUEST_SCALE_GAUSSIAN: the reference's rule from the row's mean square; QUEST_SCALE_ABSMAX: the row's largest
    // magnitude sits 7.5 steps out (a maximum is exact whatever the order, so this scale has no rounding slack)
    float s32;
    if (absmax) {
        const float m = block_max_f<BLOCK>(amax, slots_f);
        s32 = __fadd_rn(__fdiv_rn(m, 7.5f), kScaleEps);
    } else {
        float total;
        if constexpr (PLAIN) total = ordered_sum<BLOCK>(part, nchunks, slots_f);
        else total = block_sum_f<BLOCK>(sumsq, slots_f);
        s32 = scale_from_sumsq(total, K);
    }
    const uint32_t s16 = from_f32<DT>(s32);
    if (tid == 0) scale[row] = (uint16_t)s16;
    const float s = FP32 ? s32 : to_f32<DT>(s16);

    if (packed == nullptr && row_sum == nullptr) return;
    int isum = 0;
    auto put = [&](int i, uint32_t w) {
        const int c = i * BLOCK + chunk0;
        if (c < nchunks) {                      // chunks past the row's end are padding
            isum = __builtin_amdgcn_sdot8((int)w, 0x11111111, isum, false);
            if (packed != nullptr) packed[(size_t)row * nchunks + c] = w;
        }
    };
    // A NaN shows in the RMS scale but not in a maximum; the sum of squares has it either way.
    const bool nan_row = absmax && __syncthreads_or(sumsq != sumsq);
    if (!FP32 && quant_fast_ok(s) && !nan_row) {            // uniform: everything but degenerate rows
        const float inv28 = quant_inv28(s);
#pragma unroll
        for (int i = 0; i < NCHUNK; i++) {
            const uint32_t d[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
            uint32_t w = 0;
#pragma unroll
            for (int p = 3; p >= 0; p--) {
                w = push_top_nibble(w, quant_top_nibble_half<DT, 1>(d[p], inv28));
                w = push_top_nibble(w, quant_top_nibble_half<DT, 0>(d[p], inv28));
            }
            put(i, w);
        }
    } else {
        const float inv = quant_inv(s);
#pragma unroll
        for (int i = 0; i < NCHUNK; i++) {
            float v[8], q[8];
            if constexpr (!FP32) unpack8<DT>(raw[i], v);
#pragma unroll
            for (int e = 0; e < 8; e++) q[e] = quant_code_inv(FP32 ? y[FP32 ? i : 0][e] : v[e], inv);
            int unused = 0;
            put(i, pack_nibbles8(q, unused));
        }
    }
    if (row_sum != nullptr) {
        const int t = block_sum_i<BLOCK>(isum, slots_i);
        if (tid == 0) row_sum[row] = t + sum_bias;
    }
}

// ---------------------------------------------------------------------------------------------
// Stand-alone Hadamard (weights offline; activations when the caller wants the unfused steps)
// ---------------------------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256)
hadamard128_kernel(uint16_t *__restrict__ y, const uint16_t *__restrict__ x, long nchunks_total, float had_scale) {
    const int lane = threadIdx.x & 63;
    // 16 consecutive chunks (= threads) make one block; the grid strides in multiples of 256 threads
    for (long c = (long)blockIdx.x * 256 + threadIdx.x; c < nchunks_total; c += (long)gridDim.x * 256) {
        const long mine = (c & ~15L) + fwht_chunk_of((int)(c & 15));         // c is block-aligned up to the lane's part
        uint4 raw = reinterpret_cast<const uint4 *>(x)[mine];
        float v[8], factor;
        unpack8<DT>(raw, v);
        fwht128_chunk(v, lane, had_scale, factor);
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = scaled(v[e], factor);
        reinterpret_cast<uint4 *>(y)[mine] = make_uint4(pack2_rounded_products<DT>(v[0], v[1]), pack2_rounded_products<DT>(v[2], v[3]),
                                                        pack2_rounded_products<DT>(v[4], v[5]), pack2_rounded_products<DT>(v[6], v[7]));
    }
}

// ---------------------------------------------------------------------------------------------
// Scale only
// ---------------------------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256)
find_scale_kernel(uint16_t *__restrict__ scale, const uint16_t *__restrict__ x, int K) {
    __shared__ float slots_f[4];
    const int row = blockIdx.x;
    const int nchunks = K >> 3;
    const uint4 *xr = reinterpret_cast<const uint4 *>(x + (size_t)row * K);
    float sumsq = 0.f;
    for (int c = threadIdx.x; c < nchunks; c += 256) {
        float v[8];
        unpack8<DT>(xr[c], v);
#pragma unroll
        for (int e = 0; e < 8; e++) sumsq += v[e] * v[e];
    }
    const float total = block_sum_f<256>(sumsq, slots_f);
    if (threadIdx.x == 0) scale[row] = (uint16_t)from_f32<DT>(scale_from_sumsq(total, K));
}

// ---------------------------------------------------------------------------------------------
// Quantise with a given scale; every output optional
// ---------------------------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256)
quantize_kernel(uint16_t *__restrict__ x, const uint16_t *__restrict__ scale, int8_t *__restrict__ x_int,
                uint32_t *__restrict__ packed, int32_t *__restrict__ row_sum, int K, int do_dequantize) {
    __shared__ int slots_i[4];
    const int row = blockIdx.x;
    const int nchunks = K >> 3;
    uint4 *xr = reinterpret_cast<uint4 *>(x + (size_t)row * K);
    const float s = to_f32<DT>(scale[row]);
    const float half_s = __fmul_rn(s, 0.5f);
    const float inv = quant_inv(s);
    // scales in the fast range take the clamp-free form of the quantiser (in its variant for arbitrary inputs: this
    // entry point pairs any x with any scale), the others the med3 form; both equal the IEEE-divide statement
    const bool fast = quant_fast_ok(s);
    const float inv28 = quant_inv28(s);
    int isum = 0;
    // two chunks per thread and pass, both loads issued before either is used (a row of 4096 is exactly one pass)
    for (int c0 = threadIdx.x; c0 < nchunks; c0 += 512) {
        const int c1 = c0 + 256;
        const bool two = c1 < nchunks;
        uint4 raw[2];
        raw[0] = xr[c0];
        raw[1] = two ? xr[c1] : make_uint4(0, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            if (u == 1 && !two) break;
            const int c = u == 0 ? c0 : c1;
            float v[8], q[8];
            unpack8<DT>(raw[u], v);
            if (fast) {
#pragma unroll
                for (int e = 0; e < 8; e++) q[e] = (float)(quant_top_nibble_any(v[e], inv28) >> 28);
            } else {
#pragma unroll
                for (int e = 0; e < 8; e++) q[e] = quant_code_inv(v[e], inv);
            }
            if (do_dequantize) {
#pragma unroll
                for (int e = 0; e < 8; e++) v[e] = __fadd_rn(__fmul_rn(q[e], s), half_s);
                xr[c] = pack8<DT>(v);
            }
            const uint32_t w = pack_nibbles8(q, isum);
            if (packed != nullptr) packed[(size_t)row * nchunks + c] = w;
            if (x_int != nullptr) {
                uint2 b;
                b.x = ((uint32_t)(int)q[0] & 0xFFu) | (((uint32_t)(int)q[1] & 0xFFu) << 8) |
                      (((uint32_t)(int)q[2] & 0xFFu) << 16) | (((uint32_t)(int)q[3] & 0xFFu) << 24);
                b.y = ((uint32_t)(int)q[4] & 0xFFu) | (((uint32_t)(int)q[5] & 0xFFu) << 8) |
                      (((uint32_t)(int)q[6] & 0xFFu) << 16) | (((uint32_t)(int)q[7] & 0xFFu) << 24);
                reinterpret_cast<uint2 *>(x_int + (size_t)row * K)[c] = b;
            }
        }
    }
    if (row_sum != nullptr) {
        const int t = block_sum_i<256>(isum, slots_i);
        if (threadIdx.x == 0) row_sum[row] = t;
    }
}

// ---------------------------------------------------------------------------------------------
// Scale epilogue on an int32 matrix (the unfused debug path)
// ---------------------------------------------------------------------------------------------
template <int DT>
__global__ void __launch_bounds__(256)
add_mul_vv_kernel(uint16_t *__restrict__ d, const int32_t *__restrict__ a_add, const uint16_t *__restrict__ a_mul,
                  const int32_t *__restrict__ b_add, const uint16_t *__restrict__ b_mul,
                  const int32_t *__restrict__ c, int size_a, int size_b) {
    const int col_blocks = (size_b + 255) / 256;
    const int row = blockIdx.x / col_blocks;
    const int col = (blockIdx.x % col_blocks) * 256 + threadIdx.x;
    if (row >= size_a || col >= size_b) return;
    const size_t idx = (size_t)row * size_b + col;
    const float lhs = (float)(c[idx] * 2 + a_add[row] + b_add[col]);
    const float rhs = __fmul_rn(__fmul_rn(0.5f, to_f32<DT>(a_mul[row])), to_f32<DT>(b_mul[col]));
    d[idx] = (uint16_t)from_f32<DT>(__fmul_rn(lhs, rhs));
}

// ---------------------------------------------------------------------------------------------
// launchers
// ---------------------------------------------------------------------------------------------
template <int DT>
static int launch_hadamard_quantize(const void *x, void *scale, uint8_t *packed, int32_t *row_sum, void *x_had,
                                    int K, int M, float had_scale, int scale_rule, hipStream_t st, int sum_bias = 0) {
    const int nchunks = K >> 3;
    const bool fp32 = (scale_rule & QUEST_QUANT_FROM_FP32) != 0;
#define QUEST_HQ(NCH, BLK)                                                                              \
    (fp32 ? hadamard_quantize_kernel<DT, NCH, BLK, true, false> : had_scale == 0.f ? hadamard_quantize_kernel<DT, NCH, BLK, false, true> \
          : hadamard_quantize_kernel<DT, NCH, BLK, false, false>)<<<dim3(M), dim3(BLK), 0, st>>>( \
        (const uint16_t *)x, (uint16_t *)scale, (uint32_t *)packed, row_sum, (uint16_t *)x_had, K, had_scale, scale_rule & ~QUEST_QUANT_FROM_FP32, sum_bias)
    if (nchunks <= 256) QUEST_HQ(1, 256);
    else if (nchunks <= 512) QUEST_HQ(2, 256);
    else if (nchunks <= 1024) QUEST_HQ(4, 256);
    else if (nchunks <= 2048) QUEST_HQ(8, 256);
    else if (nchunks <= 8192) QUEST_HQ(8, 1024);
    else return QUEST_ERR_UNSUPPORTED;
#undef QUEST_HQ
    return launch_status();
}

// Rotary position embedding on interleaved pairs, in place (src/models/llama.py:43-62 of the reference): the first
// n_heads * head_dim elements of every row are heads of (re, im) pairs; pair i of a head at position t turns by the
// angle whose (cos, sin) is freqs[t][i].  fp32 products and sums in the reference's order, one rounding to dtype.
template <int DT>
__global__ void __launch_bounds__(256)
rope_kernel(uint16_t *__restrict__ x, const float *__restrict__ freqs, int n_rows, int seq_len, int row_stride,
            int rot_cols, int head_dim) {
    const int chunks = rot_cols >> 3;                        // 16-byte chunks (4 pairs) to rotate per row
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)n_rows * chunks) return;
    const int row = (int)(idx / chunks);
    const int col = (int)(idx % chunks) * 8;
    const int t = row % seq_len;
    const int pair0 = (col % head_dim) >> 1;
    uint4 *p = reinterpret_cast<uint4 *>(x + (size_t)row * row_stride + col);
    const float4 *f = reinterpret_cast<const float4 *>(freqs + ((size_t)t * (head_dim >> 1) + pair0) * 2);
    const uint4 v = *p;
    const float4 f01 = f[0], f23 = f[1];
    const uint32_t in[4] = {v.x, v.y, v.z, v.w};
    const float cs[4][2] = {{f01.x, f01.y}, {f01.z, f01.w}, {f23.x, f23.y}, {f23.z, f23.w}};
    uint32_t o[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const float re = lo_f32<DT>(in[i]), im = hi_f32<DT>(in[i]);
        const float c = cs[i][0], sn = cs[i][1];
        const float out_re = __fsub_rn(__fmul_rn(re, c), __fmul_rn(im, sn));
        const float out_im = __fadd_rn(__fmul_rn(re, sn), __fmul_rn(im, c));
        o[i] = from_f32<DT>(out_re) | (from_f32<DT>(out_im) << 16);
    }
    *p = make_uint4(o[0], o[1], o[2], o[3]);
}

}  // namespace quest

using namespace quest;

extern "C" int quest_find_scale_int4(void *scale, const void *x, int group_size, int batch_size, int dtype, void *stream) {
    forget_stale_error();
    if (!scale || !x) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 7)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16)) return QUEST_ERR_ALIGNMENT;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == QUEST_DTYPE_BF16)
        find_scale_kernel<0><<<dim3(batch_size), dim3(256), 0, st>>>((uint16_t *)scale, (const uint16_t *)x, group_size);
    else
        find_scale_kernel<1><<<dim3(batch_size), dim3(256), 0, st>>>((uint16_t *)scale, (const uint16_t *)x, group_size);
    return launch_status();
}

extern "C" int quest_quantize_int4(void *x, const void *scale, int8_t *x_int, uint8_t *x_int_packed,
                                   int32_t *x_int_row_sum, int group_size, int batch_size, int do_dequantize,
                                   int dtype, void *stream) {
    forget_stale_error();
    if (!x || !scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 7)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(x_int, 8) || !aligned(x_int_packed, 4)) return QUEST_ERR_ALIGNMENT;
    hipStream_t st = (hipStream_t)stream;
    if (dtype == QUEST_DTYPE_BF16)
        quantize_kernel<0><<<dim3(batch_size), dim3(256), 0, st>>>((uint16_t *)x, (const uint16_t *)scale, x_int,
                                                                    (uint32_t *)x_int_packed, x_int_row_sum, group_size, do_dequantize);
    else
        quantize_kernel<1><<<dim3(batch_size), dim3(256), 0, st>>>((uint16_t *)x, (const uint16_t *)scale, x_int,
                                                                    (uint32_t *)x_int_packed, x_int_row_sum, group_size, do_dequantize);
    return launch_status();
}

// Eight consecutive columns per thread (32 + 32 + 16 bytes in, 16 out, all as 16-byte vectors): for matrices whose rows are
// whole eights and 16-byte aligned.  Same arithmetic per element as the kernel above.
template <int DT>
__global__ void __launch_bounds__(256)
add_mul_vv_x8_kernel(uint16_t *__restrict__ d, const int32_t *__restrict__ a_add, const uint16_t *__restrict__ a_mul,
                     const int32_t *__restrict__ b_add, const uint16_t *__restrict__ b_mul,
                     const int32_t *__restrict__ c, int size_a, int size_b) {
    const int chunks = size_b >> 3;                                   // per row
    const int col_blocks = (chunks + 255) / 256;
    const int row = blockIdx.x / col_blocks;
    const int chunk = (blockIdx.x % col_blocks) * 256 + threadIdx.x;
    if (row >= size_a || chunk >= chunks) return;
    const int col = chunk * 8;
    const size_t idx = (size_t)row * size_b + col;
    const int4 c0 = *reinterpret_cast<const int4 *>(c + idx), c1 = *reinterpret_cast<const int4 *>(c + idx + 4);
    const int4 b0 = *reinterpret_cast<const int4 *>(b_add + col), b1 = *reinterpret_cast<const int4 *>(b_add + col + 4);
    const uint4 bm = *reinterpret_cast<const uint4 *>(b_mul + col);
    const int ra = a_add[row];
    const float half_am = __fmul_rn(0.5f, to_f32<DT>(a_mul[row]));
    const int cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
    const int bs[8] = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
    const uint32_t ms[4] = {bm.x, bm.y, bm.z, bm.w};
    uint32_t o[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
        const float l0 = (float)(cs[2 * j] * 2 + ra + bs[2 * j]), l1 = (float)(cs[2 * j + 1] * 2 + ra + bs[2 * j + 1]);
        const float r0 = __fmul_rn(half_am, lo_f32<DT>(ms[j])), r1 = __fmul_rn(half_am, hi_f32<DT>(ms[j]));
        o[j] = (uint32_t)from_f32<DT>(__fmul_rn(l0, r0)) | ((uint32_t)from_f32<DT>(__fmul_rn(l1, r1)) << 16);
    }
    *reinterpret_cast<uint4 *>(d + idx) = make_uint4(o[0], o[1], o[2], o[3]);
}

extern "C" int quest_add_mul_vv(void *mat_d, const int32_t *vec_a_add, const void *vec_a_mul, const int32_t *vec_b_add,
                                const void *vec_b_mul, const int32_t *mat_c, int size_a, int size_b, int dtype,
                                void *stream) {
    forget_stale_error();
    if (!mat_d || !vec_a_add || !vec_a_mul || !vec_b_add || !vec_b_mul || !mat_c) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (size_a <= 0 || size_b <= 0) return QUEST_ERR_BAD_SHAPE;
    hipStream_t st = (hipStream_t)stream;
    if ((size_b & 7) == 0 && aligned(mat_d, 16) && aligned(mat_c, 16) && aligned(vec_b_add, 16) && aligned(vec_b_mul, 16)) {
        const long nb8 = (long)((size_b / 8 + 255) / 256) * size_a;
        if (nb8 > 0x7fffffffL) return QUEST_ERR_UNSUPPORTED;
        if (dtype == QUEST_DTYPE_BF16)
            add_mul_vv_x8_kernel<0><<<dim3((unsigned)nb8), dim3(256), 0, st>>>(
                (uint16_t *)mat_d, vec_a_add, (const uint16_t *)vec_a_mul, vec_b_add, (const uint16_t *)vec_b_mul, mat_c, size_a, size_b);
        else
            add_mul_vv_x8_kernel<1><<<dim3((unsigned)nb8), dim3(256), 0, st>>>(
                (uint16_t *)mat_d, vec_a_add, (const uint16_t *)vec_a_mul, vec_b_add, (const uint16_t *)vec_b_mul, mat_c, size_a, size_b);
        return launch_status();
    }
    const long nblocks = (long)((size_b + 255) / 256) * size_a;
    if (nblocks > 0x7fffffffL) return QUEST_ERR_UNSUPPORTED;
    dim3 grid((unsigned)nblocks);
    if (dtype == QUEST_DTYPE_BF16)
        add_mul_vv_kernel<0><<<grid, dim3(256), 0, st>>>((uint16_t *)mat_d, vec_a_add, (const uint16_t *)vec_a_mul, vec_b_add,
                                                         (const uint16_t *)vec_b_mul, mat_c, size_a, size_b);
    else
        add_mul_vv_kernel<1><<<grid, dim3(256), 0, st>>>((uint16_t *)mat_d, vec_a_add, (const uint16_t *)vec_a_mul, vec_b_add,
                                                         (const uint16_t *)vec_b_mul, mat_c, size_a, size_b);
    return launch_status();
}

extern "C" int quest_hadamard128(void *y, const void *x, int group_size, int batch_size, float had_scale, int dtype,
                                 void *stream) {
    forget_stale_error();
    if (!y || !x) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 127)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(y, 16)) return QUEST_ERR_ALIGNMENT;
    hipStream_t st = (hipStream_t)stream;
    const long nchunks = (long)batch_size * (group_size >> 3);
    long blocks = (nchunks + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (dtype == QUEST_DTYPE_BF16)
        hadamard128_kernel<0><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((uint16_t *)y, (const uint16_t *)x, nchunks, had_scale);
    else
        hadamard128_kernel<1><<<dim3((unsigned)blocks), dim3(256), 0, st>>>((uint16_t *)y, (const uint16_t *)x, nchunks, had_scale);
    return launch_status();
}

// sum_bias is added to every row sum that is written
static int hadamard_quantize_any(const void *x, void *scale, uint8_t *x_int_packed, int32_t *x_int_row_sum, void *x_had,
                                 int group_size, int batch_size, float had_scale, int scale_rule, int dtype, hipStream_t st, int sum_bias) {
    if ((scale_rule & ~QUEST_QUANT_FROM_FP32) != QUEST_SCALE_ABSMAX && (scale_rule & ~QUEST_QUANT_FROM_FP32) != QUEST_SCALE_GAUSSIAN)
        return QUEST_ERR_BAD_SHAPE;
    if (!x || !scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    // the transform works on blocks of 128; without it (had_scale == 0) a row only has to be whole 16-byte chunks
    if (group_size <= 0 || batch_size <= 0 || (group_size & (had_scale != 0.f ? 127 : 7))) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(x_had, 16) || !aligned(x_int_packed, 4)) return QUEST_ERR_ALIGNMENT;
    if (scale_rule == QUEST_SCALE_GAUSSIAN && (group_size & 127) == 0) {
        // whole blocks, rows of up to 32768, a Hadamard entry the dtype holds exactly: matrix cores; anything else: the row kernel
        const int rc = launch_hadamard_quantize_mfma(0, x, nullptr, 0.f, scale, x_int_packed, x_int_row_sum, x_had, nullptr,
                                                     group_size, batch_size, had_scale, dtype, st, nullptr, nullptr, nullptr, sum_bias);
        if (rc != QUEST_ERR_UNSUPPORTED) return rc;
    }
    auto *f = dtype == QUEST_DTYPE_BF16 ? launch_hadamard_quantize<0> : launch_hadamard_quantize<1>;
    return f(x, scale, x_int_packed, x_int_row_sum, x_had, group_size, batch_size, had_scale, scale_rule, st, sum_bias);
}

extern "C" int quest_hadamard_quantize_int4(const void *x, void *scale, uint8_t *x_int_packed, int32_t *x_int_row_sum,
                                            void *x_had, int group_size, int batch_size, float had_scale, int dtype,
                                            void *stream) {
    forget_stale_error();
    return hadamard_quantize_any(x, scale, x_int_packed, x_int_row_sum, x_had, group_size, batch_size, had_scale, QUEST_SCALE_GAUSSIAN,
                                 dtype, (hipStream_t)stream, 0);
}

extern "C" int quest_hadamard_quantize_int4_rule(const void *x, void *scale, uint8_t *x_int_packed, int32_t *x_int_row_sum,
                                                 void *x_had, int group_size, int batch_size, float had_scale,
                                                 int scale_rule, int dtype, void *stream) {
    forget_stale_error();
    return hadamard_quantize_any(x, scale, x_int_packed, x_int_row_sum, x_had, group_size, batch_size, had_scale, scale_rule, dtype,
                                 (hipStream_t)stream, 0);
}

extern "C" int quest_pack_weight_int4(const void *weight, void *w_scale, uint8_t *w_int_packed, int32_t *w_add, int size_k, int size_n,
                                      float had_scale, int scale_rule, int dtype, void *stream) {
    forget_stale_error();
    if (!w_int_packed || !w_add) return QUEST_ERR_NULL_POINTER;
    return hadamard_quantize_any(weight, w_scale, w_int_packed, w_add, nullptr, size_k, size_n, had_scale, scale_rule, dtype,
                                 (hipStream_t)stream, size_k / 2);
}

extern "C" int quest_rmsnorm_hadamard_quantize_int4(const void *x, const void *norm_weight, float eps, void *scale,
                                                    uint8_t *x_int_packed, int32_t *x_int_row_sum, void *x_had,
                                                    void *x_norm, int group_size, int batch_size, float had_scale,
                                                    int dtype, void *stream) {
    forget_stale_error();
    if (!x || !norm_weight || !scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 127)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(norm_weight, 16) || !aligned(x_had, 16) || !aligned(x_norm, 16) || !aligned(x_int_packed, 16))
        return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(1, x, norm_weight, eps, scale, x_int_packed, x_int_row_sum, x_had, x_norm,
                                         group_size, batch_size, had_scale, dtype, (hipStream_t)stream);
}

extern "C" int quest_add_rmsnorm_hadamard_quantize_int4(void *x, const void *branch, const void *norm_weight, float eps,
                                                        void *scale, uint8_t *x_int_packed, int32_t *x_int_row_sum,
                                                        int group_size, int batch_size, float had_scale, int dtype,
                                                        void *stream) {
    forget_stale_error();
    if (!x || !branch || !norm_weight || !scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 127)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(branch, 16) || !aligned(norm_weight, 16) || !aligned(x_int_packed, 16))
        return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(1, x, norm_weight, eps, scale, x_int_packed, x_int_row_sum, nullptr, nullptr,
                                         group_size, batch_size, had_scale, dtype, (hipStream_t)stream, branch, x);
}

extern "C" int quest_silu_mul_hadamard_quantize_int4(const void *gate_up, void *scale, uint8_t *x_int_packed,
                                                     int32_t *x_int_row_sum, void *x_had, void *x_act, int group_size,
                                                     int batch_size, float had_scale, int dtype, void *stream) {
    forget_stale_error();
    if (!gate_up || !scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 127)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(gate_up, 16) || !aligned(x_had, 16) || !aligned(x_act, 16) || !aligned(x_int_packed, 16)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(2, gate_up, nullptr, 0.f, scale, x_int_packed, x_int_row_sum, x_had, x_act,
                                         group_size, batch_size, had_scale, dtype, (hipStream_t)stream);
}

// ---- the same kernels writing the codes as E2M3 tiles (the operand form of gemm_e2m3.hip) -------------------------------
static int e2m3_rows_check(const void *x, const void *scale, const void *tiles, int group_size, int batch_size, int dtype) {
    if (!x || !scale || !tiles) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 127)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(tiles, 16)) return QUEST_ERR_ALIGNMENT;
    return QUEST_OK;
}

extern "C" int quest_hadamard_quantize_e2m3(const void *x, void *scale, void *x_tiles, uint8_t *x_int_packed,
                                            int32_t *x_int_row_sum, void *x_had, int group_size, int batch_size,
                                            float had_scale, int dtype, void *stream) {
    forget_stale_error();
    const int rc = e2m3_rows_check(x, scale, x_tiles, group_size, batch_size, dtype);
    if (rc != QUEST_OK) return rc;
    if (!aligned(x_had, 16) || !aligned(x_int_packed, 4)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(0, x, nullptr, 0.f, scale, x_int_packed, x_int_row_sum, x_had, nullptr, group_size,
                                         batch_size, had_scale, dtype, (hipStream_t)stream, nullptr, nullptr, (uint8_t *)x_tiles);
}

extern "C" int quest_activation_before_gemm(const quest_activation *a, void *stream) {
    forget_stale_error();
    if (!a || !a->x || !a->scale || (!a->tiles && (!a->x_int_packed || !a->x_int_row_sum))) return QUEST_ERR_NULL_POINTER;
    if (a->producer < QUEST_PRODUCER_NONE || a->producer > QUEST_PRODUCER_SILU_MUL || (a->producer != QUEST_PRODUCER_RMSNORM && a->branch)) return QUEST_ERR_UNSUPPORTED;
    if (a->producer == QUEST_PRODUCER_RMSNORM && !a->norm_weight) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(a->dtype)) return QUEST_ERR_BAD_DTYPE;
    const bool padded = a->producer == QUEST_PRODUCER_NONE && a->had_scale == 0.f && a->tiles;
    if (a->size_k <= 0 || a->size_m <= 0 || (a->size_k & (padded ? 31 : 127))) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(a->x, 16) || !aligned(a->branch, 16) || !aligned(a->norm_weight, 16) || !aligned(a->x_int_packed, 16) || !aligned(a->tiles, 16)) return QUEST_ERR_ALIGNMENT;
    NextWeights next;
    if (a->next != nullptr && aligned(a->next, 16) && a->next_pitch % 16 == 0 && a->next_bytes <= a->next_pitch)
        next = {a->next, a->next_pitch, a->next_bytes & ~(size_t)15, a->next_blocks};
    return launch_hadamard_quantize_mfma(a->producer, a->x, a->norm_weight, a->eps, a->scale, a->tiles ? nullptr : a->x_int_packed, a->tiles ? nullptr : a->x_int_row_sum, nullptr, nullptr, a->size_k, a->size_m,
                                         a->had_scale, a->dtype, (hipStream_t)stream, a->branch, a->branch ? (void *)a->x : nullptr, (uint8_t *)a->tiles, 0, next);
}

extern "C" int quest_quantize_e2m3_padded(const void *x, void *scale, void *x_tiles, int group_size, int batch_size, int dtype, void *stream) {
    forget_stale_error();
    if (!x || !scale || !x_tiles) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (group_size <= 0 || batch_size <= 0 || (group_size & 31)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(x_tiles, 16)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(0, x, nullptr, 0.f, scale, nullptr, nullptr, nullptr, nullptr, group_size, batch_size, 0.f, dtype,
                                         (hipStream_t)stream, nullptr, nullptr, (uint8_t *)x_tiles);
}

extern "C" int quest_rmsnorm_hadamard_quantize_e2m3(const void *x, const void *norm_weight, float eps, void *scale,
                                                    void *x_tiles, void *x_norm, int group_size, int batch_size,
                                                    float had_scale, int dtype, void *stream) {
    forget_stale_error();
    const int rc = e2m3_rows_check(x, scale, x_tiles, group_size, batch_size, dtype);
    if (rc != QUEST_OK) return rc;
    if (!norm_weight) return QUEST_ERR_NULL_POINTER;
    if (!aligned(norm_weight, 16) || !aligned(x_norm, 16)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(1, x, norm_weight, eps, scale, nullptr, nullptr, nullptr, x_norm, group_size, batch_size,
                                         had_scale, dtype, (hipStream_t)stream, nullptr, nullptr, (uint8_t *)x_tiles);
}

extern "C" int quest_add_rmsnorm_hadamard_quantize_e2m3(void *x, const void *branch, const void *norm_weight, float eps,
                                                        void *scale, void *x_tiles, int group_size, int batch_size,
                                                        float had_scale, int dtype, void *stream) {
    forget_stale_error();
    const int rc = e2m3_rows_check(x, scale, x_tiles, group_size, batch_size, dtype);
    if (rc != QUEST_OK) return rc;
    if (!branch || !norm_weight) return QUEST_ERR_NULL_POINTER;
    if (!aligned(branch, 16) || !aligned(norm_weight, 16)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(1, x, norm_weight, eps, scale, nullptr, nullptr, nullptr, nullptr, group_size, batch_size,
                                         had_scale, dtype, (hipStream_t)stream, branch, x, (uint8_t *)x_tiles);
}

extern "C" int quest_silu_mul_hadamard_quantize_e2m3(const void *gate_up, void *scale, void *x_tiles, void *x_act,
                                                     int group_size, int batch_size, float had_scale, int dtype,
                                                     void *stream) {
    forget_stale_error();
    const int rc = e2m3_rows_check(gate_up, scale, x_tiles, group_size, batch_size, dtype);
    if (rc != QUEST_OK) return rc;
    if (!aligned(x_act, 16)) return QUEST_ERR_ALIGNMENT;
    return launch_hadamard_quantize_mfma(2, gate_up, nullptr, 0.f, scale, nullptr, nullptr, nullptr, x_act, group_size, batch_size,
                                         had_scale, dtype, (hipStream_t)stream, nullptr, nullptr, (uint8_t *)x_tiles);
}

extern "C" int quest_rope_interleaved(void *x, const float *freqs_cis, int n_rows, int seq_len, int row_stride,
                                      int rot_cols, int head_dim, int dtype, void *stream) {
    forget_stale_error();
    if (!x || !freqs_cis) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (n_rows <= 0 || seq_len <= 0 || rot_cols <= 0 || head_dim <= 0 || (head_dim & 7) || (rot_cols % head_dim) ||
        rot_cols > row_stride || (row_stride & 7))
        return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(freqs_cis, 16)) return QUEST_ERR_ALIGNMENT;
    const long work = (long)n_rows * (rot_cols >> 3);
    const unsigned blocks = (unsigned)((work + 255) / 256);
    hipStream_t st = (hipStream_t)stream;
    if (dtype == QUEST_DTYPE_BF16)
        rope_kernel<0><<<dim3(blocks), dim3(256), 0, st>>>((uint16_t *)x, freqs_cis, n_rows, seq_len, row_stride, rot_cols, head_dim);
    else
        rope_kernel<1><<<dim3(blocks), dim3(256), 0, st>>>((uint16_t *)x, freqs_cis, n_rows, seq_len, row_stride, rot_cols, head_dim);
    return launch_status();
}
