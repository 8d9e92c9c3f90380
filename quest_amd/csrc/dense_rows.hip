// The end of a model's forward for the few rows whose logits are wanted: RMSNorm of the last position of every sequence and
// the dense language-model head on those rows.
//
// The head is a (V, d) 16-bit matrix read once for at most 64 rows, so the kernel is a weight stream: 32 channels per
// workgroup, eight waves that share K in chunks of 64 (whole 128-byte lines of 16 rows per pair of loads), partial tiles
// meeting in LDS.  The library's GEMM took 285 us for 32 rows of d = 1024 against V = 32000 (65 MB) and 156 us for 2 rows
// of d = 2560 against V = 50304 (257 MB); reading those bytes takes 13 and 51 us.
#include "common.h"

namespace quest {
namespace rows {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

template <int DT>
__device__ __forceinline__ v4f mfma_k32(const v4i &a, const v4i &b, const v4f &c) {
    if constexpr (DT == QUEST_DTYPE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

// out[b] = dtype(dtype(f32(x) * rsqrt(mean(x^2) + eps)) * w) for row b of x at x + b * stride (src/models/llama.py:71-77 of the
// reference), x first replaced by dtype(x + branch) when there is a branch.  One workgroup per row.
template <int DT>
__global__ void __launch_bounds__(256)
rmsnorm_rows_kernel(uint16_t *__restrict__ out, const uint16_t *__restrict__ x, const uint16_t *__restrict__ branch,
                    const uint16_t *__restrict__ w, long stride, int cols, float eps) {
    __shared__ float slots[4];
    const uint32_t *xr = reinterpret_cast<const uint32_t *>(x + blockIdx.x * stride);
    const uint32_t *br = branch == nullptr ? nullptr : reinterpret_cast<const uint32_t *>(branch + blockIdx.x * stride);
    const uint32_t *wr = reinterpret_cast<const uint32_t *>(w);
    uint32_t *o = reinterpret_cast<uint32_t *>(out + (size_t)blockIdx.x * cols);
    auto value = [&](int i) {
        uint32_t v = xr[i];
        if (br != nullptr) {
            const uint32_t b = br[i];
            v = pack2_rounded_products<DT>(__fadd_rn(lo_f32<DT>(v), lo_f32<DT>(b)), __fadd_rn(hi_f32<DT>(v), hi_f32<DT>(b)));
        }
        return v;
    };
    float ss = 0.f;
    for (int i = threadIdx.x; i < cols / 2; i += 256) {
        const uint32_t v = value(i);
        ss += lo_f32<DT>(v) * lo_f32<DT>(v) + hi_f32<DT>(v) * hi_f32<DT>(v);
    }
    const float r = __frsqrt_rn(__fadd_rn(__fdiv_rn(block_sum_f<256>(ss, slots), (float)cols), eps));
    for (int i = threadIdx.x; i < cols / 2; i += 256) {
        const uint32_t v = value(i), g = wr[i];
        const uint32_t y = pack2_rounded_products<DT>(__fmul_rn(lo_f32<DT>(v), r), __fmul_rn(hi_f32<DT>(v), r));
        o[i] = pack2_rounded_products<DT>(__fmul_rn(lo_f32<DT>(y), lo_f32<DT>(g)), __fmul_rn(hi_f32<DT>(y), hi_f32<DT>(g)));
    }
}

constexpr int kWaves = 8;
constexpr int kUnits = 2;                 // 16-channel units per workgroup
constexpr int kChunkB = 128;              // bytes per row per chunk (64 k)
constexpr int kBatch = 2;                 // chunks whose loads are in flight together per wave

// TM = row tiles of 16 (M <= 16 TM)
template <int DT, int TM>
__global__ void __launch_bounds__(64 * kWaves)
dense_rows_kernel(uint16_t *__restrict__ out, const uint16_t *__restrict__ x, const uint16_t *__restrict__ wgt, int M, int N, int K) {
    __shared__ __attribute__((aligned(16))) float red[kWaves][kUnits * TM][64][4];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const size_t row_b = (size_t)K * 2;
    const int ch0 = blockIdx.x * 16 * kUnits;
    // rows past the end are clamped to the last one: their products are not stored
    const uint8_t *wp[kUnits], *xp[TM];
#pragma unroll
    for (int u = 0; u < kUnits; u++) wp[u] = reinterpret_cast<const uint8_t *>(wgt) + (size_t)min(ch0 + 16 * u + r, N - 1) * row_b + g * 16;
#pragma unroll
    for (int t = 0; t < TM; t++) xp[t] = reinterpret_cast<const uint8_t *>(x) + (size_t)min(16 * t + r, M - 1) * row_b + g * 16;

    v4f acc[kUnits][TM];
#pragma unroll
    for (int u = 0; u < kUnits; u++)
#pragma unroll
        for (int t = 0; t < TM; t++) acc[u][t] = v4f{0.f, 0.f, 0.f, 0.f};

    // a lane's 16 bytes of a 64-byte half chunk: both operands permute k alike, which a dot product ignores
    const int chunks = K / 64;
    for (int c0 = wave; c0 < chunks; c0 += kWaves * kBatch) {
        v4i wq[kBatch][2][kUnits], xq[kBatch][2][TM];
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            const int c = c0 + i * kWaves;
            if (i > 0 && c >= chunks) break;                          // uniform
#pragma unroll
            for (int h = 0; h < 2; h++) {
#pragma unroll
                for (int u = 0; u < kUnits; u++) wq[i][h][u] = *reinterpret_cast<const v4i *>(wp[u] + (size_t)c * kChunkB + h * 64);
#pragma unroll
                for (int t = 0; t < TM; t++) xq[i][h][t] = *reinterpret_cast<const v4i *>(xp[t] + (size_t)c * kChunkB + h * 64);
            }
        }
#pragma unroll
        for (int i = 0; i < kBatch; i++) {
            if (i > 0 && c0 + i * kWaves >= chunks) break;
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int u = 0; u < kUnits; u++)
#pragma unroll
                    for (int t = 0; t < TM; t++) acc[u][t] = mfma_k32<DT>(wq[i][h][u], xq[i][h][t], acc[u][t]);
        }
    }
#pragma unroll
    for (int u = 0; u < kUnits; u++)
#pragma unroll
        for (int t = 0; t < TM; t++) *reinterpret_cast<v4f *>(&red[wave][u * TM + t][lane][0]) = acc[u][t];
    __syncthreads();
    // wave w finishes the tiles w, w + 8, ...: lane (r, g) holds channels 4 g .. 4 g + 3 of row r of the tile
    for (int tile = wave; tile < kUnits * TM; tile += kWaves) {
        v4f s = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; w++) s += *reinterpret_cast<const v4f *>(&red[w][tile][lane][0]);
        const int row = (tile % TM) * 16 + r, ch = ch0 + (tile / TM) * 16 + 4 * g;
        if (row >= M) continue;
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (ch + e < N) out[(size_t)row * N + ch + e] = (uint16_t)from_f32<DT>(s[e]);
    }
}

}  // namespace rows
}  // namespace quest

using namespace quest;

extern "C" int quest_rmsnorm_rows(void *out, const void *x, const void *branch, const void *norm_weight, float eps, int n_rows,
                                  long row_stride, int cols, int dtype, void *stream) {
    forget_stale_error();
    if (!out || !x || !norm_weight) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (n_rows <= 0 || cols <= 0 || (cols & 1) || row_stride < cols || (row_stride & 1)) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(out, 4) || !aligned(x, 4) || !aligned(branch, 4) || !aligned(norm_weight, 4)) return QUEST_ERR_ALIGNMENT;
    auto *f = dtype == QUEST_DTYPE_BF16 ? rows::rmsnorm_rows_kernel<0> : rows::rmsnorm_rows_kernel<1>;
    f<<<dim3(n_rows), dim3(256), 0, (hipStream_t)stream>>>((uint16_t *)out, (const uint16_t *)x, (const uint16_t *)branch, (const uint16_t *)norm_weight, row_stride, cols, eps);
    return launch_status();
}

extern "C" int quest_dense_rows(void *out, const void *x, const void *weight, int size_m, int size_k, int size_n, int dtype, void *stream) {
    forget_stale_error();
    if (!out || !x || !weight) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (size_m <= 0 || size_n <= 0 || size_k <= 0 || (size_k & 63)) return QUEST_ERR_BAD_SHAPE;
    if (size_m > 64) return QUEST_ERR_UNSUPPORTED;
    if (!aligned(x, 16) || !aligned(weight, 16)) return QUEST_ERR_ALIGNMENT;
    const dim3 grid((size_n + 16 * rows::kUnits - 1) / (16 * rows::kUnits)), block(64 * rows::kWaves);
#define QUEST_ROWS(TM)                                                                                                          \
    (dtype == QUEST_DTYPE_BF16 ? rows::dense_rows_kernel<0, TM> : rows::dense_rows_kernel<1, TM>)<<<grid, block, 0, (hipStream_t)stream>>>( \
        (uint16_t *)out, (const uint16_t *)x, (const uint16_t *)weight, size_m, size_n, size_k)
    if (size_m <= 16) QUEST_ROWS(1);
    else if (size_m <= 32) QUEST_ROWS(2);
    else QUEST_ROWS(4);
#undef QUEST_ROWS
    return launch_status();
}
