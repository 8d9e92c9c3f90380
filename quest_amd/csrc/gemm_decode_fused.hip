// A W4A4 linear layer on a few tokens in one launch: every workgroup quantises the activation rows itself -- the wave program of
// hadamard_mfma.hip, and so its codes, sums and scales bit for bit -- into LDS, and multiplies its channels of the packed weights by them.
//
// Why: such a call is bound by what it costs to issue, 3.7 us for each of the two launches and 0.7 for the scratch between them, and then by the
// chain quantiser -> end of kernel -> launch -> first weights.  Here the first weights are on their way before the first activation is
// looked at, and there is neither scratch nor a second launch.  The price is the quantiser's arithmetic on every CU, so only calls whose rows are
// eight units (waves of 32 blocks of 128) at most come here: 16 tokens of 2048, 8 of 4096, 4 of 8192, 2 of 11008.
//
// A persistent workgroup of sixteen waves, one per CU, takes tiles of 16 channels.  Wave w multiplies the 256-k chunks w, w + 16, ... of
// each (as gemm_decode.hip does: the same nibble splitting and matrix instructions).  Weights travel by direct loads into a ring of kRing chunks of
// the wave's own, three chunks ahead and across tiles, so that no wave waits for another until the partial sums meet: integer additions into one
// tile in LDS, one barrier per tile, the waves finishing tiles in turn.
// What bounds it: up to 4096 channels the chain -- launch, activations, transform and quantiser, first products, sums -- of 4.3 us (K = 1024, one
// token) to 7.2 (K = 4096, eight); with more the weights' way from memory.  GPU time in a graph against the two launches, weights from HBM, us: (1,
// 4096, 4096) 5.5 / 7.1, (8, 4096, 4096) 7.1 / 7.6, (1, 1024, 4096) 4.8 / 6.2, (4, 8192, 8192) 11.3 / 13.2, (1, 4096, 22016) 12.4 / 12.9, (1, 11008, 4096)
// 8.0 / 9.8.  As calls, which the host bounds: (1, 4096, 4096) 7.0 / 11.2, (10, 1536, 1148) 7.3 / 11.5.
#include "gemm_tiles.h"
#include "hadamard_unit.h"

namespace quest {
namespace fewtok {

using hq::v4i;
using hq::v4u;

constexpr int kWaves = 16;
constexpr int kChannels = 16;
constexpr int kChunkB = 128;                       // packed bytes per row and chunk
constexpr int kRing = 3;                           // chunks of a wave's own weights in flight
constexpr int kSlotB = 2048;                       // two direct loads of a KiB: 16 rows x 64 bytes each
constexpr int kRingB = kWaves * kRing * kSlotB;
constexpr int kPad = 16;                           // behind every row of codes: a lane quarter's sixteen rows on different banks
constexpr int kMaxTokens = 16;
constexpr int kUnits = 8;                          // most units of a call (see most_tokens)
constexpr int kCodesB = kUnits * 2048 + kMaxTokens * kPad + kChunkB;       // a unit's codes are 2 KiB; the pads; what the last chunk reads past the last row
constexpr int kSumsAt = kRingB + kCodesB;
constexpr int kLdsB = kSumsAt + 2048 + 4 * 64;
static_assert(kLdsB <= 160 * 1024 && kMaxTokens <= 16 && kWaves <= 16, "LDS of a CU");

// what this wave has written to LDS is there for the others behind it; its direct loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    plain_barrier();
}

// *at += v in LDS.  (The atomic builtin waits for every direct load that is out, for they write to LDS too.)
__device__ __forceinline__ void lds_add(int *at, int v) {
    asm volatile("ds_add_u32 %0, %1" ::"v"((uint32_t)(uintptr_t)(__attribute__((address_space(3))) int *)at), "v"(v) : "memory");
}

struct Args {
    void *out;
    const uint16_t *x;
    const uint8_t *wgt;
    const int32_t *b_add;
    const uint16_t *b_mul, *bias;
    int M, N, K, tiles;
    uint32_t entry_bits;
};

// WPR, G as in hadamard_mfma.hip: waves per row, lanes of a half-wave per row
template <int DT, int WPR, int G, bool RAG>
__global__ void __launch_bounds__(64 * kWaves, 1) linear_few_tokens_kernel(Args p) {
    // (one array: with several the compiler waits for every direct load before anything is read from LDS)
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsB];
    uint8_t *const ring = lds, *const codes = lds + kRingB;
    int *const sums = reinterpret_cast<int *>(lds + kSumsAt);               // partial tiles meet here: [parity][channel of the lane's four][lane]
    float *const part_sq = reinterpret_cast<float *>(lds + kSumsAt + 2048);
    int *const part_add = reinterpret_cast<int *>(lds + kSumsAt + 2048 + 64);
    int *const a_add = reinterpret_cast<int *>(lds + kSumsAt + 2048 + 128);
    uint16_t *const a_mul = reinterpret_cast<uint16_t *>(lds + kSumsAt + 2048 + 192);
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int M = p.M, N = p.N, K = p.K;
    const int row_b = K >> 1, pitch = row_b + kPad;
    const int n_chunks = (row_b + kChunkB - 1) / kChunkB;

    // ---- the wave's stream of weight chunks: (tile, chunk) pairs in order; past the last one its loads touch no memory
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)p.wgt, 0, (int)((long)N * row_b), 0x00020000);
    uint8_t *const mine = ring + wave * (kRing * kSlotB);
    const uint32_t dead = 0x80000000u;
    int ld_tile = blockIdx.x, ld_chunk = wave;
    auto load_chunk = [&](int slot) {
        const bool any = ld_tile < p.tiles && ld_chunk < n_chunks;
        const int ch = ld_tile * kChannels + r, at = ld_chunk * kChunkB + g * 16;
        const uint32_t off = (uint32_t)ch * (uint32_t)row_b + (uint32_t)at;
#pragma unroll
        for (int hlf = 0; hlf < 2; hlf++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void *)(mine + slot * kSlotB + hlf * 1024), 16,
                                                     any && ch < N && at + 64 * hlf < row_b ? off + 64 * hlf : dead, 0, 0, 0);
        if (!any) return;
        ld_chunk += kWaves;
        if (ld_chunk >= n_chunks) {
            ld_chunk = wave;
            ld_tile += gridDim.x;
        }
    };

    // ---- the activation rows
    const int n = lane & 31, h = lane >> 5;
    const int part = wave % WPR;
    const int row = WPR == 1 ? wave * (32 / G) + n / G : wave / WPR;
    const int blk = part * 32 + n % G;
    const bool busy = (WPR == 1 ? wave * (32 / G) : wave / WPR) < M;            // uniform in the wave
    const bool live = row < M && blk < (RAG ? (K + 127) >> 7 : K >> 7);
    v4u bq[8];
    {
        const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)((long)M * K * 2), 0x00020000);
        const uint32_t ld_off = live ? (uint32_t)(row * K * 2 + blk * 256 + h * 16) : dead;
#pragma unroll
        for (int s = 0; s < 8; s++)
            bq[s] = __builtin_amdgcn_raw_buffer_load_b128(xr, (int)(!RAG || blk * 128 + 16 * s < K ? ld_off + 32 * s : dead), 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < kRing; s++) load_chunk(s);
    __builtin_amdgcn_sched_barrier(0);
    if (threadIdx.x < 512) sums[threadIdx.x] = 0;

    // the scales, sums and bias of the first tile that this wave finishes: its own number of the workgroup's tiles
    const int tok = r;
    uint32_t c_mul[4], c_bias[4] = {0, 0, 0, 0};
    v4u c_add;
    const __amdgpu_buffer_rsrc_t add_r = __builtin_amdgcn_make_buffer_rsrc((void *)p.b_add, 0, N * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t mul_r = __builtin_amdgcn_make_buffer_rsrc((void *)p.b_mul, 0, N * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t bias_r = __builtin_amdgcn_make_buffer_rsrc((void *)p.bias, 0, N * 2, 0x00020000);
    auto fetch_channels = [&](int tile) {          // (channels past the last, of tiles past the last too: zeros)
        const int ch = tile * kChannels + 4 * g;
        c_add = __builtin_amdgcn_raw_buffer_load_b128(add_r, ch * 4, 0, 0);
#pragma unroll
        for (int e = 0; e < 4; e++) c_mul[e] = __builtin_amdgcn_raw_buffer_load_b16(mul_r, ch * 2 + 2 * e, 0, 0);
        if (p.bias != nullptr) {
#pragma unroll
            for (int e = 0; e < 4; e++) c_bias[e] = __builtin_amdgcn_raw_buffer_load_b16(bias_r, ch * 2 + 2 * e, 0, 0);
        }
    };
    // Before the rows are looked at where no transform needs the registers and few waves have a row: behind them these would take the rows' registers, and waves
    // without a row wait for those and for the weights behind them (one token, no transform, (1760, 20672), weights from HBM: 10.9 us behind, 10.6 before; two tokens of
    // 10976, six waves of sixteen: 8.2 and 8.4).
    constexpr bool kEarly = RAG && WPR == 1;
    if constexpr (kEarly) fetch_channels(blockIdx.x + wave * gridDim.x);

    uint32_t yb[4][8];
    float total = 0.f;
    if (busy) {
        if constexpr (RAG) {
            total = hq::ragged_sum<DT, G>(yb, bq);
        } else {
            v4i hv[2][2];
            hq::signed_entries(hv, n, h, p.entry_bits);
            total = hq::transform<DT>(yb, bq, hv, p.entry_bits);
            total = G == 32 ? wave_sum_dpp_f(total) : hq::group_sum_f<G>(total);
        }
        if (WPR > 1 && lane == 0) part_sq[wave] = total;
    }
    if constexpr (WPR > 1) {
        lds_barrier();
        total = 0.f;
#pragma unroll
        for (int w = 0; w < WPR; w++) total += part_sq[min(wave - part + w, kWaves - 1)];          // in part order, as the activation kernel adds them
    }
    if (busy) {
        const uint32_t s16 = from_f32<DT>(scale_from_sumsq(total, K));
        uint32_t dw[8];
        hq::nibbles<DT>(dw, yb, s16, row < M);
        if constexpr (RAG) {
#pragma unroll
            for (int t = 0; t < 8; t++)
                if (blk * 128 + 64 * h + 8 * t >= K) dw[t] = 0;
        }
        int isum = 0;
#pragma unroll
        for (int t = 0; t < 8; t++) isum = __builtin_amdgcn_sdot8((int)dw[t], 0x11111111, isum, false);
        if (!live) isum = 0;
        const int t = G == 32 ? wave_sum_dpp_i(isum) : hq::group_sum_i<G>(isum);
        if (live) {
            uint8_t *dst = codes + row * pitch + blk * 64 + h * 32;
            if (!RAG || blk * 128 + 64 * h < K) *reinterpret_cast<uint4 *>(dst) = make_uint4(dw[0], dw[1], dw[2], dw[3]);
            if (!RAG || blk * 128 + 64 * h + 32 < K) *reinterpret_cast<uint4 *>(dst + 16) = make_uint4(dw[4], dw[5], dw[6], dw[7]);
        }
        if (lane % G == 0 && h == 0 && row < M) {
            if (part == 0) a_mul[row] = (uint16_t)s16;
            if constexpr (WPR == 1) a_add[row] = t; else part_add[wave] = t;
        }
    }
    if constexpr (!kEarly) fetch_channels(blockIdx.x + wave * gridDim.x);
    lds_barrier();                                 // codes, scales and sums are there
    const float t_half_mul = __fmul_rn(0.5f, to_f32<DT>(a_mul[min(tok, M - 1)]));
    int t_add = 0;
    if constexpr (WPR == 1) {
        t_add = a_add[min(tok, M - 1)];
    } else {
#pragma unroll
        for (int w = 0; w < WPR; w++) t_add += part_add[min(tok, M - 1) * WPR + w];
    }

    // ---- the tiles
    const uint8_t *const tok_codes = codes + min(tok, M - 1) * pitch + g * 16;     // (columns of tokens past M are not stored)
    int slot = 0, done = 0;                        // done: tiles before this one
    for (int tile = blockIdx.x; tile < p.tiles; tile += gridDim.x, done++) {
        v4i acc = {0, 0, 0, 0};
        for (int c = wave; c < n_chunks; c += kWaves) {
            wait_vmcnt_imm<2 * (kRing - 1)>();     // this chunk's weights have landed (whatever else is out is younger)
            asm volatile("" ::: "memory");
            v4i wq[2], aq[2];
#pragma unroll
            for (int hlf = 0; hlf < 2; hlf++) {
                wq[hlf] = *reinterpret_cast<const v4i *>(mine + slot * kSlotB + hlf * 1024 + lane * 16);
                aq[hlf] = *reinterpret_cast<const v4i *>(tok_codes + c * kChunkB + 64 * hlf);      // (past a row's end: times weights of zero)
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                      // read before the slot is loaded again
            __builtin_amdgcn_sched_barrier(0);
            load_chunk(slot);
            slot = slot + 1 == kRing ? 0 : slot + 1;
#pragma unroll
            for (int hlf = 0; hlf < 2; hlf++) {
                v4i we, wo, ae, ao;
#pragma unroll
                for (int d = 0; d < 4; d++) {
                    wo[d] = wq[hlf][d] & (int)0xF0F0F0F0u;
                    we[d] = (wq[hlf][d] << 4) & (int)0xF0F0F0F0u;
                    ao[d] = aq[hlf][d] & (int)0xF0F0F0F0u;
                    ae[d] = (aq[hlf][d] << 4) & (int)0xF0F0F0F0u;
                }
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(we, ae, acc, 0, 0, 0);
                acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(wo, ao, acc, 0, 0, 0);
            }
        }
        int *const sum = sums + (done & 1) * 256 + lane;
        if (wave < n_chunks) {
#pragma unroll
            for (int e = 0; e < 4; e++) lds_add(sum + e * 64, acc[e]);
        }
        // the tile's sums are complete behind the barrier; they are read and cleared before their reader reaches the next one, behind which
        // the tile after the next adds to the same place
        lds_barrier();
        if ((done & (kWaves - 1)) != wave) continue;
        int c[4];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            c[e] = sum[e * 64] >> 8;              // exact: every product carries 16 * 16
            sum[e * 64] = 0;
        }
        const int ch = tile * kChannels + 4 * g;
        if (tok < M && ch < N) {
            uint32_t o[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float lhs = (float)(c[e] * 2 + t_add + (int)c_add[e]);
                const float rhs = __fmul_rn(t_half_mul, to_f32<DT>(c_mul[e]));
                o[e] = from_f32<DT>(__fmul_rn(lhs, rhs));
                if (p.bias != nullptr) o[e] = from_f32<DT>(__fadd_rn(to_f32<DT>(o[e]), to_f32<DT>(c_bias[e])));
            }
            uint16_t *dst = reinterpret_cast<uint16_t *>(p.out) + (size_t)tok * N + ch;
            if ((N & 3) == 0) {
                *reinterpret_cast<uint2 *>(dst) = make_uint2(o[0] | (o[1] << 16), o[2] | (o[3] << 16));
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    if (ch + e < N) dst[e] = (uint16_t)o[e];
            }
        }
        fetch_channels(tile + kWaves * (int)gridDim.x);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");         // cleared
    }
    wait_vmcnt_imm<0>();                           // no direct load may outlive the workgroup's LDS allocation
}

template <int DT, bool RAG>
static int launch(int nb, const Args &a, int grid, hipStream_t st) {
    const dim3 blocks((unsigned)grid), threads(64 * kWaves);
    if (nb > 64) linear_few_tokens_kernel<DT, 3, 32, RAG><<<blocks, threads, 0, st>>>(a);
    else if (nb > 32) linear_few_tokens_kernel<DT, 2, 32, RAG><<<blocks, threads, 0, st>>>(a);
    else if (nb > 16) linear_few_tokens_kernel<DT, 1, 32, RAG><<<blocks, threads, 0, st>>>(a);
    else if (nb > 8) linear_few_tokens_kernel<DT, 1, 16, RAG><<<blocks, threads, 0, st>>>(a);
    else if (nb > 4) linear_few_tokens_kernel<DT, 1, 8, RAG><<<blocks, threads, 0, st>>>(a);
    else return QUEST_ERR_UNSUPPORTED;
    return launch_status();
}

// Tokens that come here: eight units of 32 blocks, and the sixteen columns of a tile.  With up to eight units the one launch is the faster one
// on the GPU as well at every size measured (K from 1024 to 11008, N from 1024 to 22016: 0.5 to 2.6 us); with more, the quantiser's
// arithmetic on every CU is longer than the second launch (K = N = 4096: eight tokens 7.2 against 7.6 us, twelve 8.6 against 7.7; (11008, 4096): two
// 9.0 against 10.1, four 10.8 against 10.2), though not than what the second launch costs the host.
static int most_tokens(int nb) {
    const int rows = nb > 16 ? 1 : nb > 8 ? 2 : 4;                  // of a unit
    const int most = nb > 64 ? kUnits / 3 : nb > 32 ? kUnits / 2 : kUnits * rows;
    return most < kMaxTokens ? most : kMaxTokens;
}

}  // namespace fewtok

static bool few_tokens_takes(int M, int K) {
    const int nb = (K + 127) / 128;
    return nb > 4 && nb <= 96 && M <= fewtok::most_tokens(nb);
}

}  // namespace quest

using namespace quest;

extern "C" int quest_linear_few_tokens_available(int size_m, int size_k) { return size_m > 0 && size_k > 0 && few_tokens_takes(size_m, size_k); }

extern "C" int quest_linear_few_tokens(void *out, const void *x, const uint8_t *w_packed, const int32_t *w_add, const void *w_scale, const void *bias,
                                       int size_m, int size_k, int size_n, float had_scale, int dtype, void *stream) {
    forget_stale_error();
    if (!out || !x || !w_packed || !w_add || !w_scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(dtype)) return QUEST_ERR_BAD_DTYPE;
    if (size_m <= 0 || size_k <= 0 || size_n <= 0 || (size_k & (had_scale != 0.f ? 127 : 31))) return QUEST_ERR_BAD_SHAPE;
    if (!aligned(x, 16) || !aligned(w_packed, 16) || !aligned(out, 8)) return QUEST_ERR_ALIGNMENT;
    uint32_t bits = 0;
    // (32-bit offsets into the weights, with the row that a last, partly filled tile reaches past them)
    if (!few_tokens_takes(size_m, size_k) || had_scale < 0.f || !representable16(had_scale, dtype, &bits) || ((long)size_n + 16) * (size_k / 2) >= (1L << 31))
        return QUEST_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const int tiles = (size_n + fewtok::kChannels - 1) / fewtok::kChannels, cus = device_cu_count(st);
    const fewtok::Args a = {out, (const uint16_t *)x, w_packed, w_add, (const uint16_t *)w_scale, (const uint16_t *)bias, size_m, size_n, size_k, tiles, bits};
    const int nb = (size_k + 127) / 128, grid = tiles < cus ? tiles : cus;
    const bool ragged = (size_k & 127) != 0;
    if (dtype == QUEST_DTYPE_BF16) return ragged ? fewtok::launch<0, true>(nb, a, grid, st) : fewtok::launch<0, false>(nb, a, grid, st);
    return ragged ? fewtok::launch<1, true>(nb, a, grid, st) : fewtok::launch<1, false>(nb, a, grid, st);
}
