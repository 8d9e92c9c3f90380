// W4A4 GEMM on the FP6 (E2M3) matrix instructions for some tens to a few hundred tokens, K split inside the workgroup.  Operands as
// E2M3 tiles and arithmetic as in gemm_e2m3.hip (every sum exact in fp32, so the order of the products does not matter), outputs
// identical bit for bit.
//
// A workgroup of four waves owns 32 TF tokens x 32 CF channels and splits K four ways: wave q multiplies the whole tile over the
// 64-k steps q, q + 4, ... .  No operand is shared between the waves, so each runs its own pipeline without a barrier: direct
// loads (1 KiB of a fragment's 1536 bytes per instruction) into a ring of kStages steps of its own in LDS, the next step's
// fragments read from there while the current one is multiplied from registers.  The four partial sums then meet in LDS in the
// [token][channel] layout that the epilogue reads eight channels at a time and stores as whole lines.
// What bounds it: the bytes into the CU (45-50 per cycle reached) and, for larger tiles, the reduction at the end (10 k cycles
// for 128 x 128, as much as the products of K = 2560: such tiles are gemm_e2m3_mid.hip's).  At (64, 11008, 4096), weights rotating
// through four copies, 9.7 us where the weight-streaming INT8 kernel took 16.0; (64, 4096, 4096) 6.0 against 7.5.
#include "e2m3_epilogue.h"

namespace quest {
namespace e2m3s {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kWaves = 4;
constexpr int kFragB = 1536;

template <int TF, int CF>
struct Tile {
    static constexpr int kTok = 32 * TF, kChn = 32 * CF, kFrags = TF + CF;
    static constexpr int kPitch = kChn + 4;       // floats per token row in LDS: sixteen lanes' 16-byte stores on different banks
    static constexpr int kTailLoads = (TF + 1) / 2 + (CF + 1) / 2;     // two fragments' tails per instruction
    static constexpr int kLoads = kFrags + kTailLoads;                 // direct loads per step
    static constexpr int kSlotB = kFrags * 1024 + kTailLoads * 1024;   // heads, then (pairs of) tails
    static constexpr int kWgPerCu = 16 * TF * CF + 12 * kFrags + 40 <= 256 && 3 * kWaves * kSlotB <= 80 * 1024 ? 2 : 1;
    static constexpr int kLdsMax = (160 / kWgPerCu) * 1024;
    static constexpr int kStages = kLdsMax / (kWaves * kSlotB) < 6 ? kLdsMax / (kWaves * kSlotB) : 6;
    static_assert(kStages >= 3 && kLoads * (kStages - 1) < 64, "steps in flight");
    static constexpr int kRingB = kWaves * kStages * kSlotB;
    // the four waves' partial sums of kPartBlocks token blocks at a time fit the LDS
    static constexpr int kPartB = kWaves * 32 * kPitch * 4;       // ... of one token block
    static constexpr int kPartBlocks = TF * kPartB <= kLdsMax ? TF : TF % 2 == 0 && TF * kPartB <= 2 * kLdsMax ? TF / 2 : 1;
    static constexpr int kLdsB = kRingB > kPartBlocks * kPartB ? kRingB : kPartBlocks * kPartB;
};

template <int DT, bool ROPE, int TF, int CF>
__device__ __forceinline__ void tile(uint8_t *lds, void *__restrict__ out, const uint8_t *__restrict__ act, const uint8_t *__restrict__ wgt,
                                     int M, int N, int K, int tiles_t, int tiles_c, const Epilogue &epi) {
    using S = Tile<TF, CF>;
    constexpr int D = S::kStages;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63;
    int tt, ct;
    if (!tile_of(tiles_t, tiles_c, tt, ct)) return;              // uniform: the whole workgroup
    const int tok0 = tt * S::kTok, ch0 = ct * S::kChn;
    const int nk = K / 64;
    const int pitch = nk * kFragB;                               // bytes per row block
    const int rbs_t = (M + 31) / 32, rbs_c = (N + 31) / 32;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)act, 0, rbs_t * pitch, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)wgt, 0, rbs_c * pitch, 0x00020000);
    // row blocks past the end of a matrix are read as its last one: their products are not stored
    int at[TF + CF];
#pragma unroll
    for (int f = 0; f < TF; f++) at[f] = min(tok0 / 32 + f, rbs_t - 1) * pitch;
#pragma unroll
    for (int f = 0; f < CF; f++) at[TF + f] = min(ch0 / 32 + f, rbs_c - 1) * pitch;

    // the epilogue's scale values set out first: a thread keeps eight channels there and walks down the tokens
    constexpr int kCols = S::kChn / 8, kRowsAtOnce = 64 * kWaves / kCols;
    const int col = (int)threadIdx.x % kCols, row0 = (int)threadIdx.x / kCols;
    const int ch = ch0 + col * 8;
    const bool works = ch < N && row0 < kRowsAtOnce;
    const bool vec16 = (N & 7) == 0;
    constexpr int kIters = (32 * S::kPartBlocks + kRowsAtOnce - 1) / kRowsAtOnce;      // rows of a thread per part
    float muls[8], t_half_mul[TF / S::kPartBlocks][kIters];
#pragma unroll
    for (int part = 0; part < TF / S::kPartBlocks; part++)
#pragma unroll
        for (int i = 0; i < kIters; i++)
            t_half_mul[part][i] = __fmul_rn(0.5f, to_f32<DT>(epi.a_mul[min(tok0 + 32 * S::kPartBlocks * part + row0 + i * kRowsAtOnce, M - 1)]));
    {   // (channels past the vector's end read as zeros: their outputs are not stored)
        const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void *)epi.b_mul, 0, (N * 2 + 2) & ~3, 0x00020000);
        const v4i m = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(br, ch * 2, 0, 0));
#pragma unroll
        for (int i = 0; i < 8; i++) muls[i] = i & 1 ? hi_f32<DT>((uint32_t)m[i >> 1]) : lo_f32<DT>((uint32_t)m[i >> 1]);
    }
    // ... and what the epilogue adds or rotates by
    Ahead<ROPE> ahead[TF / S::kPartBlocks][kIters];
    if (ROPE || epi.kind == kEpiAdd || epi.kind == kEpiBias) {   // uniform
#pragma unroll
        for (int part = 0; part < TF / S::kPartBlocks; part++)
#pragma unroll
            for (int i = 0; i < kIters; i++) {
                const int row = row0 + i * kRowsAtOnce;
                fetch_ahead<DT>(ahead[part][i], out, epi, tok0 + 32 * S::kPartBlocks * part + row, works && row < 32 * S::kPartBlocks ? ch : N, M, N, vec16);
            }
    }
    // tails: lanes 0-31 bring fragment 2 j's 512 bytes, lanes 32-63 those of 2 j + 1 of the same matrix (or nothing)
    uint32_t tail_at[S::kTailLoads];
#pragma unroll
    for (int j = 0; j < S::kTailLoads; j++) {
        const bool tok = j < (TF + 1) / 2;
        const int f0 = tok ? 2 * j : TF + 2 * (j - (TF + 1) / 2);
        const bool two = f0 + 1 < (tok ? TF : TF + CF);
        const uint32_t base = lane < 32 ? (uint32_t)at[f0] : two ? (uint32_t)at[two ? f0 + 1 : f0] : 0x80000000u;
        tail_at[j] = base + 1024 + (lane & 31) * 16;
    }
    uint8_t *const ring = lds + wave * D * S::kSlotB;
    auto load_one = [&](int slot, int step, int j) {             // steps past the end touch no memory
        uint8_t *dst = ring + slot * S::kSlotB + j * 1024;
        const bool tok = j < S::kFrags ? j < TF : j - S::kFrags < (TF + 1) / 2;
        const uint32_t off = j < S::kFrags ? (uint32_t)lane * 16 : tail_at[j < S::kFrags ? 0 : j - S::kFrags];
        __builtin_amdgcn_raw_ptr_buffer_load_lds(tok ? xr : wr, (__attribute__((address_space(3))) void *)dst, 16, step < nk ? off : 0x80000000u,
                                                 (j < S::kFrags ? at[j < S::kFrags ? j : 0] : 0) + step * kFragB, 0, 0);
    };
    struct Frags { v8i f[TF + CF]; };
    auto read_one = [&](Frags &s, int slot, int f) {
        const uint8_t *sb = ring + slot * S::kSlotB;
        const int t = f < TF ? f : (TF + 1) / 2 * 2 + (f - TF);            // place among the tails
        const v4i h = *reinterpret_cast<const v4i *>(sb + f * 1024 + lane * 16);
        const v2i l = *reinterpret_cast<const v2i *>(sb + S::kFrags * 1024 + t * 512 + lane * 8);
        v8i x = __builtin_shufflevector(h, h, 0, 1, 2, 3, -1, -1, -1, -1);
        x[4] = l[0];
        x[5] = l[1];
        s.f[f] = x;
    };
    v16f acc[TF][CF];
#pragma unroll
    for (int t = 0; t < TF; t++)
#pragma unroll
        for (int c = 0; c < CF; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][c][r] = 0.f;
    int step = wave, slot = 0;                                   // the step being multiplied, its slot (free again: it is in registers)
    // One step, one MFMA per issue slot with the rest of the pipeline spread between them and the order pinned: the direct
    // loads of the step D further on into this step's slot, then, once the next step has landed, its fragments.
    auto multiply = [&](const Frags &cur, Frags &nxt) {
        constexpr int kSlots = TF * CF, kEvents = S::kLoads + 1 + S::kFrags;
        const int next_slot = slot + 1 == D ? 0 : slot + 1;
        __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8));          // lgkmcnt(0): the fragments of this step
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < kSlots; i++) {
            const int t = i / CF, c = i % CF;
            acc[t][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(cur.f[TF + c], cur.f[t], acc[t][c], 2, 2, 0, 0, 0, 0);
#pragma unroll
            for (int e = i * kEvents / kSlots; e < (i + 1) * kEvents / kSlots; e++) {
                if (e < S::kLoads) load_one(slot, step + D * kWaves, e);
                else if (e == S::kLoads) { wait_vmcnt_imm<S::kLoads * (D - 1)>(); asm volatile("" ::: "memory"); }
                else read_one(nxt, next_slot, e - S::kLoads - 1);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        step += kWaves;
        slot = next_slot;
    };
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
        for (int j = 0; j < S::kLoads; j++) load_one(d, step + d * kWaves, j);
    wait_vmcnt_imm<S::kLoads * (D - 1)>();
    asm volatile("" ::: "memory");
    Frags u0, u1;
#pragma unroll
    for (int f = 0; f < S::kFrags; f++) read_one(u0, 0, f);
    int left = (nk - wave + kWaves - 1) / kWaves;                // this wave's steps
    for (; left >= 2; left -= 2) {
        multiply(u0, u1);
        multiply(u1, u0);
    }
    if (left > 0) multiply(u0, u1);
    wait_vmcnt_imm<0>();                                         // no direct load may still be writing when the ring is reused
    float *const red = reinterpret_cast<float *>(lds);
    constexpr int kRedPitch = S::kPartBlocks * 32 * S::kPitch;   // floats per wave

    // ---- the K slices meet in LDS, kPartBlocks token blocks at a time: register r of lane (li, lg) of tile (t, c) is token
    // 32 t + li, channel 32 c + 8 (r / 4) + 4 lg + r % 4.  Then the epilogue.
#pragma unroll
    for (int part = 0; part < TF; part += S::kPartBlocks) {                         // (whole parts: kPartBlocks divides TF)
    __syncthreads();                                             // nobody reads the ring (or the part before) any more
    {
        float *mine = red + wave * kRedPitch + (lane & 31) * S::kPitch + 4 * (lane >> 5);
#pragma unroll
        for (int t = 0; t < S::kPartBlocks; t++)
#pragma unroll
            for (int c = 0; c < CF; c++)
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const v16f &v = acc[part + t < TF ? part + t : 0][c];
                    *reinterpret_cast<float4 *>(mine + 32 * t * S::kPitch + 32 * c + 8 * q) = make_float4(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]);
                }
    }
    __syncthreads();
    const int row_end = min(32 * S::kPartBlocks, M - tok0 - 32 * part);
#pragma unroll
    for (int it = 0; it < kIters; it++) {
        const int row = row0 + it * kRowsAtOnce;
        if (!works || row >= row_end) continue;
        const int tok = tok0 + 32 * part + row;
        float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < kWaves; w++)
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const float4 v = *reinterpret_cast<const float4 *>(red + w * kRedPitch + row * S::kPitch + col * 8 + 4 * i);
                sum[4 * i] += v.x; sum[4 * i + 1] += v.y; sum[4 * i + 2] += v.z; sum[4 * i + 3] += v.w;
            }
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = __fmul_rn(__fadd_rn(sum[i], sum[i]), __fmul_rn(t_half_mul[part / S::kPartBlocks][it], muls[i]));
        uint32_t p[4];
#pragma unroll
        for (int i = 0; i < 4; i++) p[i] = pack2_rounded_products<DT>(v[2 * i], v[2 * i + 1]);
        finish_eight<DT>(out, make_uint4(p[0], p[1], p[2], p[3]), epi, ahead[part / S::kPartBlocks][it], tok, ch, N, vec16);
    }
    }
}

template <int DT, bool ROPE, int TF, int CF>
__global__ void __launch_bounds__(64 * kWaves, (Tile<TF, CF>::kWgPerCu))
gemm_e2m3_split_kernel(void *__restrict__ out, const uint8_t *__restrict__ act, const uint8_t *__restrict__ wgt, int M, int N, int K,
                       int tiles_t, int tiles_c, Epilogue epi) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[Tile<TF, CF>::kLdsB];
    tile<DT, ROPE, TF, CF>(lds, out, act, wgt, M, N, K, tiles_t, tiles_c, epi);
}

template <int DT, bool ROPE, int TF, int CF>
static int launch(void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st) {
    using S = Tile<TF, CF>;
    const int tiles_t = (M + S::kTok - 1) / S::kTok, tiles_c = (N + S::kChn - 1) / S::kChn;
    const long grid = tile_grid(tiles_t, tiles_c);
    gemm_e2m3_split_kernel<DT, ROPE, TF, CF><<<dim3((unsigned)grid), dim3(64 * kWaves), 0, st>>>(out, a, b, M, N, K, tiles_t, tiles_c, epi);
    return launch_status();
}

}  // namespace e2m3s

#define QUEST_SPLIT_SHAPES QUEST_SPLIT(1, 1) QUEST_SPLIT(1, 2) QUEST_SPLIT(2, 2) QUEST_SPLIT(4, 2)

int gemm_e2m3_split_slots(int tf, int cf) {
#define QUEST_SPLIT(TF, CF) if (tf == TF && cf == CF) return e2m3s::Tile<TF, CF>::kStages;
    QUEST_SPLIT_SHAPES
#undef QUEST_SPLIT
    return 0;
}

int launch_gemm_e2m3_split(int dtype, int tf, int cf, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st) {
#define QUEST_SPLIT_DT(DT, TF, CF) (epi.kind == kEpiRope ? e2m3s::launch<DT, true, TF, CF>(out, a, b, M, K, N, epi, st) : e2m3s::launch<DT, false, TF, CF>(out, a, b, M, K, N, epi, st))
#define QUEST_SPLIT(TF, CF) \
    if (tf == TF && cf == CF) return dtype == QUEST_DTYPE_BF16 ? QUEST_SPLIT_DT(0, TF, CF) : QUEST_SPLIT_DT(1, TF, CF);
    QUEST_SPLIT_SHAPES
#undef QUEST_SPLIT
#undef QUEST_SPLIT_DT
    return QUEST_ERR_UNSUPPORTED;
}

}  // namespace quest

