// W4A4 GEMM on the FP6 (E2M3) matrix instructions for the sizes whose 256 x 256 tiles are too few to fill the chip: some tens to
// a few thousand tokens.  Operands as E2M3 tiles and arithmetic as in gemm_e2m3.hip (every sum exact in fp32), outputs identical
// bit for bit.
//
// A workgroup of four waves owns 32 TF tokens x 32 CF channels, the waves WT x WC parts of it.  A pipeline stage is 128 k: three
// direct loads of 1 KiB per row block (the heads of its two fragments, then both tails), laid out in LDS as they come, so that a
// fragment is one ds_read_b128 and one ds_read_b64 at lane-linear addresses.  While one 64-k step is multiplied from registers the
// next one's fragments are read; one barrier per stage, in the second step, tells that the next stage has landed everywhere and
// that this stage's slot is free for the loads of the stage kStages further on.  A tile's scale values are fetched at its start, as buffer
// loads whose range check stands for the matrix' edges: with a branch per value the first stage's loads set out 0.3 to 0.8 us later ((1000,
// 512, 3072) 7.7 -> 7.0 us, (1200, 896, 2304) 8.6 -> 7.8, (333, 1024, 11000) 11.7 -> 10.8, (1000, 2560, 7680) 21.6 -> 20.3).
// What bounds it: the LDS port, which a stage's bytes cross once on their way in and twice on their way to the waves that share them
// (72 KiB per stage of a 128 x 128 tile: 576 cycles at 128 bytes a cycle, 600 measured, against 256 of matrix work), and with one
// tile per CU the trip to memory before the first stage and the epilogue after the last, together 5 us.
// 128 x 96 tiles (KS = 2) share K between the waves of a pair: each multiplies 64 x 96 of one of a stage's two 64-k steps, so that 51 KiB instead
// of 69 cross the port per stage (waves of 32 x 96 would read 48 KiB, as for 128 x 128), and at the end they trade a token block of sums each
// (96 KiB through LDS).  They fill 216 of 256 CUs where 128 x 128 has 160 tiles: (1000, 6912, 2560) 22.7 -> 20.5 us, (516, 1152, 3695)
// 15.9 -> 14.1, (197, 9600, 8324) 37.6 -> 34.2.  128 x 128 by pairs is 1 to 4 % slower than 2 x 2 waves: a stage's fragments are all read behind
// its one barrier.
// Token fragments straight into registers (no two waves of the pairs need the same ones: 27 KiB a stage through the port) with the channels'
// read a stage ahead are no faster (0.97 to 1.03 x over 12 sizes): what is left of a stage is its bytes into the CU.
// Measured against the kernels that took these sizes before (weights rotating through four copies): (200, 4096, 11008) 15.5 against
// 19.9 us, (1000, 6912, 2560) 22.2 against 27.6, (1400, 2560, 2560) 12.9 against 26.9, (1400, 6912, 2560) 24.2 against 54.3.
#include "e2m3_epilogue.h"

namespace quest {
namespace e2m3m {

typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kWaves = 4;
constexpr int kFragB = 1536;

template <int TF_, int CF_, int WT_, int WC_, int KS_ = 1>
struct Tile {
    static constexpr int TF = TF_, CF = CF_, WT = WT_, WC = WC_, KS = KS_;
    static_assert(WT * WC * KS == kWaves && TF % WT == 0 && CF % WC == 0, "whole fragments per wave");
    static constexpr int kT = TF / WT, kC = CF / WC;                   // fragments per wave
    static constexpr int kDone = kT / KS;                              // token blocks that a wave finishes
    static_assert(KS == 1 || (KS == 2 && kT == 2), "a pair's waves finish one token block each");
    static constexpr int kTok = 32 * TF, kChn = 32 * CF;
    static constexpr int kSlotB = 3072 * (TF + CF);
    static constexpr int kLoads = (3 * (TF + CF) + kWaves - 1) / kWaves;       // direct loads per wave and stage
    static constexpr bool kTwo = 24 * kT * kC + 12 * (kT + kC) + 8 * kC + kT + 50 <= 256 && 4 * kSlotB <= 80 * 1024;
    static constexpr int kWgPerCu = kTwo ? 2 : 1;
    static constexpr int kFit = ((160 / kWgPerCu) * 1024 - 1024) / kSlotB;
    static constexpr int kStages = kFit < 8 ? kFit : 8;
    static_assert(kStages >= 3 && kLoads * (kStages - 2) < 64, "stages in flight");
    static_assert(KS == 1 || kWaves * kC * 4096 <= kStages * kSlotB, "the partial sums that pairs trade");
    // (loads past the tile's last touch no memory but do write zeros: into a KiB of their own)
    static constexpr bool kSpare = 3 * (TF + CF) % kWaves != 0;
    static constexpr int kLdsB = kStages * kSlotB + (kSpare ? 1024 : 0);
};

template <int DT, bool ROPE, typename S>
__device__ __forceinline__ void tile(uint8_t *lds, void *__restrict__ out, const uint8_t *__restrict__ act, const uint8_t *__restrict__ wgt,
                                     int M, int N, int K, int tok0, int ch0, const Epilogue &epi) {
    constexpr int TF = S::TF, CF = S::CF, kT = S::kT, kC = S::kC, D = S::kStages, kDone = S::kDone;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63, li = lane & 31, lg = lane >> 5;
    const int part = wave / S::KS, half = wave % S::KS;                  // (half: which 64-k step of every stage, if each wave has one)
    const int tf0 = (part / S::WC) * kT, cf0 = (part % S::WC) * kC;      // the wave's fragments of the tile
    const int done0 = tf0 + half * kDone;                                // the token blocks that it finishes

    // the epilogue's scale values set out first: a lane finishes token li of each of its token blocks and, of each channel unit,
    // channels 8 q + 4 lg ... + 3 (values past the vectors' ends read as zeros: their outputs are not stored)
    const __amdgpu_buffer_rsrc_t ar = __builtin_amdgcn_make_buffer_rsrc((void *)epi.a_mul, 0, M * 2, 0x00020000);
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void *)epi.b_mul, 0, (N * 2 + 2) & ~3, 0x00020000);
    uint16_t t_mul[kDone];
    v2i c_mul[kC][4];
#pragma unroll
    for (int t = 0; t < kDone; t++) t_mul[t] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(ar, (tok0 + 32 * (done0 + t) + li) * 2, 0, 0);
#pragma unroll
    for (int c = 0; c < kC; c++)
#pragma unroll
        for (int q = 0; q < 4; q++) c_mul[c][q] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(br, (ch0 + 32 * (cf0 + c) + 8 * q + 4 * lg) * 2, 0, 0));
    // ... and what the epilogue adds or rotates by
    const bool vec16 = (N & 7) == 0;
    Ahead<ROPE> ahead[kDone][kC][2];
    if (ROPE || epi.kind == kEpiAdd || epi.kind == kEpiBias) {                      // uniform
#pragma unroll
        for (int t = 0; t < kDone; t++)
#pragma unroll
            for (int c = 0; c < kC; c++)
#pragma unroll
                for (int pr = 0; pr < 2; pr++)
                    fetch_ahead<DT>(ahead[t][c][pr], out, epi, tok0 + 32 * (done0 + t) + li, ch0 + 32 * (cf0 + c) + (2 * pr + lg) * 8, M, N, vec16);
    }

    const int nk = K / 128;                                      // stages
    const int pitch = (K / 64) * kFragB;                         // bytes per row block
    const int rbs_t = (M + 31) / 32, rbs_c = (N + 31) / 32;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)act, 0, rbs_t * pitch, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)wgt, 0, rbs_c * pitch, 0x00020000);
    // The wave's loads of a stage are numbers 4 j + wave of the tile's 3 (TF + CF), three per row block.  Row blocks past the end
    // of a matrix are read as its last one (their products are not stored); numbers past the tile's last touch no memory.
    uint32_t off[S::kLoads];
    bool from_x[S::kLoads];
#pragma unroll
    for (int j = 0; j < S::kLoads; j++) {
        const int l = kWaves * j + wave, rb = l / 3, kind = l - 3 * rb;
        const int at = rb < TF ? min(tok0 / 32 + rb, rbs_t - 1) : min(ch0 / 32 + rb - TF, rbs_c - 1);
        from_x[j] = rb < TF;
        off[j] = rb >= TF + CF ? 0x80000000u
                 : (uint32_t)at * (uint32_t)pitch + (kind < 2 ? kind * kFragB + lane * 16 : 1024 + (lane >> 5) * kFragB + (lane & 31) * 16);
    }
    auto load_one = [&](int slot, int stage, int j) {            // stages past the end touch no memory
        uint8_t *dst = lds + slot * S::kSlotB + (kWaves * j + wave) * 1024;
        if (kWaves * j + kWaves - 1 >= 3 * (TF + CF) && kWaves * j + wave >= 3 * (TF + CF)) dst = lds + D * S::kSlotB;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(from_x[j] ? xr : wr, (__attribute__((address_space(3))) void *)dst, 16,
                                                 stage < nk ? off[j] : 0x80000000u, stage * 2 * kFragB, 0, 0);
    };
    struct Frags { v8i t[kT], c[kC]; };
    auto read_one = [&](Frags &s, int slot, int sub, int f) {    // f: token fragments, then channel fragments
        const int rb = f < kT ? tf0 + f : TF + cf0 + f - kT;
        const uint8_t *sb = lds + slot * S::kSlotB + rb * 3072;
        const v4i h = *reinterpret_cast<const v4i *>(sb + sub * 1024 + lane * 16);
        const v2i l = *reinterpret_cast<const v2i *>(sb + 2048 + sub * 512 + lane * 8);
        v8i x = __builtin_shufflevector(h, h, 0, 1, 2, 3, -1, -1, -1, -1);
        x[4] = l[0];
        x[5] = l[1];
        if (f < kT) s.t[f] = x; else s.c[f - kT] = x;
    };
    v16f acc[kT][kC];
#pragma unroll
    for (int t = 0; t < kT; t++)
#pragma unroll
        for (int c = 0; c < kC; c++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][c][r] = 0.f;
    constexpr int kMfmas = kT * kC;
    auto mfma = [&](const Frags &s, int i) {
        const int t = i / kC, c = i % kC;
        acc[t][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(s.c[c], s.t[t], acc[t][c], 2, 2, 0, 0, 0, 0);
    };
    Frags u0, u1;
    // one stage, the MFMAs one by one with the rest of the pipeline between them, the order pinned
    constexpr int kReads = kT + kC;
    auto first_step = [&](int slot) {
#pragma unroll
        for (int i = 0; i < kMfmas; i++) {                       // first step; the second one's fragments
            mfma(u0, i);
#pragma unroll
            for (int e = i * kReads / kMfmas; e < (i + 1) * kReads / kMfmas; e++) read_one(u1, slot, 1, e);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto last_step = [&](const Frags &now, Frags &then, int stage, int slot) {      // the only step of a wave that has one per stage
        const int next_slot = slot + 1 == D ? 0 : slot + 1;
        constexpr int kEvents = S::kLoads + kReads;
#pragma unroll
        for (int i = 0; i < kMfmas; i++) {
            mfma(now, i);                                        // (waits for its fragments: the slot has been read)
            if (i == 0) {
                __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8));      // lgkmcnt(0): all of them
                wait_vmcnt_imm<S::kLoads * (D - 2)>();           // this wave's loads of the next stage have landed ...
                plain_barrier();                                 // ... and everyone else's; the slot is free
            }
            // the next stage's first fragments, then the loads into the slot
#pragma unroll
            for (int e = i * kEvents / kMfmas; e < (i + 1) * kEvents / kMfmas; e++) {
                if (e < kReads) read_one(then, next_slot, half, e); else load_one(slot, stage + D, e - kReads);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    };
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
        for (int j = 0; j < S::kLoads; j++) load_one(d, d, j);
    wait_vmcnt_imm<S::kLoads * (D - 1)>();
    plain_barrier();
#pragma unroll
    for (int f = 0; f < kT + kC; f++) read_one(u0, 0, half, f);
    int slot = 0;
    auto on = [](int x) { return x + 1 == D ? 0 : x + 1; };
    if constexpr (S::KS == 1) {
        for (int stage = 0; stage < nk; stage++, slot = on(slot)) {
            first_step(slot);
            last_step(u1, u0, stage, slot);
        }
    } else {
        int stage = 0;
        for (; stage + 2 <= nk; stage += 2) {
            last_step(u0, u1, stage, slot);
            slot = on(slot);
            last_step(u1, u0, stage + 1, slot);
            slot = on(slot);
        }
        if (stage < nk) last_step(u0, u1, stage, slot);
    }
    wait_vmcnt_imm<0>();                                         // no direct load may outlive the workgroup's LDS allocation

    // ---- a pair's waves trade the token blocks that they do not finish, a KiB of four registers at a time
    if constexpr (S::KS == 2) {
        __builtin_amdgcn_s_waitcnt(0);
        plain_barrier();                                         // nobody reads or loads a slot any more
        if (half == 1) {
#pragma unroll
            for (int c = 0; c < kC; c++) {
                const v16f x = acc[0][c];
                acc[0][c] = acc[1][c];
                acc[1][c] = x;
            }
        }
        v4f *const give = reinterpret_cast<v4f *>(lds) + wave * (kC * 256) + lane;
        const v4f *const take = reinterpret_cast<const v4f *>(lds) + (wave ^ 1) * (kC * 256) + lane;
#pragma unroll
        for (int c = 0; c < kC; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) give[(4 * c + q) * 64] = v4f{acc[1][c][4 * q], acc[1][c][4 * q + 1], acc[1][c][4 * q + 2], acc[1][c][4 * q + 3]};
        __builtin_amdgcn_s_waitcnt(0);
        plain_barrier();
#pragma unroll
        for (int c = 0; c < kC; c++)
#pragma unroll
            for (int q = 0; q < 4; q++) {
                const v4f x = take[(4 * c + q) * 64];
#pragma unroll
                for (int e = 0; e < 4; e++) acc[0][c][4 * q + e] += x[e];
            }
    }

    // ---- epilogue: register r of lane (li, lg) of block (t, c) is token 32 t + li, channel 32 c + 8 (r / 4) + 4 lg + r % 4; the
    // half-waves trade register groups, so that a lane holds eight consecutive channels
#pragma unroll
    for (int t = 0; t < kDone; t++) {
        const int tok = tok0 + 32 * (done0 + t) + li;
        const float t_half_mul = __fmul_rn(0.5f, to_f32<DT>(t_mul[t]));
#pragma unroll
        for (int c = 0; c < kC; c++) {
            const int cu = ch0 + 32 * (cf0 + c);
            uint32_t x[4][2];
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const float s = acc[t][c][4 * q + e];
                    const uint32_t m2 = (uint32_t)c_mul[c][q][e >> 1];
                    v[e] = __fmul_rn(__fadd_rn(s, s), __fmul_rn(t_half_mul, e & 1 ? hi_f32<DT>(m2) : lo_f32<DT>(m2)));
                }
                x[q][0] = pack2_rounded_products<DT>(v[0], v[1]);
                x[q][1] = pack2_rounded_products<DT>(v[2], v[3]);
            }
#pragma unroll
            for (int pr = 0; pr < 2; pr++) {
                const auto s0 = __builtin_amdgcn_permlane32_swap(x[2 * pr][0], x[2 * pr + 1][0], false, false);
                const auto s1 = __builtin_amdgcn_permlane32_swap(x[2 * pr][1], x[2 * pr + 1][1], false, false);
                const int ch = cu + (2 * pr + lg) * 8;
                if (tok >= M || ch >= N) continue;
                finish_eight<DT>(out, make_uint4(s0[0], s1[0], s0[1], s1[1]), epi, ahead[t][c][pr], tok, ch, N, vec16);
            }
        }
    }
}

template <int DT, bool ROPE, typename S>
__global__ void __launch_bounds__(64 * kWaves, (S::kWgPerCu))
gemm_e2m3_mid_kernel(void *__restrict__ out, const uint8_t *__restrict__ act, const uint8_t *__restrict__ wgt, int M, int N, int K,
                     int tiles_t, int tiles_c, Epilogue epi) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S::kLdsB];
    int tt, ct;
    if (!tile_of(tiles_t, tiles_c, tt, ct)) return;              // uniform: the whole workgroup
    tile<DT, ROPE, S>(lds, out, act, wgt, M, N, K, tt * S::kTok, ct * S::kChn, epi);
}

template <int DT, bool ROPE, typename S>
static int launch(void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st) {
    const int tiles_t = (M + S::kTok - 1) / S::kTok, tiles_c = (N + S::kChn - 1) / S::kChn;
    const long grid = tile_grid(tiles_t, tiles_c);
    gemm_e2m3_mid_kernel<DT, ROPE, S><<<dim3((unsigned)grid), dim3(64 * kWaves), 0, st>>>(out, a, b, M, N, K, tiles_t, tiles_c, epi);
    return launch_status();
}

}  // namespace e2m3m

#define QUEST_MID_SHAPES QUEST_MID(8, 4, 2, 2, 1) QUEST_MID(4, 6, 2, 2, 1) QUEST_MID(4, 4, 2, 2, 1) QUEST_MID(4, 3, 2, 1, 2) QUEST_MID(4, 2, 2, 2, 1) \
    QUEST_MID(2, 4, 2, 2, 1) QUEST_MID(2, 2, 2, 2, 1)

int gemm_e2m3_mid_slots(int tf, int cf) {
#define QUEST_MID(TF, CF, WT, WC, KS) if (tf == TF && cf == CF) return e2m3m::Tile<TF, CF, WT, WC, KS>::kStages;
    QUEST_MID_SHAPES
#undef QUEST_MID
    return 0;
}

int launch_gemm_e2m3_mid(int dtype, int tf, int cf, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st) {
#define QUEST_MID_DT(DT, T) (epi.kind == kEpiRope ? e2m3m::launch<DT, true, T>(out, a, b, M, K, N, epi, st) : e2m3m::launch<DT, false, T>(out, a, b, M, K, N, epi, st))
#define QUEST_MID(TF, CF, WT, WC, KS)                                                                                    \
    if (tf == TF && cf == CF) {                                                                                  \
        using T = e2m3m::Tile<TF, CF, WT, WC, KS>;                                                               \
        return dtype == QUEST_DTYPE_BF16 ? QUEST_MID_DT(0, T) : QUEST_MID_DT(1, T);                              \
    }
    QUEST_MID_SHAPES
#undef QUEST_MID
#undef QUEST_MID_DT
    return QUEST_ERR_UNSUPPORTED;
}

}  // namespace quest

