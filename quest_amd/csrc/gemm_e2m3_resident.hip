// W4A4 GEMM on the FP6 (E2M3) matrix instructions for many tokens and rows short enough that a channel tile's weights stay in LDS for all of
// K.  Operands as E2M3 tiles and arithmetic as in gemm_e2m3.hip (every sum exact in fp32), outputs identical bit for bit.
//
// A persistent workgroup of eight waves holds 32 kC channels x K in LDS and its waves multiply one block of 32 kT tokens after the other by
// them, each at its own pace: the weights are only read, so there is no barrier until the workgroup's next channel tile, and with two
// waves per SIMD one's epilogue runs under the other's products.  Token fragments come straight from memory in the operand's register
// order, kRing steps ahead and across the end of a block into the next one; they pass through no LDS.
//
// What bounds it: the vector ALU.  A block of 64 x 128 at K = 1024 is 128 matrix instructions (4096 cycles) and an epilogue of 1100 (plain)
// to 1700 (rotary) vector instructions (4400 to 6800), on a SIMD that has two such blocks at a time; the 256 x 256 tiles of gemm_e2m3.hip run the
// two one after the other.  Hence the doubled products (one addition per output less), four channels' scales unpacked once for both
// row blocks, and stores of 64 bytes per row (32 rows x 32 bytes at a power-of-two pitch meet in one L2 channel: rotary 55.2, now 50.3 us).
// Against the 256 x 256 kernel and the INT8 one, us, weights rotating through copies of 400 MB, K = 1024: (16384, 3072) rotary 50 / 62 / 68,
// (16384, 1024) residual 21 / 25 / 27, (16384, 5632) gated 73 / 105 / 103 (71 / 110 / 105 with the weights at hand), (3000, 2048) 9.8 / 13.8 / 15.0; (9000, 1536, 4096) 36 / 48 / 58.
// Stores past the caches (nt) take twice to three times as long, write-through ones a fifth longer.
#include "e2m3_epilogue.h"

namespace quest {
namespace e2m3r {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));
typedef int v6i __attribute__((ext_vector_type(6)));          // an FP6 operand's registers (the builtin asks for eight)
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kWaves = 8;
constexpr int kFragB = 1536;
constexpr int kT = 2, kC = 4;                               // a wave's block: row blocks of 32 tokens, of 32 channels
constexpr int kRows = 32 * kT, kChannels = 32 * kC;
constexpr int kRing = 4;                                   // 64-k steps of token fragments in flight or in use: two stages of two
constexpr int kTwo = 0x80808080, kOne = 0x7f7f7f7f;      // block scales of the products: sums come out doubled, exactly

__device__ __forceinline__ v8i eight(const v6i &x) { return __builtin_shufflevector(x, x, 0, 1, 2, 3, 4, 5, -1, -1); }

// LDS: the channel tile by 64-k steps, each the heads of its fragments, then their tails; then the channels' scales
constexpr int kStepB = kC * kFragB;
constexpr int kLoads = kC + kC / 2;                        // direct loads of a KiB per step
constexpr int kScalesAt = kResidentMaxK / 64 * kStepB;
constexpr int kLdsB = kScalesAt + kChannels * 2;
static_assert(kLdsB <= 160 * 1024, "the longest rows fit");

struct Plan {
    int groups_t, tiles_c;                                 // blocks of 32 kT tokens, tiles of 32 kC channels
    int ways_t;                                            // how many ways the eight XCDs divide the tokens; 8 / ways_t: the channels
    int per_tile;                                          // workgroups of an XCD per channel tile; 0: they divide its tiles into even runs
};

// A wave's walk over its workgroup's run of (channel tile, token group) items, the token groups of a tile dealt to the waves in turn.
struct Walk {
    int ct, g, g_end, left;                                // left: items behind this tile's
};
__device__ __forceinline__ void walk_on(Walk &w, int first, int groups) {         // to the next tile that has a group for this wave
    while (w.g >= w.g_end && w.left > 0) {
        const int n = min(w.left, groups);
        w.ct++;
        w.g = first;
        w.g_end = n;
        w.left -= n;
    }
}

template <int DT, int EPI>
__global__ void __launch_bounds__(64 * kWaves, 2)
gemm_e2m3_resident_kernel(void *__restrict__ out, const uint8_t *__restrict__ act, const uint8_t *__restrict__ wgt, int M, int N, int K, Plan plan,
                          Epilogue epi) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[kLdsB];
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int lane = (int)threadIdx.x & 63, li = lane & 31, lg = lane >> 5;
    const int nk = K / 64, pitch = nk * kFragB;                       // steps, bytes per row block

    // this XCD's part of the output, this workgroup's run of it
    const int xcd = (int)blockIdx.x & 7, rank = (int)blockIdx.x >> 3, per = (int)gridDim.x >> 3;
    const int ways_c = 8 / plan.ways_t, xt = xcd % plan.ways_t, xc = xcd / plan.ways_t;
    const int g_lo = __builtin_amdgcn_readfirstlane(plan.groups_t * xt / plan.ways_t);
    const int groups = __builtin_amdgcn_readfirstlane(plan.groups_t * (xt + 1) / plan.ways_t) - g_lo;
    const int c_lo = __builtin_amdgcn_readfirstlane(plan.tiles_c * xc / ways_c);
    const int tiles = __builtin_amdgcn_readfirstlane(plan.tiles_c * (xc + 1) / ways_c) - c_lo;
    int i0, i1;
    if (plan.per_tile > 0) {
        const int tile = __builtin_amdgcn_readfirstlane(rank / plan.per_tile), part = rank - tile * plan.per_tile;
        if (tile >= tiles) return;                                    // uniform: the whole workgroup
        i0 = tile * groups + __builtin_amdgcn_readfirstlane(groups * part / plan.per_tile);
        i1 = tile * groups + __builtin_amdgcn_readfirstlane(groups * (part + 1) / plan.per_tile);
    } else {
        i0 = __builtin_amdgcn_readfirstlane((int)((long)groups * tiles * rank / per));
        i1 = __builtin_amdgcn_readfirstlane((int)((long)groups * tiles * (rank + 1) / per));
    }
    if (i0 >= i1) return;                                             // uniform: the whole workgroup
    const int ct0 = __builtin_amdgcn_readfirstlane(i0 / groups);
    Walk seg = {c_lo + ct0, i0 - ct0 * groups, 0, 0};
    seg.g_end = min(seg.g + (i1 - i0), groups);
    seg.left = (i1 - i0) - (seg.g_end - seg.g);
    Walk mine = seg;                                                  // this wave's next block
    mine.g += wave;
    walk_on(mine, wave, groups);

    const int rbs_t = (M + 31) / 32, rbs_c = (N + 31) / 32;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)act, 0, rbs_t * pitch, 0x00020000);
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)wgt, 0, rbs_c * pitch, 0x00020000);
    // where the token fragments of a group start (row blocks past the last are read as the last one: their products are not stored)
    auto token_at = [&](const Walk &w, int t) { return min((g_lo + w.g) * kT + t, rbs_t - 1) * pitch; };
    v6i a[kRing][kT];
    auto load_token = [&](int slot, int t, int at) {
        const v4i h = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(xr, lane * 16, at, 0));
        const v2i l = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(xr, lane * 8 + 1024, at, 0));
        a[slot][t] = v6i{h[0], h[1], h[2], h[3], l[0], l[1]};
    };
#pragma unroll
    for (int s = 0; s < kRing; s++)
#pragma unroll
        for (int t = 0; t < kT; t++) load_token(s, t, token_at(mine, t) + s * kFragB);
    v6i b[kC];
    auto read_weight = [&](int step, int c) {
        const uint8_t *sb = lds + step * kStepB;
        const v4i h = *reinterpret_cast<const v4i *>(sb + c * 1024 + lane * 16);
        const v2i l = *reinterpret_cast<const v2i *>(sb + kC * 1024 + c * 512 + lane * 8);
        b[c] = v6i{h[0], h[1], h[2], h[3], l[0], l[1]};
    };
    v16f acc[kT][kC];
    int at[kT], at_next[kT];                                          // of the block being multiplied and of the wave's next one
    // two steps: slots 2 half, 2 half + 1 of the ring, refilled for the stage after the next as they are used up
    auto stage = [&](auto first_tag, int half, int step) {
        const bool over = step + kRing >= nk;
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int slot = 2 * half + u, next = step + u + 1 == nk ? 0 : step + u + 1;
#pragma unroll
            for (int c = 0; c < kC; c++) {
#pragma unroll
                for (int t = 0; t < kT; t++) {
                    acc[t][c] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(eight(b[c]), eight(a[slot][t]), decltype(first_tag)::value && u == 0 ? v16f{} : acc[t][c],
                                                                                2, 2, 0, kTwo, 0, kOne);
                    if (c == kC - 1) load_token(slot, t, (over ? at_next[t] : at[t]) + (step + u + kRing - (over ? nk : 0)) * kFragB);
                }
                read_weight(next, c);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };
    for (bool first = true;; first = false) {
        const int ch0 = seg.ct * 32 * kC;
        // ---- the tile's weights: channel blocks past the matrix arrive as zeros
        if (!first) plain_barrier();                                  // nobody reads the tile before any more
        for (int i = wave; i < nk * kLoads; i += kWaves) {
            const int step = i / kLoads, j = i - step * kLoads;
            const int rb = seg.ct * kC + (j < kC ? j : 2 * (j - kC) + lg);
            const uint32_t off = rb < rbs_c ? (uint32_t)rb * (uint32_t)pitch + step * kFragB + (j < kC ? lane * 16 : 1024 + li * 16) : 0x80000000u;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void *)(lds + step * kStepB + j * 1024), 16, off, 0, 0, 0);
        }
        uint16_t *const c_mul = reinterpret_cast<uint16_t *>(lds + kScalesAt);
        if ((int)threadIdx.x < 32 * kC) c_mul[threadIdx.x] = epi.b_mul[min(ch0 + (int)threadIdx.x, N - 1)];
        __builtin_amdgcn_s_waitcnt(0);
        plain_barrier();
        while (mine.ct == seg.ct && mine.g < mine.g_end) {
            const int tok0 = (g_lo + mine.g) * 32 * kT;
#pragma unroll
            for (int t = 0; t < kT; t++) at[t] = token_at(mine, t);
            mine.g += kWaves;
            walk_on(mine, wave, groups);
#pragma unroll
            for (int t = 0; t < kT; t++) at_next[t] = mine.g < mine.g_end ? token_at(mine, t) : at[t];
#pragma unroll
            for (int c = 0; c < kC; c++) read_weight(0, c);
            uint16_t t_mul[kT];
#pragma unroll
            for (int t = 0; t < kT; t++) t_mul[t] = epi.a_mul[min(tok0 + 32 * t + li, M - 1)];
            stage(std::true_type{}, 0, 0);
            stage(std::false_type{}, 1, 2);
            int step = kRing;
            for (; step + kRing <= nk; step += kRing) {
                stage(std::false_type{}, 0, step);
                stage(std::false_type{}, 1, step + 2);
            }
            if (step < nk) {                                          // an odd number of stages: the halves trade places
                stage(std::false_type{}, 0, step);
#pragma unroll
                for (int s = 0; s < 2; s++)
#pragma unroll
                    for (int t = 0; t < kT; t++) {
                        const v6i x = a[s][t];
                        a[s][t] = a[2 + s][t];
                        a[2 + s][t] = x;
                    }
            }

            // ---- epilogue: register r of lane (li, lg) of block (t, c) is token 32 t + li, channel 32 c + 8 (r / 4) + 4 lg + r % 4;
            // the half-waves trade register groups, so that a lane holds eight consecutive channels
            const int lg = fresh_lane_id() >> 5, li = fresh_lane_id() & 31;
            constexpr int kPieces = kT * kC, kAhead = EPI == kEpiRope ? 1 : 2;      // block piece = c kT + t
            RopeLane rl = {0, 0};
            if constexpr (EPI == kEpiRope) rl = rope_lane(epi.rope, tok0 + li, ch0);
            // (the block's rows as a buffer of their own: rows past M lie past it and are not written)
            const uint32_t row_b = (EPI == kEpiGlu ? N >> 1 : N) * 2;
            const __amdgpu_buffer_rsrc_t rows = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<uint8_t *>(out) + (size_t)tok0 * row_b, 0, min(32 * kT, M - tok0) * row_b, 0x00020000);
            // Stores write 64 bytes of a row: four lanes, one in each quarter of the wave, hold the row's 32 channels (GLU: of two blocks,
            // a unit being 32 outputs).  Store `half`: rows 16 half ... of the block.  Channels past N: past the buffer too.
            constexpr int kUnitCh = EPI == kEpiGlu ? 64 : 32;
            const int lq = li & 15, lr = li >> 4;
            const int unit_ch = lr * (kUnitCh / 2) + lg * (kUnitCh / 4);                   // of the lane's eight values, in a unit
            const uint32_t at_lane = lq * row_b + (ch0 + unit_ch) * (EPI == kEpiGlu ? 1 : 2);
            auto place = [&](int t, int unit, int half) {
                return ch0 + kUnitCh * unit + unit_ch < N ? at_lane + (32 * t + 16 * half) * row_b + 64 * unit : 0x80000000u;
            };
            auto quarters = [&](uint4 (&o)[2]) {                      // two values of row li -> rows lq and 16 + lq of the four lanes' unit
                uint32_t x[2][4] = {{o[0].x, o[0].y, o[0].z, o[0].w}, {o[1].x, o[1].y, o[1].z, o[1].w}};
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const auto s = __builtin_amdgcn_permlane16_swap(x[0][i], x[1][i], false, false);
                    x[0][i] = s[0];
                    x[1][i] = s[1];
                }
                o[0] = make_uint4(x[0][0], x[0][1], x[0][2], x[0][3]);
                o[1] = make_uint4(x[1][0], x[1][1], x[1][2], x[1][3]);
            };
            uint4 gated[kT];                                          // GLU: the even block's outputs
            // what a piece's two halves add or turn by, fetched kAhead pieces before
            float4 cs[EPI == kEpiRope ? kAhead : 1][2][2];
            uint4 other[EPI == kEpiAdd || EPI == kEpiBias ? kAhead : 1][2];
            auto fetch = [&](int piece) {
                const int c = piece / kT, t = piece % kT;
#pragma unroll
                for (int pr = 0; pr < 2; pr++) {
                    const int ch = ch0 + 32 * c + (EPI == kEpiRope ? 16 * pr + 8 * lg : unit_ch);
                    if constexpr (EPI == kEpiRope) {
                        if (ch < epi.rope.rot_cols) rope_fetch(epi.rope, rl, lg, c, t, pr, cs[piece % kAhead][pr]);
                    }
                    if constexpr (EPI == kEpiAdd || EPI == kEpiBias) {
                        if constexpr (EPI == kEpiAdd) other[piece % kAhead][pr] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rows, place(t, c, pr), 0, 0));
                        else if (ch < N) other[piece % kAhead][pr] = *reinterpret_cast<const uint4 *>(epi.rope.bias + ch);
                    }
                }
            };
            if constexpr (EPI != kEpiPlain && EPI != kEpiGlu) {
#pragma unroll
                for (int i = 0; i < kAhead; i++) fetch(i);
            }
            float t_half_mul[kT];
#pragma unroll
            for (int t = 0; t < kT; t++) t_half_mul[t] = __fmul_rn(0.5f, to_f32<DT>(t_mul[t]));
#pragma unroll
            for (int c = 0; c < kC; c++) {
                float muls[16];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint2 m4 = *reinterpret_cast<const uint2 *>(c_mul + 32 * c + 8 * q + 4 * lg);
                    muls[4 * q] = lo_f32<DT>(m4.x); muls[4 * q + 1] = hi_f32<DT>(m4.x);
                    muls[4 * q + 2] = lo_f32<DT>(m4.y); muls[4 * q + 3] = hi_f32<DT>(m4.y);
                }
#pragma unroll
                for (int t = 0; t < kT; t++) {
                    uint32_t x[4][2];
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) {
                            const float s = acc[t][c][4 * q + e];
                            v[e] = __fmul_rn(s, __fmul_rn(t_half_mul[t], muls[4 * q + e]));
                        }
                        x[q][0] = pack2_rounded_products<DT>(v[0], v[1]);
                        x[q][1] = pack2_rounded_products<DT>(v[2], v[3]);
                    }
                    constexpr bool kFetches = EPI != kEpiPlain && EPI != kEpiGlu;
                    uint4 o[2];
#pragma unroll
                    for (int pr = 0; pr < 2; pr++) {
                        const auto s0 = __builtin_amdgcn_permlane32_swap(x[2 * pr][0], x[2 * pr + 1][0], false, false);
                        const auto s1 = __builtin_amdgcn_permlane32_swap(x[2 * pr][1], x[2 * pr + 1][1], false, false);
                        const int slot = (c * kT + t) % kAhead;
                        o[pr] = make_uint4(s0[0], s1[0], s0[1], s1[1]);
                        if constexpr (EPI == kEpiRope) {
                            if (ch0 + 32 * c + 16 * pr + 8 * lg < epi.rope.rot_cols) o[pr] = rope_turn<DT>(o[pr], cs[slot][pr]);
                        }
                    }
                    if constexpr (EPI == kEpiGlu) {                   // four gates, then the four ups of the same outputs
                        const auto s0 = __builtin_amdgcn_permlane32_swap(silu_mul_pair<DT>(o[0].x, o[0].z), silu_mul_pair<DT>(o[1].x, o[1].z), false, false);
                        const auto s1 = __builtin_amdgcn_permlane32_swap(silu_mul_pair<DT>(o[0].y, o[0].w), silu_mul_pair<DT>(o[1].y, o[1].w), false, false);
                        const uint4 eight_out = make_uint4(s0[0], s1[0], s0[1], s1[1]);
                        if (c % 2 == 0) {
                            gated[t] = eight_out;
                            continue;
                        }
                        o[0] = gated[t];
                        o[1] = eight_out;
                    }
                    quarters(o);
                    if constexpr (EPI == kEpiAdd || EPI == kEpiBias) {
#pragma unroll
                        for (int pr = 0; pr < 2; pr++) o[pr] = add_eight<DT>(o[pr], other[(c * kT + t) % kAhead][pr]);
                    }
                    // the next fetch before this piece's stores: memory operations complete in order, so that whoever waits for it
                    // does not wait for them
                    if constexpr (kFetches) {
                        __builtin_amdgcn_sched_barrier(0);
                        if (c * kT + t + kAhead < kPieces) fetch(c * kT + t + kAhead);
                        __builtin_amdgcn_sched_barrier(0);
                    }
#pragma unroll
                    for (int half = 0; half < 2; half++)
                        __builtin_amdgcn_raw_buffer_store_b128(v4u{o[half].x, o[half].y, o[half].z, o[half].w}, rows, place(t, EPI == kEpiGlu ? c / 2 : c, half), 0, 0);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
        if (seg.left <= 0) break;
        const int n = min(seg.left, groups);
        seg.ct++;
        seg.g = 0;
        seg.g_end = n;
        seg.left -= n;
    }
}

// Of the ways to divide the output among the XCDs and their workgroups the one with the least estimated time, in us: 2.5 for the launch, for
// every four blocks of a workgroup (one per SIMD) 3.2 of epilogue and 1.9 per 1024 k of products, 3 for every channel tile that it loads, 0.1 per
// MB that the XCDs fetch.  Whole tiles per workgroup, or, where every XCD has an eighth of the tokens, even runs over its tiles (its L2 then
// holds its tokens; a quarter of them and half the channels is no faster on the whole: (16384, 1024, 5632) gated 70 us against 73, (16384, 1024, 3072)
// rotary 53 / 52, (16384, 1024, 1024) residual 23 / 21).  The estimate orders the
// eight plans of thirteen sizes as measured but for differences of 5 %; for one to three rounds it is within 15 % of the time itself.
static Plan make_plan(int M, int K, int N, int cus, float *us_out) {
    const int groups_t = (M + kRows - 1) / kRows, tiles_c = (N + kChannels - 1) / kChannels, per = cus / 8;
    const float four = 3.2f + 0.0019f * (float)K;
    Plan best = {groups_t, tiles_c, 8, 0};
    float best_us = 0.f;
    for (int ways = 8; ways >= 1; ways /= 2) {
        const int groups = (groups_t + ways - 1) / ways, tiles = (tiles_c * ways + 7) / 8, q = per / tiles;
        const float fetch = 2.5f + 0.1f * 0.75e-6f * (float)K * (8.f * (float)M / (float)ways + (float)N * (float)ways);
        auto consider = [&](float us, int per_tile) {
            if (best_us == 0.f || us < best_us) best = Plan{groups_t, tiles_c, ways, per_tile}, best_us = us;
        };
        if (ways == 8) {
            const float items = (float)groups * (float)tiles / (float)per, loads = 1.f + items / (float)groups;
            consider(fetch + four * (0.25f * items + 0.375f * loads) + 3.f * loads, 0);
        }
        if (q > 0) consider(fetch + four * (float)(((groups + q - 1) / q + 3) / 4) + 3.f, q);
    }
    if (us_out) *us_out = best_us;
    return best;
}

template <int DT, int EPI>
static int launch(void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, int cus, const Epilogue &epi, hipStream_t st) {
    const Plan plan = make_plan(M, K, N, cus, nullptr);
    gemm_e2m3_resident_kernel<DT, EPI><<<dim3((unsigned)(cus / 8 * 8)), dim3(64 * kWaves), 0, st>>>(out, a, b, M, N, K, plan, epi);
    return launch_status();
}

template <int DT>
static int launch_epi(void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, int cus, const Epilogue &epi, hipStream_t st) {
    switch (epi.kind) {
        case kEpiGlu: return launch<DT, kEpiGlu>(out, a, b, M, K, N, cus, epi, st);
        case kEpiAdd: return launch<DT, kEpiAdd>(out, a, b, M, K, N, cus, epi, st);
        case kEpiRope: return launch<DT, kEpiRope>(out, a, b, M, K, N, cus, epi, st);
        case kEpiBias: return launch<DT, kEpiBias>(out, a, b, M, K, N, cus, epi, st);
        default: return launch<DT, kEpiPlain>(out, a, b, M, K, N, cus, epi, st);
    }
}

}  // namespace e2m3r

float gemm_e2m3_resident_plan(int M, int K, int N, int cus, int *plan) {
    float us;
    const e2m3r::Plan p = e2m3r::make_plan(M, K, N, cus, &us);
    const int v[8] = {cus / 8 * 8, 8, p.per_tile, p.ways_t, e2m3r::kRows, e2m3r::kChannels, 1, K};
    for (int i = 0; plan != nullptr && i < 8; i++) plan[i] = v[i];
    return us;
}

int launch_gemm_e2m3_resident(int dtype, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, int cus, const Epilogue &epi,
                              hipStream_t st) {
    return dtype == QUEST_DTYPE_BF16 ? e2m3r::launch_epi<0>(out, a, b, M, K, N, cus, epi, st) : e2m3r::launch_epi<1>(out, a, b, M, K, N, cus, epi, st);
}

}  // namespace quest
