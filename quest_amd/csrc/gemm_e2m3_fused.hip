// A W4A4 linear layer on some tens of tokens of short rows in one launch, on the FP6 (E2M3) matrix instructions: every workgroup quantises the 32
// token rows of its tiles itself -- the wave program of hadamard_mfma.hip, RMSNorm in front of it where asked, and so its codes and scales bit for
// bit -- into LDS, and multiplies channel tiles of 32 by them.  Sums exact and epilogues as in gemm_e2m3_split.hip: outputs identical bit for bit.
//
// Why: at these sizes an activation kernel (4 to 5 us), a GEMM (4.5 to 5) and the gap between them are one dependent chain each of launch, trip to
// memory, arithmetic and stores.  Here the first weights are on their way before the rows are looked at, and codes and scales never leave the CU.  The
// price is the quantiser's arithmetic in every workgroup, so a tile has few tokens and a workgroup several channel tiles.
//
// G waves per workgroup for rows of up to G blocks of 128 (G = 8, 16): a wave quantises 32 / G rows (at most half of them have any: sixteen rows cost what
// eight do, 32 another 1.7 us of vector ALU, 3.2 with the norm).  Then CT channel tiles at a time are multiplied by G / CT waves each, the 64-k steps dealt
// to them in turn: a wave's token fragments stay in registers, its weight fragments come straight from memory, two rounds ahead (the first round's wait in
// LDS, where the wave's sums will be: the transform needs the registers).  The partial sums meet in LDS, and a tile's first wave finishes it.
// What bounds it: the chain -- launch, rows, transform and quantiser, products, sums -- of 4.6 us (K = 1024; 5.6 with the norm in front), then 0.8 to 1.0 us
// per further round, two barriers around the epilogue.  GPU us in a graph against the two launches (which read ahead) and the INT8 ones, weights from the
// Infinity Cache: (37, 1024, 1024) 4.7 / 6.9 / 7.2, with the norm (37, 1024, 3072) 6.2 / 8.7 / 8.6 and (37, 1024, 5632) 7.2 / 9.0 / 9.3, (16, 1024,
// 22016) 8.1 / 10.2 / 9.9, (16, 2048, 6144) 7.3 / 8.3 / 8.1.
#include "e2m3_epilogue.h"
#include "hadamard_unit.h"

namespace quest {
namespace e2m3f {

using hq::v4i;
using hq::v4u;
using hq::v16f;
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef int v8i __attribute__((ext_vector_type(8)));

constexpr int kFragB = 1536;
constexpr int kChn = 32;                           // of a tile
constexpr int kMostCus = 256;                      // of a whole device
constexpr int kMaxRows = 16;                       // tokens of a tile: half of a matrix instruction's columns are idle
constexpr int kTailAt = 2 * kMaxRows * 16;         // of a token fragment in LDS: heads, then tails, of the rows that there are
constexpr int kFragPitch = kTailAt + 2 * kMaxRows * 8 + 64;      // the blocks of a row, two fragments apart, on different banks
constexpr int kSumPitch = kChn + 4;                // floats per token row, as in gemm_e2m3_split.hip

template <int G, int CT>
struct Shape {
    static constexpr int kWaves = G, kRowsPerWave = 32 / G, kSteps = 2 * G;
    static constexpr int kShare = G / CT, kMine = 2 * CT;        // waves of a channel tile, steps of one of them
    static_assert(G % CT == 0, "whole waves per channel tile");
    static constexpr int kStageB = 32 * 256;       // a wave's rows as they come, 32 blocks
    static constexpr int kSumsAt = kSteps * kFragPitch, kWaveB = kMine * kFragB;         // of a wave's sums, and of its first weights
    static constexpr int kRowsAt = kSumsAt + kWaves * kWaveB;
    static constexpr int kNormAt = kRowsAt + kMaxRows / kRowsPerWave * kStageB, kScalesAt = kNormAt + G * 256;
    static constexpr int kLdsB = kScalesAt + kMaxRows * 2;
    static_assert(kLdsB <= 160 * 1024 && kMaxRows * kSumPitch * 4 <= kWaveB, "LDS of a CU");
};

struct Args {
    void *out;
    const uint16_t *x, *norm_w;
    const uint8_t *wgt;
    int M, N, K, tiles_t, tiles_c;                 // (tiles_c: of CT channel tiles)
    int rows, ways;                                // tokens of a tile; workgroups of an XCD per token tile
    uint32_t entry_bits;
    float eps;
    Epilogue epi;
};

// what this wave has written to LDS is there for the others behind it; its loads stay in flight
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    plain_barrier();
}

// CT: channel tiles that the waves share.  RAG: rows that are not whole 128s, without norm and transform
template <int DT, int G, int CT, bool NORM, bool ROPE, bool RAG>
__global__ void __launch_bounds__((64 * G), (G / 4)) linear_e2m3_fused_kernel(Args p) {
    using S = Shape<G, CT>;
    __shared__ __attribute__((aligned(1024))) uint8_t lds[S::kLdsB];
    float *const sums = reinterpret_cast<float *>(lds + S::kSumsAt);
    uint16_t *const scales = reinterpret_cast<uint16_t *>(lds + S::kScalesAt);
    const int lane = (int)threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int M = p.M, N = p.N, K = p.K;
    // XCD x takes the x-th eighth of the channel tiles, its workgroups the token tiles of one after the other
    const int xcd = (int)blockIdx.x & 7, local = (int)blockIdx.x >> 3;
    const int tt = local % p.tiles_t, per_xcd = (p.tiles_c + 7) >> 3;
    const int ct_end = min((xcd + 1) * per_xcd, p.tiles_c);
    int ct = xcd * per_xcd + local / p.tiles_t;
    if (ct >= ct_end) return;                      // uniform: the whole workgroup
    const int tok0 = tt * p.rows, tok_end = min(tok0 + p.rows, M);

    // ---- weights: the wave's two steps of a channel tile; steps past the row's end and tiles past the last touch no memory and are zeros
    const int nk = (K + 127) / 128 * 2, pitch = nk * kFragB;     // (rows of whole 32s, without the transform, have tiles with zeros behind them)
    const uint32_t dead = 0x80000000u;
    const int blocks_c = (N + kChn - 1) / kChn, share = wave % S::kShare, mine_c = wave / S::kShare;
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc((void *)p.wgt, 0, blocks_c * pitch, 0x00020000);
    struct Frag { v4u head; v2u tail; };
    auto step_at = [&](int tile, int i) {
        const int step = share + S::kShare * i, block = tile * CT + mine_c;
        return tile < ct_end && block < blocks_c && step < nk ? (uint32_t)(block * pitch + step * kFragB) : dead;
    };
    auto load_weights = [&](Frag (&w)[S::kMine], int tile) {
#pragma unroll
        for (int i = 0; i < S::kMine; i++) {
            const uint32_t at = step_at(tile, i);
            w[i].head = __builtin_amdgcn_raw_buffer_load_b128(wr, (int)(at + lane * 16), 0, 0);
            w[i].tail = __builtin_amdgcn_raw_buffer_load_b64(wr, (int)(at + 1024 + lane * 8), 0, 0);
        }
    };
    uint8_t *const first = lds + S::kSumsAt + wave * S::kWaveB;
    auto load_first = [&]() {                      // the heads, then two steps' tails at a time, one by lanes 0-31
        auto to_lds = [&](uint32_t at, int dst) {
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wr, (__attribute__((address_space(3))) void *)(first + dst), 16, at, 0, 0, 0);
        };
#pragma unroll
        for (int i = 0; i < S::kMine; i++) to_lds(step_at(ct, i) + lane * 16, i * 1024);
#pragma unroll
        for (int i = 0; i < S::kMine; i += 2)
            to_lds((lane < 32 ? step_at(ct, i) : step_at(ct, i + 1)) + 1024 + (lane & 31) * 16, S::kMine * 1024 + i * 512);
    };

    // ---- the wave's token rows (register layout: hadamard_unit.h)
    const int n = lane & 31, h = lane >> 5, blk = n % G;
    const int row = wave * S::kRowsPerWave + n / G;                      // of the tile
    const bool busy = tok0 + wave * S::kRowsPerWave < tok_end;           // uniform in the wave
    const bool counts = tok0 + row < tok_end;
    // They come by direct loads of a KiB, whole lines at a time, and are read from LDS in the order of the transform: 32 bytes of every block per
    // load, as the activation kernel has them, would keep the CU's one port to memory busy twice as long.  Chunk c (16 bytes) of the wave's block b waits at
    // chunk c ^ (b & 15) of its place: the lanes of a read on different banks.  Blocks past a row's end and rows past the last one are zeros.
    uint8_t *const stage = lds + S::kRowsAt + wave * S::kStageB;
    auto bring = [&](const void *from, int bytes, uint8_t *to, int i, bool rows) {
        const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void *)from, 0, bytes, 0x00020000);
        const int b = 4 * i + (lane >> 4), row_b = rows ? wave * S::kRowsPerWave + b / G : 0, at = b % G;
        const int chunk = 16 * at + ((lane & 15) ^ (b & 15));             // of the row
        const bool in = 8 * chunk < K && (!rows || tok0 + row_b < tok_end);
        const uint32_t off = in ? (uint32_t)((rows ? (tok0 + row_b) * K * 2 : 0) + chunk * 16) : dead;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)(to + i * 1024), 16, off, 0, 0, 0);
    };
    if (busy) {
#pragma unroll
        for (int i = 0; i < 8; i++) bring(p.x, M * K * 2, stage, i, true);
        if constexpr (NORM) {                      // (every wave brings the same bytes to the same place)
#pragma unroll
            for (int i = 0; i < G / 4; i++) bring(p.norm_w, K * 2, lds + S::kNormAt, i, false);
        }
    }
    load_first();
    __builtin_amdgcn_sched_barrier(0);             // all of these are in flight before anything is waited for

    // ---- what a channel tile's first wave finishes it with: eight channels of a token per lane
    const int col = lane & 3, t_row = lane >> 2;
    static_assert(kMaxRows * kChn == 8 * 64, "a lane's share");
    const bool finishes = share == 0;              // uniform in the wave
    const bool vec16 = (N & 7) == 0;
    const __amdgpu_buffer_rsrc_t br = __builtin_amdgcn_make_buffer_rsrc((void *)p.epi.b_mul, 0, (N * 2 + 2) & ~3, 0x00020000);
    v4u muls[2];                                   // of this channel tile and the next
    Ahead<ROPE> ahead[2];
    auto fetch_channels = [&](v4u &muls, Ahead<ROPE> &ahead, int tile) {          // (channels past the vector's end read as zeros: their outputs are not stored)
        if (!finishes || tile >= ct_end) return;
        const int ch = (tile * CT + mine_c) * kChn + col * 8;
        muls = __builtin_amdgcn_raw_buffer_load_b128(br, ch * 2, 0, 0);
        if (ROPE || p.epi.kind == kEpiAdd || p.epi.kind == kEpiBias) fetch_ahead<DT>(ahead, p.out, p.epi, tok0 + t_row, ch, tok_end, N, vec16);
    };

    if (busy) {
        v4i hv[2][2];
        if constexpr (!RAG) hq::signed_entries(hv, n, h, p.entry_bits);
        wait_vmcnt_imm<3 * CT>();                     // the rows (and the norm's weights) are here, the first weights need not be
        asm volatile("" ::: "memory");
        v4u bq[8];
#pragma unroll
        for (int s = 0; s < 8; s++) bq[s] = *reinterpret_cast<const v4u *>(stage + n * 256 + ((2 * s + h) ^ (n & 15)) * 16);
        if constexpr (NORM) {
            float ss = 0.f;
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int d = 0; d < 4; d++) ss = hq::dot2_self<DT>(bq[s][d], ss);
            v4u nq[8];
#pragma unroll
            for (int s = 0; s < 8; s++) nq[s] = *reinterpret_cast<const v4u *>(lds + S::kNormAt + blk * 256 + ((2 * s + h) ^ (blk & 15)) * 16);
            hq::normalise<DT>(bq, nq, hq::group_sum_f<G>(ss), K, p.eps);
        }
        uint32_t yb[4][8];
        float total;
        if constexpr (RAG) total = hq::ragged_sum<DT, G>(yb, bq);
        else total = hq::transform<DT>(yb, bq, hv, p.entry_bits);
        fetch_channels(muls[0], ahead[0], ct);     // (here: the transform needs the registers)
        if constexpr (!RAG) total = hq::group_sum_f<G>(total);
        const uint32_t s16 = from_f32<DT>(scale_from_sumsq(total, K));
        if (n % G == 0 && h == 0) scales[row] = (uint16_t)s16;
        const float sf = to_f32<DT>(s16), inv = quant_inv(sf);
        uint8_t *const frag = lds + (2 * blk + h) * kFragPitch;
        auto put = [&](int g, hq::v6u c) {
            const int slot = kMaxRows * g + row;
            if (blk * 128 + 64 * h + 32 * g >= K) c = hq::v6u{0, 0, 0, 0, 0, 0};
            *reinterpret_cast<uint4 *>(frag + slot * 16) = make_uint4(c[0], c[1], c[2], c[3]);
            *reinterpret_cast<uint2 *>(frag + kTailAt + slot * 8) = make_uint2(c[4], c[5]);
        };
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(counts && !quant_fast_ok(sf)) == 0, 1)) {
#pragma unroll
            for (int g = 0; g < 2; g++) put(g, hq::e2m3_group<DT, true>(yb, g, inv));
        } else {
#pragma unroll
            for (int g = 0; g < 2; g++) put(g, hq::e2m3_group<DT, false>(yb, g, inv));
        }
    } else {
        fetch_channels(muls[0], ahead[0], ct);
    }
    wait_vmcnt_imm<0>();                           // the first weights are in LDS
    Frag w[2][S::kMine];                                // of this channel tile and the next
    load_weights(w[1], ct + p.ways);
    fetch_channels(muls[1], ahead[1], ct + p.ways);
    lds_barrier();

    // (rows past the last token hold whatever LDS held: E2M3 has neither NaN nor Inf, and their sums are not stored)
    auto fragment = [](v4u a, v2u b) {
        v8i f = __builtin_shufflevector(__builtin_bit_cast(v4i, a), __builtin_bit_cast(v4i, a), 0, 1, 2, 3, -1, -1, -1, -1);
        f[4] = (int)b[0];
        f[5] = (int)b[1];
        return f;
    };
    v8i tok[S::kMine];
#pragma unroll
    for (int i = 0; i < S::kMine; i++) {
        w[0][i].head = *reinterpret_cast<const v4u *>(first + i * 1024 + lane * 16);
        w[0][i].tail = *reinterpret_cast<const v2u *>(first + S::kMine * 1024 + i * 512 + lane * 8);
        const uint8_t *f = lds + (share + S::kShare * i) * kFragPitch;
        const int slot = kMaxRows * h + n % kMaxRows;
        tok[i] = fragment(*reinterpret_cast<const v4u *>(f + slot * 16), *reinterpret_cast<const v2u *>(f + kTailAt + slot * 8));
    }
    const float t_half_mul = __fmul_rn(0.5f, to_f32<DT>(scales[t_row]));
    float *const mine = sums + wave * (S::kWaveB / 4) + n * kSumPitch + 4 * h;
    while (true) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            v16f acc;
#pragma unroll
            for (int r = 0; r < 16; r++) acc[r] = 0.f;
#pragma unroll
            for (int i = 0; i < S::kMine; i++) acc = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fragment(w[u][i].head, w[u][i].tail), tok[i], acc, 2, 2, 0, 0, 0, 0);
            load_weights(w[u], ct + 2 * p.ways);
            // register r of lane (li, lg) is token li, channel 8 (r / 4) + 4 lg + r % 4
            if (n < kMaxRows) {
#pragma unroll
                for (int q = 0; q < 4; q++) *reinterpret_cast<float4 *>(mine + 8 * q) = make_float4(acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]);
            }
            lds_barrier();
            if (finishes) {
                const int ch = (ct * CT + mine_c) * kChn + col * 8;
                float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
                for (int v = 0; v < S::kShare; v++)
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const float4 s = *reinterpret_cast<const float4 *>(sums + (wave + v) * (S::kWaveB / 4) + t_row * kSumPitch + col * 8 + 4 * i);
                        sum[4 * i] += s.x; sum[4 * i + 1] += s.y; sum[4 * i + 2] += s.z; sum[4 * i + 3] += s.w;
                    }
                if (tok0 + t_row < tok_end && ch < N) {
                    float v[8];
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        v[i] = __fmul_rn(__fadd_rn(sum[i], sum[i]), __fmul_rn(t_half_mul, i & 1 ? hi_f32<DT>(muls[u][i >> 1]) : lo_f32<DT>(muls[u][i >> 1])));
                    uint32_t o[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) o[i] = pack2_rounded_products<DT>(v[2 * i], v[2 * i + 1]);
                    finish_eight<DT>(p.out, make_uint4(o[0], o[1], o[2], o[3]), p.epi, ahead[u], tok0 + t_row, ch, N, vec16);
                }
            }
            ct += p.ways;
            if (ct >= ct_end) return;                  // uniform: the whole workgroup
            fetch_channels(muls[u], ahead[u], ct + p.ways);
            lds_barrier();                             // the sums have been read
        }
    }
}

template <int DT, int G, int CT>
static int launch_as(const Args &a, bool norm, hipStream_t st) {
    const dim3 grid((unsigned)(8 * a.ways * a.tiles_t)), block(64 * G);
    const bool rope = a.epi.kind == kEpiRope;
    const bool ragged = (a.K & 127) != 0;
    if (norm && rope) linear_e2m3_fused_kernel<DT, G, CT, true, true, false><<<grid, block, 0, st>>>(a);
    else if (norm) linear_e2m3_fused_kernel<DT, G, CT, true, false, false><<<grid, block, 0, st>>>(a);
    else if (rope && ragged) linear_e2m3_fused_kernel<DT, G, CT, false, true, true><<<grid, block, 0, st>>>(a);
    else if (rope) linear_e2m3_fused_kernel<DT, G, CT, false, true, false><<<grid, block, 0, st>>>(a);
    else if (ragged) linear_e2m3_fused_kernel<DT, G, CT, false, false, true><<<grid, block, 0, st>>>(a);
    else linear_e2m3_fused_kernel<DT, G, CT, false, false, false><<<grid, block, 0, st>>>(a);
    return launch_status();
}

// Tokens and channel tiles that a workgroup has at a time, and workgroups, one per CU; 0 where the two launches are the faster way, else the channel
// tiles.  A launch is its first round -- 4.6 to 5.4 us with rows of up to 1024, half a microsecond more with two channel tiles, 5.6 (eight rows) or 6.8
// (sixteen) with longer rows, with the norm 1.0, 1.3 or 2.2 more -- and for each further round 0.8 us, with two channel tiles 1.0, with longer rows 1.1.  The
// two launches take 6.7 to 8 us up to 8192 channels, 10 to 13 at 22016, with the norm 1.1 more.  So: one round of one channel tile where that is all, else
// two (K = 1024, with the norm, (37, 3072) 6.2 / 6.8, (37, 5632) 7.2 / 7.8, (128, 5632) 8.3 / 10.4; four are slower, (37, 5632) 7.4, but for 96 tokens on
// 22016 channels), and so many rounds as are faster, GPU us in a graph against the two launches.  K = 1024: (128, 8192), four rounds, 8.7 / 9.0, (192,
// 5632) with the norm, six, 11.2 / 10.9; 22016 channels, 37 tokens, five, 10.1 / 10.5, 64, six, 11.2 / 10.8.  K = 2048: (16, 6144), two, 7.3 / 8.3, (32, 6144),
// three, 8.4 / 8.3, (16, 22016), three of sixteen rows, 11.4 / 13.4, (128, 1024), one of sixteen, 6.9 / 8.1.
static int plan(Args &a, bool norm, int cus) {
    const int blocks = (a.N + kChn - 1) / kChn;
    const bool is_short = a.K <= 1024;
    for (int ct = 1; ct <= (is_short ? 2 : 1); ct++) {
        int best = 0;
        for (int rows = 8; rows <= kMaxRows; rows += 8) {
            const int tiles_t = (a.M + rows - 1) / rows, room = cus / (8 * tiles_t), per_xcd = ((blocks + ct - 1) / ct + 7) / 8;
            if (room < 1) continue;
            const int rounds = (per_xcd + room - 1) / room;
            const int most = is_short ? (ct == 1 ? 1 : 4 + a.N / 16384) : rows == 8 ? 2 + a.N / 8192 : norm ? 0 : 1 + a.N / 8192;
            if (rounds > most || (best != 0 && rounds + (is_short ? 0 : 1) >= best)) continue;
            best = rounds, a.rows = rows, a.tiles_t = tiles_t, a.tiles_c = (blocks + ct - 1) / ct, a.ways = per_xcd < room ? per_xcd : room;
        }
        if (best != 0) return ct;
    }
    return 0;
}

template <int DT>
static int launch(int ct, const Args &a, bool norm, hipStream_t st) {
    if (a.K > 1024) return launch_as<DT, 16, 1>(a, norm, st);
    return ct == 1 ? launch_as<DT, 8, 1>(a, norm, st) : launch_as<DT, 8, 2>(a, norm, st);
}

}  // namespace e2m3f
}  // namespace quest

using namespace quest;

extern "C" int quest_linear_e2m3_fused(const quest_fused_linear *l, void *stream) {
    forget_stale_error();
    if (!l || !l->out || !l->x || !l->w_tiles || !l->w_scale) return QUEST_ERR_NULL_POINTER;
    if (!check_dtype(l->dtype)) return QUEST_ERR_BAD_DTYPE;
    const int m = l->size_m, k = l->size_k, n = l->size_n;
    const bool norm = l->norm_weight != nullptr;
    if (m <= 0 || k <= 0 || n <= 0 || (k & (norm || l->had_scale != 0.f ? 127 : 31))) return QUEST_ERR_BAD_SHAPE;
    if (l->epilogue < kEpiPlain || l->epilogue > kEpiBias || m > 256 || k <= 512 || k > 2048) return QUEST_ERR_UNSUPPORTED;
    if (l->epilogue == kEpiBias && !l->bias) return QUEST_ERR_NULL_POINTER;
    if (l->epilogue == kEpiGlu && (n & 7)) return QUEST_ERR_BAD_SHAPE;
    if (l->epilogue == kEpiRope) {
        if (!l->freqs_cis) return QUEST_ERR_NULL_POINTER;
        if (l->seq_len <= 0 || l->rot_cols <= 0 || l->head_dim <= 0 || (l->head_dim & 31) || l->rot_cols % l->head_dim || l->rot_cols > n || (n & 7)) return QUEST_ERR_BAD_SHAPE;
    }
    if (!aligned(l->x, 16) || !aligned(l->w_tiles, 16) || !aligned(l->out, 16) || !aligned(l->w_scale, 4) || !aligned(l->norm_weight, 16) || !aligned(l->bias, 16) ||
        !aligned(l->freqs_cis, 16))
        return QUEST_ERR_ALIGNMENT;
    uint32_t bits = 0;
    // (32-bit offsets into the weights)
    if (l->had_scale < 0.f || !representable16(l->had_scale, l->dtype, &bits) || ((long)n + 31) / 32 * ((k + 127) / 128 * 2) * e2m3f::kFragB >= (1L << 31)) return QUEST_ERR_UNSUPPORTED;
    hipStream_t st = (hipStream_t)stream;
    const RopeArgs rope = {l->freqs_cis, l->seq_len, l->rot_cols, l->head_dim, (const uint16_t *)l->bias};
    e2m3f::Args a = {l->out, (const uint16_t *)l->x, (const uint16_t *)l->norm_weight, (const uint8_t *)l->w_tiles, m, n, k, 0, 0, 0, 0, bits,
                     l->eps, {l->epilogue, nullptr, (const uint16_t *)l->w_scale, rope}};
    // (what a whole device does not take, no partition of it does: two launches follow, and the host is not kept waiting by the question for its size)
    if (e2m3f::plan(a, norm, e2m3f::kMostCus) == 0) return QUEST_ERR_UNSUPPORTED;
    const int ct = e2m3f::plan(a, norm, device_cu_count(st));
    if (ct == 0) return QUEST_ERR_UNSUPPORTED;
    return l->dtype == QUEST_DTYPE_BF16 ? e2m3f::launch<0>(ct, a, norm, st) : e2m3f::launch<1>(ct, a, norm, st);
}
