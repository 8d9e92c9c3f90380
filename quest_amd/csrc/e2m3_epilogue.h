// What the FP6 GEMM kernels beside gemm_e2m3.hip share: the description of an epilogue and their entry points, and for the two
// smaller-tile kernels (gemm_e2m3_mid.hip, gemm_e2m3_split.hip) the way of eight consecutive channels of one token row, rounded to the dtype, to memory.
#pragma once
#include "gemm_tiles.h"

namespace quest {

struct Epilogue {
    int kind;                                     // kEpi*
    const uint16_t *a_mul, *b_mul;                // 4-byte aligned
    RopeArgs rope;                                // kEpiRope; its `bias` for kEpiBias
};

// What finish_eight needs from memory for eight channels: the residual or bias piece, or the pairs of cos and sin (ROPE).  The
// kernels fetch all of a lane's before the products and keep them in registers (there is room: one or two workgroups of four waves per
// CU): fetched piece by piece between the stores, each waits out a trip to memory (1000 x 7680 channels, K = 2560, rotary: 31.7
// us that way, 20 with the values at hand).
template <bool ROPE>
struct Ahead {
    uint4 v[ROPE ? 2 : 1];
};

// vec16: the output's rows are whole eights of channels.  (A bias is 16-byte aligned: the entry point asks for it.)
template <int DT, bool ROPE>
__device__ __forceinline__ void fetch_ahead(Ahead<ROPE> &a, const void *out, const Epilogue &epi, int tok, int ch, int M, int N, bool vec16) {
    const bool in = tok < M && ch < N;
    if constexpr (ROPE) {
        if (in && ch < epi.rope.rot_cols) {
            const int h = ch % epi.rope.head_dim;
            const uint4 *f = reinterpret_cast<const uint4 *>(epi.rope.freqs + ((size_t)(tok % epi.rope.seq_len) * (epi.rope.head_dim >> 1) + (h >> 1)) * 2);
            a.v[0] = f[0];
            a.v[1] = f[1];
        }
    } else if (vec16 && in && (epi.kind == kEpiAdd || epi.kind == kEpiBias)) {
        a.v[0] = *reinterpret_cast<const uint4 *>(epi.kind == kEpiAdd ? reinterpret_cast<const uint16_t *>(out) + (size_t)tok * N + ch : epi.rope.bias + ch);
    }
}

// p: channels ch ... ch + 7 of row tok < M, two per dword.
template <int DT, bool ROPE>
__device__ __forceinline__ void finish_eight(void *out, uint4 p, const Epilogue &epi, const Ahead<ROPE> &ahead, int tok, int ch, int N, bool vec16) {
    uint16_t *dst = reinterpret_cast<uint16_t *>(out) + (size_t)tok * N + ch;
    bool adds = false;
    if constexpr (ROPE) {
        if (ch < epi.rope.rot_cols) {
            auto f4 = [](uint4 u) { return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w)); };
            const float4 cs[2] = {f4(ahead.v[0]), f4(ahead.v[1])};
            p = rope_turn<DT>(p, cs);
        }
    } else {
        if (epi.kind == kEpiGlu) {                 // weight rows in eights: four gates, then the four ups of the same outputs
            *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(out) + (size_t)tok * (N >> 1) + (ch >> 1)) =
                make_uint2(silu_mul_pair<DT>(p.x, p.z), silu_mul_pair<DT>(p.y, p.w));
            return;
        }
        adds = epi.kind == kEpiAdd || epi.kind == kEpiBias;
    }
    if (vec16) {
        if constexpr (!ROPE) {
            if (adds) p = add_eight<DT>(p, ahead.v[0]);
        }
        *reinterpret_cast<uint4 *>(dst) = p;
        return;
    }
    const uint16_t *other = epi.kind == kEpiAdd ? dst : epi.rope.bias + ch;
    const uint32_t d[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
    for (int i = 0; i < 8; i++) {
        if (ch + i >= N) continue;
        uint32_t h = i & 1 ? d[i >> 1] >> 16 : d[i >> 1] & 0xffffu;
        if (adds) h = add_pair<DT>(h, other[i]) & 0xffffu;
        dst[i] = (uint16_t)h;
    }
}

// How the tiles of a grid of `tiles_t` token tiles x `tiles_c` channel tiles are dealt: workgroups go to the eight XCDs in turn,
// and each XCD takes a contiguous eighth of the tiles, the token tiles of a channel tile one after the other, so that its L2
// fetches few weights and no XCD has more than its share (whole channel tiles per XCD left 1400 tokens x 2560 channels with two
// rounds of 128 x 128 tiles on half of the XCDs: 24 instead of 13 us).  False: nothing for this workgroup.
__device__ __forceinline__ bool tile_of(int tiles_t, int tiles_c, int &tt, int &ct) {
    const int total = tiles_t * tiles_c, per_xcd = (total + 7) >> 3;
    const int local = (int)blockIdx.x >> 3, index = ((int)blockIdx.x & 7) * per_xcd + local;
    ct = index / tiles_t;
    tt = index - ct * tiles_t;
    return local < per_xcd && index < total;
}
inline long tile_grid(int tiles_t, int tiles_c) { return ((long)tiles_t * tiles_c + 7) / 8 * 8; }

// gemm_e2m3_mid.hip / gemm_e2m3_split.hip: tiles of 32 tf x 32 cf; QUEST_ERR_UNSUPPORTED for a shape that is not built
int launch_gemm_e2m3_mid(int dtype, int tf, int cf, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st);
int launch_gemm_e2m3_split(int dtype, int tf, int cf, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, const Epilogue &epi, hipStream_t st);
// gemm_e2m3_resident.hip: K from 256 to kResidentMaxK, whole eights of channels, at least eight CUs.  The plan's estimated time in us; `plan` (or
// null): as quest_e2m3_gemm_plan reports it.
constexpr int kResidentMaxK = 1664;
int launch_gemm_e2m3_resident(int dtype, void *out, const uint8_t *a, const uint8_t *b, int M, int K, int N, int cus, const Epilogue &epi, hipStream_t st);
float gemm_e2m3_resident_plan(int M, int K, int N, int cus, int *plan);
// LDS slots of a shape's pipeline (the split kernel's: per wave); 0 for a shape that is not built
int gemm_e2m3_mid_slots(int tf, int cf);
int gemm_e2m3_split_slots(int tf, int cf);

}  // namespace quest
