// Classes of the tiles of an attention mask that varies along the query rows and is shared by the
// heads, for the half-precision prefill kernel (mask mode 7): one pass over the mask before the
// attention, so that the attention of every head skips the tiles that block everything, treats the
// tiles that block nothing as unmasked and reads the tiles that only block as one bit per score.  Tiles
// with other values are read as float32, from the mask itself or from a copy made here.
//
// Bound by latency: a workgroup reads one 128-row tile (16 to 32 KB for a float16 mask), all loads of
// a wavefront's rows in flight; the band mask of fp16 B4 H32/8 L500 S1500 (1.5 MB, 96 tiles) takes 5.0
// us, where converting it to float32 took 10.5, and the attention after it goes from 82 to 61 us (an
// eighth of its tiles are blocked, most others clear).  A half-precision tile with other values is written
// to the copy from the registers that it was classed in (read again it took 13 us there, now 6.6).

#include "attn_common.h"

namespace {

// One workgroup per (key tile, query tile, mask batch).  Elements past L or S count as neither
// blocked nor visible (the attention kernel blocks the keys itself and does not store the rows); with a
// causal mask beside this one, tiles above the diagonal, which the attention never visits, are not read.
template <typename TM, int BN, int NW>
__global__ __launch_bounds__(64 * NW) void mask_tiles_kernel(const TM *mask, int64_t sb, int64_t sl, int64_t ss, int L, int S,
                                                         int causal, AttnMaskTiles t, float *copy) {
    constexpr int NH = BN / 64;  // 64-key halves: a wavefront's lanes are 64 keys of one row
    constexpr int ROWS = kMaskTileRows / NW;
    __shared__ int s_seen[NW];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int kt = blockIdx.x, qt = blockIdx.y, b = blockIdx.z;
    const int row0 = qt * kMaskTileRows + w * ROWS;
    uint8_t *out = const_cast<uint8_t *>(t.cls) + ((int64_t)b * gridDim.y + qt) * t.nkt + kt;
    if (causal && kt * BN >= (qt + 1) * kMaskTileRows) {
        if (threadIdx.x == 0) *out = kMaskTileBlocked;
        return;
    }
    const TM *mb = mask + b * sb;
    uint32_t *bits = const_cast<uint32_t *>(t.bits) + (int64_t)b * L * t.words;
    int seen = 0;  // 1: a visible element, 2: a blocked one, 4: a value other than 0 and -inf
    // every row's load before anything is stored (the compiler keeps a load behind a store that
    // might alias it: one round trip per row, 13.5 us instead of 6.1)
    TM v[NH][ROWS];
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
        const TM *col = mb + (int64_t)min(kt * BN + 64 * hf + lane, S - 1) * ss;
#pragma unroll
        for (int r = 0; r < ROWS; ++r) v[hf][r] = col[(int64_t)min(row0 + r, L - 1) * sl];
    }
#pragma unroll
    for (int hf = 0; hf < NH; ++hf) {
        const int key = kt * BN + 64 * hf + lane;
        uint64_t mine = 0;  // lane r: row r's 64 keys
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
            const bool in = row0 + r < L && key < S;
            bool blocked, other = false;
            if constexpr (sizeof(TM) == 1) {
                blocked = v[hf][r] == 0;
            } else {
                const float x = (float)v[hf][r];
                blocked = x == -INFINITY;
                other = !blocked && x != 0.0f;
            }
            seen |= (in && !blocked ? 1 : 0) | (in && blocked ? 2 : 0) | (in && other ? 4 : 0);
            const uint64_t vis = __builtin_amdgcn_ballot_w64(in && !blocked);
            mine = lane == r ? vis : mine;
        }
        const int word = (kt * BN + 64 * hf) / 32;
        if (lane < ROWS && row0 + lane < L) {
            uint32_t *dst = bits + (int64_t)(row0 + lane) * t.words + word;
            if (word < t.words) dst[0] = (uint32_t)mine;
            if (word + 1 < t.words) dst[1] = (uint32_t)(mine >> 32);
        }
    }
    const int any = (__builtin_amdgcn_ballot_w64(seen & 1) ? 1 : 0) | (__builtin_amdgcn_ballot_w64(seen & 2) ? 2 : 0) |
                    (__builtin_amdgcn_ballot_w64(seen & 4) ? 4 : 0);
    if (lane == 0) s_seen[w] = any;
    __syncthreads();
    int all = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) all |= s_seen[i];
    const int cls = all & 4 ? kMaskTileValues : !(all & 1) ? kMaskTileBlocked : all & 2 ? kMaskTileBits : kMaskTileClear;
    if (threadIdx.x == 0) *out = (uint8_t)cls;
    if constexpr (sizeof(TM) == 2) {
        if (cls == kMaskTileValues) {
            const int64_t pitch = attn_mask_copy_pitch(S);
#pragma unroll
            for (int hf = 0; hf < NH; ++hf) {
                const int key = kt * BN + 64 * hf + lane;
                if (key >= S) continue;
#pragma unroll
                for (int r = 0; r < ROWS; ++r) {
                    const int row = row0 + r;
                    if (row < L) copy[((int64_t)b * L + row) * pitch + key] = (float)v[hf][r];
                }
            }
        }
    }
}

template <int BN, int NW>
hipError_t launch(int kind, const void *mask, int64_t batches, int64_t sb, int64_t sl, int64_t ss, int64_t L, int64_t S,
                  int causal, const AttnMaskTiles &t, float *copy, hipStream_t s) {
    const dim3 grid((unsigned)t.nkt, (unsigned)((L + kMaskTileRows - 1) / kMaskTileRows), (unsigned)batches);
#define GT_TILES(TM) \
    hipLaunchKernelGGL((mask_tiles_kernel<TM, BN, NW>), grid, dim3(64 * NW), 0, s, (const TM *)mask, sb, sl, ss, (int)L, (int)S, causal, t, copy)
    switch (kind) {
        case 0: GT_TILES(uint8_t); break;
        case 1: GT_TILES(_Float16); break;
        case 2: GT_TILES(__bf16); break;
        default: GT_TILES(float); break;
    }
#undef GT_TILES
    return hipGetLastError();
}

}  // namespace

hipError_t launch_attn_mask_tiles(int kind, const void *mask, int64_t batches, int64_t sb, int64_t sl, int64_t ss,
                                  int64_t L, int64_t S, int bn, int causal, const AttnMaskTiles &t, float *copy,
                                  hipStream_t s) {
    // A tile's rows among 16 wavefronts while there is at most a tile for each CU (float32 values, L=S=1024,
    // tiles of 128 keys: 5.2 us, 8 wavefronts 6.3, 4 wavefronts 10), among 8 from there on (L=S=4096, tiles
    // of 64: 17 us, 16 wavefronts 21, 4 wavefronts 19).
    const int64_t tiles = (int64_t)t.nkt * ((L + kMaskTileRows - 1) / kMaskTileRows) * batches;
    if (bn == 128)
        return tiles <= 256 ? launch<128, 16>(kind, mask, batches, sb, sl, ss, L, S, causal, t, copy, s)
                            : launch<128, 8>(kind, mask, batches, sb, sl, ss, L, S, causal, t, copy, s);
    return tiles <= 256 ? launch<64, 16>(kind, mask, batches, sb, sl, ss, L, S, causal, t, copy, s)
                        : launch<64, 8>(kind, mask, batches, sb, sl, ss, L, S, causal, t, copy, s);
}
