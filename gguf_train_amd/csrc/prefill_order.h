// How the half-precision prefill deals its query tiles to workgroups (attn_prefill_half.h).
#pragma once

#include <cstdint>

// How a launch deals query tiles to workgroups.  kPairs: tiles p and nq-1-p of a head, one after
// the other (equal work for every workgroup under the causal mask).  kSingle: one tile each, the
// heaviest first (kHeadMajor: no causal mask, a head's tiles together); kFolded: one tile each where
// all workgroups are resident at once, the heavier half first and then the lighter half from its
// lightest, so that the two workgroups of a CU carry about the same together.
enum TileOrder { kPairs = 0, kSingle = 1, kFolded = 2, kHeadMajor = 3 };

// Resident workgroups of the prefill kernels: two on each of the 256 CUs.
constexpr int64_t kPrefillSlots = 512;

// Pairs keep every workgroup's work equal and load Q and set up half as often, so they are taken
// where their rounds over the slots are nearly full (causal fp16 B4 H32 L=S=2048 D128, two full
// rounds: 162 us, single tiles 171).  Fewer workgroups than that leave slots empty, and a second
// workgroup's MFMAs no longer cover the first one's softmax: single tiles then (same box, pairs
// against single: bf16 B1 H32/8 L=S=2048 D128 68.2 -> 64.9 us, fp16 B1 H32/8 L=S=1024 32.2 -> 26.8,
// fp16 B1 H8 L=S=3000 67.4 -> 58.8; over 92 causal shapes of 32 to 512 heads and L 200 to 2000, each at
// both types and head sizes, 0.70 of the time).  Short sequences (4, 6 or 8 tiles), whose set-up weighs
// more, keep pairs a little further down:
//  - causal float16 from one and a half rounds on (pairs / single: 4 tiles x 384 heads D128 52 / 57 us,
//    D64 33.2 / 33.8; 6 x 256 D128 62 / 67, D64 42.4 / 42.3; 8 x 320 D128 129 / 136, D64 75 / 78; but 4 x
//    320, one and a quarter, D128 50 / 48, and bfloat16, which does half as much again, is even or better
//    single: 8 x 320 D128 158 / 158, 4 x 384 D64 38.8 / 37.4);
//  - without the causal mask, where all tiles weigh the same, from 13 of 16 slots on at head size 64 and
//    for float16 at 128 (4 x 224 D64 fp16 26.0 / 27.7, bf16 31.4 / 32.8; 8 x 104 D64 fp16 41.7 / 44.1, D128
//    69.8 / 72.7; 4 x 500 D64 fp16 57 / 63; but bfloat16 D128 4 x 256 60 / 58.5).
// Other calls without the causal mask take single tiles, which spread better (fp16 B4 H32/8 L500 S1500 D128
// 72.3 -> 60.3 us, with an (L,S) mask 132.8 -> 93.0; bf16 B2 H16 L300 S900 D64 34.5 -> 20.0; 24 tiles x 96
// heads 310 -> 285; many rounds: even).  `light`: float16 whose
// probabilities are one operand of P.V (no training output, no dropout); `other`: mask tile classes (tiles
// of unknown weight) or dropout, which were not part of this.
constexpr TileOrder tile_order_of(bool causal, bool light, int D, bool other, int nq, int64_t BH) {
    const int64_t pairs = (int64_t)((nq + 1) / 2) * BH;
    const int64_t slots = (pairs + kPrefillSlots - 1) / kPrefillSlots * kPrefillSlots;
    const bool brief = nq % 2 == 0 && nq >= 4 && nq <= 8 && (D == 64 || D == 128) && !other;
    if (!causal) return brief && (light || D == 64) && pairs * 16 >= slots * 13 ? kPairs : kHeadMajor;
    if (nq == 1 || pairs * 16 >= slots * 15 || (brief && light && pairs * 2 >= kPrefillSlots * 3)) return kPairs;
    return nq * BH <= kPrefillSlots ? kFolded : kSingle;
}
