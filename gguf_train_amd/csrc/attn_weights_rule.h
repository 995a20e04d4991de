// When the averaged float32 weights split their heads over a workgroup's wavefronts (attn_weights.hip).
#pragma once

#include <cstdint>

// grid: workgroups of 128 query rows, nkt: 64-key tiles, of the kernel that walks all heads in each wavefront;
// that fills half of the 256 CUs where this changes over.  Split, a workgroup holds 32 rows, so there are four
// times as many, and Q and K are loaded by all of them.  Measured, walked against split, us: D64, key
// padding, H8 64 workgroups 57 against 19, H5 128 38 against 30, H4 120 32 against 21, H8 160 58 against 50,
// but H5 160 38 against 44, H8 224 60 against 66, H5 224 40 against 59; without a mask H5 120 26 against 18,
// H8 160 36 against 34, H6 160 27 against 32; D128, no mask, H8 64 55 against 26, H5 128 37 against 36, H5
// 160 41 against 50, H8 224 63 against 79.  The causal mask changes none of these by more than a tenth.
constexpr bool f32_heads_split(int64_t grid, int64_t nkt, int64_t H, int waves) { return H >= waves && grid * nkt <= 128; }
