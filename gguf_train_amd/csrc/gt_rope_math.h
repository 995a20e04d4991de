// The rotation step of RoPE, shared by the rope kernel (gt_rope.hip) and the RoPE-on-append of
// the KV cache (gt_convert.hip) so that both produce the same bits.  For a pair (lo, hi) and the
// angle's (cos, sin) = (c, s):  y_lo = lo*c - hi*s,  y_hi = lo*s + hi*c  (ggml's rotation,
// csrc/gt_ops_nn.cpp:2388-2391 -> ggml_rope_ext).  Each is one product rounded to float32 and one
// fused multiply-add, written out so that the compiler's contraction choices cannot differ
// between the call sites.  The float32 result is pinned in a register: the reference rounds it to
// float32 and then to the tensor's dtype, and without the pin the compiler may fuse the multiply-add
// with a conversion to float16 (v_fma_mix*_f16), which rounds once and differs in rare halfway cases.
#pragma once

#include <hip/hip_runtime.h>

#include "rope_rows.h"

// Angle of pair i at position p: theta_i is the float32 chain of i products (one rounding each), as
// ggml forms it; theta_{i+1} = theta_i * theta_scale continues it.  The chain's length differs between
// the lanes, so it is walked 8, 4, 2 and 1 products at a time: one product per iteration spends most of a
// wavefront's time on the loop.
__device__ inline float rope_theta(int32_t p, int i, float theta_scale) {
    float theta = (float)p;
    auto times = [&](int n) {
#pragma unroll
        for (int j = 0; j < n; ++j) theta *= theta_scale;
    };
    for (int j = i >> 3; j > 0; --j) times(8);
    if (i & 4) times(4);
    if (i & 2) times(2);
    if (i & 1) times(1);
    return theta;
}
__device__ inline float2 rope_cos_sin(float theta, float freq_scale) {
    float sn, cs;
    sincosf(freq_scale * theta, &sn, &cs);
    return make_float2(cs, sn);
}

__device__ inline float rope_rot_lo(float lo, float hi, float2 cs) {
    float r = __fmaf_rn(lo, cs.x, -(hi * cs.y));
    asm volatile("" : "+v"(r));
    return r;
}
__device__ inline float rope_rot_hi(float lo, float hi, float2 cs) {
    float r = __fmaf_rn(hi, cs.x, lo * cs.y);
    asm volatile("" : "+v"(r));
    return r;
}
