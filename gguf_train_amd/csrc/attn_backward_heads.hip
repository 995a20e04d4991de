// The float16 / bfloat16 backward kernels of head sizes 80 and 96 (attn_backward_half.h), in a file of
// their own so that they compile beside those of 64 and 128.

#include "attn_backward_half.h"

hipError_t launch_attn_bwd_heads(const AttnBwdArgs &a, int cd, hipStream_t s) {
    if (cd == GT_F16) return a.f.D == 96 ? launch_bwd_d<_Float16, 96>(a, s) : launch_bwd_d<_Float16, 80>(a, s);
    return a.f.D == 96 ? launch_bwd_d<__bf16, 96>(a, s) : launch_bwd_d<__bf16, 80>(a, s);
}
