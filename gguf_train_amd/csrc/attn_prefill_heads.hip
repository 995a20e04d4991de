// The float16 / bfloat16 prefill kernels of head sizes 80 and 96 (attn_prefill_half.h), in a file of their
// own so that they compile beside those of 64 and 128.

#include "attn_prefill_half.h"

hipError_t launch_prefill_heads(const AttnFwdArgs &a, int cd, int nq, int order, int64_t grid, hipStream_t s) {
    if (cd == GT_F16)
        return a.D == 96 ? launch_variant<_Float16, 96>(a, nq, order, grid, s) : launch_variant<_Float16, 80>(a, nq, order, grid, s);
    return a.D == 96 ? launch_variant<__bf16, 96>(a, nq, order, grid, s) : launch_variant<__bf16, 80>(a, nq, order, grid, s);
}
