// RoPE (rotary position embedding): GGUF_train's gt_rope / gt_rope_backward
// (csrc/gt_ops_nn.cpp:2298-2421), which run ggml_rope_ext / ggml_rope_ext_back with ext_factor 0,
// attn_factor 1 and no frequency factors.  With those arguments the operation is:
//   theta_scale = powf(freq_base, -2 / n_dims)            (computed on the host, C library powf)
//   pair i at position p: theta_0 = (float)p, theta_{i+1} = theta_i * theta_scale (float32, one
//   rounding per step), angle_i = freq_scale * theta_i, (c, s) = (cos, sin)(angle_i); the backward
//   uses -s (the inverse rotation).
//   NORMAL (mode 0) rotates elements (2i, 2i+1), NEOX (mode 2) rotates (i, i + n_dims/2), for
//   i < n_dims/2; elements from n_dims on pass through.  y_lo = x_lo c - x_hi s,
//   y_hi = x_lo s + x_hi c in float32, on inputs converted to float32, rounded to the output type.
//
// Few rows (kRopeInlineThreads): one kernel, each thread forming its own angles.  Otherwise two
// kernels: the angle table (one (cos, sin) pair per position and pair index, computed once per
// call and shared by every head), then the rotation, which is HBM-bound element work: one thread
// per VEC consecutive elements of a row (16-byte loads and stores for dense rows); a NeoX thread
// also loads its partner group from the other half of the same row, cache lines the neighbouring
// threads of the wave load anyway, so HBM sees each byte once.

#include "gt_internal.h"
#include "gt_rope_math.h"

#include <cmath>

namespace {

struct RopeArgs {
    const void *x;
    int64_t sb, sh, ss, sd;   // element strides of x (B, H, S, D)
    void *y;                  // dense (B, H, S, D) output
    const float2 *table;      // (table row, pair) -> (cos, sin); null: from pos
    const int32_t *pos;       // position of row s
    float theta_scale, freq_scale, sin_sign;
    int64_t tb;               // table row of (b, s) = b * tb + s
    int64_t H, S, D;
    int n_dims, half, neox;
    int64_t ngroups;          // B * H * S * D / VEC
};

template <typename T>
__device__ inline float to_f(T v) {
    return (float)v;
}
template <typename T>
__device__ inline T from_f(float v) {
    return (T)v;  // float16 / bfloat16: round to nearest even; float64: exact
}

// (cos, sin) of every (table row, pair): row r is position pos[r], or base[r / T] + r % T when
// base is given (rows appended after what each sequence holds).
__global__ void rope_table_kernel(const int32_t *__restrict__ pos, const int32_t *__restrict__ base, int64_t T,
                                  int64_t rows, int half, float theta_scale, float freq_scale, float sin_sign,
                                  float2 *__restrict__ table) {
    const int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= rows * half) return;
    const int64_t r = idx / half;
    const int i = (int)(idx - r * half);
    const int32_t p = base ? base[r / T] + (int32_t)(r % T) : pos[r];
    const float2 cs = rope_cos_sin(rope_theta(p, i, theta_scale), freq_scale);
    table[idx] = make_float2(cs.x, sin_sign * cs.y);
}

template <typename T, int VEC>
__device__ inline void load_group(const T *row, int d, int64_t sd, float *v) {
    if constexpr (VEC == 1) {
        v[0] = to_f(row[d * sd]);
    } else {
        struct alignas(sizeof(T) * VEC) G {
            T e[VEC];
        };
        const G g = *reinterpret_cast<const G *>(row + d);
#pragma unroll
        for (int j = 0; j < VEC; ++j) v[j] = to_f(g.e[j]);
    }
}

// INLINE: the angles of a.pos instead of a.table.  I: the type that indexes groups and rows (int32_t
// wherever the groups fit: a 64-bit division is about 100 dependent instructions, and a thread makes 8:
// fp16 B4 H32 L1 D128, with the angles' chain in blocks, 5.6 -> 3.9 us).
template <typename T, int VEC, bool INLINE, typename I>
__global__ void __launch_bounds__(256) rope_kernel(RopeArgs a) {
    const I g = (I)blockIdx.x * 256 + (I)threadIdx.x;
    const I gpr = (I)(a.D / VEC), S = (I)a.S, H = (I)a.H;
    __shared__ float2 s_cs[INLINE ? kRopeInlineEntries : 1];
    const I row0 = (I)blockIdx.x * 256 / gpr;  // the workgroup's first row
    if constexpr (INLINE) {
        // the rows' angles, once for all of them when they are at one position
        const I rowl = min((I)blockIdx.x * 256 + 255, (I)(a.ngroups - 1)) / gpr;
        const int n = (S == 1 ? 1 : (int)(rowl - row0 + 1)) * a.half;
        for (int e = threadIdx.x; e < n; e += 256) {
            const I s = (row0 + e / a.half) % S;
            const float2 cs = rope_cos_sin(rope_theta(a.pos[s], e % a.half, a.theta_scale), a.freq_scale);
            s_cs[e] = make_float2(cs.x, a.sin_sign * cs.y);
        }
        __syncthreads();
    }
    if (g >= a.ngroups) return;
    const I row = g / gpr;
    const int d0 = (int)(g - row * gpr) * VEC;
    const I bh = row / S, s = row - bh * S, b = bh / H, h = bh - b * H;
    const T *xr = static_cast<const T *>(a.x) + b * a.sb + h * a.sh + s * a.ss;
    float v[VEC], o[VEC];
    load_group<T, VEC>(xr, d0, a.sd, v);
    // the pairs of this group in order: first, first + 1, ...
    const int first = a.neox ? (d0 < a.half ? d0 : d0 - a.half) : d0 >> 1;
    float2 cs8[VEC];
    if (d0 < a.n_dims) {
        const int np = a.neox ? VEC : (VEC + 1) / 2;
        const float2 *tab = INLINE ? s_cs + (S == 1 ? 0 : (int)(row - row0) * a.half) : a.table + (b * a.tb + s) * a.half;
#pragma unroll
        for (int j = 0; j < VEC; ++j)
            if (j < np) cs8[j] = tab[first + j];
    }
    if (d0 >= a.n_dims) {
#pragma unroll
        for (int j = 0; j < VEC; ++j) o[j] = v[j];
    } else if (!a.neox) {
        if constexpr (VEC == 1) {
            // the pair (d0 & ~1, d0 | 1); n_dims is even, so both are rotated
            float w;
            load_group<T, 1>(xr, d0 ^ 1, a.sd, &w);
            const float2 cs = cs8[0];
            o[0] = (d0 & 1) ? rope_rot_hi(w, v[0], cs) : rope_rot_lo(v[0], w, cs);
        } else {
#pragma unroll
            for (int j = 0; j < VEC; j += 2) {
                const float2 cs = cs8[j >> 1];
                o[j] = rope_rot_lo(v[j], v[j + 1], cs);
                o[j + 1] = rope_rot_hi(v[j], v[j + 1], cs);
            }
        }
    } else {
        const bool lo = d0 < a.half;
        const int pd = lo ? d0 + a.half : d0 - a.half;
        float w[VEC];
        load_group<T, VEC>(xr, pd, a.sd, w);
#pragma unroll
        for (int j = 0; j < VEC; ++j) {
            const float2 cs = cs8[j];
            o[j] = lo ? rope_rot_lo(v[j], w[j], cs) : rope_rot_hi(w[j], v[j], cs);
        }
    }
    T *yr = static_cast<T *>(a.y) + (int64_t)row * a.D + d0;
    if constexpr (VEC == 1) {
        yr[0] = from_f<T>(o[0]);
    } else {
        struct alignas(sizeof(T) * VEC) G {
            T e[VEC];
        };
        G out;
#pragma unroll
        for (int j = 0; j < VEC; ++j) out.e[j] = from_f<T>(o[j]);
        *reinterpret_cast<G *>(yr) = out;
    }
}

template <typename T, int VEC>
hipError_t launch_rotation(RopeArgs a, int64_t numel, hipStream_t stream) {
    a.ngroups = numel / VEC;
    const int64_t blocks = (a.ngroups + 255) / 256;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    const dim3 grid((unsigned)blocks);
    if (blocks * 256 > 0x7fffffffLL) {
        if (a.table) hipLaunchKernelGGL((rope_kernel<T, VEC, false, int64_t>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((rope_kernel<T, VEC, true, int64_t>), grid, dim3(256), 0, stream, a);
    } else {
        if (a.table) hipLaunchKernelGGL((rope_kernel<T, VEC, false, int32_t>), grid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((rope_kernel<T, VEC, true, int32_t>), grid, dim3(256), 0, stream, a);
    }
    return hipGetLastError();
}

// 16-byte groups when every row starts on a group boundary and a group never straddles n_dims
// or (NeoX) the half of the rotated part.
template <typename T>
hipError_t dispatch_rotation(const RopeArgs &a, int64_t numel, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    const bool vec = V > 1 && a.sd == 1 && a.D % V == 0 && a.n_dims % V == 0 && (!a.neox || a.half % V == 0) &&
                     a.sb % V == 0 && a.sh % V == 0 && a.ss % V == 0 && ((uintptr_t)a.x % 16) == 0;
    if constexpr (V > 1) {
        if (vec) return launch_rotation<T, V>(a, numel, stream);
    }
    return launch_rotation<T, 1>(a, numel, stream);
}

}  // namespace

hipError_t gt_launch_rope_table(const int32_t *pos, const int32_t *base, int64_t T, int64_t rows, int n_dims,
                                float theta_scale, float freq_scale, int backward, void *table, hipStream_t stream) {
    const int half = n_dims / 2;
    const int64_t n = rows * half;
    if (n <= 0) return hipSuccess;
    const int64_t blocks = (n + 255) / 256;
    if (blocks > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    hipLaunchKernelGGL(rope_table_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, pos, base, T, rows, half,
                       theta_scale, freq_scale, backward ? -1.0f : 1.0f, (float2 *)table);
    return hipGetLastError();
}

bool gt_rope_inline(int64_t numel, int64_t D) { return D <= kRopeInlineMaxDim && numel / 8 <= kRopeInlineThreads; }

hipError_t gt_launch_rope(const void *x, int dtype, const int64_t *strides, void *y, const void *table,
                          int64_t table_b_stride, int64_t B, int64_t H, int64_t S, int64_t D, int n_dims, int mode,
                          hipStream_t stream, const gt_rope_angles *angles) {
    const int64_t numel = B * H * S * D;
    if (numel <= 0) return hipSuccess;
    RopeArgs a{};
    a.x = x;
    a.sb = strides[0];
    a.sh = strides[1];
    a.ss = strides[2];
    a.sd = strides[3];
    a.y = y;
    a.table = (const float2 *)table;
    if (angles) {
        a.pos = angles->pos;
        a.theta_scale = angles->theta_scale;
        a.freq_scale = angles->freq_scale;
        a.sin_sign = angles->backward ? -1.0f : 1.0f;
    } else if (!table) {
        return hipErrorInvalidValue;
    }
    a.tb = table_b_stride;
    a.H = H;
    a.S = S;
    a.D = D;
    a.n_dims = n_dims;
    a.half = n_dims / 2;
    a.neox = mode == 2;
    switch (dtype) {
        case GT_F32: return dispatch_rotation<float>(a, numel, stream);
        case GT_F16: return dispatch_rotation<_Float16>(a, numel, stream);
        case GT_BF16: return dispatch_rotation<__bf16>(a, numel, stream);
        case GT_F64: return dispatch_rotation<double>(a, numel, stream);
        default: return hipErrorInvalidValue;
    }
}
