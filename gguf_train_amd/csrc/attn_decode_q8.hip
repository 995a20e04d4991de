// Single-query (decode) attention over a GGUF Q8_0 K/V cache, fp16, bf16 or float32 query.
//
// The reference reads a Q8_0 tensor only after gt_dequantize (ggml to_float,
// csrc/gt_core.cpp:800-808: y = qs * d); passed straight to gt_flash_attention it would read
// zeros (csrc/gt_internal.h:243-259).  This kernel computes attention over exactly the
// dequantized values without materialising them: HBM traffic is the 34-byte blocks
// (1.0625 bytes per value), read once per kv head.
//
// Same streaming decomposition as the fp16 decode kernel: workgroup = (kv head of one
// sequence, split), steps of 128 keys with the next step's loads in flight, wave w owns keys
// [32w, 32w + 32) of a step with its own online softmax, one combine at the end, the last split
// merging in the kernel (or a merge launch) when there are several.
//
// Score operands: a lane reads 12 bytes (3 dwords, 4-byte aligned) of one key row in LDS: the 8
// quantized values it needs plus, for the first lane of a block, the block's fp16 scale.  qs
// starts at byte 34j + 2 of block j, 2 mod 4 for even j (the read starts 2 bytes early, on d) and 0
// mod 4 for odd j (the read starts 4 bytes early; d is the high half of the first dword).  A row
// is 34 D/32 bytes, so every read stays inside its row.
//
// fp16 queries.  Exact int8 -> fp16 without a convert per value: for u = qs ^ 0x80 (= qs + 128) the
// fp16 bit pattern 0x6400 | u is exactly 1024 + u = qs + 1152; one v_perm_b32 places two bytes under
// a zero high byte and one xor sets the 0x64 exponent and flips the sign bit.
//   scores: S^T = K . Q^T on v_mfma_f32_16x16x32_f16, one MFMA per 32-value block (the block
//           is the MFMA's k = 32): acc_j = sum (qs + 1152) q = sum qs q + 1152 sum_block q,
//           so s = sum_j d_j (acc_j - 1152 cq_j) with cq_j the block sums of q.
//   P.V:    P' = p d_v rounded to fp16, O^T += V^T . P'^T on the same MFMA; the offset 1152 is
//           removed by one more MFMA per accumulator.
//
// bf16 and float32 queries keep float32 precision throughout on v_mfma_f32_16x16x32_bf16: qs is
// exact in bf16's 8 bits (no offset), a bf16 query is its own operand and a float32 one three
// (hi + mid + lo, 24 bits: split3), and P' = p d_v in float32 enters as three operands as well.
// The products are exact and the sums float32, so only the summation order differs from
// dequantizing to float32 and attending in float32, which is what these calls did before (two
// dequantize passes, then the generic kernel for bf16 and the float32 decode kernel for float32):
// B16 H32/8 S8192 D128 bf16 1399 -> 62 us (4.6 TB/s), float32 469 -> 64 us; B4 S3001 bf16 413 -> 15
// us, float32 51 -> 16 us.  Measured error of float32 queries over that range: 1.8e-7 of the result's
// norm (2.9e-7 before).

#include "attn_common.h"
#include "decode_merge.h"
#include "gt_internal.h"
#include "q8_tile.h"

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>

namespace {

constexpr int kStep = 128;  // keys per step of a workgroup (32 per wave)
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;
constexpr float kMagic = 1152.0f;

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x3 __attribute__((ext_vector_type(3)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a4 __attribute__((aligned(4)));  // a 16-byte load from a 4-byte aligned address
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline float h2f(uint32_t bits16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits16); }
__device__ inline float hlo(uint32_t a) { return (float)__builtin_bit_cast(half2_t, a)[0]; }
__device__ inline float hhi(uint32_t a) { return (float)__builtin_bit_cast(half2_t, a)[1]; }
__device__ inline float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Eight qs bytes of a loaded 12-byte group (`odd`: block index odd, see the header), and the
// raw fp16 scale bits (meaningful in the block's first lane).
__device__ inline void extract12(u32x3 w, bool odd, uint32_t &q0, uint32_t &q1, uint32_t &dbits) {
    if (odd) {
        q0 = w[1];
        q1 = w[2];
        dbits = w[0] >> 16;
    } else {
        q0 = __builtin_amdgcn_alignbyte(w[1], w[0], 2);
        q1 = __builtin_amdgcn_alignbyte(w[2], w[1], 2);
        dbits = w[0] & 0xffffu;
    }
}

// Four bytes u = qs + 128 (the sign bit flipped) -> two packed fp16 0x64uu = 1024 + u = qs + 1152:
// one v_perm_b32 puts two bytes under 0x64 exponent bytes taken from the constant.
constexpr uint32_t kExp64 = 0x64646464u;
constexpr uint32_t kSelLo = 0x04010400u;  // (u.b0, 0x64, u.b1, 0x64)
constexpr uint32_t kSelHi = 0x04030402u;  // (u.b2, 0x64, u.b3, 0x64)
__device__ inline u32x2 magic4(uint32_t u) {
    return u32x2{__builtin_amdgcn_perm(kExp64, u, kSelLo), __builtin_amdgcn_perm(kExp64, u, kSelHi)};
}
constexpr uint32_t kFlip = 0x80808080u;

__device__ inline uint32_t pack_h2(float x, float y) {
    const half2_t v = {(_Float16)x, (_Float16)y};  // round to nearest even
    return __builtin_bit_cast(uint32_t, v);
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

// x = hi + mid + lo, three bf16 operands that together carry float32's 24 bits (each residual is
// exact in float32).  `odd`: some x may be infinite or NaN, and is then its first operand alone.
__device__ inline void split3(const float *x, bool odd, bf16x8_t *out) {
    float r[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = x[e];
#pragma unroll
    for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            out[n][e] = (__bf16)r[e];
            r[e] -= (float)out[n][e];
        }
    if (odd) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const bool fin = fabsf(x[e]) < INFINITY;
            out[1][e] = fin ? out[1][e] : (__bf16)0.0f;
            out[2][e] = fin ? out[2][e] : (__bf16)0.0f;
        }
    }
}

// Two floats that bf16 holds exactly, packed (their high halves).
__device__ inline uint32_t pack_exact(float x, float y) {
    return __builtin_amdgcn_perm(__float_as_uint(y), __float_as_uint(x), 0x07060302u);
}
__device__ inline uint32_t pack_bytes_lo(uint32_t q) {
    return pack_exact((float)(int8_t)(q & 0xffu), (float)(int8_t)((q >> 8) & 0xffu));
}
__device__ inline uint32_t pack_bytes_hi(uint32_t q) {
    return pack_exact((float)(int8_t)((q >> 16) & 0xffu), (float)(int8_t)(q >> 24));
}

// Reductions over lanes l, l ^ 16 and l, l ^ 32 with v_permlane16/32_swap (VALU, no LDS).
__device__ inline float max_x16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float max_x32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
__device__ inline float sum_x16(float v) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ inline float sum_x32(float v) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Each wavefront's 32 K rows and 32 V rows of a step (34 D / 32 bytes each,
// so a step's rows are one contiguous span per tensor) are read with 16-byte loads, 1 KiB per
// instruction, so every request the memory pipeline sees is a whole run of cache lines, and
// written raw into the wave's LDS tile; the next step's loads are in flight in registers while
// this step is computed from LDS.  Operands come from the raw rows:
//   K (scores): the 12-byte windows described at the top, read as dwords;
//   V^T (P.V MFMA A operand): byte e of lane (g = l/16, m = l%16) is row key(g, e) of dim
//     32 blk + 16 h + m, one byte read each, packed as fp16 (qs + 1152) or bf16 (qs);
//   the V block scales are read once per (row, block) into a small table, zero for keys past
//     the end (their rows may be clamped copies).
// v_mfma_f32_16x16x32_{f16,bf16} layouts, lane l: A[m = l%16][k = 8(l/16) + 0..7], B[k = 8(l/16) +
// 0..7][n = l%16], C[m = 4(l/16) + i][n = l%16].  Scores: A = key rows, B = Q^T (the G heads as
// columns), so lane l ends with keys 16kb + 4(l/16) + i of head l%16 and the softmax runs on them in
// registers; P.V: A = V^T, 16 dims x 32 keys, B = P'^T, k-slot e of lane group g being key
// 16(e/4) + 4g + e%4, the probabilities the lane already holds.
// The slices need only be 4-byte aligned: 16-byte loads from such addresses cost what aligned ones
// do (measured with the odd-length shape below), and the one piece that reaches past a slice whose
// size is no multiple of 16 is read 16 bytes before the end and shifted.  A variant that read each
// operand from global memory in 12-byte windows used to serve those slices: fp16 B16 H32/8 S8191
// D128 78.4 -> 62.5 us.
// QT: the query (and output) type.  MASK: 0 = none, 1 = bool bytes, 2 = additive float.
template <typename QT, int D, int G, int MASK>
__global__ __launch_bounds__(256, 2) void decode_q8_lds_kernel(DecodeArgs a) {
    constexpr bool WIDE = !std::is_same<QT, _Float16>::value;   // float32 precision, bf16 operands
    constexpr int NQ = std::is_same<QT, float>::value ? 3 : 1;  // operands of a query
    constexpr int NB = D / 32;                // Q8_0 blocks per row
    constexpr int RB = NB * 34;               // bytes per row
    constexpr int TB = 32 * RB;               // bytes of a wave's 32 rows (a multiple of 16)
    constexpr int NL = (TB + 1023) / 1024;    // 16-byte loads per lane and tile
    constexpr int TAIL = (TB % 1024) / 16;    // lanes of the last load that fall inside the tile (0: all)
    constexpr int SV = NB * 32 / 64;          // V scales read per lane and step
    __shared__ __attribute__((aligned(16))) uint8_t s_raw[4][2][NL * 1024];  // [wave][K, V]
    __shared__ __attribute__((aligned(16))) float s_dv[4][NB][32];       // V scales by row
    __shared__ float s_m[4][G], s_l[4][G];
    static_assert(G * D * 4 <= 2 * NL * 1024, "s_o alias");

    const AttnFwdArgs &f = a.f;
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, q4 = lane >> 4;
    // blockIdx.x = (sequence, kv head, head group), blockIdx.y = split: workgroups are dealt to
    // the XCDs round robin by linear index, so an XCD gets whole (sequence, kv head) slices rather
    // than one split position of every other slice (measured 50.2 against 50.6 us); the kv
    // head's gtot query heads run in groups of G (the last group may hold fewer, gv; its padding
    // columns are blocked)
    const int split = blockIdx.y;
    const int gtot = (int)(f.H / f.Hkv), ngrp = (gtot + G - 1) / G;
    const int64_t bkg = blockIdx.x, bk = bkg / ngrp, b = bk / f.Hkv, hk = bk % f.Hkv;
    const int hg = (int)(bkg % ngrp);
    const int h0 = (int)hk * gtot + hg * G, gv = min(G, gtot - hg * G);
    const int S = (int)f.S;
    const int span = ((S + kStep - 1) / kStep + a.nsplit - 1) / a.nsplit * kStep;
    const int kbeg = split * span, kend = min(attn_decode_end(f, b), kbeg + span);
    const int nsteps = kend > kbeg ? (kend - kbeg + kStep - 1) / kStep : 0;

    // B operand (Q^T): lane holds Q[head h0 + l16][32t + 8 q4 + 0..7]; columns l16 >= gv repeat head
    // h0 + gv - 1 and are discarded
    u32x4 qb[NQ][NB];
    f32x4 c0[NB];  // the score MFMA's initial value; fp16: -1152 x the block sums of each head's query
    {
        const QT *qr = (const QT *)f.q + b * f.q_sb + (h0 + min(l16, gv - 1)) * f.q_sh + 8 * q4;
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            if constexpr (NQ == 3) {
                const f32x4 x0 = *(const f32x4 *)(qr + 32 * t), x1 = *(const f32x4 *)(qr + 32 * t + 4);
                const float x[8] = {x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
                bf16x8_t part[3];
                split3(x, true, part);
#pragma unroll
                for (int n = 0; n < 3; ++n) qb[n][t] = __builtin_bit_cast(u32x4, part[n]);
            } else {
                qb[0][t] = *(const u32x4 *)(qr + 32 * t);
            }
        }
    }
    const half8_t neg_magic = {(_Float16)-kMagic, (_Float16)-kMagic, (_Float16)-kMagic, (_Float16)-kMagic,
                               (_Float16)-kMagic, (_Float16)-kMagic, (_Float16)-kMagic, (_Float16)-kMagic};
#pragma unroll
    for (int t = 0; t < NB; ++t) {
        c0[t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (!WIDE)
            c0[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(neg_magic, __builtin_bit_cast(half8_t, qb[0][t]), c0[t], 0, 0, 0);
    }

    const int64_t slice = (b * f.Hkv + hk) * (int64_t)S * RB;
    const uint8_t *kbase = (const uint8_t *)f.k + slice;
    const uint8_t *vbase = (const uint8_t *)f.v + slice;
    const uint32_t last16 = (uint32_t)S * RB - 16;  // last 16 bytes of the slice
    // the lane's pieces of the wave's K and V tiles of `step` (pieces past the slice read its last
    // piece; lanes of the last load past the tile re-read lane 0's line, adding no requests, and land
    // in the LDS tile's slack, never read)
    u32x4 rk[NL], rv[NL];
    auto load = [&](int step) {
        const uint32_t t0 = (uint32_t)(kbeg + step * kStep + 32 * w) * RB;
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            const bool spare = TAIL != 0 && j == NL - 1 && lane >= TAIL;
            const uint32_t off = gtq8::read_at(t0 + 1024u * j + (spare ? 0u : 16u * lane), last16);
            rk[j] = __builtin_nontemporal_load((const u32x4_a4 *)(kbase + off));
            rv[j] = __builtin_nontemporal_load((const u32x4_a4 *)(vbase + off));
        }
    };
    // the first `sh` dwords of x dropped
    auto shifted = [](u32x4 x, uint32_t sh) {
        return sh == 1 ? u32x4{x[1], x[2], x[3], 0} : sh == 2 ? u32x4{x[2], x[3], 0, 0} : u32x4{x[3], 0, 0, 0};
    };
    auto stage = [&](int step) {
        const uint32_t t0 = (uint32_t)(kbeg + step * kStep + 32 * w) * RB;
        if (gtq8::ends_inside_piece(t0, TB, last16)) {
            // the piece that straddles the end of the slice was read from last16 (t0 is a multiple
            // of 16, the slice's size here is not)
#pragma unroll
            for (int j = 0; j < NL; ++j) {
                const uint32_t early = gtq8::dwords_early(t0 + 1024u * j + 16u * lane, last16);
                if (early) {
                    rk[j] = shifted(rk[j], early);
                    rv[j] = shifted(rv[j], early);
                }
            }
        }
#pragma unroll
        for (int j = 0; j < NL; ++j) {
            *(u32x4 *)&s_raw[w][0][1024 * j + 16 * lane] = rk[j];
            *(u32x4 *)&s_raw[w][1][1024 * j + 16 * lane] = rv[j];
        }
    };

    auto in_row = [](int blk, int part) { return 34 * blk + 8 * part - ((blk & 1) ? 2 : 0); };
    const float cs = f.scale * kLog2e;
    const int64_t mrow = b * f.m_sb + (h0 + min(l16, gv - 1)) * f.m_sh;
    float m = -INFINITY, lsum = 0.0f;
    f32x4 acc[NB][2];
#pragma unroll
    for (int t = 0; t < NB; ++t) acc[t][0] = acc[t][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};

    auto compute = [&](int step) {
        const int k0 = kbeg + step * kStep + 32 * w;
        const uint8_t *kt = s_raw[w][0];
        const uint8_t *vt = s_raw[w][1];
        // ---- V block scales of the step (zero past the end: those rows may be clamped copies) ----
        bool odd = false;  // (WIDE) an infinite or NaN scale among them
#pragma unroll
        for (int j = 0; j < SV; ++j) {
            const int idx = lane + 64 * j, r = idx & 31, t = idx >> 5;
            const float d = h2f(*(const uint16_t *)(vt + r * RB + 34 * t));
            s_dv[w][t][r] = k0 + r < kend ? d : 0.0f;
            if constexpr (WIDE) odd = odd || (k0 + r < kend && !(fabsf(d) < INFINITY));
        }
        if constexpr (WIDE) odd = __builtin_amdgcn_ballot_w64(odd) != 0;
        // ---- scores ----
        // K block scales of the C rows (keys 16 kb + 4 q4 + i): d of block 2p is the low half of the
        // dword at 68 p of the row, d of block 2p + 1 the high half of the dword 32 bytes later
        float dk[2][4][NB];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t *row = (const uint32_t *)(kt + (16 * kb + 4 * q4 + i) * RB);
#pragma unroll
                for (int p2 = 0; p2 < NB / 2; ++p2) {
                    dk[kb][i][2 * p2] = h2f(row[17 * p2] & 0xffffu);
                    dk[kb][i][2 * p2 + 1] = h2f(row[17 * p2 + 8] >> 16);
                }
            }
        u32x4 ka[2][NB];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                const uint32_t *p = (const uint32_t *)(kt + (16 * kb + l16) * RB + in_row(t, q4));
                const u32x3 win = {p[0], p[1], p[2]};
                uint32_t q0, q1, db;
                extract12(win, t & 1, q0, q1, db);
                if constexpr (WIDE) {
                    ka[kb][t] = u32x4{pack_bytes_lo(q0), pack_bytes_hi(q0), pack_bytes_lo(q1), pack_bytes_hi(q1)};
                } else {
                    const u32x2 lo = magic4(q0 ^ kFlip), hi = magic4(q1 ^ kFlip);
                    ka[kb][t] = u32x4{lo[0], lo[1], hi[0], hi[1]};
                }
            }
        float sc[2][4];
        float cm = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            f32x4 sum4 = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                f32x4 c4 = c0[t];
                if constexpr (WIDE) {
                    // the smallest operand first
#pragma unroll
                    for (int n = NQ - 1; n >= 0; --n)
                        c4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ka[kb][t]),
                                                                     __builtin_bit_cast(bf16x8_t, qb[n][t]), c4, 0, 0, 0);
                } else {
                    c4 = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, ka[kb][t]),
                                                                __builtin_bit_cast(half8_t, qb[0][t]), c4, 0, 0, 0);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) sum4[i] = fmaf(dk[kb][i][t], c4[i], sum4[i]);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = k0 + 16 * kb + 4 * q4 + i;
                float x = sum4[i] * cs;
                bool blocked = key >= kend || l16 >= gv;
                if (MASK != 0) {
                    const int64_t mi = mrow + (int64_t)min(key, S - 1) * f.m_ss;
                    if (MASK == 1) blocked = blocked || !((const uint8_t *)f.mask)[mi];
                    else if constexpr (!WIDE) x = fmaf(((const float *)f.mask)[mi], kLog2e, x);
                    else {
                        // a finite value below -FLT_MAX / log2(e) (a mask of the type's lowest value) stays above
                        // -inf: a sequence with no other keys averages their values, as the generic kernel has it
                        const float mv = ((const float *)f.mask)[mi];
                        x = fmaf(mv, kLog2e, x);
                        x = x == -INFINITY && mv != -INFINITY ? -FLT_MAX : x;
                    }
                }
                x = blocked ? -INFINITY : x;
                sc[kb][i] = x;
                cm = fmaxf(cm, x);
            }
        }
        cm = max_x16(cm);
        cm = max_x32(cm);
        const float mnew = fmaxf(m, cm);
        const float msub = mnew == -INFINITY ? 0.0f : mnew;
        const float alpha = mnew == -INFINITY ? 1.0f : fast_exp2(m - mnew);
        m = mnew;
        float ps = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sc[kb][i] = fast_exp2(sc[kb][i] - msub);
                ps += sc[kb][i];
            }
        ps = sum_x16(ps);
        ps = sum_x32(ps);
        lsum = fmaf(lsum, alpha, ps);
        if (__builtin_amdgcn_ballot_w64(alpha != 1.0f) != 0) {
#pragma unroll
            for (int t = 0; t < NB; ++t) {
                acc[t][0] *= alpha;
                acc[t][1] *= alpha;
            }
        }
        // ---- P.V: k-slot e of lane group q4 is key 16(e/4) + 4 q4 + e%4 ----
#pragma unroll
        for (int t = 0; t < NB; ++t) {
            const f32x4 dv0 = *(const f32x4 *)&s_dv[w][t][4 * q4], dv1 = *(const f32x4 *)&s_dv[w][t][16 + 4 * q4];
            const uint8_t *col0 = vt + 34 * t + 2 + l16;
            if constexpr (WIDE) {
                float pv[8];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    pv[i] = sc[0][i] * dv0[i];
                    pv[4 + i] = sc[1][i] * dv1[i];
                }
                if (odd) {
                    // a key of weight 0 (masked) adds nothing whatever its values
#pragma unroll
                    for (int e = 0; e < 8; ++e) pv[e] = sc[e >> 2][e & 3] == 0.0f ? 0.0f : pv[e];
                }
                bf16x8_t bp[3];
                split3(pv, odd, bp);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    float by[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        by[e] = (float)*(const int8_t *)(col0 + 16 * h + (16 * (e >> 2) + 4 * q4 + (e & 3)) * RB);
                    u32x4 av;
#pragma unroll
                    for (int j = 0; j < 4; ++j) av[j] = pack_exact(by[2 * j], by[2 * j + 1]);
#pragma unroll
                    for (int n = 2; n >= 0; --n)
                        acc[t][h] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, av), bp[n],
                                                                            acc[t][h], 0, 0, 0);
                }
            } else {
                u32x4 pw;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    pw[j] = pack_h2(sc[0][2 * j] * dv0[2 * j], sc[0][2 * j + 1] * dv0[2 * j + 1]);
                    pw[j + 2] = pack_h2(sc[1][2 * j] * dv1[2 * j], sc[1][2 * j + 1] * dv1[2 * j + 1]);
                }
                const half8_t bp = __builtin_bit_cast(half8_t, pw);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    uint32_t by[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) by[e] = col0[16 * h + (16 * (e >> 2) + 4 * q4 + (e & 3)) * RB];
                    u32x4 av;
#pragma unroll
                    for (int j = 0; j < 4; ++j) av[j] = (by[2 * j] | (by[2 * j + 1] << 16)) ^ 0x64806480u;
                    acc[t][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, av), bp, acc[t][h],
                                                                       0, 0, 0);
                }
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    acc[t][h] = __builtin_amdgcn_mfma_f32_16x16x32_f16(neg_magic, bp, acc[t][h], 0, 0, 0);
            }
        }
    };

    // The wave's LDS tile holds the step being computed; the registers hold the next one in
    // flight.  Inside the loop the loads are unconditional (clamped) so the compiler's load
    // counters stay exact; the last step is peeled off so that no workgroup fetches the rows
    // past its split (the next split's first step, which another XCD's L2 fetches again).
    // Wave priority follows the step (progress_priority: the two workgroups on a CU stay level).
    if (nsteps > 0) {
        load(0);
        __builtin_amdgcn_s_setprio(3);
        for (int st = 0; st + 1 < nsteps; ++st) {
            progress_priority(st + 1);
            __builtin_amdgcn_wave_barrier();  // the previous step's LDS reads come before the overwrite
            stage(st);
            __builtin_amdgcn_sched_barrier(0);
            load(st + 1);
            __builtin_amdgcn_sched_barrier(0);
            __builtin_amdgcn_wave_barrier();
            compute(st);
        }
        __builtin_amdgcn_wave_barrier();
        stage(nsteps - 1);
        __builtin_amdgcn_wave_barrier();
        compute(nsteps - 1);
    }
    __builtin_amdgcn_s_setprio(3);  // the combine and the merge are the launch's tail

    // ---- combine the four waves (each wave's partial O goes into its own LDS tile) ----
    constexpr int WSTRIDE = 2 * NL * 1024 / 4;  // floats per wave region
    float *my_o = reinterpret_cast<float *>(&s_raw[w][0][0]);
    __builtin_amdgcn_wave_barrier();
    if (lane < G) {
        s_m[w][lane] = m;
        s_l[w][lane] = lsum;
    }
    if (l16 < G) {
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int i = 0; i < 4; ++i) my_o[l16 * D + 32 * t + 16 * h + 4 * q4 + i] = acc[t][h][i];
    }
    __syncthreads();
    const float *o_all = reinterpret_cast<const float *>(&s_raw[0][0][0]);
    for (int e = tid; e < gv * D; e += 256) {
        const int h = e / D, d = e % D;
        const float M = fmaxf(fmaxf(s_m[0][h], s_m[1][h]), fmaxf(s_m[2][h], s_m[3][h]));
        float o = 0.0f, L = 0.0f;
#pragma unroll
        for (int ww = 0; ww < 4; ++ww) {
            const float wg = s_m[ww][h] == -INFINITY ? 0.0f : fast_exp2(s_m[ww][h] - M);
            o = fmaf(wg, o_all[ww * WSTRIDE + h * D + d], o);
            L = fmaf(wg, s_l[ww][h], L);
        }
        const int64_t row = b * f.H + h0 + h;
        if (a.nsplit == 1) {
            ((QT *)f.o)[row * D + d] = (QT)(L > 0.0f ? o / L : 0.0f);
            if (f.lse && d == 0) ((float *)f.lse)[row] = L > 0.0f ? (M + log2f(L)) * kLn2 : INFINITY;
        } else {
            const int64_t pr = row * a.nsplit + split;
            a.part_o[pr * D + d] = o;
            if (d == 0) {
                a.part_ml[pr * 2 + 0] = M;
                a.part_ml[pr * 2 + 1] = L;
            }
        }
    }
    if (a.nsplit > 1 && a.counters) gtdecode::finish_split<QT, D>(a, bkg, b * f.H + h0, gv);
}

template <typename QT, int D>
const void *q8_kernel_d(const AttnFwdArgs &f, int G) {
    const int mode = !f.mask ? 0 : (f.mask_bool ? 1 : 2);
#define GT_QG(GG)                                                     \
    (mode == 0   ? (const void *)decode_q8_lds_kernel<QT, D, GG, 0>   \
     : mode == 1 ? (const void *)decode_q8_lds_kernel<QT, D, GG, 1>   \
                 : (const void *)decode_q8_lds_kernel<QT, D, GG, 2>)
    switch (G) {
        case 1: return GT_QG(1);
        case 2: return GT_QG(2);
        case 4: return GT_QG(4);
        case 8: return GT_QG(8);
        default: return nullptr;
    }
#undef GT_QG
}

// The query and output type is f.out_dtype (the launcher's callers stage the query so).
const void *q8_kernel(const AttnFwdArgs &f) {
    const int G = decode_head_tile(f.H / f.Hkv, kDecodeQ8MaxTile);
    switch (f.out_dtype) {
        case GT_F16: return f.D == 128 ? q8_kernel_d<_Float16, 128>(f, G) : q8_kernel_d<_Float16, 64>(f, G);
        case GT_BF16: return f.D == 128 ? q8_kernel_d<__bf16, 128>(f, G) : q8_kernel_d<__bf16, 64>(f, G);
        case GT_F32: return f.D == 128 ? q8_kernel_d<float, 128>(f, G) : q8_kernel_d<float, 64>(f, G);
        default: return nullptr;
    }
}

// Workgroups of `kernel` the device runs at once (CUs x resident workgroups per CU), cached.
int64_t resident_slots(const void *kernel) {
    static std::mutex mu;
    static std::map<std::pair<int, const void *>, int64_t> cache;
    int dev = 0;
    (void)hipGetDevice(&dev);
    std::lock_guard<std::mutex> lock(mu);
    auto it = cache.find({dev, kernel});
    if (it != cache.end()) return it->second;
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, kernel, 256, 0) != hipSuccess || per <= 0) per = 2;
    const int64_t slots = (int64_t)cus * per;
    cache[{dev, kernel}] = slots;
    return slots;
}

}  // namespace

// The merge kernel is shared with the fp16 decode path.
hipError_t launch_attn_decode_merge(const DecodeArgs &a, int out_dtype, hipStream_t s);

int attn_decode_q8_splits(const AttnFwdArgs &f) {
    const void *kernel = q8_kernel(f);
    const int64_t slots = kernel ? resident_slots(kernel) : 512;
    const int64_t steps = (f.S + kStep - 1) / kStep;
    return decode_split_count(decode_units(f.B, f.H, f.Hkv, kDecodeQ8MaxTile), steps, slots, std::min<int64_t>(64, steps));
}

bool attn_decode_q8_supported(const AttnFwdArgs &f, int q_dtype) {
    if ((q_dtype != GT_F16 && q_dtype != GT_BF16 && q_dtype != GT_F32) || f.out_dtype != q_dtype) return false;
    if (f.L != 1 || f.S <= 0 || f.D != f.Dv || (f.D != 64 && f.D != 128)) return false;
    if (f.S >= (1LL << 30) || f.S * (f.D / 32 * 34) > 0xffffffffLL) return false;  // 32-bit offsets
    // any number of query heads per kv head, in groups of up to 8
    if (decode_units(f.B, f.H, f.Hkv, kDecodeQ8MaxTile) > 65535) return false;
    const int64_t q16 = q_dtype == GT_F32 ? 4 : 8;  // query rows start 16-byte aligned
    if (f.q_sh % q16 != 0 || f.q_sb % q16 != 0 || (uintptr_t)f.q % 16 != 0) return false;
    // K/V are whole dense Q8_0 tensors.  The kernel's reads need 4-byte alignment; bases off 8 bytes keep the
    // dequantizing path, which gt_flash_attention_noalloc refuses (allocations and the tensors of a GGUF
    // file start at 32 bytes or more)
    for (const void *p : {f.k, f.v}) if ((uintptr_t)p % 8 != 0) return false;
    return true;
}

hipError_t launch_attn_decode_q8(const DecodeArgs &a, hipStream_t s) {
    const void *kernel = q8_kernel(a.f);
    if (!kernel) return hipErrorInvalidValue;
    const unsigned units = (unsigned)decode_units(a.f.B, a.f.H, a.f.Hkv, kDecodeQ8MaxTile);
    const dim3 grid(units, (unsigned)a.nsplit);
    void *args[] = {(void *)&a};
    hipError_t e = hipLaunchKernel(kernel, grid, dim3(256), args, 0, s);
    // one split, or the last split merged in the kernel: the kernel wrote the output
    if (e != hipSuccess || a.nsplit == 1 || a.counters) return e;
    return launch_attn_decode_merge(a, a.f.out_dtype, s);
}
