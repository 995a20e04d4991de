// Recompute-based attention backward on gfx950 MFMA (fp16 / bf16 inputs, fp32 gradients).
//
// Replaces the reference's Python composition (gguf_train/_functions.py:1933-1965), which
// materialises (B,H,L,S) scores, probabilities and their gradients, with two kernels that
// keep everything in registers and LDS and recompute P from the forward's log-sum-exp:
//   dQ:     the forward's structure (a workgroup owns 128 query rows, loops over key tiles);
//           each row first forms D_q = sum_d dO[q,d] * O[q,d] (= sum_s P[q,s] dP[q,s], the
//           rowsum in dS) and writes it for dK/dV, which runs after it:
//             S^T = K.Q^T, dP^T = V.dO^T, dS^T as below, dQ^T += K^T.dS^T
//   dK/dV:  a workgroup owns 128 keys of one kv head (32 per wavefront, K and V rows held in
//           registers) and walks over the query tiles of every query head of its GQA group:
//             S = Q.K^T, dP = dO.V^T          (keys on lanes: the accumulator layout)
//             P = exp2(S*scale*log2e - lse*log2e), dS = P * (dP - D_q)
//             dV += P^T.dO, dK += dS^T.Q      (P, dS feed the MFMA A operand in place; dO and Q
//                                              are read transposed from row-major LDS tiles)
// Gradients leave as float32 or, for a caller that would round them to the inputs' dtype anyway
// (g_half), in that dtype: the same bits without a float32 round trip through HBM (three
// elementwise passes of 8.3 us in the training step bf16 B8 H16 L=S=1024 D64: 199 -> 180 us).
// dK and dV of a GQA group are summed in registers (no atomics).  P and dS are split into hi +
// lo operands so the products keep ~16 bits (bf16) or ~22 (fp16): a single fp16 operand's 2^-12
// rounding accumulates in dV and dK, whose sums run over query rows (measured 1.27x the 2e-3
// bar on fp16 dV), and dQ follows the same rule.  Masks: top-left causal,
// bool / additive (read per element; an additive mask that does not depend on the query row is
// read once per key: per head in dK/dV, staged with the K/V tile in dQ), keys >= S and
// queries >= L contribute nothing.
// Dropout (DROP): dV += (P*m)^T.dO and dP = m * dO.V^T in dS = P * (dP - delta), m the
// element's multiplier (gt_philox.h).  dQ draws its lanes' Philox blocks directly (4 consecutive
// keys of one query per block, as the forward) and writes the decisions as bits, one word per
// (query row, 32 keys); dK/dV, whose lanes hold 16 queries of one key, streams those words in
// with each query step (64 rows x 4 words through LDS) instead of drawing again.  Without that
// buffer (a.dbits null: the caller bounds its size) each dK/dV thread draws its word itself, 8
// Philox blocks per step.
// Head sizes 80 and 96: tile rows of 96 values (PD).  With D = 80 the last 16 of a row repeat its dims 72
// .. 79: S and dP take D / 16 k-steps and do not read them, and the gradients' columns past D, formed in
// accumulators of their own, are not stored.
#pragma once

#include "attn_common.h"
#include "gt_internal.h"
#include "mfma_util.h"
#include "lds_dma.h"

#include <cmath>
#include <type_traits>

namespace {

using namespace gtmfma;

constexpr int BKV = 128;  // keys per dK/dV workgroup (32 per wavefront)
constexpr int BQ = 64;    // query rows per dK/dV step
constexpr int BMQ = 128;  // query rows per dQ workgroup (32 per wavefront)
constexpr int BNK = 64;   // key rows per dQ step
template <int D>
constexpr int pd_of() { return (D + 31) / 32 * 32; }  // values per tile row: whole 32-column blocks

// x * y rounded to float32: kept in a register, or the compiler would fuse the product with a
// conversion to float16 (v_fma_mix), whose single rounding differs from the float32 gradient's
__device__ inline float scaled(float x, float y) {
    float v = x * y;
    asm("" : "+v"(v));
    return v;
}

// ---- dK, dV ----------------------------------------------------------------------------------

// D = 64 fits two wavefronts per SIMD without spills (with one, the compiler parks values in
// AGPRs and moves them back and forth); D = 128 needs the whole register file.  (Dropout with the
// key-padding row spills ~60 bytes per lane at two per SIMD and is still faster there: 255 against
// 285 us for the training step with dropout.)
template <typename T, int D, bool CAUSAL, int MASK, bool DROP = false>
__global__ __launch_bounds__(256, D <= 64 ? 2 : 1) void bwd_dkdv_kernel(AttnBwdArgs a) {
    using M = Mfma<T>;
    using V8 = typename M::V8;
    constexpr int PD = pd_of<D>(), DT = D / 16, DB = PD / 32, CH = PD / 8;
    constexpr int QP = PD + 16;             // Q / dO tile pitch (transposed reads)
    constexpr int NLD = BQ * CH / 256;      // 16-byte loads per thread per tile and operand
    static_assert(NLD >= 1, "tile split over the threads");
    __shared__ __attribute__((aligned(16))) T sQ[2][BQ * QP];
    __shared__ __attribute__((aligned(16))) T sG[2][BQ * QP];  // dO
    __shared__ __attribute__((aligned(16))) float sL[2][BQ];    // lse * log2(e)
    __shared__ __attribute__((aligned(16))) float sD[2][BQ];    // -delta
    // dropout: word [w][r] = decisions of keys k0 + 32w .. +31 for query qs0 + r (bit j: key 32w + j)
    __shared__ __attribute__((aligned(16))) uint32_t sDm[DROP ? 2 : 1][DROP ? 4 * BQ : 1];

    const AttnFwdArgs &f = a.f;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lrow = lane & 31, half = lane >> 5;
    const int g16 = lane >> 4, i16 = lane & 15;
    // Key tile major: all workgroups of key tile 0 first.  Under the causal mask tile kt walks
    // the queries from k0 on, so the heaviest workgroups start first and the short ones fill
    // the tail (list scheduling over two rounds of B*Hkv*nkt = 1024 workgroups on 512 slots:
    // makespan 18 steps instead of 28 with key tiles interleaved).  The tiles of one (b, kv
    // head) sit B*Hkv apart, on the same XCD when B*Hkv % 8 == 0.
    const int64_t nbk = f.B * f.Hkv;
    const int kt = (int)(blockIdx.x / nbk);
    const int64_t bk = blockIdx.x % nbk, b = bk / f.Hkv, hk = bk % f.Hkv;
    const int G = (int)(f.H / f.Hkv);
    const int L = (int)f.L, S = (int)f.S;
    const int k0 = kt * BKV, wk0 = k0 + 32 * w, key = wk0 + lrow;  // this lane's key (n index)
    const float c = f.scale * kLog2e, inv_scale = 1.0f / f.scale;
    const float dscale = DROP ? (float)f.drop.scale : 1.0f;
    const int64_t dwords = (f.S + 31) / 32;  // decision words per query row

    // K and V rows of this lane's key as B operands (B[k = d][n = key])
    V8 kf[DT], vf[DT];
    {
        const int kk = min(key, S - 1);
        const T *kr = (const T *)f.k + b * f.k_sb + hk * f.k_sh + (int64_t)kk * f.k_ss + 8 * half;
        const T *vr = (const T *)f.v + b * f.v_sb + hk * f.v_sh + (int64_t)kk * f.v_ss + 8 * half;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            kf[t] = __builtin_bit_cast(V8, *(const u32x4 *)(kr + 16 * t));
            vf[t] = __builtin_bit_cast(V8, *(const u32x4 *)(vr + 16 * t));
        }
        // Wait for K and V here: otherwise the compiler's wait for these loads lands inside the
        // loop, where (vector memory loads completing in order) it also waits for every Q / dO
        // prefetch issued since, exposing the full global load latency on every step.
#pragma unroll
        for (int t = 0; t < DT; ++t) asm volatile("" ::"v"(kf[t]), "v"(vf[t]));
    }
    f32x16 dk[DB], dv[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dk[db][i] = dv[db][i] = 0.0f;

    // the query steps: every query head of the group, queries that can see a key of this tile
    const int qstart = CAUSAL ? (k0 / BQ) * BQ : 0;
    const int nqs = L > qstart ? (L - qstart + BQ - 1) / BQ : 0;
    const int nsteps = nqs * G;

    u32x4 qreg[NLD], greg[NLD];
    float lreg = 0.0f, dreg = 0.0f;
    uint32_t mreg = 0u;  // dropout: this thread's decision word of the step
    auto load_step = [&](int st) {
        const int hh = st / nqs, qs0 = qstart + (st % nqs) * BQ;
        const int64_t h = hk * G + hh;
        const T *qb = (const T *)f.q + b * f.q_sb + h * f.q_sh;
        const T *gb = (const T *)a.dout + ((b * f.H + h) * f.L) * D;
        if constexpr (DROP) {
            // thread t: row t % 64 of the step, key word t / 64 of the tile (words past the
            // sequence's keys repeat the last one: their keys have P = 0)
            const int r = tid % BQ, wd = min((int)(k0 / 32 + tid / BQ), (int)dwords - 1);
            const int64_t row = (b * f.H + h) * f.L + min(qs0 + r, L - 1);
            if (a.dbits) {
                mreg = a.dbits[row * dwords + wd];
            } else {
                const uint64_t n0 = (uint64_t)row * (uint64_t)((f.S + 3) / 4) + (uint64_t)(8 * wd);
                uint32_t word = 0u;
#pragma unroll 2
                for (int u = 0; u < 8; ++u) {
                    const GtWord4 x = gt_philox4x32_10(n0 + u, f.drop.offset, f.drop.seed);
#pragma unroll
                    for (int e = 0; e < 4; ++e) word |= (x.w[e] < f.drop.thresh ? 1u : 0u) << (4 * u + e);
                }
                mreg = word;
            }
        }
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int cidx = tid + 256 * i, row = cidx / CH, col = cidx % CH;
            const int q = min(qs0 + row, L - 1), at = 8 * min(col, D / 8 - 1);
            qreg[i] = *(const u32x4 *)(qb + (int64_t)q * f.q_sl + at);
            greg[i] = *(const u32x4 *)(gb + (int64_t)q * D + at);
        }
        if (tid < BQ) {
            // raw values: the arithmetic waits for the loads, so it happens at store time
            const int64_t r = (b * f.H + h) * f.L + min(qs0 + tid, L - 1);
            lreg = ((const float *)f.lse)[r];
            dreg = ((const float *)a.delta)[r];
        }
    };
    auto store_step = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int cidx = tid + 256 * i, row = cidx / CH, col = cidx % CH;
            *(u32x4 *)&sQ[buf][row * QP + 8 * col] = qreg[i];
            *(u32x4 *)&sG[buf][row * QP + 8 * col] = greg[i];
        }
        if (tid < BQ) {
            sL[buf][tid] = lreg * kLog2e;  // lse * log2(e)
            sD[buf][tid] = -dreg;          // -delta
        }
        if constexpr (DROP) sDm[buf][tid] = mreg;  // [tid / 64][tid % 64]
    };

    if (nsteps > 0) {
        load_step(0);
        store_step(0);
        if (nsteps > 1) load_step(1);
    }
    __syncthreads();
    // The first S and dP products accumulate onto (the key's mask term, -delta of each query):
    // S then holds QK^T + mask and dP holds dO.V^T - delta, with no per-element adds.
    f32x16 sinit;  // MASK 4: the mask value of this lane's key for the current head (raw units)
#pragma unroll
    for (int i = 0; i < 16; ++i) sinit[i] = 0.0f;
    for (int st = 0; st < nsteps; ++st) {
        const int buf = st & 1;
        const int hh = st / nqs, qs0 = qstart + (st % nqs) * BQ;
        if constexpr (D <= 64) progress_priority(st);  // two workgroups per CU
        const int64_t h = hk * G + hh;
        const T *cQ = sQ[buf];
        const T *cG = sG[buf];
        if (MASK == 4 && st % nqs == 0) {
            const float madd =
                ((const float *)f.mask)[b * f.m_sb + h * f.m_sh + (int64_t)min(key, S - 1) * f.m_ss] * inv_scale;
#pragma unroll
            for (int i = 0; i < 16; ++i) sinit[i] = madd;
        }
#pragma unroll
        for (int qb = 0; qb < 2; ++qb) {
            const int q0 = qs0 + 32 * qb;
            if (CAUSAL && q0 + 31 < wk0) continue;  // every query of the block precedes our keys
            // MASK 1 / 2: this lane's 16 mask values of the block (query q0 + 4half + c, c = 8(i/4) +
            // i%4), loaded before the S and dP products so that they land during them; the loads
            // are unconditional (no branch, no wait per element), an invisible element reading
            // the lane's key in the last query row instead
            constexpr bool MFULL = MASK == 1 || MASK == 2;
            float madd[MASK == 2 ? 16 : 1];
            uint32_t mbyte[MASK == 1 ? 16 : 1];
            if constexpr (MFULL) {
                const int64_t mkey = b * f.m_sb + h * f.m_sh + (int64_t)min(key, S - 1) * f.m_ss;
                const int64_t mlane = mkey + (int64_t)(q0 + 4 * half) * f.m_sl;
                const int64_t msafe = mkey + (int64_t)(L - 1) * f.m_sl;
                int lo = (CAUSAL ? key : 0) - (q0 + 4 * half);
                int span = (L - 1 - (q0 + 4 * half)) - lo;
                if (key >= S || span < 0) {
                    lo = 32;
                    span = 0;
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int cq = 8 * (i / 4) + (i % 4);
                    const int64_t mi = (uint32_t)(cq - lo) <= (uint32_t)span ? mlane + (int64_t)cq * f.m_sl : msafe;
                    if constexpr (MASK == 2) madd[i] = ((const float *)f.mask)[mi];
                    else mbyte[i] = ((const uint8_t *)f.mask)[mi];
                }
            }
            // s[i], dp[i]: query q0 + 8(i/4) + 4half + i%4, key `key`
            // (dropout: dP starts at 0, -delta is added after the multiplier)
            f32x16 s, dp;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 d4 = *(const f32x4 *)&sD[buf][32 * qb + 8 * g + 4 * half];
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[4 * g + e] = DROP ? 0.0f : d4[e];
            }
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const V8 qa = *(const V8 *)&cQ[(32 * qb + lrow) * QP + 16 * t + 8 * half];
                const V8 ga = *(const V8 *)&cG[(32 * qb + lrow) * QP + 16 * t + 8 * half];
                s = M::mma(qa, kf[t], t == 0 ? sinit : s);
                dp = M::mma(ga, vf[t], dp);
            }
            float p[16], ds[16];
            // every (query, key) of the block visible and no per-element mask: no tests
            const bool interior = (MASK == 0 || MASK == 4) && wk0 + 31 < S && q0 + 31 < L && (!CAUSAL || q0 >= wk0 + 31);
            // dropout: multiplier of entry i (query 32qb + 8(i/4) + 4half + i%4 of the step, this
            // lane's key 32w + lrow of the tile): bit lrow of word [w][query]
            uint32_t dbits = 0u;  // bit i: entry i kept
            if constexpr (DROP) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const u32x4 dw = *(const u32x4 *)&sDm[buf][w * BQ + 32 * qb + 8 * g + 4 * half];
#pragma unroll
                    for (int e = 0; e < 4; ++e) dbits |= ((dw[e] >> lrow) & 1u) << (4 * g + e);
                }
            }
            auto mult = [&](int i) { return (dbits >> i) & 1u ? dscale : 0.0f; };
            if constexpr (DROP) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 d4 = *(const f32x4 *)&sD[buf][32 * qb + 8 * g + 4 * half];
#pragma unroll
                    for (int e = 0; e < 4; ++e) dp[4 * g + e] = fmaf(dp[4 * g + e], mult(4 * g + e), d4[e]);  // m dO.V - delta
                }
            }
            if (interior) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int qi = 32 * qb + 8 * g + 4 * half;
                    const f32x4 l4 = *(const f32x4 *)&sL[buf][qi];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 4 * g + e;
                        const float pv = fast_exp2(fmaf(s[i], c, -l4[e]));
                        p[i] = DROP ? pv * mult(i) : pv;
                        ds[i] = pv * dp[i];
                    }
                }
            } else {
                // query q0 + 4half + c (c = 8(i/4) + i%4) sees this lane's key when lo <= c <= lo + span
                // (key < S, q < L, causal q >= key), as one unsigned compare per score; a
                // per-element mask is read only there, at this lane's offset plus c rows
                int lo = (CAUSAL ? key : 0) - (q0 + 4 * half);
                int span = (L - 1 - (q0 + 4 * half)) - lo;
                if (key >= S || span < 0) {
                    lo = 32;  // no c in 0..27 passes
                    span = 0;
                }
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int qi = 32 * qb + 8 * g + 4 * half;  // 4 consecutive queries
                    const f32x4 l4 = *(const f32x4 *)&sL[buf][qi];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int i = 4 * g + e;
                        float add = 0.0f;  // MASK 4: already in s
                        bool ok = (uint32_t)(8 * g + e - lo) <= (uint32_t)span;
                        if constexpr (MASK == 1) ok = ok && mbyte[i] != 0u;
                        else if constexpr (MASK == 2) add = madd[i] * inv_scale;
                        const float pv = ok ? fast_exp2(fmaf(s[i] + add, c, -l4[e])) : 0.0f;
                        p[i] = DROP ? pv * mult(i) : pv;
                        ds[i] = pv * dp[i];
                    }
                }
            }
            // P and dS as hi + lo operands for both types: dV and dK sum a key's terms over every
            // query row, so the rounding of a single fp16 operand grows with P's column sums (a
            // causal key 0 collects P of every row: measured 1.27x the 2e-3 bar on fp16 dV)
            V8 pa[2], pal[2], da[2], dal[2];
#pragma unroll
            for (int hs = 0; hs < 2; ++hs) {
                pack8_hilo<T>(p + 8 * hs, pa[hs], pal[hs]);
                pack8_hilo<T>(ds + 8 * hs, da[hs], dal[hs]);
            }
#pragma unroll
            for (int db = 0; db < DB; ++db) {
#pragma unroll
                for (int hs = 0; hs < 2; ++hs) {
                    const int row = 32 * qb + 16 * hs + 4 * (g16 >> 1) + (i16 >> 2);
                    const int col = 32 * db + 16 * (g16 & 1) + 4 * (i16 & 3);
                    const V8 gt = read_tr8<T>(&cG[row * QP + col], &cG[(row + 8) * QP + col]);
                    const V8 qt = read_tr8<T>(&cQ[row * QP + col], &cQ[(row + 8) * QP + col]);
                    dv[db] = M::mma(pa[hs], gt, dv[db]);
                    dk[db] = M::mma(da[hs], qt, dk[db]);
                    dv[db] = M::mma(pal[hs], gt, dv[db]);
                    dk[db] = M::mma(dal[hs], qt, dk[db]);
                }
            }
        }
        if (st + 1 < nsteps) {
            store_step(buf ^ 1);
            if (st + 2 < nsteps) load_step(st + 2);
        }
        __syncthreads();
    }

    // dK[key][d] (scaled) and dV[key][d]: accumulator row = key wk0 + 8(i/4) + 4half + i%4, column d
    auto store = [&](auto *dkp, auto *dvp) {
        using TG = std::remove_reference_t<decltype(*dkp)>;
#pragma unroll
        for (int db = 0; db < DB; ++db) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int kr = wk0 + 8 * (i / 4) + 4 * half + (i % 4);
                if (kr < S && (D % 32 == 0 || 32 * db + lrow < D)) {
                    dkp[(int64_t)kr * D + 32 * db + lrow] = (TG)scaled(dk[db][i], f.scale);
                    dvp[(int64_t)kr * D + 32 * db + lrow] = (TG)dv[db][i];
                }
            }
        }
    };
    const int64_t base = bk * f.S * D;
    if (a.g_half) store((T *)a.dk + base, (T *)a.dv + base);
    else store((float *)a.dk + base, (float *)a.dv + base);
}

// ---- dQ --------------------------------------------------------------------------------------

// (two per SIMD for D = 64 as in dK/dV, except with a per-element mask, which would spill)
// MASK 5 / 6: bool / float per-element mask with contiguous keys and 4-key aligned rows, read
// as a lane's 4 consecutive keys per load at the start of the tile (as the forward).
template <typename T, int D, bool CAUSAL, int MASK, bool DROP = false>
__global__ __launch_bounds__(256, D <= 64 && (MASK == 0 || MASK == 4) ? 2 : 1) void bwd_dq_kernel(AttnBwdArgs a, int nq) {
    using M = Mfma<T>;
    using V8 = typename M::V8;
    constexpr int PD = pd_of<D>(), DT = D / 16, DB = PD / 32, CH = PD / 8;
    constexpr int KP = PD + 16;  // K tile: row reads and transposed reads
    constexpr int VP = PD + 8;  // V tile: row reads
    constexpr int NLD = BNK * CH / 256;
    __shared__ __attribute__((aligned(16))) T sK[2][BNK * KP];
    __shared__ __attribute__((aligned(16))) T sV[2][BNK * VP];
    __shared__ __attribute__((aligned(16))) float sMk[MASK == 4 ? 2 : 1][BNK];  // MASK 4: the tile's mask row

    const AttnFwdArgs &f = a.f;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int lrow = lane & 31, half = lane >> 5;
    const int g16 = lane >> 4, i16 = lane & 15;
    const int64_t BH = f.B * f.H;
    const int qt = nq - 1 - (int)(blockIdx.x / BH);
    const int64_t bh = (int64_t)blockIdx.x % BH;
    const int64_t b = bh / f.H, h = bh % f.H, hk = h / (f.H / f.Hkv);
    const int L = (int)f.L, S = (int)f.S;
    const int q0 = qt * BMQ, wq0 = q0 + 32 * w, lq = wq0 + lrow;
    const int lqc = min(lq, L - 1);
    const float c = f.scale * kLog2e, inv_scale = 1.0f / f.scale;
    const float dscale = DROP ? (float)f.drop.scale : 1.0f;
    // dropout: Philox block of keys 0..3 of this lane's row
    const uint64_t drow = DROP ? (uint64_t)(bh * f.L + lq) * (uint64_t)((f.S + 3) / 4) : 0;

    V8 qf[DT], gf[DT];
    {
        const T *qr = (const T *)f.q + b * f.q_sb + h * f.q_sh + (int64_t)lqc * f.q_sl + 8 * half;
        const T *gr = (const T *)a.dout + (bh * f.L + lqc) * D + 8 * half;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            qf[t] = __builtin_bit_cast(V8, *(const u32x4 *)(qr + 16 * t));
            gf[t] = __builtin_bit_cast(V8, *(const u32x4 *)(gr + 16 * t));
        }
    }
    const float lse2 = ((const float *)f.lse)[bh * f.L + lqc] * kLog2e;
    // delta = rowsum(dO * O) of this lane's query (the two lanes of a row each hold half of it;
    // O is the training forward's float32 output when given, else the rounded one), written for
    // the dK/dV kernel that runs next; dP accumulates onto -delta (no per-element subtract)
    f32x16 dinit;
    float dlt;
    {
        float part = 0.0f;
        if (a.o_f32) {
            const float *orow = (const float *)f.o + (bh * f.L + lqc) * D + 8 * half;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const f32x4 o0 = *(const f32x4 *)(orow + 16 * t), o1 = *(const f32x4 *)(orow + 16 * t + 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    part = fmaf((float)gf[t][e], o0[e], part);
                    part = fmaf((float)gf[t][e + 4], o1[e], part);
                }
            }
        } else {
            const T *orow = (const T *)f.o + (bh * f.L + lqc) * D + 8 * half;
#pragma unroll
            for (int t = 0; t < DT; ++t) {
                const V8 ov = __builtin_bit_cast(V8, *(const u32x4 *)(orow + 16 * t));
#pragma unroll
                for (int e = 0; e < 8; ++e) part = fmaf((float)gf[t][e], (float)ov[e], part);
            }
        }
        dlt = xhalf_sum(part);
        if (half == 0 && lq < L) ((float *)a.delta)[bh * f.L + lq] = dlt;
        // (dropout: dP starts at 0, -delta is added after the multiplier)
#pragma unroll
        for (int i = 0; i < 16; ++i) dinit[i] = DROP ? 0.0f : -dlt;
    }

    f32x16 dq[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) dq[db][i] = 0.0f;

    const T *kbase = (const T *)f.k + b * f.k_sb + hk * f.k_sh;
    const T *vbase = (const T *)f.v + b * f.v_sb + hk * f.v_sh;
    const int kv_end = CAUSAL ? min(q0 + BMQ, S) : S;
    const int ntiles = (kv_end + BNK - 1) / BNK;
    u32x4 kreg[NLD], vreg[NLD];
    float mreg = 0.0f;
    const float *mrow = MASK == 4 ? (const float *)f.mask + b * f.m_sb + h * f.m_sh : nullptr;
    auto load_tile = [&](int j) {
        // the raw mask value: scaled at store time, so that nothing waits for the load here
        if (MASK == 4 && tid < BNK) mreg = mrow[(int64_t)min(j * BNK + tid, S - 1) * f.m_ss];
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int cidx = tid + 256 * i, row = cidx / CH, col = cidx % CH;
            const int kk = min(j * BNK + row, S - 1), at = 8 * min(col, D / 8 - 1);
            kreg[i] = *(const u32x4 *)(kbase + (int64_t)kk * f.k_ss + at);
            vreg[i] = *(const u32x4 *)(vbase + (int64_t)kk * f.v_ss + at);
        }
    };
    auto store_tile = [&](int buf) {
        if (MASK == 4 && tid < BNK) sMk[buf][tid] = mreg * inv_scale;
#pragma unroll
        for (int i = 0; i < NLD; ++i) {
            const int cidx = tid + 256 * i, row = cidx / CH, col = cidx % CH;
            *(u32x4 *)&sK[buf][row * KP + 8 * col] = kreg[i];
            *(u32x4 *)&sV[buf][row * VP + 8 * col] = vreg[i];
        }
    };

    if (ntiles > 0) {
        load_tile(0);
        store_tile(0);
        if (ntiles > 1) load_tile(1);
    }
    __syncthreads();
    for (int j = 0; j < ntiles; ++j) {
        const int buf = j & 1, k0 = j * BNK;
        if constexpr (D <= 64) progress_priority(j);  // two workgroups per CU with MASK 0 / 4 (one otherwise: no effect)
        const T *cK = sK[buf];
        const T *cV = sV[buf];
        if (!CAUSAL || k0 <= wq0 + 31) {
            // MASK 5 / 6: keys k0 + 32kb + 8g + 4half + 0..3 of this lane's row (starts past
            // the last 4 keys read those: their scores are blocked)
            constexpr bool MVEC = MASK >= 5;
            f32x4 mvf[MASK == 6 ? 2 : 1][4];
            uint32_t mvb[MASK == 5 ? 2 : 1][4];
            if constexpr (MVEC) {
                const int64_t mrb = b * f.m_sb + h * f.m_sh + (int64_t)lqc * f.m_sl;
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const int64_t at = mrb + min(k0 + 32 * kb + 8 * g + 4 * half, S - 4);
                        if constexpr (MASK == 5) mvb[kb][g] = *(const uint32_t *)((const uint8_t *)f.mask + at);
                        else mvf[kb][g] = *(const f32x4 *)((const float *)f.mask + at);
                    }
            }
            // s[kb][i]: key k0 + 32kb + 8(i/4) + 4half + i%4, query lq.  S accumulates onto the
            // tile's mask row (MASK 4: the keys' additive terms), dP onto -delta.
            f32x16 s[2], dp[2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                f32x16 sinit;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 mv = MASK == 4 ? *(const f32x4 *)&sMk[buf][32 * kb + 8 * g + 4 * half]
                                               : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                    for (int e = 0; e < 4; ++e) sinit[4 * g + e] = mv[e];
                }
#pragma unroll
                for (int t = 0; t < DT; ++t) {
                    const V8 ka = *(const V8 *)&cK[(32 * kb + lrow) * KP + 16 * t + 8 * half];
                    const V8 va = *(const V8 *)&cV[(32 * kb + lrow) * VP + 16 * t + 8 * half];
                    s[kb] = M::mma(ka, qf[t], t == 0 ? sinit : s[kb]);
                    dp[kb] = M::mma(va, gf[t], t == 0 ? dinit : dp[kb]);
                }
            }
            V8 sb[2][2], sl[2][2];
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                float ds[16];
                // every (query, key) of the block visible and no per-element mask: no tests
                const int kb0 = k0 + 32 * kb;
                if constexpr (DROP) {
                    // entries 4g .. 4g+3: keys kb0 + 8g + 4half + 0..3, one Philox block; the
                    // decisions also go out as bit 8g + 4half + e of the (row, 32 keys) word
                    uint32_t bits = 0u;
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        const GtWord4 x = gt_philox4x32_10(drow + (uint64_t)((kb0 + 8 * g + 4 * half) >> 2),
                                                           f.drop.offset, f.drop.seed);
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const bool keep = x.w[e] < f.drop.thresh;
                            bits |= (keep ? 1u : 0u) << (8 * g + 4 * half + e);
                            dp[kb][4 * g + e] = fmaf(dp[kb][4 * g + e], keep ? dscale : 0.0f, -dlt);
                        }
                    }
                    const auto r = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
                    if (a.dbits && half == 0 && lq < L && kb0 < S)
                        a.dbits[(bh * f.L + lq) * ((f.S + 31) / 32) + kb0 / 32] = r[0] | r[1];
                }
                const bool interior =
                    (MASK == 0 || MASK == 4) && kb0 + 31 < S && wq0 + 31 < L && (!CAUSAL || wq0 >= kb0 + 31);
                if (interior) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) ds[i] = fast_exp2(fmaf(s[kb][i], c, -lse2)) * dp[kb][i];
                } else {
                    // key kb0 + 4half + c (c = 8(i/4) + i%4) is visible to this lane's row when c <= vis
                    const int vis = (lq < L ? (CAUSAL ? min(lq, S - 1) : S - 1) : -1) - (kb0 + 4 * half);
                    // per-element mask: this lane's offset plus c keys where visible, else the
                    // lane's row at the last key (unconditional loads: no branch per element)
                    const int64_t mrow0 = b * f.m_sb + h * f.m_sh + (int64_t)lqc * f.m_sl;
                    const int64_t mlane = mrow0 + (int64_t)(kb0 + 4 * half) * f.m_ss;
                    const int64_t msafe = mrow0 + (int64_t)(S - 1) * f.m_ss;
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        float add = 0.0f;  // MASK 4: already in s
                        const int ck = 8 * (i / 4) + (i % 4);
                        bool ok = ck <= vis;
                        if constexpr (MASK == 1 || MASK == 2) {
                            const int64_t mi = ok ? mlane + (int64_t)ck * f.m_ss : msafe;
                            if constexpr (MASK == 1) ok = ok && ((const uint8_t *)f.mask)[mi] != 0;
                            else add = ((const float *)f.mask)[mi] * inv_scale;
                        } else if constexpr (MVEC) {
                            if constexpr (MASK == 5) ok = ok && ((mvb[kb][i / 4] >> (8 * (i % 4))) & 0xffu) != 0;
                            else add = mvf[kb][i / 4][i % 4] * inv_scale;
                        }
                        const float pv = ok ? fast_exp2(fmaf(s[kb][i] + add, c, -lse2)) : 0.0f;
                        ds[i] = pv * dp[kb][i];
                    }
                }
                pack8_hilo<T>(ds, sb[kb][0], sl[kb][0]);
                pack8_hilo<T>(ds + 8, sb[kb][1], sl[kb][1]);
            }
            // dQ^T += K^T . dS^T
#pragma unroll
            for (int db = 0; db < DB; ++db) {
#pragma unroll
                for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
                    for (int hs = 0; hs < 2; ++hs) {
                        const int row = 32 * kb + 16 * hs + 4 * (g16 >> 1) + (i16 >> 2);
                        const int col = 32 * db + 16 * (g16 & 1) + 4 * (i16 & 3);
                        const V8 kt = read_tr8<T>(&cK[row * KP + col], &cK[(row + 8) * KP + col]);
                        dq[db] = M::mma(kt, sb[kb][hs], dq[db]);
                        dq[db] = M::mma(kt, sl[kb][hs], dq[db]);
                    }
                }
            }
        }
        if (j + 1 < ntiles) {
            store_tile(buf ^ 1);
            if (j + 2 < ntiles) load_tile(j + 2);
        }
        __syncthreads();
    }
    if (lq < L) {
        const int64_t at = (bh * f.L + lq) * D;
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int g = 0; g < 4 && 32 * db + 8 * g < D; ++g) {
                const f32x4 v = {scaled(dq[db][4 * g], f.scale), scaled(dq[db][4 * g + 1], f.scale),
                                 scaled(dq[db][4 * g + 2], f.scale), scaled(dq[db][4 * g + 3], f.scale)};
                const int64_t e = at + 32 * db + 8 * g + 4 * half;
                if (a.g_half) *(u32x2 *)((T *)a.dq + e) = u32x2{M::pack(v[0], v[1]), M::pack(v[2], v[3])};
                else *(f32x4 *)((float *)a.dq + e) = v;
            }
    }
}

template <typename T, int D, bool CAUSAL, int MASK, bool DROP>
hipError_t launch_bwd_drop(const AttnBwdArgs &a, hipStream_t s) {
    const AttnFwdArgs &f = a.f;
    // dQ first: it computes delta = rowsum(dO * O) per query row, which dK/dV reads
    const int nq = (int)((f.L + BMQ - 1) / BMQ);
    hipLaunchKernelGGL((bwd_dq_kernel<T, D, CAUSAL, MASK, DROP>), dim3((unsigned)(nq * f.B * f.H)), dim3(256), 0, s, a, nq);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    // dK/dV reads a per-element mask one element per lane (its lanes hold one key each): modes
    // 5 / 6 are 1 / 2 there
    constexpr int MKV = MASK >= 5 ? MASK - 4 : MASK;
    const int nkt = (int)((f.S + BKV - 1) / BKV);
    hipLaunchKernelGGL((bwd_dkdv_kernel<T, D, CAUSAL, MKV, DROP>), dim3((unsigned)(nkt * f.B * f.Hkv)), dim3(256), 0, s, a);
    return hipGetLastError();
}

template <typename T, int D, bool CAUSAL, int MASK>
hipError_t launch_bwd_typed(const AttnBwdArgs &a, hipStream_t s) {
    return a.f.dropout ? launch_bwd_drop<T, D, CAUSAL, MASK, true>(a, s) : launch_bwd_drop<T, D, CAUSAL, MASK, false>(a, s);
}

template <typename T, int D>
hipError_t launch_bwd_d(const AttnBwdArgs &a, hipStream_t s) {
    // mode 4: a float mask that does not depend on the query row (key padding); 5 / 6: bool /
    // float per-element masks with contiguous, 4-key aligned keys (attn_mask_mode)
    const int mode = attn_mask_mode(a.f);
    if (a.f.causal) {
        if (mode == 0) return launch_bwd_typed<T, D, true, 0>(a, s);
        if (mode == 1) return launch_bwd_typed<T, D, true, 1>(a, s);
        if (mode == 4) return launch_bwd_typed<T, D, true, 4>(a, s);
        if (mode == 5) return launch_bwd_typed<T, D, true, 5>(a, s);
        if (mode == 6) return launch_bwd_typed<T, D, true, 6>(a, s);
        return launch_bwd_typed<T, D, true, 2>(a, s);
    }
    if (mode == 0) return launch_bwd_typed<T, D, false, 0>(a, s);
    if (mode == 1) return launch_bwd_typed<T, D, false, 1>(a, s);
    if (mode == 4) return launch_bwd_typed<T, D, false, 4>(a, s);
    if (mode == 5) return launch_bwd_typed<T, D, false, 5>(a, s);
    if (mode == 6) return launch_bwd_typed<T, D, false, 6>(a, s);
    return launch_bwd_typed<T, D, false, 2>(a, s);
}

}  // namespace
