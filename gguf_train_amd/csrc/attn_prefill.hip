// Which prefill kernel a call takes, and the float32 ones.  The float16 / bfloat16 kernels are in
// attn_prefill_half.h, instantiated here for head sizes 64 and 128 and in attn_prefill_heads.hip for 80
// and 96.

#include "attn_prefill_half.h"

namespace {

// ---- float32 --------------------------------------------------------------------------------
// Float32 prefill (D = Dv = 64 or 128, no mask or a key-padding row): the structure of
// prefill_fwd_kernel (query tiles of 128 rows in pairs, K/V tiles streamed into LDS by DMA, one
// barrier per tile, the same lazy online softmax and causal / edge handling) on
// v_mfma_f32_32x32x2_f32, whose products and sums are float32 like the generic kernel's.  The
// MFMA's k index is free as long as both operands agree:
//   S^T = K.Q^T: k-step t takes dim t + (D/2)(lane/32), so a lane's Q values are the dims
//   [(D/2)(lane/32), +D/2) of its row, held in registers, and its K values come 4 at a time from
//   one 16-byte LDS read;
//   O^T += V^T.P^T: k-step s takes key 8(s/4) + 4(lane/32) + s%4, the key of the lane's S^T
//   accumulator entry s, so P^T's operand for step s is that entry as it stands.
// 32-key tiles: 16-byte chunk c of tile row r sits at chunk c ^ (r & 15), so the 16 rows one
// quarter-wave reads land on 16 different chunks mod 16 (different LDS banks).
constexpr int F32_NW = 4, F32_BM = 32 * F32_NW, F32_BN = 32, F32_NST = 2;

__device__ inline f32x16 mfma_f32x2(float a, float b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// DROP: P.V takes P times the element's multiplier (gt_philox.h); the lane's entries 4g .. 4g+3
// are 4 consecutive keys of its row, one Philox block.  The running sum keeps the undropped P.
template <int D, bool CAUSAL, int MASK, bool DROP = false>
__global__ __launch_bounds__(64 * F32_NW, 2) void prefill_f32_kernel(AttnFwdArgs a, int nq, int npairs) {
    constexpr int NW = F32_NW, BM = F32_BM, BN = F32_BN, NST = F32_NST;
    constexpr int CH = D / 4;               // 16-byte chunks per row
    constexpr int TILE = BN * D;            // floats per tile
    constexpr int NPW = BN * CH / 64 / NW;  // 1 KB wave loads per operand, wave and tile
    constexpr int DB = D / 32;              // d blocks of O^T
    constexpr int DH = D / 2;               // dims per lane half in S^T
    constexpr bool MROW = MASK == 4;
    constexpr bool MEL = MASK == 1 || MASK == 2 || MASK >= 5;  // per-element mask
    constexpr bool MVEC = MASK >= 5;                           // 4 keys per mask load
    constexpr bool MBOOL = MASK == 1 || MASK == 5;
    constexpr int PER = 2 * NPW + (MROW ? 1 : 0);  // loads per wave and tile
    static_assert(NPW >= 1 && CH >= 16 && PER < 64, "tile split");
    __shared__ __attribute__((aligned(1024))) float sK[NST][TILE];
    __shared__ __attribute__((aligned(1024))) float sV[NST][TILE];
    __shared__ __attribute__((aligned(16))) float sMk[MROW ? NST : 1][64];  // keys k0 .. k0+63 (32 used)

    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lrow = lane & 31, half = lane >> 5;
    const int64_t BH = a.B * a.H;
    int pair;
    int64_t bh;
    if (BH % 8 == 0) {
        const int64_t hpx = BH / 8, i = blockIdx.x / 8;
        pair = (int)(i % npairs);
        bh = (int64_t)(blockIdx.x % 8) * hpx + i / npairs;
    } else {
        pair = (int)(blockIdx.x % npairs);
        bh = (int64_t)blockIdx.x / npairs;
    }
    const int64_t b = bh / a.H, h = bh % a.H, hk = h / (a.H / a.Hkv);
    const int L = (int)a.L, S = (int)a.S;
    const int nkv = attn_kv_len(a, b), qpos = attn_q_pos(a, b);
    const int qa = nq - 1 - pair, qb = pair;
    const int nparts = qa == qb ? 1 : 2;
    const int na = key_tiles<CAUSAL, BM, BN>(qa, nkv, qpos);
    const int total = na + (nparts == 2 ? key_tiles<CAUSAL, BM, BN>(qb, nkv, qpos) : 0);

    const float *kbase = (const float *)a.k + b * a.k_sb + hk * a.k_sh;
    const float *vbase = (const float *)a.v + b * a.v_sb + hk * a.v_sh;
    const float c = a.scale * kLog2e;
    const float inv_scale = 1.0f / a.scale;
    const uint32_t k_row = (uint32_t)a.k_ss * 4, v_row = (uint32_t)a.v_ss * 4;
    int lrow_n[NPW];
    uint32_t lcol_n[NPW], kofs_n[NPW], vofs_n[NPW];
#pragma unroll
    for (int n = 0; n < NPW; ++n) {
        const int slot = (w * NPW + n) * 64 + lane;
        lrow_n[n] = slot / CH;
        lcol_n[n] = 16u * (uint32_t)((slot % CH) ^ (lrow_n[n] & 15));
        kofs_n[n] = (uint32_t)lrow_n[n] * k_row + lcol_n[n];
        vofs_n[n] = (uint32_t)lrow_n[n] * v_row + lcol_n[n];
    }
    const float *mrow = MROW ? (const float *)a.mask + b * a.m_sb + h * a.m_sh : nullptr;
    auto issue = [&](int step) {
        const int kt = step < na ? step : step - na;
        const int st = step % NST;
        if constexpr (MROW)
            lds_dma4(lds_addr(&sMk[st][0]), mrow, (uint32_t)min(kt * BN + lane, S - 1) * (uint32_t)a.m_ss * 4u);
        const uint32_t dk = lds_addr(&sK[st][0]) + w * NPW * 1024;
        const uint32_t dv = lds_addr(&sV[st][0]) + w * NPW * 1024;
        if (kt * BN + BN <= S) {
            const char *kb = (const char *)kbase + (uint64_t)(kt * BN) * k_row;
            const char *vb = (const char *)vbase + (uint64_t)(kt * BN) * v_row;
#pragma unroll
            for (int n = 0; n < NPW; ++n) {
                lds_dma16(dk + n * 1024, kb, kofs_n[n]);
                lds_dma16(dv + n * 1024, vb, vofs_n[n]);
            }
        } else {
#pragma unroll
            for (int n = 0; n < NPW; ++n) {
                const uint32_t key = (uint32_t)min(kt * BN + lrow_n[n], S - 1);
                lds_dma16(dk + n * 1024, kbase, key * k_row + lcol_n[n]);
                lds_dma16(dv + n * 1024, vbase, key * v_row + lcol_n[n]);
            }
        }
    };
    // LDS float offsets of this lane's fragments within a tile, as a per-lane part plus a
    // compile-time part (the XOR swizzle only touches chunk bits 0..3, so it splits):
    //   K, dims 4u .. 4u+3 of its half: row lrow, chunk (u + (D/8) half) ^ (lrow & 15)
    //     = lrow D + (4u ^ 4 ((lrow & 15) ^ (D/8) half))  (u < D/8: u + (D/8) half = u ^ (D/8) half)
    //   V, k-step s, d block db: row r = 8(s/4) + 4half + s%4, float d = 32db + lrow, chunk
    //     (d/4) ^ (r & 15) = (8db ^ 8((s/4) & 1)) + ((lrow/4) ^ 4half ^ (s%4))
    const int kbase0 = lrow * D, kx = 4 * ((lrow & 15) ^ ((D / 8) * half));
    auto kofs = [&](int u) { return kbase0 + ((4 * u) ^ kx); };
    const int vy = (lrow >> 2) ^ (4 * half);
    int vx[4];
#pragma unroll
    for (int cc = 0; cc < 4; ++cc) vx[cc] = 4 * D * half + (lrow & 3) + 4 * (vy ^ cc);
    auto vofs = [&](int s, int db) {
        return vx[s & 3] + 8 * D * (s >> 2) + D * (s & 3) + 4 * ((8 * db) ^ (8 * ((s >> 2) & 1)));
    };

#pragma unroll
    for (int st = 0; st < NST - 1; ++st)
        if (st < total) issue(st);

    int step = 0;
    for (int part = 0; part < nparts; ++part) {
        const int qt = part == 0 ? qa : qb;
        const int ntiles = part == 0 ? na : total - na;
        const int wq0 = qt * BM + 32 * w;
        const int lq = wq0 + lrow;
        // Q^T as B operands: dims (D/2) half .. +D/2 of row lq (rows past L read row L-1)
        float qf[DH];
        {
            const float *qr = (const float *)a.q + b * a.q_sb + h * a.q_sh + (int64_t)min(lq, L - 1) * a.q_sl + DH * half;
#pragma unroll
            for (int u = 0; u < DH / 4; ++u) {
                const f32x4 x = *(const f32x4 *)(qr + 4 * u);
#pragma unroll
                for (int e = 0; e < 4; ++e) qf[4 * u + e] = x[e];
            }
#pragma unroll
            for (int u = 0; u < DH; ++u) asm volatile("" ::"v"(qf[u]));
        }
        f32x16 o[DB];
#pragma unroll
        for (int db = 0; db < DB; ++db)
#pragma unroll
            for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
        float m = -INFINITY, mthr = -INFINITY, lsum = 0.0f;
        // dropout: Philox block of keys 0..3 of this lane's row (rows past L draw unused words)
        const uint64_t drow = DROP ? (uint64_t)(bh * a.L + lq) * (uint64_t)((a.S + 3) / 4) : 0;
        // per-element mask: element offset of this lane's mask row
        const int64_t mrb = MEL ? b * a.m_sb + h * a.m_sh + (int64_t)min(lq, L - 1) * a.m_sl : 0;

        for (int j = 0; j < ntiles; ++j, ++step) {
            const int k0 = j * BN;
            const int later = min(NST - 2, total - 1 - step);
            if (later >= 1) wait_vm<PER>();
            else wait_vm<0>();
            __syncthreads();
            const float *cK = sK[step % NST];
            const float *cV = sV[step % NST];
            // MVEC: the mask of keys k0 + 8g + 4half + 0..3 of this lane's row, loaded before the
            // MFMAs (groups past the last 4 keys read those: their scores are blocked below)
            f32x4 mvf[MVEC && !MBOOL ? 4 : 1];
            uint32_t mvb[MVEC && MBOOL ? 4 : 1];
            if constexpr (MVEC) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int64_t at = mrb + min(k0 + 8 * g + 4 * half, S - 4);
                    if constexpr (MBOOL) mvb[g] = *(const uint32_t *)((const uint8_t *)a.mask + at);
                    else mvf[g] = *(const f32x4 *)((const float *)a.mask + at);
                }
            }
            // ---- S^T = K . Q^T: s[i] is key k0 + 8(i/4) + 4half + i%4, query lq ----
            f32x16 s;
            if constexpr (MROW) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 mv4 = *(const f32x4 *)&sMk[step % NST][8 * g + 4 * half];
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * g + e] = mv4[e] * inv_scale;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) s[i] = 0.0f;
            }
#pragma unroll
            for (int u = 0; u < DH / 4; ++u) {
                const f32x4 kv = *(const f32x4 *)&cK[kofs(u)];
#pragma unroll
                for (int e = 0; e < 4; ++e) s = mfma_f32x2(kv[e], qf[4 * u + e], s);
            }
            // the next tile's loads into the stage every wavefront finished with before the barrier
            if (step + NST - 1 < total) issue(step + NST - 1);

            const bool edge = k0 + BN > nkv || (CAUSAL && k0 + BN - 1 > wq0 + qpos);
            if (MEL || edge) {
                const int vis = min(nkv - 1, CAUSAL ? lq + qpos : nkv - 1) - (k0 + 4 * half);
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    float x = s[i];
                    if constexpr (MVEC) {
                        if constexpr (MBOOL) x = (mvb[i / 4] >> (8 * (i % 4))) & 0xffu ? x : -INFINITY;
                        else x = fmaf(mvf[i / 4][i % 4], inv_scale, x);
                    } else if constexpr (MEL) {
                        const int key = min(k0 + 8 * (i / 4) + 4 * half + (i % 4), S - 1);
                        const int64_t mi = mrb + (int64_t)key * a.m_ss;
                        if constexpr (MBOOL) x = ((const uint8_t *)a.mask)[mi] ? x : -INFINITY;
                        else x = fmaf(((const float *)a.mask)[mi], inv_scale, x);
                    }
                    const bool blocked = 8 * (i / 4) + (i % 4) > vis;
                    s[i] = blocked ? -INFINITY : x;
                }
            }
            float tmax = max3(s[0], s[1], s[2]);
#pragma unroll
            for (int i = 3; i < 15; i += 2) tmax = max3(tmax, s[i], s[i + 1]);
            tmax = max3(tmax, s[15], s[15]);
            tmax = xhalf_max(tmax);
            const float tm = tmax * c;
            const bool move = tm > mthr;
            if (!__all(!move)) {
                const float mnew = move ? tm + huge_margin(tm) : m;
                const float alpha = move ? fast_exp2(m - mnew) : 1.0f;
                lsum *= alpha;
#pragma unroll
                for (int db = 0; db < DB; ++db)
#pragma unroll
                    for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
                m = mnew;
                mthr = m + kLazy - 0.5f * huge_margin(m);
            }
            const float msub = m == -INFINITY ? 0.0f : m;
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                s[i] = fast_exp2(fmaf(s[i], c, -msub));
                lsum += s[i];
            }
            if constexpr (DROP) {
                const float dscale = (float)a.drop.scale;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const GtWord4 x = gt_philox4x32_10(drow + (uint64_t)((k0 + 8 * g + 4 * half) >> 2), a.drop.offset,
                                                       a.drop.seed);
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[4 * g + e] *= x.w[e] < a.drop.thresh ? dscale : 0.0f;
                }
            }
            // ---- O^T += V^T . P^T ----
#pragma unroll
            for (int st2 = 0; st2 < 16; ++st2)
#pragma unroll
                for (int db = 0; db < DB; ++db) o[db] = mfma_f32x2(cV[vofs(st2, db)], s[st2], o[db]);
        }

        const float ltot = xhalf_sum(lsum);
        const float inv = ltot > 0.0f ? 1.0f / ltot : 0.0f;
        if (lq < L) {
            float *orow = (float *)a.o + (bh * a.L + lq) * D;
            float *row32 = a.o32 ? (float *)a.o32 + (bh * a.L + lq) * D : nullptr;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 v = {o[db][4 * g] * inv, o[db][4 * g + 1] * inv, o[db][4 * g + 2] * inv,
                                     o[db][4 * g + 3] * inv};
                    *(f32x4 *)(orow + 32 * db + 8 * g + 4 * half) = v;
                    if (row32) *(f32x4 *)(row32 + 32 * db + 8 * g + 4 * half) = v;
                }
            if (a.lse && half == 0)
                ((float *)a.lse)[bh * a.L + lq] = ltot > 0.0f ? (m + log2f(ltot)) * kLn2 : INFINITY;
        }
    }
}

// Float32 prefill for small grids (few heads of short sequences, where prefill_f32_kernel has
// fewer workgroups than the GPU has CUs and each wavefront's walk over the key tiles is the whole
// time): one workgroup per 32 query rows, its 4 wavefronts splitting the key tiles (tile t to
// wavefront t % 4) with an online softmax each, then merging the four (max, sum, O) states
// through LDS.  The operand mapping is prefill_f32_kernel's (S^T = K.Q^T with k-step t = dim
// t + (D/2)(lane/32) and Q in registers; O^T += V^T.P^T with k-step s = the key of accumulator
// entry s), but each wavefront reads its K rows (16-byte pieces) and V^T values straight from
// memory: they are few and stay in L2.  Masks, dropout and KV-cache lengths as prefill_f32_kernel
// takes them (the mask read per score, or 4 keys per load for modes 5 and 6).
template <int D, bool CAUSAL, int MASK, bool DROP>
__global__ __launch_bounds__(256) void prefill_f32_split_kernel(AttnFwdArgs a, int ng) {
    constexpr int DH = D / 2, DB = D / 32, OP = D + 4;  // OP: LDS row pitch of the partial O
    constexpr bool MVEC = MASK >= 5;                    // 4 keys per mask load
    constexpr bool MBOOL = MASK == 1 || MASK == 5;
    __shared__ __attribute__((aligned(16))) float sO[4][32][OP];
    __shared__ float sM[4][32], sL[4][32];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int lrow = lane & 31, half = lane >> 5;
    const int64_t bh = blockIdx.x / ng;
    const int rg = (int)(blockIdx.x % ng);
    const int64_t b = bh / a.H, h = bh % a.H, hk = h / (a.H / a.Hkv);
    const int L = (int)a.L, S = (int)a.S;
    const int q0 = 32 * rg, lq = q0 + lrow, lqc = min(lq, L - 1);
    const int nkv = attn_kv_len(a, b), qpos = attn_q_pos(a, b);
    const int kv_end = CAUSAL ? min(q0 + 32 + qpos, nkv) : nkv;  // keys any row of the group sees
    const int nt = kv_end > 0 ? (kv_end + 31) / 32 : 0;
    const float c = a.scale * kLog2e;
    // element offset of this lane's mask row (MASK 4: the key-padding row, m_sl = 0)
    const int64_t mrb = MASK != 0 ? b * a.m_sb + h * a.m_sh + (int64_t)lqc * a.m_sl : 0;
    // dropout: Philox block of keys 0..3 of this lane's row (rows past L draw unused words)
    const uint64_t drow = DROP ? (uint64_t)(bh * a.L + lq) * (uint64_t)((a.S + 3) / 4) : 0;

    float qf[DH];  // Q of row lqc, dims DH half .. +DH (B operand of S^T)
    {
        const float *qr = (const float *)a.q + b * a.q_sb + h * a.q_sh + (int64_t)lqc * a.q_sl + DH * half;
#pragma unroll
        for (int u = 0; u < DH / 4; ++u) {
            const f32x4 x = *(const f32x4 *)(qr + 4 * u);
#pragma unroll
            for (int e = 0; e < 4; ++e) qf[4 * u + e] = x[e];
        }
    }
    const float *kbase = (const float *)a.k + b * a.k_sb + hk * a.k_sh;
    const float *vbase = (const float *)a.v + b * a.v_sb + hk * a.v_sh;
    f32x16 o[DB];
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[db][i] = 0.0f;
    float m = -INFINITY, lsum = 0.0f;  // running max (log2 domain) and this half's share of the sum

    for (int t = w; t < nt; t += 4) {
        const int k0 = 32 * t;
        // S^T: s[i] is key k0 + 8(i/4) + 4half + i%4, query lq
        const float *kr = kbase + (int64_t)min(k0 + lrow, S - 1) * a.k_ss + DH * half;
        f32x16 s;
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
        for (int u = 0; u < DH / 4; ++u) {
            const f32x4 kv = *(const f32x4 *)(kr + 4 * u);
#pragma unroll
            for (int e = 0; e < 4; ++e) s = mfma_f32x2(kv[e], qf[4 * u + e], s);
        }
        const int vis = min(nkv - 1, CAUSAL ? lq + qpos : nkv - 1) - (k0 + 4 * half);
        // MVEC: the mask of keys k0 + 8g + 4half + 0..3 (groups past the last 4 keys read those:
        // their scores are blocked)
        f32x4 mvf[MVEC && !MBOOL ? 4 : 1];
        uint32_t mvb[MVEC && MBOOL ? 4 : 1];
        if constexpr (MVEC) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int64_t at = mrb + min(k0 + 8 * g + 4 * half, S - 4);
                if constexpr (MBOOL) mvb[g] = *(const uint32_t *)((const uint8_t *)a.mask + at);
                else mvf[g] = *(const f32x4 *)((const float *)a.mask + at);
            }
        }
        float tmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float x = s[i] * c;
            bool blocked = 8 * (i / 4) + (i % 4) > vis;
            if constexpr (MVEC) {
                if constexpr (MBOOL) blocked = blocked || ((mvb[i / 4] >> (8 * (i % 4))) & 0xffu) == 0u;
                else x = fmaf(mvf[i / 4][i % 4], kLog2e, x);
            } else if constexpr (MASK != 0) {
                const int64_t mi = mrb + (int64_t)min(k0 + 8 * (i / 4) + 4 * half + (i % 4), S - 1) * a.m_ss;
                if constexpr (MBOOL) blocked = blocked || ((const uint8_t *)a.mask)[mi] == 0;
                else x = fmaf(((const float *)a.mask)[mi], kLog2e, x);
            }
            s[i] = blocked ? -INFINITY : x;
            tmax = fmaxf(tmax, s[i]);
        }
        const float mnew = fmaxf(m, xhalf_max(tmax));
        const float msub = mnew == -INFINITY ? 0.0f : mnew;
        if (mnew != m) {
            const float alpha = fast_exp2(m - msub);  // m = -inf: 0 (O and the sum are 0)
            lsum *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[db][i] *= alpha;
            m = mnew;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            s[i] = fast_exp2(s[i] - msub);  // -inf -> 0
            lsum += s[i];
        }
        if constexpr (DROP) {
            // entries 4g .. 4g+3 are keys k0 + 8g + 4half + 0..3: one Philox block
            const float dscale = (float)a.drop.scale;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const GtWord4 x = gt_philox4x32_10(drow + (uint64_t)((k0 + 8 * g + 4 * half) >> 2), a.drop.offset,
                                                   a.drop.seed);
#pragma unroll
                for (int e = 0; e < 4; ++e) s[4 * g + e] *= x.w[e] < a.drop.thresh ? dscale : 0.0f;
            }
        }
        // O^T += V^T . P^T: k-step s2 is key k0 + 8(s2/4) + 4half + s2%4, A = V[that key][32 db + lrow]
#pragma unroll
        for (int s2 = 0; s2 < 16; ++s2) {
            const float *vr = vbase + (int64_t)min(k0 + 8 * (s2 >> 2) + 4 * half + (s2 & 3), S - 1) * a.v_ss + lrow;
#pragma unroll
            for (int db = 0; db < DB; ++db) o[db] = mfma_f32x2(vr[32 * db], s[s2], o[db]);
        }
    }

    // ---- merge the four wavefronts' states ----
    const float ltot = xhalf_sum(lsum);
    if (half == 0) {
        sM[w][lrow] = m;
        sL[w][lrow] = ltot;
    }
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const f32x4 v = {o[db][4 * g], o[db][4 * g + 1], o[db][4 * g + 2], o[db][4 * g + 3]};
            *(f32x4 *)&sO[w][lrow][32 * db + 8 * g + 4 * half] = v;
        }
    __syncthreads();
    // thread: row r of the group, dims (D/8) part .. +D/8
    const int r = threadIdx.x >> 3, part = threadIdx.x & 7;
    float M = -INFINITY;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) M = fmaxf(M, sM[ww][r]);
    float wg[4], Lt = 0.0f;
#pragma unroll
    for (int ww = 0; ww < 4; ++ww) {
        wg[ww] = sM[ww][r] == -INFINITY ? 0.0f : fast_exp2(sM[ww][r] - M);
        Lt = fmaf(wg[ww], sL[ww][r], Lt);
    }
    const float inv = Lt > 0.0f ? 1.0f / Lt : 0.0f;
    if (q0 + r < L) {
        float *orow = (float *)a.o + (bh * a.L + q0 + r) * D + (D / 8) * part;
#pragma unroll
        for (int j = 0; j < D / 32; ++j) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int ww = 0; ww < 4; ++ww) {
                const f32x4 x = *(const f32x4 *)&sO[ww][r][(D / 8) * part + 4 * j];
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = fmaf(wg[ww], x[e], acc[e]);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[e] *= inv;
            *(f32x4 *)(orow + 4 * j) = acc;
        }
        if (a.lse && part == 0) ((float *)a.lse)[bh * a.L + q0 + r] = Lt > 0.0f ? (M + log2f(Lt)) * kLn2 : INFINITY;
    }
}

// The calls prefill_f32_split_kernel takes: at most 64 workgroups of prefill_f32_kernel
// (B * H * query-tile pairs) and at most 4096 keys.  Measured
// against the tiled kernel: faster at every grid of up to 64 of its workgroups (B2 H8 L=S=1024
// D128: 107 against 276 us; B1 H8 L=S=2048 D128 causal: 207 against 295 us), mixed at 128,
// twice as slow at 256 (each 32-row group reads its keys' K and V itself, where the tiled
// kernel shares a tile among 128 rows).
bool prefill_f32_split(const AttnFwdArgs &f) {
    if (f.o32 || f.rope_q || f.S > 4096) return false;
    const int64_t pairs = ((f.L + F32_BM - 1) / F32_BM + 1) / 2;
    return f.B * f.H * pairs <= 64;
}

bool prefill_f32_supported(const AttnFwdArgs &f) {
    if (f.out_dtype != GT_F32 || f.D != f.Dv || (f.D != 64 && f.D != 128)) return false;
    if (f.rope_q) return false;
    const int mode = attn_mask_mode(f);
    // fewer than 16 query rows: one mostly empty 128-row tile per head walking every key; the
    // generic kernel measured as fast or faster there (one row: 1.14 against 2.02 ms at B32
    // H32/8 S4096 D128; 16 rows: even).  The small-grid kernel takes them (32-row groups,
    // 4 wavefronts per key range): 4 rows B1 H32/8 S4096 D128 229 us against the generic 538
    if ((f.L < 16 && !prefill_f32_split(f)) || f.L < 1 || f.S < 1 || !(f.scale > 0.0f)) return false;
    if (f.L >= (1LL << 30) || f.S >= (1LL << 30)) return false;
    const int64_t strides[] = {f.q_sb, f.q_sh, f.q_sl, f.k_sb, f.k_sh, f.k_ss, f.v_sb, f.v_sh, f.v_ss};
    for (int64_t st : strides) if (st % 4 != 0 || st < 0) return false;  // 16-byte rows
    for (const void *p : {f.q, f.k, f.v, (const void *)f.o}) if ((uintptr_t)p % 16 != 0) return false;
    if (f.o32 && (uintptr_t)f.o32 % 16 != 0) return false;
    if ((f.S - 1) * f.k_ss * 4 + f.D * 4 > 0xffffffffLL) return false;
    if ((f.S - 1) * f.v_ss * 4 + f.Dv * 4 > 0xffffffffLL) return false;
    if (mode == 4 && (f.m_ss < 0 || (f.S - 1) * f.m_ss * 4 + 4 > 0xffffffffLL)) return false;
    return true;
}

template <int D, bool CAUSAL, bool DROP>
hipError_t launch_prefill_f32_cd(const AttnFwdArgs &a, int nq, int npairs, int64_t grid, hipStream_t s) {
#define GT_F32_LAUNCH(MK) \
    hipLaunchKernelGGL((prefill_f32_kernel<D, CAUSAL, MK, DROP>), dim3((unsigned)grid), dim3(64 * F32_NW), 0, s, a, nq, npairs)
    switch (attn_mask_mode(a)) {
        case 0: GT_F32_LAUNCH(0); break;
        case 1: GT_F32_LAUNCH(1); break;
        case 2: GT_F32_LAUNCH(2); break;
        case 4: GT_F32_LAUNCH(4); break;
        case 5: GT_F32_LAUNCH(5); break;
        case 6: GT_F32_LAUNCH(6); break;
        default: return hipErrorInvalidValue;
    }
#undef GT_F32_LAUNCH
    return hipGetLastError();
}

template <int D>
hipError_t launch_prefill_f32_d(const AttnFwdArgs &a, int nq, int npairs, int64_t grid, hipStream_t s) {
    if (a.dropout)
        return a.causal ? launch_prefill_f32_cd<D, true, true>(a, nq, npairs, grid, s)
                        : launch_prefill_f32_cd<D, false, true>(a, nq, npairs, grid, s);
    return a.causal ? launch_prefill_f32_cd<D, true, false>(a, nq, npairs, grid, s)
                    : launch_prefill_f32_cd<D, false, false>(a, nq, npairs, grid, s);
}

template <int D, bool CAUSAL, bool DROP>
hipError_t launch_split(const AttnFwdArgs &a, dim3 grid, int ng, hipStream_t s) {
#define GT_SPLIT(MK) hipLaunchKernelGGL((prefill_f32_split_kernel<D, CAUSAL, MK, DROP>), grid, dim3(256), 0, s, a, ng)
    switch (attn_mask_mode(a)) {
        case 0: GT_SPLIT(0); break;
        case 1: GT_SPLIT(1); break;
        case 2: GT_SPLIT(2); break;
        case 4: GT_SPLIT(4); break;
        case 5: GT_SPLIT(5); break;
        case 6: GT_SPLIT(6); break;
        default: return hipErrorInvalidValue;
    }
#undef GT_SPLIT
    return hipGetLastError();
}

hipError_t launch_prefill_f32(const AttnFwdArgs &a, hipStream_t s) {
    if (prefill_f32_split(a)) {
        const int ng = (int)((a.L + 31) / 32);
        const dim3 grid((unsigned)(a.B * a.H * ng));
        if (a.D == 128) {
            if (a.dropout) return a.causal ? launch_split<128, true, true>(a, grid, ng, s) : launch_split<128, false, true>(a, grid, ng, s);
            return a.causal ? launch_split<128, true, false>(a, grid, ng, s) : launch_split<128, false, false>(a, grid, ng, s);
        }
        if (a.dropout) return a.causal ? launch_split<64, true, true>(a, grid, ng, s) : launch_split<64, false, true>(a, grid, ng, s);
        return a.causal ? launch_split<64, true, false>(a, grid, ng, s) : launch_split<64, false, false>(a, grid, ng, s);
    }
    const int nq = (int)((a.L + F32_BM - 1) / F32_BM);
    const int npairs = (nq + 1) / 2;
    const int64_t grid = (int64_t)npairs * a.B * a.H;
    if (grid <= 0) return hipSuccess;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    return a.D == 128 ? launch_prefill_f32_d<128>(a, nq, npairs, grid, s) : launch_prefill_f32_d<64>(a, nq, npairs, grid, s);
}

}  // namespace

int attn_prefill_key_tile(const AttnFwdArgs &f) { return f.D == 64 ? bn_of<64>() : bn_of<128>(); }  // (80, 96: as 128)

bool attn_prefill_f32_split(const AttnFwdArgs &f, int cd) {
    return cd == GT_F32 && prefill_f32_supported(f) && prefill_f32_split(f);
}

bool attn_prefill_supported(const AttnFwdArgs &f, int cd) {
    if (cd == GT_F32) return prefill_f32_supported(f);
    if (cd != GT_F16 && cd != GT_BF16) return false;
    if (f.rope_q && f.mask && (f.mask_bool || f.m_sl != 0)) return false;  // fused RoPE: no mask or key padding
    if (f.rope_q && f.dropout) return false;
    if (f.out_dtype != cd || f.D != f.Dv || !attn_half_head(f.D, f.L)) return false;
    // 80 and 96: no fused rotation, and a caller's own output off the 8 bytes of a store goes to the generic kernel
    if (f.D != 64 && f.D != 128 && (f.rope_q || (uintptr_t)f.o % 8 != 0)) return false;
    if (f.L < 1 || f.S < 1 || !(f.scale > 0.0f)) return false;
    if (f.L >= (1LL << 30) || f.S >= (1LL << 30)) return false;  // 32-bit row indices
    const int64_t strides[] = {f.q_sb, f.q_sh, f.q_sl, f.k_sb, f.k_sh, f.k_ss, f.v_sb, f.v_sh, f.v_ss};
    for (int64_t st : strides) if (st % 8 != 0 || st < 0) return false;
    for (const void *p : {f.q, f.k, f.v}) if ((uintptr_t)p % 16 != 0) return false;
    // K/V tiles are addressed by 32-bit byte offsets from the (batch, kv head) base
    if ((f.S - 1) * f.k_ss * 2 + f.D * 2 > 0xffffffffLL) return false;
    if ((f.S - 1) * f.v_ss * 2 + f.Dv * 2 > 0xffffffffLL) return false;
    // a query-independent float mask row is addressed the same way
    if (f.mask && !f.mask_bool && f.m_sl == 0 && (f.m_ss < 0 || (f.S - 1) * f.m_ss * 4 + 4 > 0xffffffffLL)) return false;
    return true;
}

hipError_t launch_attn_prefill(const AttnFwdArgs &a, int cd, hipStream_t s) {
    if (cd == GT_F32) return launch_prefill_f32(a, s);
    if (attn_prefill_asm_supported(a, cd)) return launch_attn_prefill_asm(a, s);
    const int BM = a.D == 64 ? bm_of<64>() : bm_of<128>();
    const int nq = (int)((a.L + BM - 1) / BM);
    const int order = tile_order(a, nq);
    const int64_t grid = (int64_t)(order == kPairs ? (nq + 1) / 2 : nq) * a.B * a.H;
    if (grid <= 0) return hipSuccess;
    if (grid > 0x7fffffffLL) return hipErrorInvalidConfiguration;
    if (a.D != 64 && a.D != 128) return launch_prefill_heads(a, cd, nq, order, grid, s);
    if (cd == GT_F16)
        return a.D == 128 ? launch_variant<_Float16, 128>(a, nq, order, grid, s)
                          : launch_variant<_Float16, 64>(a, nq, order, grid, s);
    return a.D == 128 ? launch_variant<__bf16, 128>(a, nq, order, grid, s)
                      : launch_variant<__bf16, 64>(a, nq, order, grid, s);
}
