// Which rows of a KV-cache append a thread and its workgroup handle, and where the workgroup keeps the
// RoPE angles that it forms for them (kv_append_vec_kernel), plain arithmetic that a host program can
// check.  256 threads per workgroup, each 8 elements of a row.
#pragma once

#include <cstdint>

// Threads (of a kernel that rotates up to 8 elements each) up to which a workgroup forms its rows' angles
// itself, into LDS; more of them share a table made by a launch before, since a prompt's workgroups
// would repeat each angle for every head.  A decode step's rows then take one launch: RoPE of fp16 B4
// H32 D128 3.2 + 5.2 -> 3.9 us.  (Every thread forming its own 8 angles took 7.6 us: one accurate
// sincosf after the other.)
constexpr int64_t kRopeInlineThreads = 65536;
constexpr int kRopeInlineMaxDim = 256;  // head size up to which the angles of a workgroup's rows fit
// Angles of a 256-thread workgroup's rows: 8 elements per thread are 2048 / D rows, and one more at
// either end when rows straddle workgroups.
constexpr int kRopeInlineEntries = 1024 + kRopeInlineMaxDim;

// Elements d0 .. d0 + 7 of source row `row` = (b, h, t).  Threads past the last row (not live) take the
// first one, so that their loads stay inside the source; they rotate and store nothing.
template <typename I>
struct KvAppendThread {
    bool live;
    I row, b;
    int h, t, d0;
    constexpr KvAppendThread(I i, I n8, int D, int Hkv, int T) : live(i < n8), row(0), b(0), h(0), t(0), d0(0) {
        const I ic = live ? i : 0;
        const int per = D / 8;
        row = ic / per;
        d0 = 8 * (int)(ic - row * per);
        const I bh = row / T;
        t = (int)(row - bh * T);
        b = bh / Hkv;
        h = (int)(bh - b * Hkv);
    }
    // an idle thread's row need not be one of its workgroup's, whose angles alone are in LDS
    constexpr bool rotates(int n_dims) const { return live && d0 < n_dims; }
};

// The rows whose angles a workgroup forms: r0 .. rl, or (single tokens: T == 1) their sequences, whose
// heads share a position.
template <typename I>
struct KvAngleRows {
    I r0, b0;
    int count;
    constexpr KvAngleRows(uint32_t block, I n8, int D, int Hkv, int T) : r0((I)block * 256 / (D / 8)), b0(0), count(0) {
        const I last = (I)block * 256 + 255, rl = (last < n8 - 1 ? last : n8 - 1) / (D / 8);
        b0 = T == 1 ? r0 / Hkv : 0;
        count = (int)(T == 1 ? rl / Hkv - b0 + 1 : rl - r0 + 1);
    }
    // the place (of `count`) of a rotating thread's angles
    constexpr int place(const KvAppendThread<I> &th, int T) const { return (int)(T == 1 ? th.b - b0 : th.row - r0); }
};
