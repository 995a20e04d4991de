"""Rows and angles of a KV-cache append's threads (csrc/rope_rows.h), compiled for the host: every thread
that rotates finds its row's angles among those its workgroup formed, threads past the last row read
none, and a workgroup's angles fit their array.  Sequences, heads and tokens that do and do not fill
whole workgroups."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gguf_train_amd" / "csrc"

PROGRAM = r"""
#include "rope_rows.h"
#include <cstdio>
#include <initializer_list>

template <typename I>
static bool append_ok(I B, int Hkv, int T, int D) {
    const I n8 = B * Hkv * T * (D / 8);
    for (uint32_t block = 0; (int64_t)block * 256 < n8; ++block) {
        const KvAngleRows<I> ang(block, n8, D, Hkv, T);
        for (int n_dims = 16; n_dims <= D; n_dims += 16) {
            const int half = n_dims / 2, formed = ang.count * half;
            if (ang.count < 1 || formed > kRopeInlineEntries) return false;
            for (int tid = 0; tid < 256; ++tid) {
                const I i = (I)block * 256 + tid;
                const KvAppendThread<I> th(i, n8, D, Hkv, T);
                if (th.live != (i < n8) || th.d0 < 0 || th.d0 + 8 > D || th.row < 0 || th.row >= B * Hkv * T) return false;
                if (th.live && (th.row * (D / 8) + th.d0 / 8 != i || (th.b * Hkv + th.h) * T + th.t != th.row)) return false;
                if (!th.rotates(n_dims)) continue;
                const int place = ang.place(th, T);
                if (!th.live || place < 0 || place >= ang.count) return false;
                if (T == 1 ? ang.b0 + place != th.b : ang.r0 + place != th.row) return false;
                // both pairings read `pairs` angles from `first` on
                for (int neox : {0, 1}) {
                    const int first = neox ? (th.d0 < half ? th.d0 : th.d0 - half) : th.d0 / 2, pairs = neox ? 8 : 4;
                    if (first < 0 || first + pairs > half) return false;
                }
            }
        }
    }
    return true;
}

int main() {
    int bad = 0;
    for (int D : {16, 48, 64, 80, 120, 128, 256})
        for (int Hkv : {1, 2, 5, 8})
            for (int T : {1, 2, 3, 17, 100})
                for (int B : {1, 2, 3, 30, 300}) {
                    if ((int64_t)B * Hkv * T * (D / 8) > kRopeInlineThreads || D > kRopeInlineMaxDim) continue;
                    if (!append_ok<int32_t>(B, Hkv, T, D) || !append_ok<int64_t>(B, Hkv, T, D)) {
                        printf("B %d Hkv %d T %d D %d\n", B, Hkv, T, D);
                        ++bad;
                    }
                }
    return bad != 0;
}
"""


def test_rotating_threads_find_their_angles(tmp_path):
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O2", f"-I{CSRC}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
