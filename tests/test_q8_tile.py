"""The byte offsets of the Q8_0 decode kernel's tiles (csrc/q8_tile.h), compiled for the host: every dword
of a row that exists reaches its place in the tile, for slices of every remainder and those that end
within a tile of 4 GiB, where a tile's end passes 2^32."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gguf_train_amd" / "csrc"

PROGRAM = r"""
#include "q8_tile.h"
#include <cstdio>
#include <initializer_list>

// The tile of 32 rows at key `key`, as the kernel loads and stages it: dword i of the piece at `pos` holds
// dword read_at / 4 + early + i of the slice.
static bool tile_ok(uint64_t S, uint32_t rb, uint64_t key) {
    const uint32_t size = (uint32_t)(S * rb), last16 = size - 16, tb = 32 * rb, t0 = (uint32_t)(key * rb);
    const bool ends = gtq8::ends_inside_piece(t0, tb, last16);
    for (uint32_t pos = 0; pos < tb; pos += 16) {
        const uint32_t off = t0 + pos, at = gtq8::read_at(off, last16);
        if (at > last16) return false;  // inside the slice
        const uint32_t early = ends ? gtq8::dwords_early(off, last16) : 0;
        for (uint32_t i = 0; i < 4; ++i) {
            const uint64_t want = key * rb + pos + 4 * i;
            if (want >= S * rb) continue;  // past the last row
            if (i + early >= 4 || at + 4 * (uint64_t)(early + i) != want) return false;
        }
    }
    return true;
}

int main() {
    int bad = 0;
    for (uint32_t rb : {68u, 136u}) {  // head sizes 64 and 128
        const uint64_t most = 0xffffffffull / rb;
        auto check = [&](uint64_t S) {
            for (uint64_t key = S > 200 ? (S - 200) / 32 * 32 : 0; key < S; key += 32)
                if (!tile_ok(S, rb, key)) {
                    printf("row bytes %u S %llu key %llu\n", rb, (unsigned long long)S, (unsigned long long)key);
                    ++bad;
                }
        };
        for (uint64_t S = 1; S < 400; ++S) check(S);
        for (uint64_t S : {3001, 8191, 8192, 100003}) check(S);
        for (uint64_t S = most - 400; S <= most; ++S) check(S);
    }
    return bad != 0;
}
"""


def test_every_dword_of_a_row_reaches_its_place(tmp_path):
    (tmp_path / "t.cpp").write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", f"-I{CSRC}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    r = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
