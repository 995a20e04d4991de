"""Which way the half-precision prefill deals query tiles to workgroups (csrc/prefill_order.h), compiled
for the host: pairs of tiles where they were measured to be the faster, single tiles where those were."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gguf_train_amd" / "csrc"

# (causal, float16 with one operand of P.V, D, tile classes or dropout, query tiles, heads) -> the order
PAIRS, SINGLE, FOLDED, HEAD_MAJOR = range(4)
MEASURED = [
    # causal: nearly full rounds; short float16 sequences from 1.5 rounds on; else single
    (1, 1, 128, 0, 16, 128, PAIRS), (1, 0, 64, 0, 8, 128, PAIRS), (1, 1, 128, 0, 1, 3, PAIRS), (1, 0, 128, 0, 16, 32, FOLDED),
    (1, 1, 128, 0, 4, 384, PAIRS), (1, 1, 64, 0, 6, 384, PAIRS), (1, 1, 128, 0, 8, 192, PAIRS), (1, 1, 64, 0, 8, 320, PAIRS),
    (1, 1, 128, 0, 4, 320, SINGLE), (1, 0, 128, 0, 4, 384, SINGLE), (1, 0, 64, 0, 8, 320, SINGLE), (1, 1, 64, 0, 3, 384, SINGLE),
    (1, 1, 128, 0, 16, 96, SINGLE), (1, 1, 64, 0, 11, 192, SINGLE), (1, 1, 128, 1, 4, 384, SINGLE), (1, 1, 80, 0, 4, 384, SINGLE),
    # without the causal mask
    (0, 1, 64, 0, 4, 208, PAIRS), (0, 0, 64, 0, 8, 104, PAIRS), (0, 1, 128, 0, 8, 112, PAIRS), (0, 1, 64, 0, 4, 500, PAIRS),
    (0, 0, 128, 0, 4, 256, HEAD_MAJOR), (0, 1, 64, 0, 8, 160, HEAD_MAJOR), (0, 1, 128, 0, 8, 200, HEAD_MAJOR),
    (0, 1, 128, 0, 4, 128, HEAD_MAJOR), (0, 1, 64, 0, 2, 512, HEAD_MAJOR), (0, 1, 64, 0, 24, 96, HEAD_MAJOR),
    (0, 1, 64, 1, 4, 256, HEAD_MAJOR),
]


def test_the_order_of_measured_shapes(tmp_path):
    rows = "".join(f"{{{', '.join(map(str, m[:6]))}}}, " for m in MEASURED)
    (tmp_path / "t.cpp").write_text(
        f'#include "prefill_order.h"\n#include <cstdio>\nint main() {{ const int m[][6] = {{{rows}}};\n'
        'for (auto &x : m) printf("%d", (int)tile_order_of(x[0], x[1], x[2], x[3], x[4], x[5])); }\n')
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, check=True).stdout
    assert out == "".join(str(m[6]) for m in MEASURED)
