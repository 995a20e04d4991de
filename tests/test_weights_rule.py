"""When the averaged float32 weights split their heads over the wavefronts (csrc/attn_weights_rule.h),
compiled for the host: where it was measured to be the faster one, and nowhere that it was the slower."""

import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parent.parent / "gguf_train_amd" / "csrc"

# (B, H, L, S): split the faster one / the slower one (fp32, head sizes 64 and 128, causal or not, padded or not)
FASTER = [(1, 4, 128, 128), (8, 4, 256, 256), (8, 8, 256, 256), (4, 8, 512, 512), (4, 5, 512, 512), (3, 5, 512, 512),
          (15, 5, 250, 250), (15, 4, 256, 256), (1, 8, 1024, 900)]
SLOWER = [(7, 5, 512, 512), (7, 4, 512, 512), (7, 8, 512, 512), (6, 5, 512, 512), (5, 5, 512, 512), (5, 6, 512, 512),
          (1, 5, 1024, 1900), (20, 5, 256, 256), (28, 5, 250, 250), (7, 12, 512, 512), (8, 3, 256, 256)]


def test_the_line_lies_between_the_measured_shapes(tmp_path):
    shapes = "".join(f"{{{', '.join(map(str, s))}}}, " for s in FASTER + SLOWER)
    (tmp_path / "t.cpp").write_text(
        f'#include "attn_weights_rule.h"\n#include <cstdio>\nint main() {{ const int64_t s[][4] = {{{shapes}}};\n'
        'for (auto &x : s) printf("%d", (int)f32_heads_split((x[2] + 127) / 128 * x[0], (x[3] + 63) / 64, x[1], 4)); }\n')
    subprocess.run(["g++", "-std=c++17", f"-I{CSRC}", str(tmp_path / "t.cpp"), "-o", str(tmp_path / "t")], check=True)
    out = subprocess.run([str(tmp_path / "t")], capture_output=True, text=True, check=True).stdout
    assert out == "1" * len(FASTER) + "0" * len(SLOWER)
