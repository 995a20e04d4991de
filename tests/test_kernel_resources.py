"""Kernels whose time is a chain of latencies keep their values in registers: the compiler's resource
report of the KV-cache append names no private memory."""

import re
import subprocess
import sys
from pathlib import Path

import pytest

PKG = Path(__file__).resolve().parent.parent / "gguf_train_amd"


def _reports(source, tmp_path):
    """{kernel: bytes of private memory per lane} of one source, as the library's build compiles it."""
    sys.path.insert(0, str(PKG))
    try:
        import _build
    finally:
        sys.path.remove(str(PKG))
    if not Path(_build.HIPCC).exists():
        pytest.skip("no hipcc")
    p = subprocess.run([_build.HIPCC, *_build.HIP_FLAGS, "-Rpass-analysis=kernel-resource-usage", "--offload-device-only",
                        "-x", "hip", "-c", str(PKG / "csrc" / source), "-o", str(tmp_path / "o")], capture_output=True, text=True)
    assert p.returncode == 0, p.stderr
    names = re.findall(r"Function Name: (\S+)", p.stderr)
    sizes = re.findall(r"ScratchSize \[bytes/lane\]: (\d+)", p.stderr)
    assert names and len(names) == len(sizes)
    return dict(zip(names, map(int, sizes)))


def test_the_append_uses_no_private_memory(tmp_path):
    appends = {n: s for n, s in _reports("gt_convert.hip", tmp_path).items() if "kv_append_vec_kernel" in n}
    assert len(appends) == 24  # 3 sources, 4 caches, 2 index types
    assert not any(appends.values()), appends
