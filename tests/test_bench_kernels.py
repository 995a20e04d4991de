"""The kernels whose counters and durations bench.py summarises are in the built library under the names it
looks for (a template parameter more or less would leave a configuration out)."""

import importlib.util
import re
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def _bench():
    spec = importlib.util.spec_from_file_location("_bench_names", ROOT / "bench.py")
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def test_every_summarised_kernel_is_in_the_library():
    bench = _bench()
    lib = (ROOT / "gguf_train_amd" / "libgt_attn.so").read_bytes()
    names = {n.decode() for n in re.findall(rb"_ZN12_GLOBAL__N_1[A-Za-z0-9_]+", lib)}
    shown = subprocess.run(["c++filt"], input="\n".join(sorted(names)), capture_output=True, text=True, check=True).stdout
    for table in (bench.TRAFFIC_KERNELS, bench.TRACE_KERNELS):
        for config, patterns in table.items():
            for p in [patterns] if isinstance(patterns, str) else patterns:
                # rocprofv3 prints names that its demangler knows not (float16 parameters) as they are
                assert any(p in n for n in names) or p in shown, (config, p)
