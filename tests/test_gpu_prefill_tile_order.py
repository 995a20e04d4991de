"""Every way the half-precision prefill deals query tiles to workgroups (pairs of tiles, single tiles
heaviest first, single tiles folded, head by head), with heads that do and do not divide among the 8
XCDs and odd tile counts.  The output is the caller's own, NaN before the call, so a row that no
workgroup writes shows; every head is compared with the float32 kernels, whose workgroups are dealt
otherwise, and a few with the float64 oracle."""

import pytest
import torch

import gguf_train_amd as g
from gguf_train_amd import _C

from _util import assert_close, oracle_forward, randn
from test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu


def _order(causal, light, D, nq, heads):
    """The rule under test, restated: 512 resident workgroups."""
    pairs = (nq + 1) // 2 * heads
    slots = (pairs + 511) // 512 * 512
    brief = nq in (4, 6, 8) and D in (64, 128)
    if not causal:
        return "pairs" if brief and (light or D == 64) and pairs * 16 >= slots * 13 else "head major"
    if nq == 1 or pairs * 16 >= slots * 15 or (brief and light and pairs >= 768):
        return "pairs"
    return "folded" if nq * heads <= 512 else "single"


@pytest.mark.parametrize("dtype,B,H,Hkv,L,S,D,causal,order", [
    (torch.float16, 1, 3, 1, 300, 300, 128, True, "folded"),
    (torch.bfloat16, 2, 8, 4, 257, 400, 64, True, "folded"),
    (torch.float16, 1, 8, 2, 129, 129, 64, True, "folded"),
    (torch.float16, 1, 32, 32, 2300, 300, 64, True, "single"),
    (torch.bfloat16, 1, 36, 12, 2305, 200, 64, True, "single"),
    (torch.float16, 4, 64, 64, 500, 200, 64, True, "pairs"),
    (torch.float16, 2, 5, 5, 128, 128, 128, True, "pairs"),
    (torch.bfloat16, 1, 6, 2, 400, 130, 128, False, "head major"),
    (torch.float16, 2, 8, 8, 385, 100, 64, False, "head major"),
    (torch.float16, 6, 64, 8, 390, 70, 64, True, "pairs"),  # four tiles, one and a half rounds
    (torch.bfloat16, 6, 64, 8, 390, 70, 64, True, "single"),
    (torch.bfloat16, 4, 54, 54, 390, 70, 64, False, "pairs"),  # 13.5 of 16 slots
    (torch.float16, 6, 35, 7, 500, 90, 128, False, "pairs"),
    (torch.bfloat16, 6, 35, 7, 500, 90, 128, False, "head major"),
])
def test_every_tile_order(dev, dtype, B, H, Hkv, L, S, D, causal, order):
    assert _order(causal, dtype == torch.float16, D, (L + 127) // 128, B * H) == order
    q, k, v = (randn((B, h, n, D), i + L, dtype) for i, (h, n) in enumerate(((H, L), (Hkv, S), (Hkv, S))))
    qd, kd, vd = (t.to(dev) for t in (q, k, v))
    got = torch.full((B, H, L, D), float("nan"), dtype=dtype, device=dev)
    assert noalloc(qd, kd, vd, None, 0.0, causal, got) == 0, _C.last_error()
    assert _C.last_launch().startswith(f"prefill {'f16' if dtype == torch.float16 else 'bf16'} D={D} "), _C.last_launch()
    every = g.flash_attention(qd.float(), kd.float(), vd.float(), None, 0.0, causal)
    assert_close(got, every.double().cpu().numpy(), dtype, "every head")
    assert torch.equal(g.flash_attention(qd, kd, vd, None, 0.0, causal), got)
    G = H // Hkv
    for b, h in {(0, 0), (B - 1, H - 1), (0, H // 2)}:
        kv = slice(h // G, h // G + 1)
        want = oracle_forward(q[b:b + 1, h:h + 1], k[b:b + 1, kv], v[b:b + 1, kv], is_causal=causal)
        assert_close(got[b:b + 1, h:h + 1], want, dtype, f"head {b},{h}")
