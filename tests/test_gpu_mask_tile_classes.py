"""Masks whose tiles are of several classes at once in the half-precision prefill: a window of blocked,
clear and partly blocked tiles with finite values in some of them, so that a workgroup's list mixes tiles
that are skipped, unmasked, read as bits and read as values.  Sequences off the 4-key groups (half masks,
whose values are read from a copy), one mask for all sequences and one for each, with the causal mask
(whose unvisited tiles are not classed) and without; and that the calls do take the tile classes."""

import numpy as np
import pytest
import torch

import gguf_train_amd as g
from gguf_train_amd import _C

from _util import assert_close, oracle_forward, randn

pytestmark = pytest.mark.gpu


def _mask(batches, L, S, seed, low):
    rng = np.random.default_rng(seed)
    m = torch.zeros((batches, L, S))
    band = torch.ones((L, S), dtype=torch.bool).tril(S - L)
    keep = band & ~torch.ones((L, S), dtype=torch.bool).tril(S - L - 400)
    m.masked_fill_(~keep, float("-inf"))
    for b in range(batches):
        # finite values in scattered 40 x 50 patches, inside the window and past it
        for r0 in range(30 * (b + 1), L, 150):
            for c0 in range(0, S, 230):
                patch = torch.from_numpy(rng.standard_normal((min(40, L - r0), min(50, S - c0))).astype(np.float32))
                m[b, r0:r0 + 40, c0:c0 + 50] = torch.where(torch.isinf(m[b, r0:r0 + 40, c0:c0 + 50]), low, patch)
    return m


@pytest.mark.parametrize("dtype,D", [(torch.float16, 64), (torch.bfloat16, 64), (torch.float16, 128), (torch.bfloat16, 80)])
@pytest.mark.parametrize("L,S,batches,causal", [(300, 1201, 1, False), (300, 1204, 2, False), (1090, 1090, 2, True),
                                                (1031, 1100, 1, True)])
@pytest.mark.parametrize("mdtype", ["same", torch.float32])
@pytest.mark.parametrize("low", [-1e4, float("-inf")])
def test_lists_of_several_classes(dev, dtype, D, L, S, batches, causal, mdtype, low):
    B, H, Hkv = 2, 8, 4
    q, k, v = (randn((B, h, n, D), L + i, dtype) for i, (h, n) in enumerate(((H, L), (Hkv, S), (Hkv, S))))
    mask = _mask(batches, L, S, L + S, low).to(dtype if mdtype == "same" else mdtype)
    mask = mask[0] if batches == 1 else mask[:, None]
    want = oracle_forward(q, k, v, mask=mask.float(), is_causal=causal)
    qd, kd, vd, md = (t.to(dev) for t in (q, k, v, mask))
    got = g.flash_attention(qd, kd, vd, md, 0.0, causal)
    # float32 values are read in place: whole 4-key groups; of any mask, 8 or (half) 4 key tiles
    tiles = mdtype == "same" or S % 4 == 0
    assert _C.last_launch().endswith(" mask_tiles") == tiles, _C.last_launch()
    assert_close(got, want, dtype, "out")
    out, lse, out32 = g.flash_attention_train(qd, kd, vd, md, 0.0, causal)
    assert_close(out32, want, dtype, "out32", out_dtype=torch.float32)
    wide = torch.full((*mask.shape[:-1], S + 5), 7.0, dtype=mask.dtype, device=dev)  # rows off the 4-key groups
    wide[..., :S] = md
    view = g.flash_attention(qd, kd, vd, wide[..., :S], 0.0, causal)
    assert _C.last_launch().endswith(" mask_tiles") == (mdtype == "same"), _C.last_launch()
    assert_close(view, want, dtype, "view")


@pytest.mark.parametrize("nkt,mdtype,tiles", [(3, "same", False), (4, "same", True), (7, torch.float32, False), (8, torch.float32, True),
                                              (7, torch.bool, False), (8, torch.bool, True)])
@pytest.mark.parametrize("D,bn", [(64, 128), (128, 64)])
def test_the_line_is_a_number_of_key_tiles(dev, D, bn, nkt, mdtype, tiles):
    B, H, L, S = 1, 4, 40, nkt * bn
    q, k, v = (randn((B, H, n, D), n + i, torch.float16) for i, n in enumerate((L, S, S)))
    keep = torch.ones((L, S), dtype=torch.bool).tril(S - L)
    mask = keep if mdtype == torch.bool else torch.zeros((L, S), dtype=torch.float16 if mdtype == "same" else mdtype).masked_fill(
        ~keep, float("-inf"))
    got = g.flash_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev))
    assert _C.last_launch().endswith(" mask_tiles") == tiles, _C.last_launch()
    assert_close(got, oracle_forward(q, k, v, mask=mask if mdtype == torch.bool else mask.float()), torch.float16, "out")
