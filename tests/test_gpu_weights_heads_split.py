"""Averaged float32 weights of small grids: a workgroup's wavefronts take the heads in turn and add their
tiles.  Grids on both sides of the rule (up to 128 workgroups of 128 rows and 64 keys), head counts that are and
are not whole rounds of the four wavefronts, rows and keys that are not whole tiles, against the mean of
the weights per head."""

import pytest
import torch

import gguf_train_amd as g
from gguf_train_amd import _ops

from _util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,L,S,D", [(1, 4, 4, 1, 5, 64), (2, 5, 5, 33, 64, 64), (1, 8, 2, 130, 257, 128), (3, 3, 3, 70, 66, 64),
                                           (8, 9, 9, 100, 1000, 64), (8, 4, 4, 100, 1025, 64),
                                           (8, 9, 9, 100, 1985, 64), (8, 4, 4, 100, 2049, 64)])
@pytest.mark.parametrize("causal,mkind", [(False, None), (True, "pad"), (False, "bool")])
def test_average_is_the_mean_of_the_heads(dev, B, H, Hkv, L, S, D, causal, mkind):
    q, k, v = (randn((B, h, n, D), L + S + i).to(dev) for i, (h, n) in enumerate(((H, L), (Hkv, S), (Hkv, S))))
    mask = None
    if mkind == "pad":
        mask = torch.zeros((B, 1, 1, S), device=dev)
        mask[0, ..., S - S // 3:] = float("-inf")
    elif mkind == "bool":
        mask = randn((L, S), 7).to(dev) > -0.5
        mask[:, 0] = True
    _, lse = g.flash_attention_lse(q, k, v, mask, 0.0, causal)
    each = _ops.attention_weights(q, k, mask, lse, 0.0, causal, False).double().mean(1)
    got = _ops.attention_weights(q, k, mask, lse, 0.0, causal, True).double()
    # weights are at most 1: H products by 1 / H and H - 1 sums, each within 2^-24 of a value below 1
    assert (got - each).abs().max().item() <= 2 * H * 2.0 ** -24
