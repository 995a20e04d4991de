"""bfloat16 and float32 queries over Q8_0 keys with an additive mask that blocks by its type's lowest
value, which is finite: a sequence whose keys are all so masked averages their values (adding a score to
that value leaves it), one with some keys visible sees only those, and -inf still blocks."""

import pytest
import torch

import gguf_train_amd as g
import oracle
from gguf_train_amd import _C

from _util import assert_close, oracle_forward, randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mdtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,G,S", [(128, 4, 5), (64, 1, 130), (128, 8, 3001)])
def test_masks_of_the_lowest_value(dev, dtype, mdtype, D, G, S):
    B, Hkv = 4, 2
    q = randn((B, Hkv * G, 1, D), S + D, dtype)
    blocks = [oracle.q8_0_quantize(randn((B, Hkv, S, D), S + i).numpy()) for i in (1, 2)]
    k, v = (torch.from_numpy(oracle.q8_0_dequantize(b).reshape(B, Hkv, S, D)) for b in blocks)
    m = torch.zeros((B, 1, 1, S), dtype=mdtype)
    m[0] = torch.finfo(mdtype).min
    m[1, ..., S // 2:] = torch.finfo(mdtype).min
    m[2] = torch.finfo(mdtype).min
    m[2, ..., S // 3:] = float("-inf")
    m[3] = float("-inf")
    qt = [g.QuantizedTensor(torch.from_numpy(b).to(dev), (B, Hkv, S, D)) for b in blocks]
    got = g.flash_attention(q.to(dev), *qt, m.to(dev), 0.0, False)
    assert _C.last_launch().startswith("decode q8_0"), _C.last_launch()
    assert_close(got, oracle_forward(q, k, v, mask=m.float()), dtype, f"{dtype} {mdtype} D={D} S={S}")
