"""Gradients written in the inputs' dtype equal the float32 gradients rounded once, on the MFMA
kernels (head sizes of their own and padded ones), the generic kernels and with dropout."""

import pytest
import torch

import gguf_train_amd as g
from gguf_train_amd import _ops

from _util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32, torch.float64])
@pytest.mark.parametrize("D,L,S,Hkv,causal,p", [(64, 129, 130, 2, True, 0.0), (128, 33, 200, 4, False, 0.0),
                                                (80, 65, 65, 4, True, 0.0), (100, 40, 40, 2, False, 0.0),
                                                (160, 17, 19, 4, True, 0.0), (64, 70, 70, 4, True, 0.2), (1, 1, 1, 4, False, 0.0)])
def test_gradients_in_the_inputs_dtype(dev, dtype, D, L, S, Hkv, causal, p):
    B, H, seed = 2, 4, 11
    q, dout = (randn((B, H, L, D), D + i, dtype).to(dev) for i in (0, 1))
    k, v = (randn((B, Hkv, S, D), D + i, dtype).to(dev) for i in (2, 3))
    if p:
        out, lse, out32 = g.flash_attention_dropout(q, k, v, None, 0.0, causal, p, seed)
        want = g.flash_attention_dropout_backward(dout, q, k, v, None, out if out32 is None else out32, lse, 0.0, causal, p, seed)
    else:
        out, lse, out32 = g.flash_attention_train(q, k, v, None, 0.0, causal)
        want = g.flash_attention_backward(dout, q, k, v, None, out if out32 is None else out32, lse, 0.0, causal)
    got = _ops.input_gradients(dout, q, k, v, None, out if out32 is None else out32, lse, 0.0, causal, p, seed)
    for a, b in zip(got, want):
        assert a.dtype == dtype
        assert torch.equal(a, b.to(dtype))


def test_mixed_dtypes_keep_float32_gradients(dev):
    q = randn((1, 2, 20, 64), 1, torch.float16).to(dev)
    k, v = (randn((1, 2, 20, 64), i, torch.bfloat16).to(dev) for i in (2, 3))
    dout = randn((1, 2, 20, 64), 4, torch.float16).to(dev)
    out, lse, out32 = g.flash_attention_train(q, k, v, None, 0.0, True)
    res = out if out32 is None else out32
    got = _ops.input_gradients(dout, q, k, v, None, res, lse, 0.0, True)
    want = g.flash_attention_backward(dout, q, k, v, None, res, lse, 0.0, True)
    assert all(a.dtype == torch.float32 and torch.equal(a, b) for a, b in zip(got, want))
