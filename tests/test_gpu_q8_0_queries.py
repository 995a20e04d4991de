"""Single-query attention straight from Q8_0 K/V for every query dtype, at slice sizes that are and
are not multiples of 16 bytes (a slice is S rows of 34 D / 32 bytes), against the oracle on the
dequantized values.

Float32 queries are held to a bound of their own: the products are exact and each of the S + D
float32 additions and the exponential round by at most 2^-24 relative, so the error of a row is within
a few 2^-24 sqrt(S) of the weighted sum of |v| (random signs); 2^-20 of max|v| covers S up to 3001
(sqrt(3001) = 55, with scores of up to 8 whose own rounding moves p by 2^-21)."""

import numpy as np
import pytest
import torch

import oracle
from _util import assert_close, oracle_forward, randn

pytestmark = pytest.mark.gpu


def _cache(dev, shape, seed):
    blocks = oracle.q8_0_quantize(randn(shape, seed).numpy())
    values = torch.from_numpy(oracle.q8_0_dequantize(blocks).reshape(shape))
    return blocks, values


@pytest.fixture(scope="module")
def g():
    import gguf_train_amd

    return gguf_train_amd


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D,G,S", [(128, 4, 1), (64, 1, 1), (64, 2, 3), (128, 4, 127), (128, 1, 129), (64, 8, 130), (64, 3, 515),
                                   (128, 4, 3001), (128, 12, 1024)])
@pytest.mark.parametrize("mask", ["none", "pad", "bool"])
def test_single_query_of_every_dtype(dev, g, dtype, D, G, S, mask):
    from gguf_train_amd import _C

    B, Hkv = 2, 2
    q = randn((B, Hkv * G, 1, D), S + D + G, dtype)
    (kb, k), (vb, v) = _cache(dev, (B, Hkv, S, D), S + 1), _cache(dev, (B, Hkv, S, D), S + 2)
    m = None
    if mask == "pad":
        m = torch.zeros((B, 1, 1, S))
        m[1, ..., (S + 1) // 2:] = float("-inf")
    elif mask == "bool":
        m = torch.from_numpy(np.random.default_rng(S).random((B, Hkv * G, 1, S)) < 0.7)
        m[..., 0] = True
    qt = [g.QuantizedTensor(torch.from_numpy(x).to(dev), (B, Hkv, S, D)) for x in (kb, vb)]
    got = g.flash_attention(q.to(dev), *qt, m.to(dev) if m is not None else None, 0.0, False)
    assert _C.last_launch().startswith(f"decode q8_0 D={D}"), _C.last_launch()
    assert got.dtype == dtype
    want = oracle_forward(q, k, v, mask=m)
    assert_close(got, want, dtype, f"{dtype} D={D} G={G} S={S} {mask}")
    if dtype == torch.float32:
        err = np.abs(got.double().cpu().numpy() - np.asarray(want, np.float64)).max()
        assert err <= 2.0 ** -20 * max(1.0, float(v.abs().max())), err


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_masked_keys_of_infinite_scale_add_nothing(dev, g, dtype):
    B, H, S, D = 1, 4, 200, 128
    q = randn((B, H, 1, D), 5, dtype)
    (kb, k), (vb, v) = _cache(dev, (B, 1, S, D), 6), _cache(dev, (B, 1, S, D), 7)
    keep = torch.ones((1, 1, 1, S), dtype=torch.bool)
    keep[..., 150:] = False
    vb = vb.reshape(S, 4, 34).copy()
    vb[160:, 1, :2] = np.array([0x00, 0x7C], np.uint8)  # float16 infinity
    qt = [g.QuantizedTensor(torch.from_numpy(np.ascontiguousarray(x).reshape(-1)).to(dev), (B, 1, S, D)) for x in (kb, vb)]
    got = g.flash_attention(q.to(dev), *qt, keep.to(dev), 0.0, False)
    assert_close(got, oracle_forward(q, k[:, :, :150], v[:, :, :150]), dtype, "masked infinite scales")
