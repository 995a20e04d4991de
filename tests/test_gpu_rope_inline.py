"""RoPE angles formed inside the rotating kernels (few rows) against those of the table kernel (many
rows): the same bits, for single tokens and small groups, rows that straddle workgroups, both pairings
and partial rotations; and the KV cache's lengths after one-launch appends."""

import pytest
import torch

import gguf_train_amd as g

from _util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16, torch.float64])
@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("H,S,D,n_dims", [(3, 1, 64, 64), (32, 1, 128, 128), (5, 7, 80, 48), (2, 3, 256, 256), (1, 1, 6, 4),
                                          (7, 5, 24, 16)])
def test_rope_of_few_rows(dev, dtype, mode, H, S, D, n_dims):
    n = -(-2 ** 20 // (H * D))  # enough rows for the table
    pos = torch.randint(0, 5000, (n,), dtype=torch.int32, generator=torch.Generator().manual_seed(D)).to(dev)
    x = randn((1, H, n, D), D + H, dtype).to(dev)
    want = g.rope(x, pos, n_dims, mode)
    at = n // 2
    got = g.rope(x[:, :, at:at + S], pos[at:at + S], n_dims, mode)
    assert torch.equal(got, want[:, :, at:at + S])


@pytest.mark.parametrize("store", ["q8_0", torch.float16, torch.float32])
@pytest.mark.parametrize("mode,n_dims", [(0, 64), (2, 64), (2, 32)])
@pytest.mark.parametrize("B,Hkv,D", [(3, 5, 64), (1, 8, 128), (300, 1, 64)])
def test_single_token_appends_equal_one_long_append(dev, store, mode, n_dims, B, Hkv, D):
    T, extra = 6, -(-2 ** 19 // (B * Hkv * D)) + 1  # the long append is past the inline limit
    k, v = (randn((B, Hkv, T + extra, D), B + i, torch.float16).to(dev) for i in (0, 1))
    rope = {"mode": mode, "n_dims": n_dims}
    one, many = (g.KVCache(B, Hkv, T + extra, D, store, dev) for _ in range(2))
    one.append(k, v, rope=rope)
    for lo, hi in [(0, 1), (1, 2), (2, 5), (5, 6), (6, T + extra)]:
        many.append(k[:, :, lo:hi], v[:, :, lo:hi], rope=rope)
        assert many.lengths == [hi] * B
    data = lambda t: t.data if store == "q8_0" else t
    assert torch.equal(data(one.keys()), data(many.keys())) and torch.equal(data(one.values()), data(many.values()))
    many.clear(B - 1)
    if B > 1:
        assert many.lengths == [T + extra] * (B - 1) + [0]
    q = randn((B, Hkv, 1, D), 9, torch.float16).to(dev)
    full = one.attention(q)
    many.clear()
    many.append(k, v, rope=rope)
    assert torch.equal(many.attention(q), full)


def test_keys_and_values_of_two_dtypes(dev):
    c = g.KVCache(2, 2, 8, 64, torch.float16, dev)
    k, v = randn((2, 2, 3, 64), 1, torch.float32).to(dev), randn((2, 2, 3, 64), 2, torch.bfloat16).to(dev)
    for _ in range(2):
        c.append(k, v)
    assert c.lengths == [6, 6]
    assert torch.equal(c.keys()[:, :, 3:6], k.half()) and torch.equal(c.values()[:, :, 3:6], v.half())
    q = randn((2, 2, 1, 64), 3, torch.float16).to(dev)
    want = g.flash_attention(q, c.keys()[:, :, :6], c.values()[:, :, :6])
    assert torch.allclose(c.attention(q).float(), want.float(), atol=2e-3)
