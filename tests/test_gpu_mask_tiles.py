"""Forward calls whose mask varies along the query rows and is shared by the heads: the half-precision
prefill walks a list of key tiles by class (blocked throughout, clear, only blocking, other values).
Masks of every dtype, with sequences that are and are not whole tiles or 4-key groups, strides other
than dense, rows and tiles that are blocked throughout, against the float64 oracle."""

import numpy as np
import pytest
import torch

import gguf_train_amd as g

from _util import assert_close, oracle_forward, randn

pytestmark = pytest.mark.gpu


def _mask(kind, batches, L, S, seed):
    rng = np.random.default_rng(seed)
    band = torch.ones((L, S), dtype=torch.bool).tril(S - L)
    if kind == "band":
        m = band[None].repeat(batches, 1, 1)
    elif kind == "window":  # clear, mixed and blocked tiles on both sides
        m = (band & ~torch.ones((L, S), dtype=torch.bool).tril(S - L - 150))[None].repeat(batches, 1, 1)
        m[..., : L // 3, :] = False  # whole rows blocked
    else:
        m = torch.from_numpy(rng.random((batches, L, S)) < 0.5)
    bias = torch.from_numpy(rng.standard_normal((batches, L, S)).astype(np.float32))
    return m, bias


@pytest.mark.parametrize("dtype,D", [(torch.float16, 128), (torch.bfloat16, 64), (torch.float16, 80)])
@pytest.mark.parametrize("L,S,batches,causal", [(130, 590, 1, False), (257, 1025, 2, False), (1030, 1030, 1, True), (2, 64, 1, False),
                                                (129, 1031, 1, False), (100, 1024, 2, True)])
@pytest.mark.parametrize("kind,mdtype", [("band", torch.bool), ("window", torch.bool), ("band", "same"), ("window", torch.float32),
                                         ("bias", "same"), ("bias", torch.float32), ("random", torch.bool)])
def test_masks_shared_by_the_heads(dev, dtype, D, L, S, batches, causal, kind, mdtype):
    B, H, Hkv = 2, 8, 4
    mdtype = dtype if mdtype == "same" else mdtype
    q, k, v = (randn((B, h, n, D), L + i, dtype) for i, (h, n) in enumerate(((H, L), (Hkv, S), (Hkv, S))))
    keep, bias = _mask(kind, batches, L, S, L + S)
    if mdtype == torch.bool:
        mask = keep
    elif kind == "bias":  # values, some blocked, and (with a band) clear tiles are none
        mask = bias.masked_fill(~keep, float("-inf")).to(mdtype)
    else:
        mask = torch.zeros(keep.shape, dtype=mdtype).masked_fill(~keep, float("-inf"))
    mask = mask[0] if batches == 1 else mask[:, None]
    got = g.flash_attention(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), 0.0, causal)
    want = oracle_forward(q, k, v, mask=mask.float() if mdtype != torch.bool else mask, is_causal=causal)
    assert_close(got, want, dtype, f"{kind} {mdtype}")
    # the same mask as a view with another layout
    wide = torch.zeros((*mask.shape[:-1], S + 3), dtype=mask.dtype, device=dev)
    wide[..., :S] = mask.to(dev)
    view = g.flash_attention(q.to(dev), k.to(dev), v.to(dev), wide[..., :S], 0.0, causal)
    if mdtype == torch.float32:  # rows off the 4-key groups: read as given, in another order of operations
        assert_close(view, want, dtype, f"{kind} view")
    else:
        assert torch.equal(view, got)
    turned = mask.to(dev).transpose(-1, -2).contiguous().transpose(-1, -2)
    assert_close(g.flash_attention(q.to(dev), k.to(dev), v.to(dev), turned, 0.0, causal), want, dtype, "turned")


@pytest.mark.parametrize("dtype,D", [(torch.float16, 64), (torch.bfloat16, 128)])
def test_training_forward_and_lse(dev, dtype, D):
    B, H, L, S = 1, 8, 190, 700
    q, k, v = (randn((B, H, n, D), 3 + i, dtype) for i, n in enumerate((L, S, S)))
    keep, bias = _mask("window", 1, L, S, 9)
    mask = torch.zeros((L, S), dtype=dtype).masked_fill(~keep[0], float("-inf"))
    out, lse, out32 = g.flash_attention_train(q.to(dev), k.to(dev), v.to(dev), mask.to(dev), 0.0, False)
    want, want_lse = oracle_forward(q, k, v, mask=mask.float(), return_lse=True)
    assert_close(out32, want, dtype, "out32", out_dtype=torch.float32)
    seen = np.isfinite(want_lse)
    assert np.array_equal(np.isfinite(lse.cpu().numpy()), seen)
    assert np.abs(lse.cpu().double().numpy() - want_lse)[seen].max() < 1e-4
