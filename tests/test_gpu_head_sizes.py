"""Head sizes 80 and 96 in float16 and bfloat16: the prefill and backward kernels read, compute and write
them without padding.  Sizes around the tiles (128 query rows and 128 or 64 keys), GQA, causal or not,
masks and dropout against the float64 oracle; rows the kernels cannot read in place are copied and give
the same bits; sizes between pad to the next of them; what lies beyond a row's 80 values is never read
into a result."""

import numpy as np
import pytest
import torch

import gguf_train_amd as g
import oracle
from gguf_train_amd import _C

from _util import assert_close, oracle_forward, randn, to_oracle

pytestmark = pytest.mark.gpu


def _mask(kind, B, L, S, seed):
    rng = np.random.default_rng(seed)
    if kind == "bool":
        m = torch.from_numpy(rng.random((L, S)) < 0.7)
        m[:, 0] = True
        return m
    if kind == "add":
        return torch.from_numpy(rng.standard_normal((B, 1, L, S)).astype(np.float32))
    m = torch.zeros(B, 1, 1, S)
    m[0, ..., S - S // 4:] = float("-inf")
    return m


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [80, 96, 72])
@pytest.mark.parametrize("L,S,H,Hkv,causal,mkind", [(2, 3, 2, 2, False, None), (31, 65, 4, 2, False, "pad"), (128, 128, 2, 2, True, None),
                                                    (129, 257, 4, 1, True, "pad"), (200, 120, 2, 1, True, "bool"),
                                                    (130, 192, 4, 4, False, "add")])
def test_forward_and_backward(dev, dtype, D, L, S, H, Hkv, causal, mkind):
    B, seed = 2, L + S + D
    q, k, v, dout = (randn((B, h, n, D), seed + i, dtype) for i, (h, n) in enumerate(((H, L), (Hkv, S), (Hkv, S), (H, L))))
    mask = None if mkind is None else _mask(mkind, B, L, S, seed)
    md = None if mask is None else mask.to(dev)
    want = oracle_forward(q, k, v, mask=mask, is_causal=causal)
    assert_close(g.flash_attention(q.to(dev), k.to(dev), v.to(dev), md, 0.0, causal), want, dtype, "inference")
    out, lse, out32 = g.flash_attention_train(q.to(dev), k.to(dev), v.to(dev), md, 0.0, causal)
    assert f"D={max(D, 80)} " in _C.last_launch() and _C.last_launch().startswith("prefill "), _C.last_launch()
    assert_close(out32, want, dtype, "out32", out_dtype=torch.float32)
    grads = g.flash_attention_backward(dout.to(dev), q.to(dev), k.to(dev), v.to(dev), md, out32, lse, 0.0, causal)
    assert _C.last_launch().endswith(f"backward mfma {'f16' if dtype == torch.float16 else 'bf16'} D={max(D, 80)}"), _C.last_launch()
    wants = oracle.flash_attention_backward(to_oracle(dout), to_oracle(q), to_oracle(k), to_oracle(v),
                                            mask=None if mask is None else to_oracle(mask), is_causal=causal)
    for name, got, ref in zip(("dq", "dk", "dv"), grads, wants):
        assert_close(got, ref, torch.bfloat16, name, out_dtype=torch.float32)


@pytest.mark.parametrize("D", [80, 96])
def test_views_read_in_place_and_rows_that_are_copied(dev, D):
    B, H, L = 2, 4, 150
    base = [randn((B, L, H, D), 40 + i, torch.bfloat16).to(dev) for i in range(4)]
    dense = [t.transpose(1, 2).contiguous() for t in base]
    want = g.flash_attention_train(*dense[:3], None, 0.0, True)
    wgrad = g.flash_attention_backward(dense[3], *dense[:3], None, want[2], want[1], 0.0, True)
    wide = torch.zeros((B, H, L, D + 9), dtype=torch.bfloat16, device=dev)  # rows off 16 bytes
    odd = []
    for t in dense:
        w = wide.clone()
        w[..., 1:1 + D] = t
        odd.append(w[..., 1:1 + D])
    for views in ([t.transpose(1, 2) for t in base], odd):
        got = g.flash_attention_train(*views[:3], None, 0.0, True)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        grads = g.flash_attention_backward(views[3], *views[:3], None, got[2], got[1], 0.0, True)
        assert all(torch.equal(a, b) for a, b in zip(grads, wgrad))


@pytest.mark.parametrize("L", [1, 70])
def test_what_follows_a_row_stays_out(dev, L):
    # rows of 80 inside rows of 96 whose last 16 are NaN
    B, H, S, D = 1, 2, 90, 80
    q, k, v = (randn((B, H, n, D), 50 + i, torch.float16) for i, n in enumerate((L, S, S)))
    views = []
    for t in (q, k, v):
        w = torch.full((*t.shape[:-1], 96), float("nan"), dtype=torch.float16, device=dev)
        w[..., :D] = t.to(dev)
        views.append(w[..., :D])
    assert_close(g.flash_attention(*views, None, 0.0, False), oracle_forward(q, k, v), torch.float16, "out")


def test_dropout(dev):
    B, H, L, D, p, seed = 1, 2, 150, 96, 0.2, 23
    q, k, v, dout = (randn((B, H, L, D), i + 60, torch.float16) for i in range(4))
    out, lse, out32 = g.flash_attention_dropout(q.to(dev), k.to(dev), v.to(dev), None, 0.0, True, p, seed)
    grads = g.flash_attention_dropout_backward(dout.to(dev), q.to(dev), k.to(dev), v.to(dev), None, out32, lse, 0.0, True, p, seed)
    keep = oracle.dropout_keep(B, H, L, L, p, seed)
    ref, refs = oracle.attention_dropout(to_oracle(q), to_oracle(k), to_oracle(v), keep, p, is_causal=True,
                                         dout=to_oracle(dout), out_dtype=oracle.F64)
    assert_close(out32, ref, torch.float16, "out32", out_dtype=torch.float32)
    for name, got, want in zip(("dq", "dk", "dv"), grads, refs):
        assert_close(got, want, torch.bfloat16, name, out_dtype=torch.float32)


@pytest.mark.parametrize("offset", [0, 1, 4])
def test_callers_output_off_the_stores_alignment(dev, offset):
    from test_zz_no_alloc import noalloc

    B, H, L, D = 1, 2, 40, 80
    q, k, v = (randn((B, H, L, D), 70 + i, torch.float16).to(dev) for i in range(3))
    flat = torch.zeros(B * H * L * D + offset, dtype=torch.float16, device=dev)
    out = flat[offset:].view(B, H, L, D)
    assert noalloc(q, k, v, causal=True, out=out) == 0
    assert _C.last_launch().startswith("generic" if offset % 4 else "prefill f16 D=80"), _C.last_launch()
    assert_close(out, oracle_forward(q.cpu(), k.cpu(), v.cpu(), is_causal=True), torch.float16, f"offset {offset}")
