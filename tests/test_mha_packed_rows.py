"""Self-attention projects q, k and v in one product while rows of 3E keep the MFMA kernels' 32-bit byte
offsets, and apart past them, where rows of E still do.  Shapes only (meta tensors)."""

import pytest
import torch

from gguf_train_amd.nn.modules import transformer


@pytest.mark.parametrize("dtype,E,L,packed", [(torch.float16, 4096, 174762, True), (torch.float16, 4096, 174763, False),
                                              (torch.float16, 4096, 400000, False), (torch.float32, 1024, 349525, True),
                                              (torch.float32, 1024, 349526, False), (torch.bfloat16, 64, 3, True)])
@pytest.mark.parametrize("batch_first", [True, False])
def test_the_projection_by_length(monkeypatch, dtype, E, L, packed, batch_first):
    m = transformer.MultiheadAttention(E, E // 64, batch_first=batch_first, device="meta", dtype=dtype)
    seen = {}

    def attend(q, k, v, **kw):
        seen["strides"] = [t.stride(2) for t in (q, k, v)]
        return torch.empty(q.shape, dtype=q.dtype, device="meta")

    monkeypatch.setattr(transformer.F, "scaled_dot_product_attention", attend)
    x = torch.empty((1, L, E) if batch_first else (L, 1, E), dtype=dtype, device="meta")
    out, _ = m(x, x, x, need_weights=False)
    assert out.shape == x.shape
    assert seen["strides"] == [3 * E if packed else E] * 3
    assert (L - 1) * seen["strides"][1] * m.in_proj_weight.element_size() < 2 ** 32  # what the kernels check
