"""MultiheadAttention of one tensor (self-attention) projects q, k and v in one product; the same module on
equal tensors that are not one object projects them separately.  Outputs, weights and every gradient agree,
and gradients that arrive as transposed views equal those of dense ones."""

import pytest
import torch

import gguf_train_amd as g
from gguf_train_amd.nn import MultiheadAttention

from _util import randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,L,E,H,bias,batch_first", [(2, 50, 128, 2, True, True), (3, 17, 64, 4, False, False), (1, 130, 256, 2, True, True)])
@pytest.mark.parametrize("need_weights,dropout", [(True, 0.0), (False, 0.0), (True, 0.2)])
def test_one_projection_equals_three(dev, B, L, E, H, bias, batch_first, need_weights, dropout):
    torch.manual_seed(3)
    m = MultiheadAttention(E, H, dropout=dropout, bias=bias, batch_first=batch_first, device=dev)
    x0 = randn((B, L, E) if batch_first else (L, B, E), 5).to(dev)
    pad = torch.zeros((B, L), dtype=torch.bool, device=dev)
    pad[0, L - L // 4:] = True
    res = []
    for one in (True, False):
        x = x0.clone().requires_grad_(True)
        torch.manual_seed(11)
        out, w = m(x, x, x, key_padding_mask=pad, need_weights=need_weights) if one else m(
            x, x * 1.0, x * 1.0, key_padding_mask=pad, need_weights=need_weights)
        grads = torch.autograd.grad((out * torch.linspace(-1, 1, out.numel(), device=dev).reshape(out.shape)).sum(),
                                    [x, *m.parameters()])
        res.append([out, *([w] if w is not None else []), *grads])
    for a, b in zip(*res):
        # float32 sums of up to 3E products in another order
        assert (a - b).abs().max().item() <= 1e-5 * max(1.0, b.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [64, 36, 128])
def test_gradients_of_transposed_outputs(dev, dtype, D):
    B, H, L = 2, 4, 70
    q, k, v = (randn((B, H, L, D), i, dtype).to(dev) for i in range(3))
    flat = randn((B * L * H * D + 1,), 9, dtype).to(dev)
    out, lse, out32 = g.flash_attention_train(q, k, v, None, 0.0, True) if dtype != torch.float32 else (
        *g.flash_attention_lse(q, k, v, None, 0.0, True), None)
    res = out if out32 is None else out32
    for start in (0, 1):  # 1: rows off 16 bytes
        view = flat[start:start + B * L * H * D].view(B, L, H, D).transpose(1, 2)
        want = g.flash_attention_backward(view.contiguous(), q, k, v, None, res, lse, 0.0, True)
        got = g.flash_attention_backward(view, q, k, v, None, res, lse, 0.0, True)
        assert all(torch.equal(a, b) for a, b in zip(got, want))
