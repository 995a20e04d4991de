"""The native bridge between PyTorch tensors and the library's handles, without a GPU: what a borrowed
handle says of its tensor, who owns what, and how errors come out."""

import gc
import sys

import pytest
import torch

from gguf_train_amd import _bridge, _C


@pytest.mark.parametrize("dtype", list(_bridge.TORCH_TO_GT))
def test_borrowed_handles_describe_the_tensor(dtype):
    base = torch.arange(2 * 3 * 4 * 6).reshape(2, 3, 4, 6).to(dtype)
    for t in (base, base.transpose(1, 3), base[:, 1:, ::2], base[0, 0, 0, 0], base[:, :0]):
        h = _bridge.borrow(t)
        n = _C.lib.gt_tensor_ndim(h.ptr)
        shape = (_C.c_int64 * max(n, 1))()
        _C.lib.gt_tensor_shape(h.ptr, shape)
        assert n == t.ndim and list(shape)[:n] == list(t.shape)
        assert _C.lib.gt_tensor_dtype(h.ptr) == _bridge.TORCH_TO_GT[dtype]
        assert _C.lib.gt_tensor_device_type(h.ptr) == _C.GT_DEV_CPU
        if t.numel():
            assert h.keep is t and _C.lib.gt_tensor_data_ptr(h.ptr) == t.data_ptr()
            assert torch.equal(_bridge.adopt(_C.lib.gt_tensor_clone(h.ptr)), t)


def test_a_handle_pins_its_tensor_until_it_is_dropped():
    t = torch.zeros(8)
    before = sys.getrefcount(t)
    h = _bridge.borrow(t)
    assert sys.getrefcount(t) == before + 1
    del h
    gc.collect()
    assert sys.getrefcount(t) == before
    for _ in range(1500):  # past the release queue's drains
        _bridge.borrow(t)
    assert sys.getrefcount(t) == before


def test_released_handles_give_up_the_tensor():
    lent = _bridge.borrow(torch.ones(3))  # must outlive the call that uses its address
    h = _bridge.Handle(_C.lib.gt_tensor_clone(lent.ptr), keep=None)
    p = h.release()
    assert p and h.ptr == 0 and h.keep is None
    assert torch.equal(_bridge.adopt(p), torch.ones(3))


def test_what_cannot_be_lent_raises():
    with pytest.raises(TypeError, match="is not supported by libgt_attn"):
        _bridge.borrow(torch.zeros(2, dtype=torch.complex64))
    with pytest.raises(TypeError):
        _bridge.borrow([1.0])
    with pytest.raises(RuntimeError):  # a C++ exception
        _bridge.borrow(torch.zeros(2, 2).to_sparse())
    with pytest.raises(RuntimeError):  # more dimensions than the ABI has
        _bridge.borrow(torch.zeros((1,) * 20))
    with pytest.raises(RuntimeError):
        _bridge.adopt(0, "test")
