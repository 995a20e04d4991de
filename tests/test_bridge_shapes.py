"""A QuantizedTensor's shape may hold whatever int() takes, as a division or NumPy leaves it."""

import numpy as np
import pytest
import torch

from gguf_train_amd import QuantizedTensor, _bridge, _C


@pytest.mark.parametrize("shape", [(2, 32), (2.0, 32.0), (np.int64(2), np.float32(32)), (torch.tensor(2), 64 / 2), [2, 32],
                                   torch.Size([2, 32])])
def test_shapes_of_other_numbers(shape):
    h = _bridge.borrow(QuantizedTensor(torch.zeros(2 * 34, dtype=torch.uint8), shape))
    dims = (_C.c_int64 * 2)()
    _C.lib.gt_tensor_shape(h.ptr, dims)
    assert _C.lib.gt_tensor_ndim(h.ptr) == 2 and list(dims) == [2, 32]


def test_a_shape_of_no_numbers_raises():
    with pytest.raises((TypeError, ValueError)):
        _bridge.borrow(QuantizedTensor(torch.zeros(2 * 34, dtype=torch.uint8), (2, "rows")))
    with pytest.raises(RuntimeError, match="Negative"):
        _bridge.borrow(QuantizedTensor(torch.zeros(2 * 34, dtype=torch.uint8), (2, -32)))
