"""Moves PyTorch tensors across the C ABI without copies.

Inputs are lent to the library as borrowed handles (gt_tensor_from_device_ptr for HIP
memory, gt_tensor_from_external for host memory); results come back as library-owned
handles and are adopted by PyTorch through DLPack (gt_tensor_to_dlpack), so the memory the
kernels wrote is the memory the caller reads.  Both steps run in the native module _gt_bridge.  Every native call is made on the caller's
current PyTorch stream (gt_set_stream), which keeps the library ordered with PyTorch work.

PyTorch is plumbing here: device memory and streams.  No attention math happens in PyTorch.
"""

from __future__ import annotations

import ctypes
import itertools
from dataclasses import dataclass

import torch

from . import _C

TORCH_TO_GT = {
    torch.float32: _C.GT_F32,
    torch.float16: _C.GT_F16,
    torch.bfloat16: _C.GT_BF16,
    torch.float64: _C.GT_F64,
    torch.int8: _C.GT_I8,
    torch.uint8: _C.GT_U8,
    torch.int16: _C.GT_I16,
    torch.int32: _C.GT_I32,
    torch.int64: _C.GT_I64,
    torch.bool: _C.GT_BOOL,
}
GT_TO_TORCH = {v: k for k, v in TORCH_TO_GT.items()}

_tokens = itertools.count(1)

Handle = _C.bridge.Handle  # owns one gt_tensor* (`ptr`), freed with it; `keep` pins borrowed memory


@dataclass
class QuantizedTensor:
    """A GGUF Q8_0 tensor: `data` holds the ggml blocks (fp16 d + 32 int8, 34 bytes per 32
    values along the flattened logical shape) as a uint8 tensor; `shape` is the logical shape.
    Mirrors the reference's quantized Tensor (dtype code 108, gguf_train/_dtype.py:85)."""

    data: torch.Tensor
    shape: tuple
    gt_dtype: int = _C.GT_Q8_0

    @property
    def device(self) -> torch.device:
        return self.data.device

    @property
    def ndim(self) -> int:
        return len(self.shape)

    def numel(self) -> int:
        n = 1
        for s in self.shape:
            n *= int(s)
        return n


def _i64(vals) -> ctypes.Array:
    vals = [int(v) for v in vals]
    return (ctypes.c_int64 * max(len(vals), 1))(*vals)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def bind_stream(device: torch.device) -> None:
    """Makes the library enqueue on PyTorch's current stream of `device`."""
    if device.type != "cuda":
        _C.bridge.set_stream(0)
    elif _raw_stream is not None and device.index is not None and torch.cuda.is_initialized():
        _C.bridge.set_stream(_raw_stream(device.index))
    else:
        _C.bridge.set_stream(torch.cuda.current_stream(device).cuda_stream)


def borrow(t) -> Handle:
    """A Handle (its `ptr` a gt_tensor*) on the memory of a PyTorch tensor or QuantizedTensor, without a
    copy; it frees the gt_tensor when dropped and pins the memory until then."""
    if not isinstance(t, QuantizedTensor):
        return _C.bridge.borrow(t)
    d = t.data
    h = _C.bridge.borrow_q8(d, t.shape) if type(t.shape) is tuple and t.gt_dtype == _C.GT_Q8_0 else None
    if h is not None:
        return h
    if not d.is_cuda:
        nb = d.numel()
        ptr = _C.lib.gt_tensor_from_data(len(t.shape), _i64(t.shape), _C.GT_Q8_0, _C.GT_DEV_CPU, 0,
                                         ctypes.c_void_p(d.contiguous().data_ptr()), nb)
        return Handle(_C.check_ptr(ptr, "borrow"))
    if not d.is_contiguous() or d.dtype != torch.uint8:
        raise ValueError("QuantizedTensor.data must be a contiguous uint8 tensor")
    strides = []
    acc = 1
    for s in reversed(t.shape):
        strides.append(acc)
        acc *= int(s)
    strides.reverse()
    ptr = _C.lib.gt_tensor_from_device_ptr(len(t.shape), _i64(t.shape), _i64(strides), _C.GT_Q8_0,
                                           d.device.index or 0, ctypes.c_void_p(d.data_ptr()), next(_tokens))
    return Handle(_C.check_ptr(ptr, "borrow"), keep=d)


def adopt(ptr: int, ctx: str = "") -> torch.Tensor:
    """Turns a library-owned result handle into a PyTorch tensor (zero-copy, via DLPack)."""
    t = _C.bridge.adopt(_C.check_ptr(ptr, ctx))
    if t is None:
        _C.check_ptr(0, ctx)
    return t


def adopt_quantized(ptr: int, shape, ctx: str = "") -> QuantizedTensor:
    return QuantizedTensor(adopt(ptr, ctx), tuple(int(s) for s in shape))
