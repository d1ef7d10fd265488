"""Device addresses of a step's tensors and its stream, at little host cost.

Below some 10000 particles the host work of a call is longer than its kernels
(one launch runs in 3 us at 1000 particles).  Unpacking nine rows as tensors
takes 6.6 us and torch.cuda.current_stream() 2.8 us, so the common argument, a
plain (3, n) float32 tensor with contiguous rows, is read by its base address
and row stride.  Host time a call on MI355X: forward 18.7 -> 5.9 us, adjoint
31 -> 10.8, both together 39 -> 12.0.  Everything else (sequences of tensors, subclasses, other
shapes, types and strides) takes the caller's general checks.
"""
from __future__ import annotations

_tensor = _f32 = _device = _raw_stream = None


def _bind() -> None:
    global _tensor, _f32, _device, _raw_stream
    import torch

    _f32 = torch.float32
    _device = getattr(torch._C, "_cuda_getDevice", None)
    _raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)
    _tensor = torch.Tensor


def row_ptrs(t, n: int | None):
    """(x, y, z) addresses of a plain (3, >= n) CUDA tensor (n None: any
    length), or None where the general checks have to look at it."""
    if _tensor is None:
        _bind()
    if type(t) is not _tensor or not t.is_cuda or t.dtype is not _f32:
        return None
    shape = t.shape
    if len(shape) != 2 or shape[0] != 3 or shape[1] < (n or 1):
        return None
    row, one = t.stride()
    if one != 1:
        return None
    a = t.data_ptr()
    return a, a + 4 * row, a + 8 * row


def row_length(t) -> int:
    """Values in the first row."""
    if type(t) is _tensor and t.is_cuda:
        shape = t.shape
        if len(shape) == 2 and shape[0] == 3:
            return shape[1]
    return int(t[0].numel())


def stream_ptr(stream) -> int:
    """The raw stream of a torch stream, or of the current one for None."""
    if stream is not None:
        return stream.cuda_stream
    import torch

    if _raw_stream is None or _device is None or not torch.cuda.is_initialized():
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(_device())
